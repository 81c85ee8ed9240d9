"""Prompt attention (of the stacks, and of GGUF models) in halves of a block and where two groups of waves share the keys: walks of one tile (the second group has none), of two and of odd counts, windows, keys
of one group only that outweigh the other's, and the choice between the forms."""
import types

import numpy as np
import pytest
import torch

from nats_llm_studio_amd import ops
from nats_llm_studio_amd.models.stack import _prompt_waves
from nats_llm_studio_amd.ops import stack as K

RUNS = [(0, 130), (61, 3), (64, 1), (128, 200), (0, 64), (700, 150)]          # first position, rows
T = sum(n for _, n in RUNS)
NX = sum(p + n for p, n in RUNS)


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def table():
    blocks, a, x = [], 0, 0
    for i, (p, n) in enumerate(RUNS):
        blocks += [(a + o, min(128, n - o), i, p + o, x, 0, 0, 0) for o in range(0, n, 128)]
        a, x = a + n, x + p + n
    return i32(blocks), len(blocks)


def check(out, q, k, v, scale, gate=None, window=0, keep=0, sink=False):
    """out [T, H, V] against f64 of q [T, H, D], k [NX, H, D], v [NX, H, V], row by row. Weights and outputs are rounded to bf16 (2^-9 each)."""
    a = x = 0
    for p, n in RUNS:
        s = torch.einsum("thd,khd->htk", q[a:a + n].double(), k[x:x + p + n].double()) * scale
        i, j = torch.arange(p, p + n, device="cuda")[:, None], torch.arange(p + n, device="cuda")[None]
        see = (j <= i) & ((i - j < window) | (j < keep)) if window else j <= i
        s = s.masked_fill(~see, -torch.inf)
        if sink:
            s = torch.cat([s, torch.zeros_like(s[..., :1])], -1)
        w = torch.softmax(s, -1)[..., :p + n]
        want = (w @ v[x:x + p + n].double().transpose(0, 1)).transpose(0, 1)
        if gate is not None:
            want = want * gate[a:a + n].double()[..., None]
        e = (out[a:a + n].double() - want).norm(dim=-1) / want.norm(dim=-1)
        assert float(e.max()) < 8e-3, (p, n, float(e.max()))
        a, x = a + n, x + p + n


def loud(k, q):
    """A late key (of the other group's tile) far above the others for some rows, and an early one for others."""
    x = a = 0
    for p, n in RUNS:
        for r, at in ((n - 1, p + n - 1), (n // 2, 0), (n // 3, (p + n // 3) // 2)):
            k[x + at] = 6 * q[a + r] / q[a + r].float().norm(dim=-1, keepdim=True).to(q.dtype) * q.shape[-1] ** 0.25
        x, a = x + p + n, a + n


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D", [(4, 2, 32), (5, 1, 64), (8, 2, 128), (2, 2, 256)])
@pytest.mark.parametrize("window,keep,sink", [(0, 0, False), (0, 0, True), (70, 5, True), (200, 0, False)])
def test_paged(H, G, D, window, keep, sink):
    g = torch.Generator(device="cuda").manual_seed(D)
    q = torch.randn(T, H, D, generator=g, device="cuda").bfloat16()
    k, v = (torch.randn(NX, G, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    loud(k, q[:, ::H // G])
    slot = torch.randperm(NX, generator=torch.Generator().manual_seed(1)).cuda()
    kc, vc = torch.empty_like(k), torch.empty_like(v)
    kc[slot], vc[slot] = k, v
    gate = torch.rand(T, H, generator=g, device="cuda")
    out = torch.full((T + 1, H * D), 7.0, dtype=torch.bfloat16, device="cuda")
    blocks, n = table()
    K.gqa_prefill(q.view(T, -1), kc, vc, slot.int(), blocks, n, 4, gate, out, H, G, D, D ** -0.5, K.stream(q.device), window, keep, sink, groups=2)
    assert (out[T] == 7).all()
    check(out[:T].view(T, H, D), q, k.repeat_interleave(H // G, 1), v.repeat_interleave(H // G, 1), D ** -0.5, gate, window, keep, sink)


@pytest.mark.gpu
@pytest.mark.parametrize("dku,dr,dv,vdim", [(32, 32, 32, 30), (64, 32, 128, 128), (128, 64, 128, 100), (128, 64, 32, 32), (32, 64, 64, 64)])
def test_expanded(dku, dr, dv, vdim):
    H, g = 3, torch.Generator(device="cuda").manual_seed(dku + dr + dv)
    qn = torch.randn(T, H, dku, generator=g, device="cuda").bfloat16()
    qr = torch.randn(T, H, dr, generator=g, device="cuda").bfloat16()
    kx = torch.randn(NX, H, dku, generator=g, device="cuda").bfloat16()
    vx = torch.randn(NX, H, dv, generator=g, device="cuda").bfloat16()
    rot = torch.randn(NX, dr, generator=g, device="cuda").bfloat16()
    loud(kx, qn)
    slot = torch.randperm(NX, generator=torch.Generator().manual_seed(1)).cuda()
    cache = torch.zeros(NX, 64 + dr, dtype=torch.bfloat16, device="cuda")
    cache[slot, 64:] = rot
    q = torch.cat([torch.zeros(T, H, 64, dtype=torch.bfloat16, device="cuda"), qr], -1)       # (the rotated part at column 64, as in the cache)
    gate = torch.rand(T, H, generator=g, device="cuda")
    out = torch.full((T + 1, H * vdim), 7.0, dtype=torch.bfloat16, device="cuda")
    blocks, n = table()
    scale = (dku + dr) ** -0.5
    K.latent_prefill(qn.view(T, -1), dku, q.view(T, -1), 64, 64 + dr, kx, vx, cache, slot.int(), blocks, n, 4, gate, out, H, dku, dr, dv, vdim,
                     scale, K.stream(q.device), groups=2)
    assert (out[T] == 7).all()
    check(out[:T].view(T, H, vdim), torch.cat([qn, qr], -1), torch.cat([kx, rot[:, None].expand(-1, H, -1)], -1), vx[..., :vdim], scale, gate)


@pytest.mark.parametrize("heads,window,spans,want", [
    (32, 0, [(0, 1000)], (4, 2)),            # few workgroups
    (32, 0, [(0, 300)], (4, 1)),             # short walks
    (32, 0, [(0, 2000)], (4, 2)),            # the longest walk outlasts the rest
    (32, 1024, [(0, 2000)], (4, 1)),         # ... not in a window
    (32, 0, [(0, 650)] * 6, (4, 1)),
    (32, 0, [(0, 3500)], (8, 1)),            # long walks fill the chip
    (16, 0, [(0, 3500)], (4, 2)),
    (16, 0, [(3000, 128)], (4, 2)),          # a run behind a long context
])
def test_choice(heads, window, spans, want):
    att = [types.SimpleNamespace(cfg=types.SimpleNamespace(heads=heads, window=window))]
    assert _prompt_waves(att, [(0, n, 0, p, 0, p + n, 0, 0) for p, n in spans]) == want


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("kvt", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("D,G,Hkv", [(128, 4, 2), (64, 8, 1)])
def test_gguf_forms(form, kvt, D, G, Hkv):
    bs, g, H = 16, torch.Generator(device="cuda").manual_seed(D), G * Hkv
    pages = max(-(-(p + n) // bs) for p, n in RUNS)
    bt = torch.randperm(len(RUNS) * pages, generator=torch.Generator().manual_seed(1)).view(len(RUNS), pages).int().cuda()
    q = torch.randn(T, H, D, generator=g, device="cuda").bfloat16()
    k, v = (torch.randn(NX, Hkv, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    loud(k, q[:, ::G])
    k, v = k.to(kvt), v.to(kvt)
    kc, vc = (torch.zeros(bt.numel() * bs, Hkv, D, device="cuda").to(kvt) for _ in range(2))
    x = 0
    for r, (p, n) in enumerate(RUNS):
        at = torch.arange(p + n, device="cuda")
        at = bt[r, at // bs].long() * bs + at % bs
        for c, t in ((kc, k), (vc, v)):
            c.view(torch.uint8 if kvt.itemsize == 1 else torch.int16)[at] = t[x:x + p + n].view(torch.uint8 if kvt.itemsize == 1 else torch.int16)
        x += p + n
    seq = np.concatenate([np.full(n, r) for r, (_, n) in enumerate(RUNS)])
    pos = np.concatenate([np.arange(p, p + n) for p, n in RUNS])
    qb = ops.prefill_blocks(seq, pos, T)
    out = torch.full((T + 1, H * D), 7.0, dtype=ops.ACT_DTYPE, device="cuda")
    ops.attention_prefill(q.view(T, -1), kc, vc, bt, torch.from_numpy(qb).cuda(), len(qb), None, None, out, T, H, Hkv, D, bs, D ** -0.5, form)
    assert (out[T] == 7).all()
    check(out[:T].view(T, H, D), q, k.float().repeat_interleave(G, 1), v.float().repeat_interleave(G, 1), D ** -0.5)


@pytest.mark.parametrize("units,runs,want", [
    (8, [(0, 21)], 1), (8, [(0, 300)], 1), (8, [(0, 1000)], 2), (8, [(0, 2000)], 2), (8, [(0, 3000)], 1), (8, [(0, 4096)], 0), (4, [(0, 3000)], 2),
    (8, [(4000, 1000)], 2), (8, [(0, 60)] * 64, 1), (8, [(0, 20)] * 300, 0), (4, [(0, 8000)], 0)])
def test_gguf_choice(units, runs, want):
    seq = np.concatenate([np.full(n, r) for r, (_, n) in enumerate(runs)])
    pos = np.concatenate([np.arange(p, p + n) for p, n in runs])
    assert ops.prefill_form(ops.prefill_blocks(seq, pos, len(seq)), units) == want


@pytest.mark.parametrize("units,runs,want", [
    (16, [(0, 229), (0, 1006)], 1), (16, [(p, 24) for p in [0] * 96 + [30, 80, 200, 500] * 7 + [3973] * 4], 0), (16, [(795, 23)] + [(0, 23)] * 15, 0), (2, [(4781, 18)] * 8 + [(0, 18)] * 56, 2)])
def test_gguf_choice_of_unlike_runs(units, runs, want):
    """us of forms 0 / 1 / 2: 45 / 41 / 49 for the first, 100 / 112 / 126 for the second, 27 / 29 / 25 for one like the third."""
    seq = np.concatenate([np.full(n, r) for r, (_, n) in enumerate(runs)])
    pos = np.concatenate([np.arange(p, p + n) for p, n in runs])
    assert ops.prefill_form(ops.prefill_blocks(seq, pos, len(seq)), units) == want


def test_choice_of_many_short_runs_behind_contexts():
    """Walks of one tile waste a second group of waves: 90 us with four waves, 160 with two groups, 149 with eight."""
    att = [types.SimpleNamespace(cfg=types.SimpleNamespace(heads=32, window=0))]
    assert _prompt_waves(att, [(0, 19, 0, p, 0, p + 19, 0, 0) for p in [0] * 96 + [30, 80, 200, 500] * 7 + [1971] * 4]) == (4, 1)


@pytest.mark.gpu
def test_grown_scratch_of_a_queued_step():
    """A scratch that a queued launch of a side stream still uses is not handed out again when a larger one takes its place."""
    from nats_llm_studio_amd.models.stack import StackModel
    m, b = types.SimpleNamespace(dtype=torch.float32, device="cuda"), types.SimpleNamespace(shared={})
    t = StackModel.grown(m, b, "x", 1024, 4096)
    at, side = t.data_ptr(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(50_000_000)
        t.fill_(3.0)
        del t
        StackModel.grown(m, b, "x", 2048, 4096)
    assert not side.query()
    other = torch.empty(1024, 4096, device="cuda")
    assert other.data_ptr() != at
    torch.cuda.synchronize()
