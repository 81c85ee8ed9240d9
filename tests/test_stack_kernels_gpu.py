"""Launch forms of the stack kernels at the sizes where their tiles, splits and groups end."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nats_llm_studio_amd.ops import stack
    stack.lib()
    return stack


def st():
    return torch.cuda.current_stream().cuda_stream


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)


def relerr(got, want):
    want = want.double()
    return float((got.double().cpu() - want).norm() / want.norm())


# heads, key heads, key and value columns: groups that do and do not divide 16, single heads, widths with a part of a block
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (6, 2, 20), (3, 3, 64), (20, 1, 32), (2, 1, 300), (1, 1, 600)])
@pytest.mark.parametrize("window,keep,sink", [(0, 0, False), (40, 5, True)])
def test_plain_attention_rows_of_many_sequences(K, dt, H, G, D, window, keep, sink):
    """Runs of several lengths beside single tokens and a padded row, more than 64 rows: a workgroup's tokens are of one sequence, of
    several, or end before the batch does."""
    d = {"f32": torch.float32, "bf16": torch.bfloat16}[dt]
    Dp, _ = K.head_pad(D)
    bs, scale = 16, 0.8 / math.sqrt(D)
    runs = [(0, 50), (33, 1), (100, 3), (0, 17), (7, 1), (15, 2)]            # first position, rows
    nb = 7
    T = sum(n for _, n in runs) + 1
    assert T > 64
    perm = torch.randperm(len(runs) * nb, generator=torch.Generator().manual_seed(5)).view(-1, nb)
    kc, vc = (torch.zeros(perm.numel() * bs, G, Dp, dtype=d) for _ in range(2))
    q = torch.zeros(T, H, Dp, dtype=d)
    q[..., :D] = rnd(T, H, D, seed=1).to(d)
    gate, want = rnd(T, H, seed=3).float(), torch.zeros(T, H, D, dtype=torch.float64)
    seq, ctx, t = torch.zeros(T, dtype=torch.int32), torch.zeros(T, dtype=torch.int32), 0
    for i, (p0, n) in enumerate(runs):
        N = p0 + n
        k, v = rnd(N, G, D, seed=10 + i).to(d), rnd(N, G, D, seed=50 + i).to(d)
        pos = torch.arange(N)
        slot = perm[i][pos // bs] * bs + pos % bs
        kc[slot, :, :D], vc[slot, :, :D] = k, v
        for p in range(p0, N):
            s = torch.einsum("hd,khd->hk", q[t, :, :D].double(), k.double().repeat_interleave(H // G, 1)) * scale
            see = (pos <= p) & ((p - pos < window) | (pos < keep) if window else torch.ones(N, dtype=torch.bool))
            s = s.masked_fill(~see, -math.inf)
            if sink:
                s = torch.cat([s, torch.zeros(H, 1, dtype=torch.float64)], 1)
            w = torch.softmax(s, 1)[:, :N]
            want[t] = torch.einsum("hk,khd->hd", w, v.double().repeat_interleave(H // G, 1)) * gate[t].double()[:, None]
            seq[t], ctx[t] = i, p + 1
            t += 1
    out = torch.full((T + 1, H * Dp), 7.0, dtype=d, device="cuda")
    part = tuple(torch.zeros(1, device="cuda") for _ in range(3))
    K.gqa_attention(q.view(T, -1).cuda(), kc.view(-1, G * Dp).cuda(), vc.view(-1, G * Dp).cuda(), gate.cuda(), out, part,
                    perm.int().cuda(), bs, seq.cuda(), ctx.cuda(), T, H, G, Dp, False, 1, scale, st(), window=window, keep=keep, sink=sink)
    o = out.view(T + 1, H, Dp)
    # f32: the sums of a row; bf16: the output's rounding
    assert relerr(o[:T, :, :D], want) < (2e-6 if dt == "f32" else 3e-3)
    assert (o[:T, :, D:] == 0).all() and (o[T - 1] == 0).all() and (o[T] == 7).all()
