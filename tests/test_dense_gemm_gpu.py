"""The dense f16 GEMM (mode 10) where its row blocks change between 192 and 256 rows, and its RoPE epilogue for head widths that its
8-byte stores take and that they do not."""
import numpy as np
import pytest
import torch

from nats_llm_studio_amd import ops
from nats_llm_studio_amd.gguf.constants import GGMLType
from nats_llm_studio_amd.gguf.quants import random_blocks

pytestmark = pytest.mark.gpu


def weight(rows, K, seed=0):
    w = ops.QWeight(random_blocks(GGMLType.Q8_0, rows * K, 0.02, np.random.default_rng(seed)), GGMLType.Q8_0, rows, K, "cuda", "w")
    w.expand_dense()
    return w


def acts(M, K, seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((M + 63) // 64 * 64, K, generator=g, device="cuda").to(torch.float16)


def relerr(got, want):
    return float((got.double() - want.double()).norm() / want.double().norm())


# rows: 101 weight tiles of 256 (202 of 128) make 192-row blocks the shorter walk at 190, 384 and 700 rows and 256-row blocks at
# 193 .. 256 and 512 rows, for one of the two tile widths at least
@pytest.mark.parametrize("rt", [1, 2])
@pytest.mark.parametrize("M", [190, 193, 256, 257, 384, 385, 512, 700])
@pytest.mark.parametrize("epi", ["f32", "swiglu"])
def test_row_blocks(M, rt, epi):
    rows, K = 25700 - 4 if epi == "f32" else 25600, 256
    w, x = weight(rows, K), acts(M, K)
    z = x[:M].float() @ w.d16.float().T
    if epi == "swiglu":
        v = z.view(M, rows // 16, 2, 8)
        z = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, rows // 2)
    y = torch.full((x.shape[0], z.shape[1]), 7.0, device="cuda", dtype=torch.float32 if epi == "f32" else torch.float16)
    ops.qgemv([ops.Seg(w)], x, y, M, epi=epi, mode=10, waves=8, rt=rt, ks=1)
    # sums of 256 products in f32; f16 outputs round to 2^-11
    assert relerr(y[:M], z) < (1e-6 if epi == "f32" else 5e-4)
    assert (y[M:] == 7).all()


@pytest.mark.parametrize("cfg", [(10, 8, 1, 1), (10, 8, 2, 1), (4, 16, 2, 1), (4, 8, 4, 1)])
@pytest.mark.parametrize("D,bias", [(64, False), (128, True), (34, True)])
@pytest.mark.parametrize("M", [70, 300])
def test_rope_epilogue(cfg, D, bias, M):
    """Against the same product rotated on the CPU: rows without a cache slot, shuffled slots."""
    Hq, Hkv, K = 16, 8, 256
    ws = [weight(h * D, K, s) for s, h in enumerate((Hq, Hkv, Hkv))]
    segs = [ops.Seg(ws[0], 0), ops.Seg(ws[1], Hq * D), ops.Seg(ws[2], (Hq + Hkv) * D)]
    x, n = acts(M, K), (Hq + 2 * Hkv) * D
    pad = x.shape[0]
    cs = ops.rope_table(400, D, 10000.0, torch.device("cuda"))
    pos = (torch.arange(pad, dtype=torch.int32, device="cuda") * 7) % 400
    slot = torch.randperm(pad, generator=torch.Generator().manual_seed(2)).int().cuda()
    slot[[0, 17, M - 1]] = -1
    b = torch.randn(n, generator=torch.Generator().manual_seed(3)).cuda() if bias else None
    outs = []
    for c, fuse in ((cfg, True), (cfg, False)):
        q = torch.full((pad, Hq * D), 776.0, dtype=torch.bfloat16, device="cuda")
        kc, vc = (torch.full((pad, Hkv, D), 776.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        qkv = torch.zeros(pad, n, device="cuda")
        if fuse:
            ops.qkv_rope_kv(segs, x, qkv, pos, slot, cs, q, kc, vc, M, Hq, Hkv, D, cfg=c, bias=b)
        else:
            ops.qgemv(segs, x, qkv, M, mode=c[0], waves=c[1], rt=c[2], ks=1)
            q, kc, vc = q.cpu(), kc.cpu(), vc.cpu()
            ops.rope_kv(qkv.cpu(), pos.cpu(), slot.cpu(), cs.cpu(), q, kc, vc, M, Hq, Hkv, D, bias=None if b is None else b.cpu())
        outs.append((q.cpu(), kc.cpu(), vc.cpu()))
    for a, b in zip(*outs):      # one bf16 rounding apart at most, and the same places written
        assert relerr(a, b) < 2e-3 and ((a == 776) == (b == 776)).all()


@pytest.mark.parametrize("cfg", [(10, 8, 1), (10, 8, 2), (5, 16, 2), (4, 8, 2)])
@pytest.mark.parametrize("rows,K", [(1024, 2304), (1020, 2048), (2048, 1024), (388, 2048), (1536, 2560)])
def test_split_reduce(cfg, rows, K):
    """Slabs of a split product and their sum: whole and part workgroups of columns and of rows, where a workgroup has the tile's columns
    and where it has 1024; every kind of output, two slabs to nine."""
    w = weight(rows, K)
    for M in (70, 129, 258, 263):
        x = acts(M, K)
        z = x[:M].double() @ w.d16.double().T
        for ks in (2, 3, 4, 5, 8, 9):
            for epi, dt in (("f32", torch.float32), ("add", torch.float32), ("act", torch.float16)):
                y = torch.full((M + 1, rows + 4), 7.0, device="cuda", dtype=dt)
                ops.qgemv([ops.Seg(w, 4)], x, y, M, epi=epi, mode=cfg[0], waves=cfg[1], rt=cfg[2], ks=ks)
                # f32 sums of K products; f16 outputs round to 2^-11
                assert relerr(y[:M, 4:] - (7 if epi == "add" else 0), z) < (5e-4 if epi == "act" else 4e-6), (M, ks, epi)
                assert (y[M] == 7).all() and (y[:, :4] == 7).all()


# 320-row blocks with 128 weight rows: 201 weight tiles take them at 257 .. 320 and 513 .. 640 rows; one K step (no successor to stage) to twelve
@pytest.mark.parametrize("M", [257, 271, 319, 320, 321, 513, 640])
@pytest.mark.parametrize("K", [256, 768])
def test_blocks_of_320(M, K):
    rows = 25700 - 4
    w, x = weight(rows, K), acts(M, K)
    z = x[:M].double() @ w.d16.double().T
    for epi, ks in (("f32", 1), ("add", 1), ("add", 4)):
        y = torch.full((x.shape[0] + 1, rows), 7.0, device="cuda")
        ops.qgemv([ops.Seg(w)], x, y, M, epi=epi, mode=10, waves=8, rt=2, ks=ks)
        assert relerr(y[:M] - (7 if epi == "add" else 0), z) < 4e-6, (epi, ks)       # sums of K products in f32
        assert (y[M:] == 7).all()


@pytest.mark.parametrize("M", [257, 300, 320, 513, 640])
def test_blocks_of_320_gate_and_head(M):
    """The other epilogues of 320-row blocks: SwiGLU, and a head's arg-max with its logits and alone."""
    rows, K = 25600, 256                         # 200 weight tiles
    w, x = weight(rows, K), acts(M, K)
    z = x[:M].double() @ w.d16.double().T
    v = z.view(M, rows // 16, 2, 8)
    want = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, rows // 2)
    y = torch.full((x.shape[0] + 1, rows // 2), 7.0, device="cuda", dtype=torch.float16)
    ops.qgemv([ops.Seg(w)], x, y, M, epi="swiglu", mode=10, waves=8, rt=2, ks=1)
    assert relerr(y[:M], want) < 5e-4 and (y[M:] == 7).all()                       # f16 outputs round to 2^-11
    logits = torch.full((M + 1, rows), 7.0, device="cuda")
    for epi in ("f32", "argmax"):
        keys, ids = torch.zeros(M + 1, dtype=torch.int64, device="cuda"), torch.full((M + 1,), -1, dtype=torch.int32, device="cuda")
        ops.qgemv([ops.Seg(w)], x, logits, M, epi=epi, argmax=keys, mode=10, waves=8, rt=2, ks=1)
        ops.argmax_unpack(keys, M, ids)
        assert (ids[:M].long() == logits[:M].argmax(1)).all() and int(keys[M]) == 0 and int(ids[M]) == -1, epi
    assert relerr(logits[:M], z) < 4e-6 and (logits[M:] == 7).all()


def test_blocks_of_320_rope():
    """144 weight tiles in three segments; D = 34 takes the general stores."""
    M, K = 300, 256
    for D, Hq, Hkv in ((128, 128, 8), (34, 504, 24)):
        ws = [weight(h * D, K, s) for s, h in enumerate((Hq, Hkv, Hkv))]
        segs = [ops.Seg(ws[0], 0), ops.Seg(ws[1], Hq * D), ops.Seg(ws[2], (Hq + Hkv) * D)]
        x, n = acts(M, K), (Hq + 2 * Hkv) * D
        pad = x.shape[0]
        cs = ops.rope_table(400, D, 10000.0, torch.device("cuda"))
        pos = (torch.arange(pad, dtype=torch.int32, device="cuda") * 7) % 400
        slot = torch.randperm(pad, generator=torch.Generator().manual_seed(2)).int().cuda()
        slot[[0, 17, M - 1]] = -1
        outs = []
        for fuse in (True, False):
            q = torch.full((pad, Hq * D), 776.0, dtype=torch.bfloat16, device="cuda")
            kc, vc = (torch.full((pad, Hkv, D), 776.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
            qkv = torch.zeros(pad, n, device="cuda")
            if fuse:
                ops.qkv_rope_kv(segs, x, qkv, pos, slot, cs, q, kc, vc, M, Hq, Hkv, D, cfg=(10, 8, 2, 1))
            else:
                ops.qgemv(segs, x, qkv, M, mode=4, waves=16, rt=2, ks=1)
                q, kc, vc = q.cpu(), kc.cpu(), vc.cpu()
                ops.rope_kv(qkv.cpu(), pos.cpu(), slot.cpu(), cs.cpu(), q, kc, vc, M, Hq, Hkv, D)
            outs.append((q.cpu(), kc.cpu(), vc.cpu()))
        for a, b in zip(*outs):      # one bf16 rounding apart at most, and the same places written
            assert relerr(a, b) < 2e-3 and ((a == 776) == (b == 776)).all()
