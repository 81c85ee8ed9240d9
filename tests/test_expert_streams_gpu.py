"""Grouped expert products at few rows to an expert (path B of the quantised GEMV: per-expert active tiles) and the rule that sends
launches there."""
import numpy as np
import pytest
import torch

from nats_llm_studio_amd import ops
from nats_llm_studio_amd.gguf import quants as Q
from nats_llm_studio_amd.gguf.constants import GGMLType
from nats_llm_studio_amd.ops import tuning


@pytest.mark.gpu
@pytest.mark.parametrize("waves,rt", [(4, 1), (4, 2), (8, 2)])
@pytest.mark.parametrize("counts", [(1, 0, 4), (16, 15, 9), (17, 16, 1, 0), (32, 31, 33, 16), (48, 17, 64, 0, 1), (47, 32, 90, 128)])
@pytest.mark.parametrize("qt", [GGMLType.Q4_K, GGMLType.Q5_K, GGMLType.Q6_K, GGMLType.Q8_0])
def test_active_tiles(gpu, waves, rt, counts, qt):
    """Counts at the edges of the 16-row tiles, rows short of a workgroup's tile, a single super-block of K and an odd number. x and
    the dequantised weights are f16 (a weight is rounded at most twice, d * q and its difference to the minimum), products are summed
    in 32 bits: |error| <= 2^-9 sum |x| |w|."""
    rng = np.random.default_rng(len(counts))
    T = max(max(counts), 4)
    for N, K in ((272, 256), (144, 1280)):
        raw = [Q.random_blocks(qt, N * K, 0.05, rng) for _ in counts]
        ws = [ops.QWeight(r, qt, N, K, gpu) for r in raw]
        W = [ops.QWeight(r, qt, N, K, "cpu").dense().double() for r in raw]
        x = torch.randn(T, K, device=gpu).to(ops.ACT_DTYPE)
        xm = [torch.randperm(T)[:c] for c in counts]
        y = torch.full((sum(counts) + 1, N), 3.0, device=gpu)
        act = torch.full((sum(counts) + 1, N // 2), 3.0, device=gpu, dtype=ops.ACT_DTYPE)
        segs, y0 = [], 0
        for w, c, m in zip(ws, counts, xm):
            pad = torch.zeros(T, dtype=torch.int32)
            pad[:c] = m
            ym = torch.zeros(T, dtype=torch.int32)
            ym[:c] = torch.arange(y0, y0 + c)
            segs.append(ops.Seg(w, 0, pad.to(gpu), ym.to(gpu), torch.tensor([c], dtype=torch.int32, device=gpu)))
            y0 += c
        ops.qgemv(segs, x, y, T, epi="f32", mode=1, waves=waves, rt=rt, ks=1)
        ops.qgemv(segs, x, act, T, epi="swiglu", mode=1, waves=waves, rt=rt, ks=1)
        xd, y0 = x.cpu().double(), 0
        for c, m, w in zip(counts, xm, W):
            ref, e = xd[m] @ w.t(), (xd[m].abs() @ w.abs().t()) * 2.0 ** -9
            assert ((y[y0:y0 + c].cpu().double() - ref).abs() <= e).all()
            g, u = (ref.view(c, N // 16, 2, 8)[:, :, i] for i in (0, 1))
            eg, eu = (e.view(c, N // 16, 2, 8)[:, :, i] for i in (0, 1))
            want = torch.nn.functional.silu(g) * u
            bound = 1.1 * eg * (u.abs() + eu) + torch.nn.functional.silu(g).abs() * eu + want.abs() * 2.0 ** -10 + 2.0 ** -14
            assert ((act[y0:y0 + c].cpu().double() - want.reshape(c, N // 2)).abs() <= bound.reshape(c, N // 2)).all()
            y0 += c
        assert (y[y0:] == 3.0).all() and (act[y0:] == 3.0).all()


class _W:
    def __init__(self, rows, type=12):
        self.rows, self.type = rows, type


def test_expert_rule():
    """Path B only where its grid covers the chip, for the quantised types, and never above 128 tokens."""
    up, small = [_W(8192)] * 8, [_W(2048)] * 8
    assert [tuning.expert_heuristic(up, T, T / 4) for T in (1, 3, 4, 32, 128, 129)] == [None, None] + [(1, 8, 2, 1)] * 2 + [None] * 2
    assert tuning.expert_heuristic([_W(28672)] * 8, 32, 8) == (1, 4, 2, 1) and tuning.expert_heuristic([_W(28672)] * 8, 33, 8.25) == (1, 8, 2, 1)
    assert [tuning.expert_heuristic(small, T, T / 4) for T in (16, 17, 64, 65)] == [None, (1, 4, 1, 1), (1, 4, 1, 1), None]
    assert tuning.expert_heuristic([_W(4096)] * 8, 5, 1.25) == (1, 4, 1, 1) and tuning.expert_heuristic([_W(4096)] * 8, 4, 1) is None
    assert tuning.expert_heuristic([_W(8192)], 32, 8) is None and tuning.expert_heuristic([_W(8192, 1)] * 8, 32, 8) is None
    assert tuning.expert_heuristic([_W(2048)] * 4 + [_W(2048, 99)] * 4, 32, 8) is None


def test_dense_rule_counts_an_xcds_rounds():
    """28 weight tiles give four XCDs a tile more than the others: three parts of K, or nine blocks of rows, are two rounds there. us of what the
    rule took when it counted the whole chip's workgroups and of what it must take: 3584 x 3584 at 300 rows 31 / 23, at 513 35 / 31, at 2880
    114 / 76; 3584 x 18944 at 513 118 / 100, at 2880 557 / 345; 20480 x 8192 at 1920 631 / 575; 12288 x 4096 at 3200 358 / 313; 57344 x 8192 at
    320 391 / 347 (an entry)."""
    def pick(rows, K, M):
        w = _W(rows)
        w.K = K
        return tuning.select_dense([ops.Seg(w)], M)
    for rows, K, M, slow in ((3584, 3584, 300, (4, 16, 2, 3)), (3584, 3584, 513, (10, 8, 2, 3)), (3584, 3584, 2880, (10, 8, 2, 1)),
                             (3584, 18944, 513, (10, 8, 2, 3)), (3584, 18944, 2880, (10, 8, 2, 1)), (20480, 8192, 1920, (10, 8, 2, 1)),
                             (12288, 4096, 3200, (10, 8, 2, 1)), (57344, 8192, 320, (10, 8, 2, 1))):
        assert pick(rows, K, M) != slow, (rows, K, M)
    # blocks of 320 rows where they are the shorter walk
    assert pick(28672, 4096, 300) == pick(28672, 4096, 640) == pick(128256, 4096, 320) == (10, 8, 2, 1)


def test_environment_entries_stay(monkeypatch):
    """A launch config given in the environment is what runs: not split for a head's arg-max, and also above the tuned row counts."""
    class W(_W):
        K = 4096
    head, dense = [ops.Seg(W(32000, 14))], [ops.Seg(W(4096))]
    monkeypatch.setattr(tuning, "_TABLE", None)
    monkeypatch.setenv("NLS_TUNING_EXTRA", '{"14:32000:4096:16": [1, 4, 1, 1], "d:4096:4096:2048": [5, 8, 4, 2]}')
    try:
        assert tuning.argmax_config(tuning.select(head, 12), head, 12) == (1, 4, 1, 1)
        assert tuning.argmax_config((1, 4, 1, 1), head, 24) == (1, 8, 2, 2)          # another row count's own
        assert tuning.select_dense(dense, 3000) == (5, 8, 4, 2) and tuning.select_dense(dense, 1024) != (5, 8, 4, 2)
    finally:
        tuning._TABLE = None
        tuning._FORCED.clear()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 15, 17, 33, 64])
@pytest.mark.parametrize("rows,K,qt", [(8192, 1024, GGMLType.Q6_K), (8209, 1280, GGMLType.Q4_K), (32000, 2048, GGMLType.Q8_0)])
def test_head_argmax(gpu, M, rows, K, qt):
    """A head's own config: split in two with the maxima from the reduce. The keys are those of the logits it stored (the lowest of
    equal columns: every row of the second half is there twice), and a second launch into the same keys changes nothing."""
    raw = Q.random_blocks(qt, rows * K, 0.05, np.random.default_rng(5)).reshape(rows, -1)
    raw[rows // 2:2 * (rows // 2)] = raw[:rows // 2]
    seg = [ops.Seg(ops.QWeight(raw.reshape(-1), qt, rows, K, gpu))]
    assert tuning.argmax_config(ops.gemv_config(seg, M), seg, M)[3] > 1 or ops.gemv_config(seg, M)[0] != 1
    x = torch.zeros(64, K, dtype=ops.ACT_DTYPE, device=gpu)
    x[:M] = torch.randn(M, K, device=gpu)
    y, only = (torch.zeros(64, rows, device=gpu) for _ in range(2))
    keys, keys2 = (torch.zeros(64, dtype=torch.int64, device=gpu) for _ in range(2))
    ids = torch.zeros(64, dtype=torch.int32, device=gpu)
    for _ in range(2):
        ops.qgemv(seg, x, y, M, argmax=keys)
    ops.qgemv(seg, x, only, M, epi="argmax", argmax=keys2)
    assert torch.equal(keys, keys2) and not only.any() and not keys[M:].any()
    ops.argmax_unpack(keys, M, ids)
    assert ids[:M].tolist() == y[:M].cpu().numpy().argmax(1).tolist()
    W = ops.QWeight(raw.reshape(-1), qt, rows, K, "cpu").dense().double()
    ref, bound = x[:M].cpu().double() @ W.t(), (x[:M].cpu().double().abs() @ W.abs().t()) * 2.0 ** -9
    assert ((y[:M].cpu().double() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,D,E,k", [(5, 256, 4, 2), (24, 2048, 8, 2), (33, 1280, 2, 1), (64, 4096, 8, 8), (70, 512, 8, 3)])
@pytest.mark.parametrize("ksplit", [0, 2, 3, 4])
def test_add_rmsnorm_route(gpu, monkeypatch, M, D, E, k, ksplit):
    """Projection, residual, norm and route in one call: the rows as qgemv_add_rmsnorm leaves them, and the lists, weights and experts
    moe_route makes of the logits it reports; those are the f16 rows' products in 32 bits (|error| <= D 2^-24 sum |h| |w|)."""
    rng = np.random.default_rng(3)
    raw = Q.random_blocks(GGMLType.Q4_K, D * 1280, 0.05, rng)
    seg = ops.Seg(ops.QWeight(raw, GGMLType.Q4_K, D, 1280, gpu))
    monkeypatch.setattr(ops, "gemv_config", lambda segs, M: (1, 8, 1, ksplit) if ksplit else (0, 4, 1, 1))
    xin, h, h2 = torch.zeros(128, 1280, dtype=ops.ACT_DTYPE, device=gpu), *(torch.zeros(128, D, dtype=ops.ACT_DTYPE, device=gpu) for _ in range(2))
    xin[:M] = torch.randn(M, 1280, device=gpu)
    x = torch.randn(128, D, device=gpu)
    x2, nw = x.clone(), torch.rand(D, device=gpu) + 0.5
    wr = (torch.randn(E, D, device=gpu) * 0.1).to(ops.ACT_DTYPE)
    cap = M + 3

    def state():
        return dict(logits=torch.zeros(128, E, device=gpu), topw=torch.zeros(128 * k, device=gpu),
                    counts=torch.zeros(E, dtype=torch.int32, device=gpu), xrows=torch.full((E * cap,), -1, dtype=torch.int32, device=gpu),
                    yrows=torch.full((E * cap,), -1, dtype=torch.int32, device=gpu), sel=torch.zeros(128 * k, dtype=torch.int32, device=gpu))
    a, b = state(), state()
    assert ops.qgemv_add_rmsnorm_route(seg, xin, x, nw, h, M, 0.7, 1e-5, wr, a["logits"], k, a["topw"], a["counts"], a["xrows"], a["yrows"],
                                       cap, sel=a["sel"])
    ops.qgemv_add_rmsnorm(seg, xin, x2, nw, h2, M, 0.7, 1e-5)
    assert torch.equal(x, x2) and (h.float() - h2.float()).abs().max() <= 2.0 ** -10 * h2.float().abs().max()
    hd, wd = h[:M].cpu().double(), wr.cpu().double()
    assert ((a["logits"][:M].cpu().double() - hd @ wd.t()).abs() <= D * 2.0 ** -24 * (hd.abs() @ wd.abs().t())).all()
    ops.moe_route(a["logits"], M, k, b["topw"], b["counts"], b["xrows"], b["yrows"], cap, sel=b["sel"])
    for n in ("topw", "counts", "sel"):
        assert torch.equal(a[n], b[n])
    for n in ("xrows", "yrows"):
        assert torch.equal(a[n].view(E, cap).sort(1).values, b[n].view(E, cap).sort(1).values)
    assert not ops.qgemv_add_rmsnorm_route(seg, xin, x, nw, h, M, 0.7, 1e-5, wr[:1], a["logits"][:, :1], 1, a["topw"], a["counts"], a["xrows"],
                                           a["yrows"], cap)


@pytest.mark.gpu
@pytest.mark.parametrize("bound", [False, True])
@pytest.mark.parametrize("rows", [(0, 1, 257, 256), (96, 97, 0, 0, 600, 5), (0, 0, 0), (255, 64, 128, 129, 300, 1, 0, 40)])
@pytest.mark.parametrize("mode,waves,rt", [(2, 8, 4), (2, 8, 2), (3, 4, 6), (4, 8, 2), (9, 8, 2)])
def test_grouped_blocks(gpu, mode, waves, rt, rows, bound):
    """Blocks of rows of a grouped launch: experts without rows, with whole blocks, with one row more; the number of rows known and not; rows
    of y that no expert has stay as they are."""
    E, K, N, T = len(rows), 512, 272, 640
    raw = [Q.random_blocks(GGMLType.Q5_K, N * K, 0.05, np.random.default_rng(60 + e)) for e in range(E)]
    ws = [ops.QWeight(r, GGMLType.Q5_K, N, K, gpu) for r in raw]
    if mode == 4:
        for w in ws:
            w.expand_dense()
    g = torch.Generator().manual_seed(7)
    x = torch.randn(T, K, generator=g).to(ops.ACT_DTYPE).to(gpu)
    lists = [torch.randperm(T, generator=g)[:n] for n in rows]
    at = np.cumsum([0] + list(rows))
    xr, yr = torch.zeros(E * T, dtype=torch.int32), torch.zeros(E * T, dtype=torch.int32)
    for e, t in enumerate(lists):
        xr[e * T:e * T + len(t)] = t.int()
        yr[e * T:e * T + len(t)] = torch.arange(at[e], at[e + 1]).int()
    xr, yr, counts = xr.to(gpu), yr.to(gpu), torch.tensor(rows, dtype=torch.int32, device=gpu)
    y = torch.full((int(at[-1]) + 3, N), 5.0, device=gpu)
    segs = [ops.Seg(w, 0, xr[e * T:], yr[e * T:], counts[e:e + 1]) for e, w in enumerate(ws)]
    ops.qgemv(segs, x, y, T, epi="f32", mode=mode, waves=waves, rt=rt, ks=1, routed=int(at[-1]) if bound else 0)
    assert (y[int(at[-1]):] == 5.0).all()
    for e, t in enumerate(lists):
        if len(t):
            W, xd = ops.QWeight(raw[e], GGMLType.Q5_K, N, K, "cpu").dense().double(), x.cpu().double()[t]
            got = y[int(at[e]):int(at[e + 1])].cpu().double()
            assert ((got - xd @ W.t()).abs() <= (xd.abs() @ W.abs().t()) * 2.0 ** -9).all()      # (the bound of test_active_tiles)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [256, 5120])
@pytest.mark.parametrize("mode,waves,rt,ks", [(2, 8, 4, 1), (2, 8, 2, 1), (2, 8, 2, 2), (3, 4, 6, 1), (3, 4, 6, 2), (4, 8, 2, 1), (9, 8, 2, 1)])
def test_grouped_lists(gpu, mode, waves, rt, ks, K):
    """Grids that number the blocks with rows: all experts' blocks for a weight tile in turn (K 256), and expert by expert (K 5120); 19 weight
    tiles of 128 and 10 of 256, so the XCDs have unequal shares; K whole and split."""
    rows, N, T = (0, 1, 257, 256, 513, 96, 600, 40), 2320, 640
    E, n, g = len(rows), sum(rows), torch.Generator().manual_seed(K)
    ws = [ops.QWeight(Q.random_blocks(GGMLType.Q5_K, N * K, 0.05, np.random.default_rng(e)), GGMLType.Q5_K, N, K, gpu) for e in range(2)]
    dense = [w.dense(torch.float32).double() for w in ws]
    if mode == 4:
        for w in ws:
            w.expand_dense()
    x = torch.randn(T, K, generator=g).to(ops.ACT_DTYPE).to(gpu)
    lists, at = [torch.randperm(T, generator=g)[:c] for c in rows], np.cumsum((0,) + rows)
    ys = torch.randperm(n, generator=g).int()
    xr, yr = torch.zeros(E * T, dtype=torch.int32), torch.zeros(E * T, dtype=torch.int32)
    for e, t in enumerate(lists):
        xr[e * T:e * T + len(t)], yr[e * T:e * T + len(t)] = t.int(), ys[at[e]:at[e + 1]]
    xr, yr, counts = xr.to(gpu), yr.to(gpu), torch.tensor(rows, dtype=torch.int32, device=gpu)
    segs = [ops.Seg(ws[e % 2], 0, xr[e * T:], yr[e * T:], counts[e:e + 1]) for e in range(E)]
    y = torch.full((n + 1, N), 5.0, device=gpu)
    ops.qgemv(segs, x, y, n if ks > 1 else T, epi="f32", mode=mode, waves=waves, rt=rt, ks=ks, routed=n)
    assert (y[n] == 5.0).all()
    for e, t in enumerate(lists):
        W, xd = dense[e % 2], x[t.to(gpu)].double()
        got = y[ys[at[e]:at[e + 1]].long().to(gpu)].double()
        assert ((got - xd @ W.t()).abs() <= (xd.abs() @ W.abs().t()) * 2.0 ** -9).all(), e      # (the bound of test_active_tiles)


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [GGMLType.Q4_K, GGMLType.Q5_K, GGMLType.Q6_K, GGMLType.Q8_0])
@pytest.mark.parametrize("rows", [(0, 1, 257, 256), (96, 513, 0)])
def test_grouped_gate_and_down(gpu, qt, rows):
    """Mode 9 as the experts of long prompts run it: gate and up with the gate applied to scattered rows, then the down projection from them;
    weight rows that are no multiple of 256, one super-block of K and several. Bounds: test_active_tiles."""
    E, T, n = len(rows), 600, sum(rows)
    rng, g = np.random.default_rng(n), torch.Generator().manual_seed(n)
    for K, F in ((256, 768), (1280, 256)):
        N = 2 * F - 112                                       # (a whole number of 16-row tiles)
        gu, dn = ([Q.random_blocks(qt, a * b, 0.05, rng) for _ in rows] for a, b in ((N, K), (K - 16, F)))
        wg, wd = [ops.QWeight(r, qt, N, K, gpu) for r in gu], [ops.QWeight(r, qt, K - 16, F, gpu) for r in dn]
        lists, at = [torch.randperm(T, generator=g)[:c] for c in rows], np.cumsum((0,) + rows)
        ys = torch.randperm(n, generator=g).int()             # (an expert's rows of y are anywhere)
        xr, yr = torch.zeros(E * T, dtype=torch.int32), torch.zeros(E * T, dtype=torch.int32)
        for e, t in enumerate(lists):
            xr[e * T:e * T + len(t)], yr[e * T:e * T + len(t)] = t.int(), ys[at[e]:at[e + 1]]
        x = torch.randn(T, K, generator=g).to(ops.ACT_DTYPE).to(gpu)
        act = torch.full((n + 1, F), 3.0, device=gpu, dtype=ops.ACT_DTYPE)
        act[:n, N // 2:] = 0
        y = torch.full((n + 1, K - 16), 3.0, device=gpu)
        xr, yr, counts = xr.to(gpu), yr.to(gpu), torch.tensor(rows, dtype=torch.int32, device=gpu)
        for ws, a, b, epi in ((wg, x, act, "swiglu"), (wd, act, y, "f32")):
            segs = [ops.Seg(w, 0, (xr if a is x else yr)[e * T:], yr[e * T:], counts[e:e + 1]) for e, w in enumerate(ws)]
            ops.qgemv(segs, a, b, T, epi=epi, mode=9, waves=8, rt=2, ks=1, routed=n)
        assert (act[n] == 3.0).all() and (y[n] == 3.0).all() and (act[:n, N // 2:] == 0).all()
        for e, t in enumerate(lists):
            W, at_y = ops.QWeight(gu[e], qt, N, K, "cpu").dense().double(), ys[at[e]:at[e + 1]].long()
            xd, c = x.cpu().double()[t], len(t)
            ref, err = xd @ W.t(), (xd.abs() @ W.abs().t()) * 2.0 ** -9
            a, u, ea, eu = (v.view(c, N // 16, 2, 8)[:, :, i].reshape(c, N // 2) for v in (ref, err) for i in (0, 1))
            want = torch.nn.functional.silu(a) * u
            bound = 1.1 * ea * (u.abs() + eu) + torch.nn.functional.silu(a).abs() * eu + want.abs() * 2.0 ** -10 + 2.0 ** -14
            assert ((act.cpu().double()[at_y, :N // 2] - want).abs() <= bound).all()
            D, ad = ops.QWeight(dn[e], qt, K - 16, F, "cpu").dense().double(), act.cpu().double()[at_y]
            assert ((y.cpu().double()[at_y] - ad @ D.t()).abs() <= (ad.abs() @ D.abs().t()) * 2.0 ** -9).all()


def test_expert_gemm_few_rows():
    """Few rows of narrow products: mode 2, the fastest measured (2048 x 4096, 4096 x 14336, 1536 x 2048), not mode 3; wide ones mode 3; long
    prompts mode 9."""
    def mode(N, K, type, per):
        ws = [_W(N, type) for _ in range(8)]
        for w in ws:
            w.K = K
        return tuning.expert_gemm(ws, per)[0]
    for N, K, type in ((2048, 4096, 14), (2048, 4096, 8), (4096, 4096, 12), (4096, 14336, 14), (2816, 2048, 12), (1536, 2048, 12), (2048, 768, 14)):
        assert {mode(N, K, type, per) for per in (3, 10, 17, 24, 32, 40, 50)} == {2}, (N, K)
    assert {mode(N, K, 12, per) for N, K in ((28672, 4096), (8192, 4096), (8192, 2048)) for per in (17, 32, 50)} == {3}
    assert {mode(N, 4096, 12, per) for N in (28672, 8192) for per in (768, 1500)} == {9}


def test_expert_gemm_rule():
    """Configs that exist, of types their modes take; the DMA GEMM only where it is allowed."""
    for type in (7, 8, 12, 13, 14):
        for N, K in ((8192, 2048), (2048, 4096), (28672, 4096), (4096, 14336), (272, 512)):
            for E in (1, 2, 4, 8):
                for per in (0.5, 9, 33, 64, 96, 250, 540, 1000, 4096):
                    ws = [_W(N, type) for _ in range(E)]
                    for w in ws:
                        w.K = K
                    for dma in (True, False):
                        mode, waves, rt, ks = tuning.expert_gemm(ws, per, dma)
                        assert ks == 1 and (mode, waves, rt) in ((2, 8, 4), (2, 8, 2), (3, 4, 6), (9, 8, 2))
                        assert mode == 2 or type != 7
                        assert mode != 3 or (dma and type != 8)
