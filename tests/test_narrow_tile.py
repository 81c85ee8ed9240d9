"""The 64 x 32 tile of the GEMM: steps of K, rows and columns around its edges, and the launches that take it."""
import ctypes

import pytest
import torch

from nats_llm_studio_amd.ops import stack as S


def launch(N, Kd, slabs=1):
    w = type("W", (), dict(groups=1, N=N, K=Kd, f32=False, nsub=S.act_ld(Kd) // 32))()
    L = S.LinLaunch.__new__(S.LinLaunch)
    L.f32, L.plan, L._rows = 0, None, 512 if slabs > 1 else 0
    L.segs = [type("Seg", (), dict(w=w, slabs=slabs, s=S.LinSeg(), y=type("Y", (), dict(shape=(4096, N)))()))()]
    return L


def test_rule():
    """Wide launches of 13 to 32 rows take it up to one tile for each CU, larger ones the balanced tiles; narrow ones stream; launches with slabs of 17
    rows on take as many splits as there are CUs for."""
    for N in (8256, 10240, 16384):
        assert [launch(N, 4096).config(M) for M in (13, 16, 17, 32)] == [(True, 12)] * 4
        assert launch(N, 4096).config(12)[0] is False and launch(N, 4096).config(33) == (True, 5)
    assert launch(16448, 4096).config(16) != (True, 12) and launch(8192, 4096).config(16)[0] is False
    assert [launch(4096, 17408, 8).choice(M) for M in (16, 24, 32)] == [((True, 12), 4)] * 3
    assert launch(2048, 8704, 8).choice(24) == ((True, 12), 8) and launch(2048, 8704, 8).choice(16)[0][0] is False


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 31, 32, 33, 70])
def test_edges(M):
    """One to nineteen steps of K, whole and in two splits, rows at and past a tile's edge. |error| <= 2^-24 K sum |x| |w|."""
    K, N = S, 200
    for steps in range(1, 20):
        Kd = steps * 64 - 3
        g = torch.Generator().manual_seed(steps)
        x, w = (torch.randn(n, Kd, generator=g).bfloat16() for n in (M, N))
        xa = torch.zeros(M, K.act_ld(Kd), dtype=torch.bfloat16, device="cuda")
        xa[:, :Kd] = x
        y = torch.full((2 * M + 1, N), 9.0, device="cuda")
        p = K.PackedLinear(w, False, "cuda")
        a = K.LinLaunch([K.Seg(p, xa, y, slabs=2, slab_rows=M)]).a
        a.s[0].M = M
        want, bound = x.double() @ w.double().T, 2.0 ** -24 * (Kd + 8) * (x.double().abs() @ w.double().abs().T)
        for ks in (1, 2)[:min(2, steps)]:
            a.s[0].ks = ks
            K._check(K.lib().nls_lin_gemm(ctypes.byref(a), 0, 12, torch.cuda.current_stream().cuda_stream), "gemm")
            got = y[:2 * M].view(2, M, N)[:ks].sum(0).cpu().double()
            assert ((got - want).abs() <= bound + 2.0 ** -23 * want.abs()).all() and (y[-1] == 9).all(), (steps, ks)


def test_splits_stay_in_one_round():
    """Splits of the tile give each CU one workgroup at most, at widths that 256 is no multiple of too; short launches stream."""
    for N in (640, 2560, 3072, 4096, 5120, 6144, 10240, 17000):
        for M in (16, 17, 32):
            c, ks = launch(N, 8192, 8).choice(M)
            assert c[0] == (M > 16 or N >= 4096) and (not c[0] or ks == 1 or ks * -(-N // 64) <= 256)
    for N, Kd in ((2048, 2048), (1024, 4096), (3072, 2048), (96, 4096)):
        assert launch(N, Kd, 8).choice(24)[0][0] is False
