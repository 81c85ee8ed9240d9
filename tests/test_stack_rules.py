"""Launch rules of the linear layers of the stacks, on the host alone."""
import pytest

from nats_llm_studio_amd.ops import stack as S


class _W:
    groups = 1

    def __init__(self, N, Kd, f32):
        self.N, self.K, self.f32, self.nsub = N, Kd, f32, S.act_ld(Kd) // (16 if f32 else 32)


def launch(N, Kd, f32=False, rows=0, slabs=1, slab_rows=0):
    """A launch of one N x Kd layer without its buffers; y: `rows` rows."""
    L = S.LinLaunch.__new__(S.LinLaunch)
    seg = type("Seg", (), dict(w=_W(N, Kd, f32), slabs=slabs, s=S.LinSeg(), y=type("Y", (), dict(shape=(rows, N)))()))()
    L.f32, L.segs, L.plan, L._rows = int(f32), [seg], None, slab_rows
    return L


@pytest.mark.parametrize("Kd", [2090, 4096, 17408])
@pytest.mark.parametrize("N", [1030, 2048, 3072, 4096, 4112, 6144, 8192])
def test_few_rows(N, Kd):
    """17 to 64 rows of up to 8192 outputs: the smallest tiles with at most a workgroup for each CU, and all of them cover the rows."""
    for M in range(17, 65):
        gemm, mt, nw, rt = launch(N, Kd).config(M)
        grids = {t: -(-N // (16 * t[1])) * -(-M // (16 * t[0])) for t in ((2, 1), (2, 2), (4, 2))}
        assert not gemm and nw == 8 and grids[mt, rt] <= 256
        smaller = [t for t in grids if t[0] * t[1] < mt * rt and grids[t] <= 256]
        assert all(t == (2, 2) and M <= 48 for t in smaller)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("N,Kd", [(4096, 17408), (4096, 6144), (2048, 5632), (640, 4096), (36000, 2048), (1030, 2090), (96, 8192)])
@pytest.mark.parametrize("pad", [64, 512, 4096])
def test_splits_of_a_launch(N, Kd, pad, f32):
    """What a launch with slabs runs, over the rows a buffer of `pad` takes: no more splits than slabs, than fit the buffer's rows at the
    distance the launch sets, or than leave 8 sub-tile pairs to each; a config that exists and takes the launch."""
    bound = min(pad, 512)
    rows = max(pad, 8 * bound)
    L = launch(N, Kd, f32, rows, 8, bound)
    nsub = L.segs[0].w.nsub
    for M in sorted({m for b in (1, 9, 16, 17, 32, 33, 64, 65, 128, 129, 200, 256, 300, 512, 513, 601, 1000, 1365, 2047, 2049, 3001, 4096)
                     for m in (b, pad) if m <= pad}):
        (gemm, c, *more), ks = L.choice(M)
        step = L.slab_step(M)
        assert step >= M and step % 4 == 0 and 1 <= ks <= 8 and ks * step <= max(rows, step)
        assert ks == 1 or nsub // ks >= 16
        if gemm:
            assert c in S.GEMM_TILES and (c != 7 or (not f32 and nsub // 2 // ks >= 3))
        else:
            assert c in (1, 2, 4) and more[0] in (4, 8, 16) and more[1] in (1, 2, 4)


def test_tiles_of_some_hundred_rows():
    """The tiles of lin_pair.hip: above 128 rows, where their workgroups fill the chip and whole rounds of the phased tile do not; never for row maps."""
    pair = lambda L, M: L.config(M)[1] >= 256
    for N, Kd, M in ((10240, 4096, 300), (14336, 2048, 200), (24576, 4096, 300), (10240, 2048, 800), (17944, 2048, 400), (6144, 4096, 640)):
        L = launch(N, Kd)
        assert pair(L, M) and not pair(L, 128)
        L.segs[0].s.xmap = 1
        assert not pair(L, M)
    for N, Kd, M in ((2048, 2048, 200), (3072, 2048, 512), (1024, 4096, 1024), (24576, 4096, 512), (35888, 4096, 3000)):
        assert not pair(launch(N, Kd), M)


def test_equal_rounds():
    """Wide launches of few rows whose rounds sum up to the same weight rows on two tiles: 64 rows to a tile up to 40 rows, then 128."""
    for N in (26880, 32000, 32768):
        assert [launch(N, 4096).config(M) for M in (17, 32, 40, 41, 64)] == [(True, 0)] * 3 + [(True, 10)] * 2
    assert [launch(35888, 4096).config(M) for M in (24, 64)] == [(True, 9)] * 2


def test_short_expert_products():
    """Experts of a few dozen rows: tiles by rounds only where the inputs are many."""
    for N, Kd, want in ((512, 2048, 0), (2048, 512, 0), (3072, 2048, 0), (4096, 6144, 10), (6144, 4096, 8)):
        L = launch(N, Kd)
        L.plan, L.segs[0].s.rows = S.MoePlan(120, 8, 2, 1, 1, 1.0, "cpu"), 1
        L.segs[0].w.groups = 8
        assert L.plan.bm(120) == 64 and L.config(120) == (True, want), (N, Kd)


def test_tiles_of_32_bits():
    """One workgroup to a CU at most: the f32 MFMA, unless the inputs are few; more of them: bf16 parts. Splits of K count as workgroups."""
    for N, Kd, M in ((4096, 12288, 65), (4096, 12288, 256), (16384, 4096, 64), (2048, 512, 512), (1030, 2090, 900)):
        assert launch(N, Kd, True).config(M) == (True, 5)
    for N, Kd, M in ((4096, 12288, 257), (16384, 4096, 65), (35888, 4096, 33), (2048, 64, 200), (2048, 128, 200)):
        assert launch(N, Kd, True).config(M)[1] in (0, 1, 2)
    assert launch(2048, 8704, True, 4096, 8, 512).choice(64) == ((True, 5), 8)
    for N, Kd, T, want in ((4096, 3072, 150, (5,)), (2048, 4096, 32, (5,)), (8192, 2048, 150, (0, 1)), (4096, 3072, 300, (0, 1))):
        L = launch(N, Kd, True)
        L.plan, L.segs[0].s.rows = S.MoePlan(T, 8, 2, 1, 1, 1.0, "cpu"), 1
        L.segs[0].w.groups = 8
        assert L.plan.bm(T) == 64 and L.config(T)[1] in want, (N, Kd, T)
    assert launch(2048, 8704, True, 8192, 8, 512).choice(900)[0][1] in (0, 1, 2)
