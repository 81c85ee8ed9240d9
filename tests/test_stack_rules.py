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
