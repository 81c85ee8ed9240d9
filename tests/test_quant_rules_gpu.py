"""The rules that choose the launch of quantised projections without a tuned entry, and the launches they choose."""
import numpy as np
import pytest
import torch

from nats_llm_studio_amd import ops
from nats_llm_studio_amd.gguf import quants as Q
from nats_llm_studio_amd.gguf.constants import GGMLType
from nats_llm_studio_amd.ops import tuning


class _W:
    def __init__(self, type, rows, K):
        self.type, self.rows, self.K = type, rows, K


@pytest.mark.parametrize("types", [(8,), (12,), (13,), (14,), (12, 12, 14), (13, 13, 14), (8, 8, 14)])
def test_rules_give_launches(types):
    """Every config is one the launcher takes: path A up to 32 rows, a split leaves two super-blocks of K to a part, no LDS-DMA GEMM for Q8_0."""
    for rows in (16, 208, 2048, 16384, 128256):
        for K in (256, 512, 768, 2048, 14336):
            segs = [ops.Seg(_W(t, rows, K), i * rows) for i, t in enumerate(types)]
            for M in (2, 8, 9, 16, 17, 32, 33, 64, 65, 96, 97, 128, 129, 192, 255, 256, 700):
                mode, waves, rt, ks = tuning.heuristic(segs, M)
                assert ks >= 1 and (ks == 1 or ks * 2 <= K // 256)
                assert {0: M <= 32 and ks == 1 and waves == 4 and rt in (1, 2), 1: M <= 64 and waves in (4, 8) and rt in (1, 2),
                        2: M > 64 and waves == 8 and rt in (1, 2, 4), 3: M > 64 and waves == 4 and rt in (4, 6) and 8 not in types,
                        9: M >= 256}[mode], (types, rows, K, M, mode, waves, rt, ks)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2, 8, 9, 17, 33, 64, 65, 96, 97, 129, 193, 255])
@pytest.mark.parametrize("qt,rows,K", [(GGMLType.Q4_K, 2048, 2048), (GGMLType.Q4_K, 209, 2048), (GGMLType.Q5_K, 4111, 512), (GGMLType.Q6_K, 1040, 4096),
                                       (GGMLType.Q8_0, 2048, 2048), (GGMLType.Q8_0, 77, 256), (GGMLType.Q8_0, 3000, 1536)])
def test_chosen_launch(gpu, M, qt, rows, K):
    """Rows short of a tile, single super-blocks and splits, y's columns at an odd place; x also with rows that are not 16 bytes apart. x and the
    dequantised weights are f16 (a weight is rounded at most twice), products are summed in 32 bits: |error| <= 2^-9 sum |x| |w|."""
    raw = Q.random_blocks(qt, rows * K, 0.05, np.random.default_rng(M))
    seg = [ops.Seg(ops.QWeight(raw, qt, rows, K, gpu), 3)]
    W = ops.QWeight(raw, qt, rows, K, "cpu").dense().double()
    wide = torch.randn(256, K + 12, device=gpu).to(ops.ACT_DTYPE)
    for x in (wide[:, :K].contiguous(), wide[:, :K]) if M > 64 else (wide[:, :K].contiguous(),):
        y = torch.full((257, rows + 5), 3.0, device=gpu)
        ops.qgemv(seg, x, y, M)
        xd = x[:M].cpu().double()
        err = (y[:M, 3:3 + rows].cpu().double() - xd @ W.t()).abs()
        assert (err <= (xd.abs() @ W.abs().t()) * 2.0 ** -9).all(), (tuning.select(seg, M), err.max())
        assert (y[M:] == 3.0).all() and (y[:, :3] == 3.0).all() and (y[:, 3 + rows:] == 3.0).all()
