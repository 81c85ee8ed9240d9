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


def test_launches_fit_their_rows():
    """Rows of x that are not 16 bytes apart (or start elsewhere), and y's columns that are not at fours, go to launches that take them; the others
    stay with what the sizes choose."""
    from types import SimpleNamespace as NS

    def rows_of(stride, at=0):
        return NS(stride=lambda d: stride, data_ptr=lambda: at)
    for t in (8, 12, 14):
        for rows, K in ((16384, 2048), (2048, 8192), (2048, 2048), (49155, 2048)):
            for M in (65, 96, 255, 256, 300, 3000):
                cfg = tuning.heuristic([ops.Seg(_W(t, rows, K))], M)
                for x in (rows_of(K), rows_of(K + 4), rows_of(K + 1), rows_of(K, 8)):
                    for y in (rows_of(rows), rows_of(rows + 1), rows_of(rows + 5), None):
                        for ycol in (0, 3):
                            for epi in ("f32", "add", "act", "swiglu", "argmax"):
                                segs = [ops.Seg(_W(t, rows, K), ycol)]
                                got = ops.fitting_config(cfg, segs, M, x, y, epi)
                                regular = x.stride(0) % 8 == 0 and x.data_ptr() == 0
                                stores = ycol == 0 and (epi == "argmax" and cfg[3] == 1 or rows % 4 == 0
                                                        and (y is None or y.stride(0) % 4 == 0 or epi in ("swiglu", "argmax")))
                                assert got == (cfg if regular and (stores or cfg[0] < 9) or cfg[0] < 3 else tuning.any_rows(segs, M))
                                assert got[0] in (1, 2) or (regular and (stores or got[0] < 9))


def test_stores_of_four_are_refused():
    """The launcher itself takes no rows for modes 9 to 11 that their stores do not fit, with any epilogue but an unsplit arg-max."""
    from nats_llm_studio_amd.ops import _lib
    for mode, waves, rt, t in ((9, 8, 2, 8), (10, 8, 1, 1), (11, 8, 512 + 16 * 3 + 3, 1)):
        for ks in (1, 2):
            arr = (_lib.NlsSeg * 1)(_lib.NlsSeg(4096, None, None, None, t, 8195, 2048, 0))
            for epi in ("f32", "add", "act", "slabs") + (("argmax",) if ks > 1 else ()):
                assert _lib.lib().nls_qgemv(arr, 1, 4096, 2048, 4096, 8196, 300, 1.0, ops.EPI[epi], None, waves, rt, mode, ks, 4096, None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("M", [256, 300])
@pytest.mark.parametrize("qt,rows,K", [(GGMLType.Q8_0, 8195, 2048), (GGMLType.Q8_0, 1030, 2304), (GGMLType.Q8_0, 2048, 2048), (GGMLType.Q4_K, 4099, 1024),
                                       (GGMLType.Q6_K, 130, 512)])
def test_many_rows_anywhere(gpu, M, qt, rows, K):
    """256 rows and more of wide, down and square shapes: y in an odd place with rows of odd length, with and without an arg-max, x's rows 8 bytes off a
    multiple of 16, and starting there. Bound as above."""
    raw = Q.random_blocks(qt, rows * K, 0.05, np.random.default_rng(M))
    w = ops.QWeight(raw, qt, rows, K, gpu)
    W = ops.QWeight(raw, qt, rows, K, "cpu").dense().double()
    wide = torch.randn(320, K + 8, device=gpu).to(ops.ACT_DTYPE)
    for x in (wide[:, :K].contiguous(), wide.view(-1)[:320 * (K + 4)].view(320, K + 4)[:, :K], wide[:, 4:4 + K]):
        xd = x[:M].cpu().double()
        z, bound = xd @ W.t(), (xd.abs() @ W.abs().t()) * 2.0 ** -9
        for at, ld in ((0, rows + (-rows) % 4), (3, rows + 5), (0, rows + (-rows) % 2 + 1)):
            y = torch.full((M + 1, ld), 3.0, device=gpu)
            ops.qgemv([ops.Seg(w, at)], x, y, M)
            assert ((y[:M, at:at + rows].cpu().double() - z).abs() <= bound).all(), (at, ld)
            assert (y[M:] == 3.0).all() and (y[:, :at] == 3.0).all() and (y[:, at + rows:] == 3.0).all()
        for at in (0, 3):
            for epi in ("f32", "argmax"):
                keys = torch.zeros(M + 1, dtype=torch.int64, device=gpu)
                if epi == "f32":
                    logits = torch.full((M, at + rows), 3.0, device=gpu)
                ops.qgemv([ops.Seg(w, at)], x, logits, M, epi=epi, argmax=keys)
                ids = torch.full((M,), -1, dtype=torch.int32, device=gpu)
                ops.argmax_unpack(keys, M, ids)
                assert ((logits[:, at:].cpu().double() - z).abs() <= bound).all() and int(keys[M]) == 0
                top = z.gather(1, ids.cpu().long()[:, None] - at)[:, 0]
                assert (top >= (z - 2 * bound).amax(1)).all() and (epi == "argmax" or (ids.long() - at == logits[:, at:].argmax(1)).all())
