"""The dense f16 GEMM whose wave groups take alternate k-steps (mode 11): every form, at the edges of its tiles and of its ring of K-tiles."""
import pytest
import torch

from nats_llm_studio_amd import ops
from nats_llm_studio_amd.ops import tuning
from test_dense_gemm_gpu import acts, relerr, weight

FORMS = [512 + 16 * mt + nt for mt in (3, 4, 5) for nt in (3, 4, 5, 6, 7, 8)]


class _W:
    d16 = None

    def __init__(self, rows, K):
        self.type, self.rows, self.K = 12, rows, K


def test_one_product_is_one_buffer():
    """Copies count as one product's rows where they are neighbours in one buffer, not where the allocator has put two behind each other."""
    from types import SimpleNamespace as NS

    def seg(rows, at, buf):
        return NS(w=NS(rows=rows, K=64, d16=NS(data_ptr=lambda: at, untyped_storage=lambda: NS(data_ptr=lambda: buf))))
    assert tuning._launch_rows([seg(96, 0, 0), seg(32, 96 * 128, 0), seg(32, 128 * 128, 0)]) == (160,)
    assert tuning._launch_rows([seg(96, 0, 0), seg(32, 96 * 128, 96 * 128), seg(32, 128 * 128, 96 * 128)]) == (96, 64)
    assert tuning._launch_rows([seg(96, 0, 0), seg(32, 97 * 128, 0)]) == (96, 32)


def test_rule_gives_built_forms():
    """The forms that the rule can choose are those that are built, with at least six K-tiles to a part; none for rows that its stores do not take."""
    for rows in (256, 2048, 4100, 6144, 16384, 28672):
        for K in (256, 512, 2048, 14336):
            for M in (128, 190, 257, 640, 1000, 2560, 2561):
                t, (mode, waves, rt, ks) = tuning._best11((rows,), K, M, False)
                assert t > 0 and mode == 11 and waves == 8 and rt in FORMS and (ks == 1 or K // 64 // ks >= 6)
                cfg = tuning.select_dense([ops.Seg(_W(rows, K))], M)
                assert cfg[0] != 11 or M <= 2560
            assert tuning.select_dense([ops.Seg(_W(rows + 1, K))], 300)[0] != 11


@pytest.mark.parametrize("rt", [0, 512, 512 + 16 * 3 + 2, 512 + 16 * 3 + 9, 512 + 16 * 2 + 3, 512 + 16 * 6 + 3, 512 + 48, 256 + 51, 768 + 51, 1024 + 51, -1, 4096 + 563])
def test_unbuilt_forms_are_refused(rt):
    """The launcher refuses forms that are not built, those of no weight rows among them."""
    from nats_llm_studio_amd.ops import _lib
    arr = (_lib.NlsSeg * 1)(_lib.NlsSeg(4096, None, None, None, 1, 2048, 2048, 0))
    assert _lib.lib().nls_qgemv(arr, 1, 4096, 2048, 4096, 2048, 300, 1.0, ops.EPI["f32"], None, 8, rt, 11, 1, None, None) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("rt", FORMS)
@pytest.mark.parametrize("rows,K", [(772, 256), (64, 512), (1020, 1536)])
def test_forms(gpu, rt, rows, K):
    """Rows short of a weight tile and of a row block; fewer K-tiles than the ring holds, splits with parts of one K-tile more than others."""
    w = weight(rows, K)
    for M in (1, 95, 96, 161, 320, 333):
        x = acts(M, K)
        z = x[:M].double() @ w.d16.double().T
        for epi, dt, ks in (("f32", torch.float32, 1), ("add", torch.float32, 1), ("act", torch.float16, 1), ("f32", torch.float32, 3)):
            y = torch.full((M + 1, rows + 4), 7.0, device="cuda", dtype=dt)
            ops.qgemv([ops.Seg(w, 4)], x, y, M, epi=epi, mode=11, waves=8, rt=rt, ks=ks)
            # f32 sums of K products; f16 outputs round to 2^-11
            assert relerr(y[:M, 4:] - (7 if epi == "add" else 0), z) < (5e-4 if epi == "act" else 4e-6), (M, ks, epi)
            assert (y[M] == 7).all() and (y[:, :4] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rt", [563, 583, 599, 600])
@pytest.mark.parametrize("M", [130, 300])
def test_gate_and_head(gpu, rt, M):
    """SwiGLU over a row count that no tile divides, a head's arg-max with its logits."""
    rows, K = 2000, 512
    w, x = weight(rows, K), acts(M, K)
    z = x[:M].double() @ w.d16.double().T
    v = z.view(M, rows // 16, 2, 8)
    want = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, rows // 2)
    y = torch.full((M + 1, rows // 2), 7.0, device="cuda", dtype=torch.float16)
    ops.qgemv([ops.Seg(w)], x, y, M, epi="swiglu", mode=11, waves=8, rt=rt, ks=1)
    assert relerr(y[:M], want) < 5e-4 and (y[M:] == 7).all()                       # f16 outputs round to 2^-11
    logits = torch.full((M + 1, rows), 7.0, device="cuda")
    keys, ids = torch.zeros(M + 1, dtype=torch.int64, device="cuda"), torch.full((M + 1,), -1, dtype=torch.int32, device="cuda")
    ops.qgemv([ops.Seg(w)], x, logits, M, epi="f32", argmax=keys, mode=11, waves=8, rt=rt, ks=1)
    ops.argmax_unpack(keys, M, ids)
    assert (ids[:M].long() == logits[:M].argmax(1)).all() and int(keys[M]) == 0 and relerr(logits[:M], z) < 4e-6


@pytest.mark.gpu
@pytest.mark.parametrize("rt", [563, 599])
@pytest.mark.parametrize("D,bias", [(128, True), (34, True), (64, False)])
def test_rope(gpu, rt, D, bias):
    """Three segments with RoPE and the cache rows, against mode 10."""
    Hq, Hkv, K, M = 16, 8, 64 * 4, 200
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
    for cfg in ((11, 8, rt, 1), (10, 8, 2, 1)):
        q = torch.full((pad, Hq * D), 776.0, dtype=torch.bfloat16, device="cuda")
        kc, vc = (torch.full((pad, Hkv, D), 776.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        ops.qkv_rope_kv(segs, x, torch.zeros(pad, n, device="cuda"), pos, slot, cs, q, kc, vc, M, Hq, Hkv, D, cfg=cfg, bias=b)
        outs.append((q, kc, vc))
    for a, b in zip(*outs):      # one bf16 rounding apart at most, and the same places written
        assert relerr(a, b) < 2e-3 and ((a == 776) == (b == 776)).all()


def ragged(x, how):
    """x's rows as they are, 8 bytes off a multiple of 16, or from there on."""
    M, K = x.shape
    if how == "regular":
        return x
    wide = torch.zeros(M, K + 8, dtype=x.dtype, device=x.device)
    v = wide.view(-1)[:M * (K + 4)].view(M, K + 4)[:, :K] if how == "stride" else wide[:, 4:4 + K]
    return v.copy_(x)


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["regular", "stride", "start"])
@pytest.mark.parametrize("copies", [True, False])
@pytest.mark.parametrize("M", [128, 192, 300])
def test_fused_launches_take_any_rows(gpu, how, copies, M):
    """Q, K and V with RoPE, and projections with residual, norm and route, as chosen by size, for rows that the copies to LDS do not take; with f16 copies
    and without. Against the launches of irregular rows done on regular ones: the same products of f16 values, summed in 32 bits."""
    D, Hq, Hkv, K = 128, 16, 8, 2048
    ws = [weight(h * D, K, s) for s, h in enumerate((Hq, Hkv, Hkv))]
    o = weight(K, K, 5)
    for w in (*ws, o) if not copies else ws:
        w.d16 = None
    if copies:
        ops.QWeight.expand_dense_group(ws)               # (one buffer, as a loaded model has them)
    segs = [ops.Seg(ws[0], 0), ops.Seg(ws[1], Hq * D), ops.Seg(ws[2], (Hq + Hkv) * D)]
    x, n = acts(M, K), (Hq + 2 * Hkv) * D
    pad = x.shape[0]
    cs = ops.rope_table(400, D, 10000.0, torch.device("cuda"))
    pos, slot = (torch.arange(pad, dtype=torch.int32, device="cuda") * 7) % 400, torch.arange(pad, dtype=torch.int32, device="cuda")
    assert ops.gemv_config(segs, M)[0] == (11 if copies else 2) and (M > 192 or ops.gemv_config([ops.Seg(o)], M)[0] == (11 if copies else 2))
    nw, wr = torch.randn(K, device="cuda"), (torch.randn(4, K, device="cuda") * 0.05).half()
    res = torch.randn(pad, K, device="cuda")

    def run(x):
        q = torch.zeros(pad, Hq * D, dtype=torch.bfloat16, device="cuda")
        kc, vc = (torch.zeros(pad, Hkv, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        ops.qkv_rope_kv(segs, x, torch.zeros(pad, n, device="cuda"), pos, slot, cs, q, kc, vc, M, Hq, Hkv, D)
        a, h = res.clone(), torch.zeros(pad, K, dtype=torch.float16, device="cuda")
        ops.qgemv_add_rmsnorm(ops.Seg(o), x, a, nw, h, M, 0.5, 1e-5)
        b, h2, lg = res.clone(), torch.zeros_like(h), torch.zeros(pad, 4, device="cuda")
        ints = [torch.zeros(m, dtype=torch.int32, device="cuda") for m in (4, 4 * pad, 4 * pad)]
        assert ops.qgemv_add_rmsnorm_route(ops.Seg(o), x, b, nw, h2, M, 0.5, 1e-5, wr, lg, 2, torch.zeros(pad * 2, device="cuda"), *ints, pad)
        return q[:M], kc[:M], vc[:M], a[:M], h[:M], b[:M], h2[:M], lg[:M]
    for got, want, tol in zip(run(ragged(x, how)), run(x), (2e-3, 2e-3, 2e-3, 4e-6, 5e-4, 4e-6, 5e-4, 2e-3)):
        assert relerr(got, want) < tol
    z = x[:M].double() @ torch.cat([w.dense().double().to("cuda") for w in ws]).T
    assert relerr(run(x)[2].view(M, -1), z[:, (Hq + Hkv) * D:]) < 4e-3              # (bf16 rows: 2^-9; f16 copies round once more)
