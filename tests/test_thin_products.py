"""Products of up to 128 inputs straight from memory, and the epilogues taken out of a tile's blocks."""
import pytest
import torch

from nats_llm_studio_amd.ops import stack as ops


def test_rule():
    """From two workgroups of 64 x 128 to a CU on, in 16 bits, for up to four sub-tiles of K."""
    class W:
        def __init__(self, N, nsub):
            self.N, self.nsub, self.groups, self.K = N, nsub, 1, 32 * nsub

    class S:
        rows, ng = None, 1

    class Seg:
        def __init__(self, N, nsub):
            self.w, self.s = W(N, nsub), S()

    def config(M, N, nsub, f32=0):
        L = object.__new__(ops.LinLaunch)
        L.segs, L.plan, L.f32 = [Seg(N, nsub)], None, f32
        return L.config(M)
    for M, N in ((2048, 2048), (4096, 1024), (16384, 256)):
        assert config(M, N, 2) == config(M, N, 4) == (True, ops.THIN)
        assert config(M - 128, N, 4) == (True, 0) and config(M, N, 6)[1] != ops.THIN and config(M, N, 4, 1)[1] != ops.THIN


@pytest.mark.gpu
@pytest.mark.parametrize("epi", ["none", "silu", "tanh", "sigmoid", "relu2", "decay", "sigpow", "gate", "siluglu"])
@pytest.mark.parametrize("M,N,Kin,act", [(65, 64, 16, False), (129, 72, 128, True), (300, 200, 64, False), (127, 70, 100, False), (257, 20, 33, True)])
def test_thin(epi, M, N, Kin, act):
    """The bits of the 64 x 64 tile (the same order of sums), in whole groups of four columns and, with rows that are not, one by one;
    nothing else is written. Against 64 bits: products of 128 inputs in 32 bits and functions of them, 2^-7 in bf16, 2^-13 else."""
    K = ops
    K.lib()
    g = torch.Generator().manual_seed(M + N)
    w, x = torch.randn(N, Kin, generator=g).to(torch.bfloat16), torch.zeros(M, K.act_ld(Kin), dtype=torch.bfloat16)
    x[:, :Kin] = (torch.randn(M, Kin, generator=g) / Kin ** 0.5).to(torch.bfloat16)
    b, gt = torch.randn(N, generator=g) - 1, torch.rand(M, 1, generator=g)
    p, xd, bd, gd = K.PackedLinear(w, False, "cuda"), x.cuda(), b.cuda(), gt.cuda()
    glu, dt, out = epi == "siluglu", torch.bfloat16 if act else torch.float32, []
    if glu and not act:
        pytest.skip("gated outputs are in the activation type")
    n = N // 2 if glu else N
    for cfg in (0, K.THIN):
        for ld in (K.pad_to(n, 8) + 8, K.pad_to(n, 8) + 9):
            y = torch.full((M + 1, ld), 7.0, dtype=dt, device="cuda")
            L = K.LinLaunch([K.Seg(p, xd, y, epi, bias=bd if epi in ("decay", "sigpow") else None, gate=gd if epi == "gate" else None,
                                   alpha=0.25 if epi == "sigpow" else 1.0)])
            L._cfg[M] = ((True, cfg), 1)
            L.run(M, torch.cuda.current_stream().cuda_stream)
            y = y.cpu()
            assert (y[M] == 7).all() and (y[:, n:] == 7).all()
            out.append(y[:M, :n])
    assert all(torch.equal(out[0], o) for o in out[1:])
    v = x[:, :Kin].double() @ w.double().T
    if epi in ("decay", "sigpow"):
        v = v + b.double()
    f = dict(none=lambda v: v, silu=torch.nn.functional.silu, tanh=torch.tanh, sigmoid=torch.sigmoid, relu2=lambda v: v.relu() ** 2,
             decay=lambda v: torch.exp(-torch.exp(v)), sigpow=lambda v: torch.sigmoid(v) ** 0.25, gate=lambda v: v * gt.double(),
             siluglu=lambda v: torch.nn.functional.silu(v[:, ::2]) * v[:, 1::2])[epi]
    want = f(v)
    assert ((out[0].double() - want).abs() <= (2.0 ** -7 if act else 2.0 ** -13) * (want.abs() + 1)).all()
