"""Single-token steps of the recurrences: states loaded ahead of the inputs (few workgroups) and behind them give the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind,H,D,V", [("gla", 32, 64, 128), ("gla", 27, 20, 128), ("gla", 40, 128, 60), ("gla", 33, 48, 1024), ("wkv", 40, 64, 64),
                                        ("wkv", 33, 128, 128), ("wkv", 36, 100, 100)])
def test_forms(dtype, kind, H, D, V):
    """Forty tokens in one launch (more than two workgroups to a CU), and the same tokens one and ten at a time; first tokens and unused rows among them."""
    from nats_llm_studio_amd.ops import stack as K
    T = 40
    g = torch.Generator().manual_seed(D)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    lo = K.act_ld(H * (2 * D + V))
    z, gate, norm = rnd(T, lo + 64), rnd(T, H * V), torch.rand(H * V, generator=g).cuda()
    q, k, v, low = z, z[:, H * D:], z[:, 2 * H * D:], z[:, lo:]
    a2, a2b, u = rnd(H * D, 16), torch.randn(H * D, generator=g).cuda(), torch.randn(H * D, generator=g).cuda()
    w, x = torch.rand(T, H * D, generator=g).cuda(), torch.randn(T, H * D, generator=g).cuda()
    S0 = torch.randn(T, H * D * V, generator=g).cuda()
    runs = torch.tensor([[i, 1, -1 if i % 7 == 5 else i, i % 3] for i in range(T)], dtype=torch.int32).cuda()
    st = torch.cuda.current_stream().cuda_stream

    def run(n):
        S, out, prev = S0.clone(), torch.full((T, H * V), 7.0, dtype=dtype, device="cuda"), torch.zeros(T, H * D, device="cuda")
        for i in range(0, T, n):
            if kind == "gla":
                K.gla_step(q, k, v, None, (low, a2, a2b, 0.3), 0.5, S, runs[i:i + n], n, norm, gate, out, H, D, V, 1e-5, st)
            else:
                K.wkv_step(q, k, v, w, u, S, x, prev, runs[i:i + n], n, norm, gate, out, H, D, 1e-5, st)
        return S, out, prev
    one = run(T)
    for n in (1, 10):
        assert all(torch.equal(a, b) for a, b in zip(one, run(n))), n
    assert not torch.equal(one[0], S0) and torch.equal(one[0][5], S0[5]) and (one[1][5] == 7).all()
