"""The wkv scan of few runs: ends of its chunks and of eight tokens, runs of their own lengths, a run cut anywhere, both types."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nats_llm_studio_amd.ops import stack
    stack.lib()
    return stack


@pytest.mark.parametrize("D,H", [(64, 3), (128, 2), (256, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens", [[1, 7], [8, 0], [31, 33], [70], [16, 17, 100]], ids=str)
def test_few_runs(K, D, H, dtype, lens):
    """|error| <= 2^-24 (i + D + 8) of the magnitudes behind token i: each token adds two roundings to a state and an output sums D of them. The same run
    in two pieces gives the same bits."""
    assert H * len(lens) * (D // 8) <= 512                       # (the launch's rule)
    g = torch.Generator().manual_seed(D + len(lens))
    T, W = sum(lens), H * D
    r, k, v = (torch.randn(T, W, generator=g).to(dtype).cuda() for _ in range(3))
    w, u = torch.sigmoid(torch.randn(T, W, generator=g) + 1).cuda(), torch.randn(W, generator=g).cuda()
    x = torch.randn(T, W, generator=g).cuda()
    S0 = torch.randn(len(lens), H * D * D, generator=g).cuda()
    starts = [sum(lens[:i]) for i in range(len(lens))]
    pos = [5 * (i & 1) for i in range(len(lens))]                # every second run goes on from its slot

    def run(runs, state, prev):
        o = torch.full((T + 1, W), 7.0, device="cuda")
        K.wkv_scan(r, k, v, w, u, o, state, x, prev, torch.tensor(runs, dtype=torch.int32, device="cuda"), len(runs), H, D,
                   torch.cuda.current_stream().cuda_stream)
        assert (o[T] == 7).all()
        return o[:T]
    state, prev = S0.clone(), torch.zeros(len(lens), W, device="cuda")
    o = run([[s, n, i, p] for i, (s, n, p) in enumerate(zip(starts, lens, pos))] , state, prev)
    st2, pv2 = S0.clone(), torch.zeros_like(prev)
    cut = [n // 3 for n in lens]
    a = run([[s, c, i if c else -1, p] for i, (s, c, p) in enumerate(zip(starts, cut, pos))], st2, pv2)
    b = run([[s + c, n - c, i, p + c] for i, (s, c, n, p) in enumerate(zip(starts, cut, lens, pos))], st2, pv2)
    for i, (s, c, n) in enumerate(zip(starts, cut, lens)):
        if not n:
            assert torch.equal(state[i], S0[i])
            continue
        assert torch.equal(o[s:s + c], a[s:s + c]) and torch.equal(o[s + c:s + n], b[s + c:s + n]) and torch.equal(state[i], st2[i])
        assert torch.equal(prev[i], x[s + n - 1]) and torch.equal(pv2[i], prev[i])
        S = S0[i].double().view(H, D, D) * (pos[i] > 0)
        A = S.abs()
        uu = u.double().view(H, D, 1)
        for t in range(n):
            rr, kk, vv, ww = (q[s + t].double().view(H, D) for q in (r, k, v, w))
            kv = kk[:, :, None] * vv[:, None, :]
            want, mag = ((S + uu * kv) * rr[:, :, None]).sum(1), ((A + uu.abs() * kv.abs()) * rr.abs()[:, :, None]).sum(1)
            assert ((o[s + t].double().view(H, D) - want).abs() <= 2.0 ** -24 * (t + D + 8) * mag).all(), (i, t)
            S, A = ww[:, :, None] * S + kv, ww[:, :, None] * A + kv.abs()
        assert ((state[i].double().view(H, D, D) - S).abs() <= 2.0 ** -24 * (2 * n + 2) * A).all()
