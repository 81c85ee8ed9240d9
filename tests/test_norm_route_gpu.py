"""Norm, router and route of 2 to 4 tokens at once, at the edges of its columns and behind them."""
import pytest
import torch

from nats_llm_studio_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [2, 3, 4])
@pytest.mark.parametrize("E", [2, 4, 8])
@pytest.mark.parametrize("D", [256, 1020, 1028, 4092, 4096, 4100])
def test_tokens_at_once(T, E, D):
    """Rows: f16 of the norm, half an ulp and the sum's error off (2^-10); logits of those rows in 32 bits (D 2^-24 of the summed magnitudes);
    the same experts and lists as the route of those logits."""
    k, cap = 2, 8
    g = torch.Generator().manual_seed(T + D)
    x, nw = (torch.randn(cap, D, generator=g) * 3).cuda(), (torch.rand(D, generator=g) + 0.5).cuda()
    wr = (torch.randn(E, D, generator=g) * 0.05).half().cuda()
    h = torch.full((cap, D + 4), 7.0, dtype=ops.ACT_DTYPE, device="cuda")
    lg, lists = torch.zeros(cap, E, device="cuda"), []
    for fused in (True, False):
        tw = torch.zeros(cap * k, device="cuda")
        c, xr, yr, sel = (torch.full((n,), 5, dtype=torch.int32, device="cuda") for n in (E, E * cap, E * cap, cap * k))
        if fused:
            assert ops.moe_norm_route(x, nw, 1e-5, wr, h, lg, T, k, tw, c, xr, yr, cap, sel=sel)
        else:
            ops.moe_route(lg, T, k, tw, c, xr, yr, cap, sel=sel)
        rows = [sorted(xr[e * cap:e * cap + int(c[e])].tolist()) for e in range(E)]
        lists.append((tw.cpu(), c.cpu(), sel.cpu(), rows))
    assert all(torch.equal(a, b) for a, b in zip(lists[0][:3], lists[1][:3])) and lists[0][3] == lists[1][3]
    xs, hh = x[:T].double().cpu(), h[:T, :D].double().cpu()
    want = xs * torch.rsqrt(xs.pow(2).mean(1, keepdim=True) + 1e-5) * nw.double().cpu()
    assert ((hh - want).abs() <= 2.0 ** -10 * want.abs() + 1e-7).all() and (h[T:] == 7).all() and (h[:, D:] == 7).all()
    w = wr.double().cpu()
    assert ((lg[:T].double().cpu() - hh @ w.T).abs() <= D * 2.0 ** -24 * (hh.abs() @ w.abs().T)).all()
