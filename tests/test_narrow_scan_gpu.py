"""Chunked recurrences over 128 channels with 64 value columns to a workgroup: the shapes that the models' launches choose."""
import pytest
import torch

import bibapel_oracle as O
from nats_llm_studio_amd.ops import stack as K
from test_bibapel_gpu import DT, delta_data, i32, relerr, st

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,G,D,V", [(2, 1, 128, 128), (1, 1, 68, 65), (3, 3, 100, 192)])
@pytest.mark.parametrize("nseg", [1, 3])
def test_delta(dt, H, G, D, V, nseg):
    """Two sequences and an empty run, two or three column blocks, the last one partly filled; then the norm's launch. Three times the same."""
    d, n, eps = DT[dt], 330, 1e-3
    (q, k, v, fac, beta, a), plain = delta_data(d, H, G, D, V, n)
    GD, HD, HV = G * D, H * D, H * V
    cat = lambda t: torch.cat([t[0], t[1]]).cuda()      # noqa: E731
    z = torch.cat([cat(q), cat(k), cat(v)], 1)
    runs = i32([[0, n, 3, 0], [n, n, 1, 0], [0, 0, -1, 0]])
    seg = (torch.full((3 * nseg * HD * V,), 5.0, device="cuda"), torch.full((3 * nseg * HD * D,), 5.0, device="cuda"))
    norm, gate = torch.randn(HV, device="cuda"), torch.randn(2 * n, HV, device="cuda").to(d)
    first = None
    for _ in range(3):
        S, o = torch.full((4, HD * V), 9.0, device="cuda"), torch.full((2 * n, HV), 7.0, device="cuda")
        K.delta_scan(z, z[:, GD:], z[:, 2 * GD:], cat(fac), cat(beta), cat(a), o, norm, gate, None, S, runs, 3, H, G, D, V, eps, (nseg, 1), seg, st())
        y = torch.zeros(2 * n, HV, dtype=d, device="cuda")
        K.scan_out(o, norm, gate, y, H, V, 2 * n, eps, st())
        if first is None:
            first = o.clone(), S.clone()
        assert torch.equal(o, first[0]) and torch.equal(S, first[1])
    for i, slot in ((0, 3), (1, 1)):
        want, Sx = O.delta_scan(*(t[i] for t in plain))
        assert relerr(o[i * n:(i + 1) * n].view(n, H, V), want) < 2e-5 and relerr(S[slot].view(H, D, V), Sx) < 2e-5
    assert (S[0] == 9).all() and (S[2] == 9).all()
    want = O.rms(o.cpu().double().view(2 * n, H, V), eps).view(2 * n, HV) * norm.cpu().double() * gate.cpu().double()
    assert relerr(y, want) < (2e-5 if dt == "f32" else 5e-3)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("D,V", [(132, 40), (200, 128), (256, 192)])
@pytest.mark.parametrize("nseg,nt", [(1, 1), (3, 1), (1, 2), (3, 2)])
def test_wide(dt, D, V, nseg, nt):
    """The kernels whose lanes hand each other most through LDS, in place, and whose registers spill: more than 128 channels, in both forms. Three times the
    same, and what the plain implementation gives."""
    d, n, eps, H = DT[dt], 150, 1e-3, 2
    (q, k, v, fac, beta, a), plain = delta_data(d, H, H, D, V, n)
    GD, HD = H * D, H * D
    cat = lambda t: torch.cat([t[0], t[1]]).cuda()      # noqa: E731
    z = torch.cat([cat(q), cat(k), cat(v)], 1)
    runs = i32([[0, n, 3, 0], [n, n, 1, 0]])
    seg = (torch.full((2 * nseg * HD * V,), 5.0, device="cuda"), torch.full((2 * nseg * HD * D,), 5.0, device="cuda"))
    first = None
    for _ in range(3):
        S, o = torch.full((4, HD * V), 9.0, device="cuda"), torch.full((2 * n, H * V), 7.0, device="cuda")
        K.delta_scan(z, z[:, GD:], z[:, 2 * GD:], cat(fac), cat(beta), cat(a), o, None, None, None, S, runs, 2, H, H, D, V, eps, (nseg, nt), seg, st())
        first = first or (o.clone(), S.clone())
        assert torch.equal(o, first[0]) and torch.equal(S, first[1])
    for i, slot in ((0, 3), (1, 1)):
        want, Sx = O.delta_scan(*(t[i] for t in plain))
        assert relerr(o[i * n:(i + 1) * n].view(n, H, V), want) < 2e-5 and relerr(S[slot].view(H, D, V), Sx) < 2e-5
    assert (S[0] == 9).all() and (S[2] == 9).all()


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("nseg", [1, 3])
def test_plain(dt, nseg):
    """Lightning's form against workgroups of 128 columns: the same sums in another split of the columns, bit for bit."""
    d, H, D, V, n = DT[dt], 2, 128, 128, 330
    z = (torch.randn(2 * n, H * (2 * D + V), device="cuda") * 0.2).to(d)
    a = torch.rand(1, H * D, device="cuda")
    runs = i32([[0, n, 1, 0], [n, n, 0, 0]])
    got = []
    for nt in (2, 1):
        S, o = torch.zeros(2, H * D * V, device="cuda"), torch.zeros(2 * n, H * V, device="cuda")
        seg = (torch.zeros(2 * nseg * H * D * V, device="cuda"), torch.zeros(2 * nseg * H * D, device="cuda"))
        K.gla_scan(z, z[:, H * D:], z[:, 2 * H * D:], a.expand(2 * n, -1).contiguous(), 1.0, o, None, None, None, S, runs, 2, H, D, V, 1e-3, (nseg, nt), seg, st())
        got.append((o, S))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
