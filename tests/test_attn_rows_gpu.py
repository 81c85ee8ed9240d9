"""Queries and keys of many rows, whose weights and angles are loaded with the row, against few rows at a time."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,D,rot", [(8, 2, 128, 128), (24, 8, 128, 64), (40, 2, 64, 30), (20, 7, 52, 12), (50, 10, 128, 128), (3, 1, 24, 0)])
@pytest.mark.parametrize("norm", ["", "q", "k", "qk", "heads"])
@pytest.mark.parametrize("own", [True, False])
def test_many_rows(H, G, D, rot, norm, own):
    """Sums of up to 6400 squares in another order (2^-24 of it each, a norm takes half of that) and a rotation: 2^-20 of a pair's
    magnitude; values and rows without a slot are the same bits."""
    from nats_llm_studio_amd.ops import stack as K
    K.lib()
    if norm == "heads" and (D & (D - 1) or not rot):
        pytest.skip("plain rows kernel")
    T, g = 70, torch.Generator().manual_seed(D)
    z = torch.randn(T, (H + (2 if own else 1) * G) * D, generator=g).cuda()
    k, v = z[:, H * D:], z[:, (H + G) * D:] if own else z[:, H * D:]
    qn = torch.rand(H * D, generator=g).cuda() if "q" in norm else None
    kn = torch.rand(G * D, generator=g).cuda() if norm in ("k", "qk") else None
    cs = torch.randn(512, max(rot, 1), generator=g).cuda() if rot else None
    pos, slot = torch.randint(0, 512, (T,), generator=g).int().cuda(), torch.randperm(80, generator=g)[:T].int().cuda()
    slot[5] = -1
    Dp, out = K.pad_to(D, 8), []
    for n in (T, 7):
        qo, kc, vc = torch.zeros(T, H * Dp).cuda(), torch.full((80, G * Dp), 7.0).cuda(), torch.full((80, G * Dp), 7.0).cuda()
        for t in range(0, T, n):
            K.attn_rows(z[t:], k[t:], v[t:], qn, kn, cs, pos[t:], slot[t:], qo[t:], kc, vc, n, H, G, D, Dp, rot, 1e-5,
                        torch.cuda.current_stream().cuda_stream, V=D, head_norm=norm == "heads")
        out.append((qo.cpu(), kc.cpu(), vc.cpu()))
    for a, b in zip(out[0][:2], out[1][:2]):
        assert ((a - b).abs() <= 2.0 ** -20 * (b.abs() + b.abs().max())).all()
    assert torch.equal(out[0][2], out[1][2]) and (out[0][1] == 7).all(1).sum() == 11
