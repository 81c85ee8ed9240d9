"""Experts chosen and listed in one launch and in two, at the edges of the one: 16 tokens, 256 experts, every expert chosen."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,top,groups,keep", [(8, 2, 1, 1), (8, 8, 1, 1), (256, 4, 8, 3), (256, 256, 1, 1), (257, 3, 1, 1)])
@pytest.mark.parametrize("T", [1, 15, 16, 17])
@pytest.mark.parametrize("score", ["sigmoid", "softmax"])
def test_one_launch_and_two(E, top, groups, keep, T, score):
    """The same scores and choices as in a step of many rows, an expert's list holds its rows that have keys, its tiles cover the list."""
    from nats_llm_studio_amd.ops import stack as K
    K.lib()
    g = torch.Generator().manual_seed(E + T)
    z, ctx = torch.randn(40, E, generator=g).cuda(), (torch.rand(40, generator=g) > 0.3).int().cuda()
    st = torch.cuda.current_stream().cuda_stream
    a, b = (K.MoePlan(40, E, top, groups, keep, 0.5, "cuda", score=score) for _ in range(2))
    a.run(z, T, st, ctx)
    b.run(z, 40, st, ctx)
    n = T * top
    assert torch.equal(a.topw[:n], b.topw[:n]) and torch.equal(a.sel[:n], b.sel[:n])
    sel, rows, live = a.sel.cpu(), a.rows.cpu(), ctx.cpu()
    tiles = a.tiles[:int(a.ntiles[0])].cpu().tolist()
    seen = {}
    for e, first, cnt, _ in tiles:
        assert 1 <= cnt <= a.bm(T)
        seen.setdefault(e, []).extend(rows[first:first + cnt].tolist())
    for e in range(E):
        want = [i for i in range(n) if int(sel[i]) == e and int(live[i // top])]
        assert sorted(seen.get(e, [])) == want
