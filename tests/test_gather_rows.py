"""Rows for the head, and the memo of launch configs."""
import pytest
import torch

from nats_llm_studio_amd import ops
from nats_llm_studio_amd.ops import tuning


def check(dev, n, D, cap, ld):
    x = torch.randn(50, ld, device=dev).half()[:, :D]
    rows = torch.randint(0, 50, (n + 3,), dtype=torch.int32, device=dev)
    out = torch.full((cap, D), 7.0, device=dev).half()
    h = ops.gather_rows(x, rows, n, out)
    assert h.shape == ((n + 15) // 16 * 16, D) and torch.equal(h[:n], x[rows[:n].long()]) and (h[n:] == 0).all()
    assert (out[len(h):] == 7).all()
    return h.data_ptr() == out.data_ptr()


def test_rows_on_the_host():
    assert not check("cpu", 5, 24, 16, 24) and not check("cpu", 16, 24, 16, 40)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [8, 2040, 2048, 2056, 8192])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 48])
def test_rows(n, D):
    """One to several blocks of 16, rows narrower and wider than a workgroup takes at once; what the launch does not take goes the general way."""
    assert check("cuda", n, D, 64, D + 16) and check("cuda", n, D, (n + 15) // 16 * 16, D)
    assert not check("cuda", n, D, (n + 15) // 16 * 16 - 1, D) and not check("cuda", n, D - 1 if D > 8 else 4, 64, D + 16)


@pytest.mark.gpu
def test_rows_that_lie_elsewhere():
    """Rows and buffers that do not start at a multiple of 16 bytes, columns that are not neighbours, and no rows at all go the general way."""
    wide, rows = torch.randn(50, 80, device="cuda").half(), torch.arange(49, -1, -1, dtype=torch.int32, device="cuda")
    buf = torch.full((65 * 64,), 7.0, device="cuda").half()
    for h in (wide[:, :64], wide[:, 4:68], wide[:, 1:65], wide[:, 8:72], torch.randn(128, 50, device="cuda").half().t()[:, :64]):
        for at in (0, 4, 8):
            out = buf[at:at + 64 * 64].view(64, 64)
            for n in (0, 5, 16):
                got = ops.gather_rows(h, rows, n, out)
                assert got.shape == ((n + 15) // 16 * 16, 64) and torch.equal(got[:n], h[rows[:n].long()]) and (got[n:] == 0).all()


def test_configs_are_kept_by_what_the_rules_see(monkeypatch):
    """The memo gives what the rules give, for layers alike and unlike, and forgets with the table."""
    from types import SimpleNamespace as NS

    def seg(rows, K, t, d16=None, ycol=0, xmap=None):
        return NS(w=NS(rows=rows, K=K, type=t, d16=d16), ycol=ycol, xmap=xmap, ymap=xmap)
    one = torch.zeros(1)
    for M in (1, 24, 64, 65, 200, 900):
        for s in ([seg(4096, 4096, 12)], [seg(4096, 4096, 14)], [seg(4096, 2048, 12)], [seg(4096, 4096, 12, one)], [seg(4096, 4096, 12, one, 2)],
                  [seg(2048, 2048, 12, one), seg(512, 2048, 12, one, 2048)], [seg(2048, 2048, 12), seg(512, 2048, 14, None, 2048)]):
            want = (tuning.select_dense(s, M) if ops.dense_ok(s, M) else None) or tuning.select(s, M)
            assert ops.gemv_config(s, M) == want == ops.gemv_config(s, M)
    s = [seg(4096, 4096, 12)]
    monkeypatch.setattr(tuning, "_TABLE", {tuning.key(s, 24): (0, 4, 1, 1)})
    assert ops.gemv_config(s, 24) == (0, 4, 1, 1)
