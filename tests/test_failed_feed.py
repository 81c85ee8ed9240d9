"""A feed step that fails in the middle of its batches."""
import pytest

import sekolorn_models as S
from test_sekolorn import _FakeRecurrent

from nats_llm_studio_amd.engine.engine import Engine


def test_failed_step_moves_tokens_and_places_together(monkeypatch):
    """The second of three row batches raises: each request's tokens are as many as its places, those of the batches that were begun."""
    m = _FakeRecurrent()
    eng = Engine(m, None, max_batch=2, num_blocks=20, max_prefill_tokens=16, ctx=96, use_graphs=False)
    a, b = S.tokens(30, 64, 1), S.tokens(18, 64, 2)
    eng.feed([("a", a[:4], []), ("b", b[:3], [])])
    forward, calls = m.forward, []

    def second_fails(*args, **kw):
        calls.append(1)
        if len(calls) == 2:
            raise RuntimeError("step")
        return forward(*args, **kw)
    monkeypatch.setattr(m, "forward", second_fails)
    with pytest.raises(RuntimeError, match="step"):
        eng.feed([("a", a[4:], []), ("b", b[3:], [])])
    s, t = eng._fed["a"], eng._fed["b"]
    assert (s.n_fed, t.n_fed) == (30, 9) and s.tokens == a and t.tokens == b[:9]
