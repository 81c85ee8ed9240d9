"""What the engine tells a model about the runs of a batch: stand-ins with and without recurrent states, that take the longest run or do not."""
import pytest
import torch

import sekolorn_models as S
from test_sekolorn import _FakeRecurrent, _fake_next

from nats_llm_studio_amd.engine.engine import Engine, GenRequest
from nats_llm_studio_amd.engine.sampling import SamplingParams


class _Fake(_FakeRecurrent):
    """Answers with a counter over the tokens of its cached rows, whatever its states; keeps each prefill's keywords."""

    def __init__(self, recurrent, lengths):
        super().__init__()
        self.recurrent, self.calls, self.cached = recurrent, [], {}
        if lengths is not None:
            self.run_lengths = lengths

    def forward(self, b, kc, vc, T, bs, ns=1, logit_rows=None, n_logits=None, qblocks=None, nqb=0, feed_prev=False,
                need_logits=True, **told):
        if feed_prev:
            b.ids[:T] = torch.where(b.use_prev[:T] != 0, b.next_ids[:T], b.ids[:T])
        else:
            self.calls.append((told, b.tok_seq[:T].bincount().max().item(), int(b.tok_seq[T - 1]) + 1))
        slots = [(b.block_tables[b.tok_seq[t], torch.arange(b.ctx_len[t]) // bs] * bs + torch.arange(b.ctx_len[t]) % bs).tolist()
                 for t in range(T)]
        for t in range(T):
            if b.ctx_len[t]:
                assert slots[t][-1] == b.slot[t]
                self.cached[slots[t][-1]] = int(b.ids[t])
        pick = range(T) if logit_rows is None else logit_rows[:n_logits].tolist()
        b.logits[:len(pick)] = 0
        for i, t in enumerate(pick):
            b.logits[i, _fake_next([self.cached[s] for s in slots[t]])] = 1.0
        b.next_ids[:len(pick)] = b.logits[:len(pick)].argmax(1).int()
        return len(pick)


@pytest.mark.parametrize("recurrent", [False, True])
@pytest.mark.parametrize("lengths", [None, False, True])
def test_longest_run(recurrent, lengths):
    """Prompts of several lengths, fed and generated from, up to eight runs in a batch and more: a model with states gets states and runs, the
    longest run only one that takes it, and then the rows it has; a model without gets none of them, and both answer."""
    m = _Fake(recurrent, lengths)
    eng = Engine(m, None, max_batch=12, num_blocks=200, max_prefill_tokens=256, ctx=96, use_graphs=False)
    for n in (1, 3, 12):
        p = [S.tokens(1 + (7 * i + n) % 30, 64, i) for i in range(n)]
        got = eng.feed([(i, t, [len(t) - 1]) for i, t in enumerate(p)] if n > 1 else [(0, p[0], [])])
        if n > 1:
            assert [int(g[0].argmax()) for g in got] == [_fake_next(t) for t in p]
        got = eng.feed([(i, [5, 6][:1 + i % 2], [0]) for i in range(n)])
        assert [int(g[0].argmax()) for g in got] == [_fake_next(t + [5]) for t in p]
        for i in range(n):
            eng.feed_end(i)
        futs = [eng.submit(GenRequest(t, SamplingParams(max_tokens=3, ignore_eos=True))) for t in p]
        for _ in range(30):
            eng.step()
        for t, f in zip(p, futs):
            w = list(t)
            for _ in range(3):
                w.append(_fake_next(w))
            assert f.result(0).token_ids == w[len(t):]
    assert len(m.calls) >= 8
    for told, longest, nruns in m.calls:
        want = {"state": eng.state, "nruns": nruns} if recurrent else {}
        if recurrent and lengths:
            want["longest"] = longest
        assert told == want
