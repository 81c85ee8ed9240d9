"""Segments of the chunked recurrences: the count a launch takes, from its rows, runs and longest run."""

import pytest

from nats_llm_studio_amd.ops import stack as K


@pytest.mark.parametrize("kind", ["gla", "delta"])
@pytest.mark.parametrize("D, V", [(64, 64), (65, 65), (128, 128), (96, 300), (129, 128)])
@pytest.mark.parametrize("T, n, longest", [(1, 1, None), (64, 1, 64), (65, 1, 65), (2000, 1, 2000), (3900, 6, 650), (3900, 6, None),
                                           (700, 101, 600), (4000, 64, 64), (7, 7, 1), (16384, 1, 16384)])
@pytest.mark.parametrize("H", [1, 16, 200])
def test_counts(kind, D, V, T, n, longest, H):
    """No more segments than whole chunks of 64 tokens, and scratch for no more of them than twice (delta: once) the CUs, or one
    per run; a launch that fills the chip with whole runs is not cut."""
    f = (lambda *a: K.gla_shape(T, n, H, V, D, *a)) if kind == "gla" else (lambda *a: K.delta_shape(T, n, H, D, V, *a))
    nseg, nt = f(longest)
    wgs = H * -(-V // (64 * nt)) * n
    assert 1 <= nseg <= 16 and nseg <= max(1, -(-(longest or T - n + 1) // 64)) and nt == (1 if V <= 64 else 2)
    assert (nseg - 1) * wgs < (512 if kind == "gla" else 256)
    if 64 < D <= 128 and V > 64:
        tokens = longest or -(-T // n)
        one = H * -(-V // 128) * T / tokens
        us = [K.segments_us(kind, tokens, one, s) for s in range(1, nseg + 1)]
        assert us[-1] == min(us)
