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


@pytest.mark.parametrize("H, D, V", [(32, 64, 128), (16, 64, 64), (8, 32, 64), (16, 128, 128), (32, 128, 128), (16, 96, 256), (8, 256, 128)])
def test_short_runs_are_not_cut(H, D, V):
    """Segments cost three launches: none up to 128 tokens, however few runs; from 256 on one run of few heads has as many as chunks, or as
    the model of whole rounds says."""
    for n in (64, 65, 100, 128):
        for runs in (1, 2):
            assert K.gla_shape(n * runs, runs, H, V, D, n)[0] == K.delta_shape(n * runs, runs, H, D, V, n)[0] == 1
    assert K.gla_shape(256, 1, H, V, D, 256)[0] == (4 if D <= 64 or D > 128 else K.segments("gla", 256, 256, H * -(-V // 128), 16))
    assert K.gla_shape(256, 1, H, V, D, 256)[0] >= 3


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("kind", ["gla", "delta"])
def test_narrow_workgroups(kind, f32):
    """64 value columns to a workgroup where they are all under way at once, in no more segments than whole chunks and no more scratch; never for other
    widths than the kernels that gain."""
    shape = lambda T, n, H, V, D, l: K.gla_shape(T, n, H, V, D, l) if kind == "gla" else K.delta_shape(T, n, H, D, V, l)
    for H, n, tokens in ((16, 1, 40), (16, 6, 650), (16, 7, 86), (32, 1, 330), (32, 3, 700), (16, 8, 300), (16, 1, 2000), (1, 64, 60), (32, 214, 16)):
        T, old = n * tokens, shape(n * tokens, n, H, 128, 128, tokens)
        nseg, nt = K.narrow_shape(kind, old, T, n, H, 128, 128, tokens, f32)
        if nt == 2:
            assert (nseg, nt) == old
        else:
            assert 1 <= nseg <= max(1, -(-tokens // 64)) and (nseg - 1) * H * n < (512 if kind == "gla" else 256)
            assert 2 * H * n * nseg <= 256 or (f32 and kind == "delta" and nseg == 1)
        assert not (kind == "delta" and 2 * H * n <= 256 and tokens < 1000) or nt == 1
        for V, D in ((64, 128), (128, 64), (128, 129)):
            old = shape(T, n, H, V, D, tokens)
            assert K.narrow_shape(kind, old, T, n, H, V, D, tokens, f32) == old
