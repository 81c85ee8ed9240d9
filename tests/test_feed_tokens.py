"""Tokens of a feed as an array: every form of a whole number that int() takes, each once."""
import numpy as np
import pytest
import torch

from nats_llm_studio_amd.engine.engine import Engine


@pytest.mark.parametrize("toks", [
    [0, 5, 31999], (0, 5, 31999), np.array([0, 5, 31999], np.int32), torch.tensor([0, 5, 31999]), [np.int64(0), True + 4, np.int32(31999)],
    [0.0, 5.9, "31999"], [torch.tensor(0), 5, 31999], bytearray([0, 5]), [-1, 5, 1 << 62]], ids=str)
def test_forms(toks):
    a = Engine._token_array(toks)
    assert a.dtype == np.int64 and a.tolist() == [int(t) for t in toks]


@pytest.mark.parametrize("toks", [[1, 1 << 63], [-(1 << 63) - 1, 0], (1 << 70, 2), [1 << 64, 2.5]], ids=str)
def test_past_64_bits(toks):
    assert Engine._token_array(toks) is None
