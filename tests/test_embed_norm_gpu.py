"""The embedding and the first norm in one launch, against the two launches."""
import numpy as np
import pytest
import torch

from nats_llm_studio_amd import ops
from nats_llm_studio_amd.gguf import quants as Q
from nats_llm_studio_amd.gguf.constants import GGMLType

pytestmark = pytest.mark.gpu
T_ = GGMLType


@pytest.mark.parametrize("t", [T_.F32, T_.F16, T_.BF16, T_.Q8_0, T_.Q4_K, T_.Q5_K, T_.Q6_K, T_.Q5_1])
@pytest.mark.parametrize("K", [256, 2048, 2304, 8192])
def test_embed_norm(t, K):
    """Rows that fill a part of the workgroup to all of its registers (and a type that takes the two launches); ids outside the table are clamped;
    chained ids are written back; counters are cleared, their neighbours not. The same products in both, but for a contraction: values differ by
    2^-22 of the row's largest term at most, the norms' f16 by an ulp."""
    V, T, n = 40, 19, 13
    raw = Q.random_blocks(t, V * K, 0.05, np.random.default_rng(3))
    w = ops.QWeight(raw, t, V, K, "cuda", layout="rows")
    nw = torch.randn(K, device="cuda")
    for chained in (False, True):
        ids = torch.randint(0, V, (T,), dtype=torch.int32, device="cuda")
        ids[3], ids[4] = -1, V + 5
        nxt, use = torch.randint(0, V, (T,), dtype=torch.int32, device="cuda"), torch.randint(0, 2, (T,), dtype=torch.int32, device="cuda")
        prev = (nxt, use) if chained else None
        got, want = [], []
        for out, one in ((want, False), (got, True)):
            i = ids.clone()
            x, h = torch.full((T + 1, K), 7.0, device="cuda"), torch.full((T + 1, K), 7.0, device="cuda").half()
            z = torch.full((n + 2,), 5, dtype=torch.int32, device="cuda")
            if one:
                ops.embed_norm(i, w, x, T, nw, h, 1e-5, 1.5, prev=prev, zero=z[1:n + 1])
            else:
                ops.embed(i, w, x, T, 1.5, prev=prev)
                ops.rmsnorm(x, nw, h, T, 1e-5)
                z[1:n + 1] = 0
            out += [i, x, h, z]
        assert torch.equal(got[0], want[0]) and torch.equal(got[3], want[3])
        assert (got[1] - want[1]).abs().max() <= 2.0 ** -22 * want[1].abs().max()
        assert ((got[2].float() - want[2].float()).abs() <= 2.0 ** -10 * want[2].float().abs() + 1e-6).all()
