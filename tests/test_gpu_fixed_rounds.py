"""The fixed-point value kernel at the edges of its rounds of 256 positions: the rounds in flight
before the softmax (1024 positions), the ones after, the largest context.  Equal integers."""

import numpy as np
import pytest

from llm_accelerator_amd import fixed as X
from oracle import q4_fixed as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [256, 257, 768, 769, 1024, 1025, 1281, 4096])
def test_value_rounds_match_oracle(dev, t):
    rng = np.random.default_rng(t)
    q = rng.integers(-(1 << 11), 1 << 11, (16, 128))
    k = rng.integers(-(1 << 23), 1 << 23, (t, 8, 128))
    v = rng.integers(-(1 << 23), 1 << 23, (t, 8, 128))
    k[:, ::2] //= 4096  # every other kv head: moderate scores, a spread of LUT indices
    print(f"[fixed] value rounds T={t}", flush=True)
    r = X.attention_score_value(q, k, v, 189812531)
    ref = F.attention_score_value(q, k, v, 189812531, F.build_exp_lut())
    for key in ("lut_indices", "probs", "output"):
        np.testing.assert_array_equal(r[key].cpu().numpy().astype(np.int64), ref[key], err_msg=key)
