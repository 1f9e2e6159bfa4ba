"""The attention launch whose workgroups' halves divide the keys
(flash_attn.hip, two groups), at the edges of its blocks, against the oracle."""

import numpy as np
import pytest

import oracle
from tests.conftest import announce
from tests.parity import BF16_ABS, assert_max_abs
from tests.test_gpu_flash_attn import randn16, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("case", [
    # batch, heads, kv_heads, seq_q, seq_k, head_dim; 64-key blocks
    (1, 2, 1, 33, 64, 64),     # one block: the second half sees none
    (1, 3, 3, 64, 65, 128),    # a second block of one key
    (2, 4, 2, 65, 129, 64),    # three blocks, a second workgroup of one query
    (1, 2, 2, 200, 256, 128),  # four blocks
    (1, 2, 2, 300, 70, 64),    # more queries than keys: rows that see none
    (1, 2, 2, 300, 70, 128),
    (1, 4, 1, 700, 1000, 64),  # many blocks, a tail of 40 keys
    (1, 16, 4, 260, 260, 128)])
def test_two_groups_match_oracle(hiplib, case, causal, rng):
    announce(f"flash attn two groups {case} causal={causal}")
    b, h, hk, sq, sk, d = case
    q16, k16, v16 = randn16(rng, (b, h, sq, d)), randn16(rng, (b, hk, sk, d)), randn16(rng, (b, hk, sk, d))
    rows = oracle.attention_all_rows(b, h, sq)
    for scale in (d ** -0.5, -(d ** -0.5)):
        o, lse = run(hiplib, q16, k16, v16, h, hk, scale, causal, poison=True)
        wo, wl = oracle.attention_rows(q16, k16, v16, h, hk, scale, causal, rows)
        assert_max_abs(o.reshape(-1, d), wo, BF16_ABS, f"o {case}")
        seen = np.isfinite(wl)
        assert np.array_equal(np.isfinite(lse.ravel()), seen)
        assert_max_abs(lse.ravel()[seen], wl[seen], 1e-3, f"lse {case}")
        assert np.all(o.reshape(-1, d)[~seen] == 0)
