"""The attention launch whose workgroups' halves divide the keys
(flash_attn.hip, two groups), at the edges of its blocks, and the undivided
one of one group, against the oracle."""

import numpy as np
import pytest

import oracle
from tests.conftest import announce
from tests.parity import BF16_ABS, assert_max_abs
from tests.test_gpu_flash_attn import CASES, randn16, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("case", [
    # batch, heads, kv_heads, seq_q, seq_k, head_dim; 64-key blocks
    (1, 2, 1, 33, 64, 64),     # one block: one group
    (1, 3, 3, 64, 65, 128),    # two blocks of head size 128: one group
    (1, 2, 1, 33, 65, 64),     # a second block of one key
    (1, 3, 3, 64, 193, 128),   # a fourth block of one key
    (2, 3, 1, 100, 100, 64),   # causal: the first queries' second half sees none
    (1, 2, 2, 300, 200, 128),  # more queries than keys, four blocks
    (1, 200, 50, 129, 320, 64),  # more than half a round: five blocks
    (2, 4, 2, 65, 129, 64),    # three blocks, a second workgroup of one query
    (1, 2, 2, 200, 256, 128),  # four blocks
    (1, 2, 2, 300, 70, 64),    # more queries than keys: rows that see none
    (1, 2, 2, 300, 70, 128),   # one group
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


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("case", CASES + [
    (1, 2, 1, 33, 64, 64), (1, 3, 3, 64, 65, 64), (1, 2, 2, 300, 70, 64), (1, 4, 1, 700, 1000, 64),
    (1, 4, 1, 300, 457, 128), (2, 4, 2, 129, 513, 64)])
def test_one_group_matches_oracle(hiplib, case, causal, rng):
    """The undivided launch of 128-query workgroups, which larger grids take:
    a forced split count of 1."""
    announce(f"flash attn one group {case} causal={causal}")
    b, h, hk, sq, sk, d = case
    q16, k16, v16 = randn16(rng, (b, h, sq, d)), randn16(rng, (b, hk, sk, d)), randn16(rng, (b, hk, sk, d))
    hiplib.force_fa_splits(1)
    try:
        o, lse = run(hiplib, q16, k16, v16, h, hk, d ** -0.5, causal, poison=True)
    finally:
        hiplib.force_fa_splits(0)
    wo, wl = oracle.attention_rows(q16, k16, v16, h, hk, d ** -0.5, causal, oracle.attention_all_rows(b, h, sq))
    assert_max_abs(o.reshape(-1, d), wo, BF16_ABS, f"o {case}")
    seen = np.isfinite(wl)
    assert np.array_equal(np.isfinite(lse.ravel()), seen)
    assert_max_abs(lse.ravel()[seen], wl[seen], 1e-3, f"lse {case}")
    assert np.all(o.reshape(-1, d)[~seen] == 0)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("case", [
    # batch, heads, kv_heads, seq_q, seq_k, head_dim: each side of the choice
    (1, 64, 32, 513, 577, 64), (1, 64, 8, 512, 577, 64),  # past one round of two groups, and one
    (2, 32, 8, 300, 300, 128), (1, 32, 8, 500, 512, 128),
    (64, 32, 32, 20, 130, 128), (16, 32, 4, 9, 130, 128),  # one group, few rows
    (4, 128, 32, 20, 255, 64), (4, 129, 43, 20, 255, 64),
    (1, 256, 256, 17, 384, 128), (1, 255, 255, 17, 384, 128)])
def test_grids_beside_the_choices(hiplib, case, causal, rng):
    announce(f"flash attn grids {case} causal={causal}")
    b, h, hk, sq, sk, d = case
    q16, k16, v16 = randn16(rng, (b, h, sq, d)), randn16(rng, (b, hk, sk, d)), randn16(rng, (b, hk, sk, d))
    o, lse = run(hiplib, q16, k16, v16, h, hk, d ** -0.5, causal, poison=True)
    assert np.isfinite(o).all() and np.isfinite(lse).all()
    rows = np.array(sorted({(bi, hi, qi) for bi in (0, b - 1) for hi in range(0, h, max(1, h // 16))
                            for qi in {0, sq - 1, *rng.integers(0, sq, 6).tolist()}}), np.int64)
    wo, wl = oracle.attention_rows(q16, k16, v16, h, hk, d ** -0.5, causal, rows)
    at = (rows[:, 0], rows[:, 1], rows[:, 2])
    assert_max_abs(o[at], wo, BF16_ABS, f"o {case}")
    assert_max_abs(lse[at], wl, 1e-3, f"lse {case}")
