"""Attention of few queries a head (flash_rows.hip) against the oracle: the
edges of its blocks of 32 keys and tiles of 16 rows, head groups, splits."""

import numpy as np
import pytest

import oracle
from tests.conftest import announce
from tests.parity import BF16_ABS, assert_max_abs
from tests.test_gpu_flash_attn import fa_workspaces, randn16, run
from vx_amd import abi
from vx_amd.abi import bf16_to_f32, f32_to_bf16
from vx_amd.runtime import DeviceArray, HipTimer, flash_attention_fwd

pytestmark = pytest.mark.gpu

CASES = [
    # batch, heads, kv_heads, seq_q, seq_k, head_dim, splits (0: as chosen)
    (1, 1, 1, 1, 128, 128, 0),    # the shortest cache, one row of a tile
    (2, 16, 1, 1, 129, 64, 0),    # a tile filled by a group's heads, one key past a block
    (1, 17, 1, 1, 160, 128, 0),   # one row past a tile
    (3, 6, 2, 11, 159, 128, 0),   # 33 rows: two readings, the second of one row
    (1, 8, 8, 32, 288, 64, 0),    # the most queries, no group
    (2, 8, 2, 32, 1000, 128, 0),  # 128 rows: four tiles on each reading
    (1, 4, 2, 3, 4097, 128, 16),  # splits, the last with one key more
    (1, 2, 1, 16, 300, 64, 64),   # more splits than blocks of keys (clamped)
    (4, 32, 4, 1, 2049, 128, 0),  # splits as chosen
]


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("case", CASES)
def test_few_queries_match_oracle(hiplib, case, causal, rng):
    announce(f"flash rows {case} causal={causal}")
    b, h, hk, sq, sk, d, splits = case
    q16, k16, v16 = randn16(rng, (b, h, sq, d)), randn16(rng, (b, hk, sk, d)), randn16(rng, (b, hk, sk, d))
    scale = 1.0 / np.sqrt(d)
    rows = oracle.attention_all_rows(b, h, sq)
    for sc in (scale, -scale):
        hiplib.force_fa_splits(splits)
        try:
            o, lse = run(hiplib, q16, k16, v16, h, hk, sc, causal)
            again, _ = run(hiplib, q16, k16, v16, h, hk, sc, causal, with_lse=False)
        finally:
            hiplib.force_fa_splits(0)
        wo, wl = oracle.attention_rows(q16, k16, v16, h, hk, sc, causal, rows)
        assert_max_abs(o.reshape(-1, d), wo, BF16_ABS, f"o {case}")
        assert_max_abs(lse.ravel(), wl, 1e-3, f"lse {case}")
        assert np.array_equal(o, again)


def test_scores_rise_along_the_keys(hiplib, rng):
    """Each block of keys scores higher than the one before, by more than the
    headroom of the stale maximum: every block rescales the sums."""
    announce("flash rows, rising scores")
    b, h, hk, sq, sk, d = 1, 2, 1, 4, 512, 128
    q16, v16 = randn16(rng, (b, h, sq, d)), randn16(rng, (b, hk, sk, d))
    k = np.abs(bf16_to_f32(randn16(rng, (b, hk, sk, d)))) * (1 + np.arange(sk)[None, None, :, None] // 32)
    q16 = f32_to_bf16(np.abs(bf16_to_f32(q16)))
    k16 = f32_to_bf16(k.astype(np.float32))
    scale = 1.0 / np.sqrt(d)
    o, lse = run(hiplib, q16, k16, v16, h, hk, scale, True)
    wo, wl = oracle.attention_rows(q16, k16, v16, h, hk, scale, True, oracle.attention_all_rows(b, h, sq))
    assert_max_abs(o.reshape(-1, d), wo, BF16_ABS, "o")
    # scores of up to 16 x 13 in f32: 2^-24 of them, 128 terms
    assert_max_abs(lse.ravel(), wl, 2e-3, "lse")


def test_what_follows_the_cache_stays_out_and_capture_runs_unsplit(hiplib, rng):
    """The rows after the last key are NaN in memory; a captured launch takes
    no workspace and each replay equals the eager unsplit result; a split
    launch's workspace goes with its stream."""
    announce("flash rows: capture, NaN past the cache")
    b, h, hk, sq, sk, d = 1, 8, 1, 2, 1029, 128
    q16, k16, v16 = randn16(rng, (b, h, sq, d)), randn16(rng, (b, hk, sk, d)), randn16(rng, (b, hk, sk, d))
    nan = np.full((40, d), 0x7fc0, np.uint16)
    dq = DeviceArray.of(hiplib, q16, abi.DTYPE_BF16)
    dk = DeviceArray.of(hiplib, np.concatenate((k16.reshape(sk, d), nan)), abi.DTYPE_BF16)
    dv = DeviceArray.of(hiplib, np.concatenate((v16.reshape(sk, d), nan)), abi.DTYPE_BF16)
    do = DeviceArray(hiplib, (b, h, sq, d), abi.DTYPE_BF16)
    dl = DeviceArray(hiplib, (b, h, sq), abi.DTYPE_F32)

    def call():
        assert flash_attention_fwd(hiplib, dq.ptr, dk.ptr, dv.ptr, do.ptr, dl.ptr, b, h, hk, sq, sk, d,
                                   d ** -0.5, True) == 0

    wo, wl = oracle.attention_rows(q16, k16, v16, h, hk, d ** -0.5, True,
                                   oracle.attention_all_rows(b, h, sq))
    t = HipTimer()
    s = t.stream_create()
    ex = None
    try:
        hiplib.force_fa_splits(1)
        call()
        o1, l1 = do.numpy().copy(), dl.numpy().copy()
        hiplib.force_fa_splits(4)
        base = fa_workspaces(hiplib)[0]
        hiplib.lib.vx_hip_set_stream(s)
        call()
        assert fa_workspaces(hiplib)[0] == base + 1
        t.sync()
        o4 = do.numpy().copy()
        ex = t.capture(s, call)
        hiplib.lib.vx_hip_set_stream(None)
        t.sync()
        assert fa_workspaces(hiplib)[0] == base
        for o in (o1, o4):
            assert_max_abs(bf16_to_f32(o).reshape(-1, d), wo, BF16_ABS, "o")
        assert_max_abs(l1.ravel(), wl, 1e-3, "lse")
        for _ in range(3):
            call()  # eager, split
            hiplib.wait()
            t.graph_launch(ex, s)
            t.sync()
            assert np.array_equal(do.numpy(), o1) and np.array_equal(dl.numpy(), l1)
    finally:
        hiplib.force_fa_splits(0)
        hiplib.lib.vx_hip_set_stream(None)
        if ex is not None:
            t.graph_destroy(ex)
        t.stream_destroy(s)
        for x in (dq, dk, dv, do, dl):
            x.free()
