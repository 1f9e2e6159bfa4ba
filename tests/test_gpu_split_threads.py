"""Launches that divide a tile's or a query's work over workgroups, from
several threads at once. They meet in workspaces kept by stream, and every
result must equal, bit for bit, the one that the same call gives alone."""

import threading

import numpy as np
import pytest

from tests.conftest import announce
from tests.test_gpu_flash_attn import fa_workspaces, randn16
from vx_amd import abi
from vx_amd.abi import f32_to_bf16
from vx_amd.runtime import DeviceArray, HipTimer, flash_attention_fwd, matmul

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread: one handle, a stream of each thread

GEMMS = [  # m, n, k, dtype: few rows, a small grid of 128x128 tiles, f32
    (8, 4096, 4096, abi.DTYPE_BF16), (256, 512, 8192, abi.DTYPE_BF16), (128, 2048, 4096, abi.DTYPE_F32)]
ATTENTIONS = [  # batch, heads, kv_heads, seq_q, seq_k, head_dim
    (2, 32, 4, 1, 4096, 128), (1, 32, 4, 512, 2048, 128)]


def operands(rng):
    """Host arrays and what makes the call on device copies of them."""
    jobs = []
    for m, n, k, dt in GEMMS:
        a = rng.normal(0, 1, (m, k)).astype(np.float32)
        b = rng.normal(0, k ** -0.5, (k, n)).astype(np.float32)
        if dt == abi.DTYPE_BF16:
            a, b = f32_to_bf16(a), f32_to_bf16(b)

        def gemm(lib, x, c, dt=dt):
            matmul(lib, x[0].descriptor(), dt, x[1].descriptor(), dt, c.descriptor(), abi.DTYPE_F32)

        jobs.append(((a, b), dt, (m, n), abi.DTYPE_F32, gemm))
    for b, h, hk, sq, sk, d in ATTENTIONS:
        def attn(lib, x, o, s=(b, h, hk, sq, sk, d)):
            assert flash_attention_fwd(lib, x[0].ptr, x[1].ptr, x[2].ptr, o.ptr, None, *s, s[5] ** -0.5,
                                       True) == 0

        jobs.append(((randn16(rng, (b, h, sq, d)), randn16(rng, (b, hk, sk, d)), randn16(rng, (b, hk, sk, d))),
                     abi.DTYPE_BF16, (b, h, sq, d), abi.DTYPE_BF16, attn))
    return jobs


def run_all(lib, jobs, order, want, errors, tag):
    arrays = []
    try:
        dev = []
        for host, dt, shape, out, _ in jobs:
            x = [DeviceArray.of(lib, h, dt) for h in host]
            c = DeviceArray(lib, shape, out)
            arrays += [*x, c]
            dev.append((x, c))
        got = {}
        for i in order:
            x, c = dev[i]
            for _ in range(3):  # the same workspace again, before anything waits
                jobs[i][4](lib, x, c)
            got[i] = c.numpy().copy()
            if want is not None and not np.array_equal(got[i].view(np.uint8), want[i].view(np.uint8)):
                errors.append((tag, i, "differs from the call alone"))
        return got
    finally:
        for x in arrays:
            x.free()


@pytest.mark.parametrize("per_thread", [False, True])
def test_split_launches_from_threads(hiplib, per_thread):
    announce(f"split launches from four threads, hipStreamPerThread {per_thread}")
    jobs = operands(np.random.default_rng(7))
    order = list(range(len(jobs)))

    def spaces():
        return hiplib.gemm_workspaces()["blocks"] + fa_workspaces(hiplib)[0]

    if per_thread:
        hiplib.lib.vx_hip_set_stream(PER_THREAD)
    before = spaces()
    try:
        want = run_all(hiplib, jobs, order, None, [], "alone")
        assert not per_thread or spaces() == before  # kept by no such handle
    finally:
        hiplib.lib.vx_hip_set_stream(None)
    errors = []

    def work(tid):
        t = HipTimer()
        s = PER_THREAD if per_thread else t.stream_create()
        try:
            hiplib.lib.vx_hip_set_stream(s)
            for it in range(2):
                run_all(hiplib, jobs, order[tid % len(order):] + order[:tid % len(order)], want, errors, (tid, it))
        except Exception as e:  # reported below, with the thread that raised it
            errors.append((tid, -1, repr(e)))
        finally:
            hiplib.lib.vx_hip_set_stream(None)
            t.sync()
            if not per_thread:
                t.stream_destroy(s)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join(timeout=90)
    assert not any(th.is_alive() for th in threads), "a launching thread did not finish"
    assert not errors, errors
    if per_thread:
        assert spaces() == before
