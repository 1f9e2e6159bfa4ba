"""The 128x128- and 256x128-tile GEMM (gemm_ring.hip) at the edges of its tiles, ring and
splits, against the f64 product, with the bound of f32 sums in any order."""

import numpy as np
import pytest

from tests.conftest import announce
from tests.test_gpu_gemm_direct import BF, F32, HF, check, holder, narrow, widen
from vx_amd import abi
from vx_amd.runtime import DeviceArray, HipTimer, matmul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 32), (128, 128, 64), (127, 136, 96), (129, 264, 160),  # 1, 2, 3 and 5 stages of the ring
    (257, 120, 192), (640, 1000, 1024),  # 6 stages, 32 and a tile per two CUs
    (300, 264, 8192), (512, 1024, 4096),  # split along k
    (1200, 4104, 288),  # more tiles than CUs
    (300, 11000, 2048), (2049, 2040, 2080)])  # 256x128 tiles, 64 and 65 stages
@pytest.mark.parametrize("dt,out,pad", [(BF, F32, 0), (BF, BF, 8), (HF, F32, 16), (HF, HF, 8)])
def test_ring_gemm(hiplib, rng, m, n, k, dt, out, pad):
    announce(f"ring gemm {m}x{n}x{k} {dt}->{out} pad {pad}")
    a16 = narrow(rng.normal(0, 1, (m, k)).astype(np.float32), dt)
    b16 = narrow(rng.normal(0, k ** -0.5, (k, n)).astype(np.float32), dt)
    fa, lda = holder(a16, pad, 0, 0x7fff)
    fb, ldb = holder(b16, pad, 0, 0x7fff)
    da, db = DeviceArray.of(hiplib, fa, dt), DeviceArray.of(hiplib, fb, dt)
    ldc = n + (3 if out == BF else pad)
    dc = DeviceArray.of(hiplib, np.full((m + 2, ldc), 7, np.float32 if out == F32 else np.uint16), out)
    hiplib.force_gemm_kernel(abi.GEMM_MFMA_RING)
    try:
        before = hiplib.stats()["gemm_mfma"]
        runs = []
        for _ in range(2):
            matmul(hiplib, da.descriptor(sizes=(m, k), strides=(lda, 1)), dt,
                   db.descriptor(sizes=(k, n), strides=(ldb, 1)), dt,
                   dc.descriptor(sizes=(m, n), strides=(ldc, 1), offset=ldc), out)
            runs.append(dc.numpy().copy())
        assert hiplib.stats()["gemm_mfma"] == before + 2
    finally:
        hiplib.force_gemm_kernel(abi.GEMM_AUTO)
        for x in (da, db, dc):
            x.free()
    assert np.array_equal(runs[0], runs[1])
    c = runs[0][1:m + 1, :n]
    rest = runs[0].copy()
    rest[1:m + 1, :n] = 7
    assert np.all(rest == 7)
    check(c.astype(np.float64) if out == F32 else widen(np.ascontiguousarray(c), out),
          widen(a16, dt), widen(b16, dt), out)


def test_split_ring_under_capture(hiplib, rng):
    """A captured launch takes no workspace; eager split launches of other
    operands run between its replays."""
    announce("ring gemm: split, capture")
    m, n, k = 256, 512, 8192
    a16 = narrow(rng.normal(0, 1, (m, k)).astype(np.float32), BF)
    b16 = narrow(rng.normal(0, k ** -0.5, (k, n)).astype(np.float32), BF)
    da, db = DeviceArray.of(hiplib, a16, BF), DeviceArray.of(hiplib, b16, BF)
    dx = DeviceArray.of(hiplib, np.ascontiguousarray(a16[::-1]), BF)
    dc, dy = DeviceArray(hiplib, (m, n), F32), DeviceArray(hiplib, (m, n), F32)
    t = HipTimer()
    s = t.stream_create()
    ex = None
    hiplib.force_gemm_kernel(abi.GEMM_MFMA_RING)

    def call(a, c):
        matmul(hiplib, a.descriptor(), BF, db.descriptor(), BF, c.descriptor(), F32)

    try:
        held = hiplib.gemm_workspaces()["blocks"]
        hiplib.lib.vx_hip_set_stream(s)
        call(da, dy)
        assert hiplib.gemm_workspaces()["blocks"] == held + 1
        t.sync()
        split = dy.numpy().copy()
        ex = t.capture(s, lambda: call(da, dc))
        hiplib.lib.vx_hip_set_stream(None)
        t.sync()
        assert hiplib.gemm_workspaces()["blocks"] == held
        replays = []
        for _ in range(3):
            call(dx, dy)
            t.graph_launch(ex, s)
            t.sync()
            replays.append(dc.numpy().copy())
            assert np.array_equal(dy.numpy()[::-1], split)
        for c in (replays[0], split):
            check(c.astype(np.float64), widen(a16, BF), widen(b16, BF), F32)
        assert all(np.array_equal(r, replays[0]) for r in replays)
    finally:
        hiplib.force_gemm_kernel(abi.GEMM_AUTO)
        hiplib.lib.vx_hip_set_stream(None)
        if ex is not None:
            t.graph_destroy(ex)
        t.stream_destroy(s)
        for x in (da, db, dx, dc, dy):
            x.free()
