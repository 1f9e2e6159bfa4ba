"""The register GEMM (16-bit operands straight into MFMA registers): edges of
its tiles, splits along k, any alignment and stride, against the f64 product.

The tolerance is the bound of f32 sums of exact products in any order:
|C - AB| <= K 2^-24 (|A| |B|), plus half a unit of a 16-bit result."""

import numpy as np
import pytest

from tests.conftest import announce
from vx_amd import abi
from vx_amd.abi import bf16_to_f32, f32_to_bf16
from vx_amd.runtime import DeviceArray, HipTimer, matmul

pytestmark = pytest.mark.gpu

BF, HF, F32 = abi.DTYPE_BF16, abi.DTYPE_F16, abi.DTYPE_F32


def narrow(x, dt):
    return f32_to_bf16(x) if dt == BF else x.astype(np.float16).view(np.uint16)


def widen(x, dt):
    return (bf16_to_f32(x) if dt == BF else x.view(np.float16)).astype(np.float64)


def check(got, a, b, out):
    """`got` f64; a, b the f64 values of the operands."""
    k = a.shape[1]
    bound = k * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 1e-30
    want = a @ b
    if out != F32:
        bound += np.abs(want) * (2.0 ** -8 if out == BF else 2.0 ** -11) * 1.01 + 2.0 ** -24
    worst = np.max(np.abs(got - want) / bound)
    assert worst <= 1.0, f"{worst} times the bound"


def holder(x, pad, lead, fill):
    """x's rows `pad` elements apart more than they are long, from element
    `lead` on, everything else `fill`: the buffer, and the row stride."""
    rows, cols = x.shape
    full = np.full(lead + rows * (cols + pad), fill, np.uint16)
    view = full[lead:].reshape(rows, cols + pad)
    view[:, :cols] = x
    return full, cols + pad


SHAPES = [
    (1, 8, 32800), (1, 64, 4100), (3, 136, 2048), (16, 128, 1024), (17, 129, 1023),  # few rows
    (8, 1000, 4096), (33, 1031, 2081), (64, 127, 8195),  # split along k
    (500, 501, 1301), (1000, 777, 1111), (512, 512, 512),  # every CU a tile or so
    (2049, 4099, 97), (4100, 2055, 160),  # 256-row tiles, the last of 1 or 4 rows
]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dt,out,lead_a,pad_a,lead_b,pad_b", [
    (BF, F32, 0, 0, 0, 0), (BF, BF, 1, 0, 0, 3), (HF, F32, 0, 1, 3, 0), (HF, HF, 2, 2, 1, 1)])
def test_register_gemm(hiplib, rng, m, n, k, dt, out, lead_a, pad_a, lead_b, pad_b):
    """What lies around the operands is NaN and must not reach C; what lies
    around C must stay as it is."""
    announce(f"register gemm {m}x{n}x{k} {dt}->{out} lead {lead_a},{lead_b} pad {pad_a},{pad_b}")
    nan = 0x7fff
    a16 = narrow(rng.normal(0, 1, (m, k)).astype(np.float32), dt)
    b16 = narrow(rng.normal(0, k ** -0.5, (k, n)).astype(np.float32), dt)
    fa, lda = holder(a16, pad_a, lead_a, nan)
    fb, ldb = holder(b16, pad_b, lead_b, nan)
    da, db = DeviceArray.of(hiplib, fa, dt), DeviceArray.of(hiplib, fb, dt)
    ldc = n + pad_a
    dc = DeviceArray.of(hiplib, np.full((m + 2, ldc), 7, np.float32 if out == F32 else np.uint16), out)
    hiplib.force_gemm_kernel(abi.GEMM_MFMA_DIRECT)
    try:
        before = hiplib.stats()["gemm_mfma"]
        runs = []
        for _ in range(2):
            matmul(hiplib, da.descriptor(sizes=(m, k), strides=(lda, 1), offset=lead_a), dt,
                   db.descriptor(sizes=(k, n), strides=(ldb, 1), offset=lead_b), dt,
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


def test_infinities_and_nans_reach_their_row_and_column_only(hiplib, rng):
    announce("register gemm, an infinite and a NaN element")
    m, n, k = 40, 200, 1030
    a = rng.normal(0, 1, (m, k)).astype(np.float32)
    b = rng.normal(0, 1, (k, n)).astype(np.float32)
    a[7, k - 1], b[3, 11] = np.inf, np.nan
    a16, b16 = f32_to_bf16(a), f32_to_bf16(b)
    da, db = DeviceArray.of(hiplib, a16, BF), DeviceArray.of(hiplib, b16, BF)
    dc = DeviceArray(hiplib, (m, n), F32)
    matmul(hiplib, da.descriptor(), BF, db.descriptor(), BF, dc.descriptor(), F32)
    c = dc.numpy().copy()
    for x in (da, db, dc):
        x.free()
    bad = np.zeros((m, n), bool)
    bad[7, :], bad[:, 11] = True, True
    assert np.isnan(c[:, 11]).all() and np.isinf(np.delete(c[7], 11)).all()
    assert np.isfinite(c[~bad]).all()


def test_splits_on_two_streams_and_under_capture(hiplib, rng):
    """Two streams' split launches, each with a workspace of its own that
    goes when the thread's caller stream moves off it; a captured launch
    takes none, and each replay gives the same result."""
    announce("register gemm: splits on streams, capture")
    m, n, k = 8, 512, 8192
    a16 = f32_to_bf16(rng.normal(0, 1, (m, k)).astype(np.float32))
    b16 = f32_to_bf16(rng.normal(0, k ** -0.5, (k, n)).astype(np.float32))
    da, db = DeviceArray.of(hiplib, a16, BF), DeviceArray.of(hiplib, b16, BF)
    dc = [DeviceArray(hiplib, (m, n), F32) for _ in range(3)]

    def call(i):
        matmul(hiplib, da.descriptor(), BF, db.descriptor(), BF, dc[i].descriptor(), F32)

    t = HipTimer()
    streams = [t.stream_create() for _ in range(2)]
    ex = None
    try:
        held = hiplib.gemm_workspaces()["blocks"]
        for i, s in enumerate(streams):
            hiplib.lib.vx_hip_set_stream(s)
            for _ in range(3):
                call(i)
            assert hiplib.gemm_workspaces()["blocks"] == held + 1
        hiplib.lib.vx_hip_set_stream(streams[0])
        ex = t.capture(streams[0], lambda: call(2))
        hiplib.lib.vx_hip_set_stream(None)
        t.sync()
        assert hiplib.gemm_workspaces()["blocks"] == held
        first = dc[0].numpy().copy()
        assert np.array_equal(first, dc[1].numpy())
        check(first.astype(np.float64), widen(a16, BF), widen(b16, BF), F32)
        replays = []
        for _ in range(3):
            t.graph_launch(ex, streams[0])
            t.sync()
            replays.append(dc[2].numpy().copy())
            call(0)
        check(replays[0].astype(np.float64), widen(a16, BF), widen(b16, BF), F32)
        assert all(np.array_equal(r, replays[0]) for r in replays)
    finally:
        hiplib.lib.vx_hip_set_stream(None)
        t.sync()
        if ex is not None:
            t.graph_destroy(ex)
        for s in streams:
            t.stream_destroy(s)
        for x in (da, db, *dc):
            x.free()
