"""Every routed 16-bit MFMA GEMM records its clock counters when asked to."""

import numpy as np
import pytest

from tests.conftest import announce
from vx_amd import abi
from vx_amd.abi import f32_to_bf16
from vx_amd.runtime import DeviceArray, matmul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,m,n,k", [
    (abi.GEMM_MFMA_PP, 512, 512, 512),
    (abi.GEMM_MFMA_RING, 256, 264, 256), (abi.GEMM_MFMA_RING, 256, 512, 8192),  # whole, K divided
    (abi.GEMM_MFMA_RING, 300, 11000, 2048),  # 256x128 tiles
    (abi.GEMM_MFMA_DIRECT, 8, 264, 256), (abi.GEMM_MFMA_DIRECT, 8, 4096, 4096),  # whole, K divided
    (abi.GEMM_MFMA_DIRECT, 1500, 2048, 288)])  # waves along the rows
def test_stamps_are_written(hiplib, rng, kernel, m, n, k):
    announce(f"clock stamps of kernel {kernel}, {m}x{n}x{k}")
    a = f32_to_bf16(rng.normal(0, 1, (m, k)).astype(np.float32))
    b = f32_to_bf16(rng.normal(0, 1, (k, n)).astype(np.float32))
    da, db = DeviceArray.of(hiplib, a, abi.DTYPE_BF16), DeviceArray.of(hiplib, b, abi.DTYPE_BF16)
    dc = DeviceArray(hiplib, (m, n), abi.DTYPE_F32)
    got = np.zeros((3, 4), np.uint64)
    ring = hiplib.transfer(got)
    hiplib.force_gemm_kernel(kernel)
    hiplib.clock_stamps(ring, 3)
    try:
        for _ in range(2):
            matmul(hiplib, da.descriptor(), abi.DTYPE_BF16, db.descriptor(), abi.DTYPE_BF16, dc.descriptor(),
                   abi.DTYPE_F32)
        hiplib.wait()
        hiplib.fetch(ring, got)
    finally:
        hiplib.clock_stamps(None, 0)
        hiplib.force_gemm_kernel(abi.GEMM_AUTO)
        hiplib.free(ring)
        for x in (da, db, dc):
            x.free()
    assert np.all(got[:2, 2] > got[:2, 0]) and np.all(got[:2, 3] >= got[:2, 1]) and np.all(got[:2, 1] > 0)
    assert not got[2].any()
