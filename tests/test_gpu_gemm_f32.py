"""The f32 GEMM on bf16 planes, and on f32 MFMAs where K is short
(gemm_f32.hip): what its planes cannot hold, and the edges of its stages,
against the f64 product. The tolerance is the bound of f32 sums of products in
any order plus what the planes' products left out come to, 2^-24 of each:
|C - AB| <= (K + 2) 2^-24 (|A| |B|)."""

import numpy as np
import pytest

from tests.conftest import announce
from vx_amd import abi
from vx_amd.runtime import DeviceArray, matmul

pytestmark = pytest.mark.gpu


def product(lib, a, b, pad=0):
    """a @ b on the GPU; with `pad`, from and into rows that much longer,
    whose padding is NaN and must stay."""
    (m, k), n = a.shape, b.shape[1]

    def padded(x):
        full = np.full((x.shape[0], x.shape[1] + pad), np.nan, np.float32)
        full[:, :x.shape[1]] = x
        return full

    da, db = DeviceArray.of(lib, padded(a), abi.DTYPE_F32), DeviceArray.of(lib, padded(b), abi.DTYPE_F32)
    dc = DeviceArray.of(lib, np.full((m, n + pad), np.nan, np.float32), abi.DTYPE_F32)
    lib.force_gemm_kernel(abi.GEMM_F32_MFMA)
    try:
        before = lib.stats()["gemm_mfma"]
        matmul(lib, da.descriptor(sizes=(m, k), strides=(k + pad, 1)), abi.DTYPE_F32,
               db.descriptor(sizes=(k, n), strides=(n + pad, 1)), abi.DTYPE_F32,
               dc.descriptor(sizes=(m, n), strides=(n + pad, 1)), abi.DTYPE_F32)
        full = dc.numpy().copy()
        assert lib.stats()["gemm_mfma"] == before + 1
    finally:
        lib.force_gemm_kernel(abi.GEMM_AUTO)
        for x in (da, db, dc):
            x.free()
    assert np.isnan(full[:, n:]).all()
    return full[:, :n]


def check(c, a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    bound = (a.shape[1] + 2) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 2.0 ** -149
    assert np.max(np.abs(c - a @ b) / bound) <= 1.0


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (128, 128, 31), (129, 127, 32), (127, 130, 33), (5, 300, 64),
                                   (300, 5, 95), (256, 384, 96), (130, 131, 129), (200, 200, 1000),
                                   (130, 131, 2047), (20, 1000, 4100), (1, 1, 127), (130, 131, 128),
                                   (129, 127, 160), (127, 130, 161), (60, 300, 257), (300, 60, 288), (33, 70, 320)])
@pytest.mark.parametrize("pad", [0, 1])
def test_edges_of_stages_and_tiles(hiplib, rng, m, n, k, pad):
    announce(f"f32 gemm {m}x{n}x{k} pad {pad}")
    a = rng.uniform(-1, 1, (m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (k, n)).astype(np.float32)
    c = product(hiplib, a, b, pad)
    check(c, a, b)
    assert np.array_equal(c, product(hiplib, a, b, pad))


@pytest.mark.parametrize("k", [90, 260])  # on f32 MFMAs, and in planes
@pytest.mark.parametrize("lo,hi,other", [(-60, 60, 0), (-126, -100, 100), (90, 126, -100)])
def test_magnitudes(hiplib, rng, lo, hi, other, k):
    """Elements of every magnitude f32 has, times ones that keep the products
    inside its range."""
    announce(f"f32 gemm, magnitudes 2^{lo} .. 2^{hi}")
    m, n = 150, 140

    def draw(shape, exponents):
        return (rng.uniform(1, 2, shape) * rng.choice([-1, 1], shape) * 2.0 ** exponents).astype(np.float32)

    a = draw((m, k), rng.integers(lo, hi, (m, k)).astype(np.float64))
    b = draw((k, n), float(other))
    check(product(hiplib, a, b), a, b)
    at, bt = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    check(product(hiplib, bt, at), bt, at)


@pytest.mark.parametrize("k", [100, 330])
def test_rows_and_columns_too_small_for_the_planes(hiplib, rng, k):
    """A row of A and a column of B of subnormal and other tiny values, next
    to zeros, in tiles of ordinary ones."""
    announce("f32 gemm, tiny rows")
    m, n = 260, 300
    a = rng.uniform(-1, 1, (m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (k, n)).astype(np.float32)
    a[140] = (rng.uniform(-1, 1, k) * 2.0 ** -120).astype(np.float32)
    a[141] = 0
    b[:, 10] = (rng.uniform(-1, 1, k) * 2.0 ** -118).astype(np.float32)
    c = product(hiplib, a, b)
    check(c, a, b)
    assert not c[141].any()


def test_tiny_and_infinite_rows_over_splits(hiplib, rng):
    """K divided over workgroups: a row that is tiny in some of its splits
    only, one that is tiny in all, one with an infinity in one split."""
    announce("f32 gemm, splits, tiny and infinite rows")
    m, n, k = 200, 140, 3000
    a = rng.uniform(-1, 1, (m, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (k, n)).astype(np.float32)
    a[20, :2000] *= np.float32(2.0 ** -118)
    a[30] *= np.float32(2.0 ** -118)
    check(product(hiplib, a, b), a, b)
    a[199, 2500] = np.inf
    c = product(hiplib, a, b)
    check(c[:199], a[:199], b)
    assert np.array_equal(c[199], np.where(b[2500] > 0, np.inf, -np.inf))


@pytest.mark.parametrize("k", [70, 200])
def test_infinities_and_nans(hiplib, rng, k):
    """As f32 arithmetic has them: an infinity times a finite value is an
    infinity of the product's sign, times zero NaN; nothing else is touched."""
    announce("f32 gemm, infinities and NaNs")
    m, n = 260, 260
    a = rng.uniform(0.5, 1, (m, k)).astype(np.float32)
    b = rng.uniform(0.5, 1, (k, n)).astype(np.float32)
    a[3, 69], a[200, 0], b[5, 150], b[69, 7] = np.inf, np.nan, -np.inf, 0.0
    c = product(hiplib, a, b)
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(c), np.isnan(want))
    assert np.array_equal(np.isposinf(c), np.isposinf(want)) and np.array_equal(np.isneginf(c), np.isneginf(want))
    ok = np.isfinite(want)
    assert np.max(np.abs(c - want)[ok] / np.abs(want)[ok]) < (k + 2) * 2.0 ** -24
    assert np.isnan(c[3, 7]) and np.isnan(c[3, 150]) and np.isposinf(c[3, 0])


@pytest.mark.parametrize("k", [140, 3000])  # in one workgroup a tile, and divided
@pytest.mark.parametrize("exponent", [-101, -112, -124, -134, -140])
def test_tiny_elements_of_ordinary_rows(hiplib, rng, k, exponent):
    """Rows that hold ordinary values opposite zeros and tiny ones opposite
    large ones: each sum is of the tiny ones' products alone."""
    announce(f"f32 gemm, elements of 2^{exponent} in ordinary rows, k {k}")
    m, n = 150, 140
    a = rng.uniform(1, 2, (m, k)) * rng.choice([-1, 1], (m, k))
    b = rng.uniform(1, 2, (k, n)) * rng.choice([-1, 1], (k, n))
    a, b = a.astype(np.float32), b.astype(np.float32)
    tiny = rng.choice(k, 5, replace=False)
    a[17, tiny] *= np.float32(2.0 ** exponent)
    b[:, 99] = 0
    b[tiny, 99] = (rng.uniform(1, 2, 5) * 2.0 ** 120).astype(np.float32)
    check(product(hiplib, a, b), a, b)
    at, bt = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    check(product(hiplib, bt, at), bt, at)


@pytest.mark.parametrize("k", [1, 31, 128, 140, 2100])
def test_single_products(hiplib, rng, k):
    """One value in each row of A: every sum is one product, whose error is
    its rounding (2^-24) and the products of planes left out (2^-24, of values
    whose planes are worst the most)."""
    announce(f"f32 gemm, single products, k {k}")
    m, n = 140, 150
    a = np.zeros((m, k), np.float32)
    values = np.float32(1 + 2.0 ** -7 - 2.0 ** -23) * rng.choice([1, -1], m)
    values[m // 2:] = rng.uniform(1, 2, m - m // 2)
    a[np.arange(m), rng.integers(0, k, m)] = values
    b = np.full((k, n), 1 + 2.0 ** -7 - 2.0 ** -23, np.float32)
    b[:, n // 2:] = rng.uniform(1, 2, (k, n - n // 2))
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.max(np.abs(product(hiplib, a, b) - want) / np.abs(want)) <= 2.1 * 2.0 ** -24
