"""GPU parity of float64 products whose last tiles are moved inside the
operands: extents just above a tile, odd ones, a K that ends inside a slab,
slices and shares of K, every layout.  Whole numbers: every sum is exact."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb,tc", [(False, False, False), (True, False, False),
                                      (False, True, False), (True, True, False),
                                      (False, False, True), (True, True, True)])
@pytest.mark.parametrize("m,n,k", [
    # (K under 16 or 4e9 products and more: between them small tiles share out K)
    (128, 2050, 14), (2049, 128, 15), (386, 516, 20402),    # one tile across; slices of K
    (514, 516, 15), (515, 1031, 13), (640, 513, 9),         # odd extents go through copies
    (1028, 1030, 3802), (1500, 1502, 1802),                 # slices, shares
    (2050, 2052, 970), (2048, 2048, 970),                   # 289 tiles; only K is cut short
])
def test_products_of_whole_numbers(hip, m, n, k, ta, tb, tc):
    from numba_mlir_amd.mlir import math_runtime, ops
    rng = np.random.default_rng(m + n + k)
    lay = lambda x, t: hip.asarray(np.ascontiguousarray(x.T)).T if t else hip.asarray(x)
    a = rng.integers(-99, 99, (m, k), endpoint=True).astype(np.float64)
    b = rng.integers(-99, 99, (k, n), endpoint=True).astype(np.float64)
    c0 = rng.integers(-99, 99, (m, n), endpoint=True).astype(np.float64)
    c = lay(c0.copy(), tc)
    ops.gemm(lay(a, ta), lay(b, tb), c, 3.0, -2.0)
    assert "dgemm_mfma_128x128_ragged" in math_runtime.last_kernel()
    assert np.array_equal(c.asnumpy(), 3.0 * (a @ b) - 2.0 * c0)
    c = lay(np.full((m, n), np.nan), tc)
    ops.gemm(lay(a, ta), lay(b, tb), c, 1.0, 0.0)
    assert np.array_equal(c.asnumpy(), a @ b)


@pytest.mark.parametrize("dtype,m,n,k,kernel", [
    # rounds of whole tiles first, then one to two rounds in shares
    (np.float64, 4100, 4100, 242, "dgemm_mfma_128x128_ragged_even"),      # 1089 tiles: 2.1 rounds
    (np.float64, 4096, 4224, 240, "dgemm_mfma_128x128_even"),             # 1056 whole tiles
    (np.float32, 6144, 6144, 160, "sgemm_mfma_256x256_even"),             # 576: 2.25
    (np.float32, 6100, 6000, 3520, "sgemm_mfma_256x256_even+packed"),
    (np.float32, 5888, 8192, 144, "sgemm_mfma_256x256"),                  # 736: 0.96 full, whole
])
@pytest.mark.parametrize("tc", [False, True])
def test_whole_rounds_before_the_shares(hip, dtype, m, n, k, kernel, tc):
    """Every element, alpha and beta once each, the same bits again.  (Whole
    numbers below 2^24: exact in float32 too.)"""
    from numba_mlir_amd.mlir import math_runtime, ops
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-9, 9, (m, k), endpoint=True).astype(dtype)
    b = rng.integers(-9, 9, (k, n), endpoint=True).astype(dtype)
    c0 = rng.integers(-99, 99, (m, n), endpoint=True).astype(dtype)
    want = 3 * (a @ b) - 2 * c0
    for _ in range(2):
        c = hip.asarray(np.asfortranarray(c0)) if tc else hip.asarray(c0)
        ops.gemm(hip.asarray(a), hip.asarray(b), c, 3.0, -2.0)
        if not tc:
            assert math_runtime.last_kernel() == kernel
        assert np.array_equal(c.asnumpy(), want)
