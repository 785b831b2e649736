"""GPU parity of the products that waves share out by K (small results, short
rounds of tiles): edges of their tiles and of K, every layout, both types."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env(hip):
    from numba_mlir_amd.mlir import math_runtime, ops

    def gemm(*args):
        ops.gemm(*args)
        kernel = math_runtime.last_kernel()
        assert kernel.split("_")[1] == "fine", kernel
        return kernel
    return hip, gemm


def _dev(hip, a, transposed, off):
    """A device view of `a` in either layout; off: one element into wider rows."""
    flat = np.ascontiguousarray(a.T if transposed else a)
    if off:
        wide = np.full((flat.shape[0], flat.shape[1] + 3), np.nan, a.dtype)
        wide[:, 1:-2] = flat
        view = hip.asarray(wide)[:, 1:-2]
    else:
        view = hip.asarray(flat)
    return view.T if transposed else view


def _norm_room(dtype, k):
    """2-norm of the error over that of a product of normal operands: the i-th of n
    roundings in turn moves a sum of size sqrt(i) by 2^-p / sqrt(3) of it in the mean, all of
    them together by 2^-p sqrt(n / 6) of the whole; no sum in registers has more than 64
    terms (float32) or 160, and those sums' own sum, the slices' and the scale have another
    2^-p.  (Measured 1.0 to 3.6 2^-24 and 1.3 to 4.5 2^-53, of 2.6 to 4.3 and to 6.2.  Operands
    of 16 bits are far beyond; sums left in the registers 5.2 2^-24 at K = 1200.)"""
    return (1 + (min(k, 64 if dtype == np.float32 else 160) / 6) ** 0.5) * np.finfo(dtype).eps / 2


# (no tile, one tile, one row or column more or less than whole tiles of 16, 32 and
# 48; K of one chunk of 16 and one more or less than whole chunks of 4 and 8 waves,
# of a run and of slices)
SHAPES = [(1, 1, 16), (15, 17, 17), (16, 16, 31), (17, 33, 63), (31, 47, 64), (33, 49, 65),
          (47, 33, 129), (49, 97, 255), (97, 49, 257), (310, 1, 506), (1, 127, 1000),
          (200, 300, 641), (129, 143, 1025), (500, 350, 33), (1000, 1100, 80), (64, 48, 5000),
          (159, 1, 6745)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_against_higher_precision(env, dtype, m, n, k):
    """A sum of K products in any order is within K roundings of |a| |b|: K / 2 of
    its last place to nearest; the error's 2-norm within _norm_room."""
    hip, gemm = env
    rng = np.random.default_rng(m + 10 * n + 100 * k)
    a, b = rng.standard_normal((m, k)).astype(dtype), rng.standard_normal((k, n)).astype(dtype)
    c0 = rng.standard_normal((m, n)).astype(dtype)
    high = np.float64 if dtype == np.float32 else np.longdouble
    product = a.astype(high) @ b.astype(high)
    bound = (k + 4) * np.finfo(dtype).eps / 2 * (np.abs(a).astype(high) @ np.abs(b).astype(high))
    norm_room = _norm_room(dtype, k) * np.sqrt((product ** 2).sum())
    for ta in (False, True):
        for tb in (False, True):
            for off in (False, True):
                d_a, d_b = _dev(hip, a, ta, off), _dev(hip, b, tb, off)
                d_c = hip.asarray(np.full((m, n), np.nan, dtype))
                gemm(d_a, d_b, d_c, 1.0, 0.0)
                got = d_c.asnumpy()
                assert (np.abs(got - product) <= bound).all(), (ta, tb, off)
                assert np.sqrt(((got - product) ** 2).sum()) <= norm_room, (ta, tb, off)
                gemm(d_a, d_b, d_c, 1.0, 0.0)
                assert np.array_equal(d_c.asnumpy(), got)
    wide = rng.standard_normal((m, n + 2)).astype(dtype)
    d_w = hip.asarray(wide)
    gemm(d_a, d_b, d_w[:, 1:n + 1], 1.5, -0.5)
    got = d_w.asnumpy()
    assert np.array_equal(got[:, 0], wide[:, 0]) and np.array_equal(got[:, n + 1], wide[:, n + 1])
    want = 1.5 * product - 0.5 * wide[:, 1:n + 1].astype(high)
    room = 1.5 * bound + 4 * np.finfo(dtype).eps * (1.5 * np.abs(product) + np.abs(wide[:, 1:n + 1]))
    assert (np.abs(got[:, 1:n + 1] - want) <= room).all()
    d_t = hip.asarray(np.ascontiguousarray(c0.T)).T      # a column-major C
    gemm(d_a, d_b, d_t, 1.0, 0.0)
    assert (np.abs(d_t.asnumpy() - product) <= bound).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", [(9, 9, 100_003), (16, 16, 2064), (31, 33, 50_021), (63, 63, 9000),
                                   (20, 150, 4113), (1, 63, 70_001), (48, 85, 16_411)])
def test_many_slices_of_a_long_k(env, dtype, m, n, k):
    """Small results of a long K in 16 slices and more, the last one shorter or
    longer by a few: every element within its products' roundings, alpha and beta
    once, nothing beside C, the same bits again."""
    hip, gemm = env
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(dtype), rng.standard_normal((k, n)).astype(dtype)
    high = np.float64 if dtype == np.float32 else np.longdouble
    product = a.astype(high) @ b.astype(high)
    bound = (k + 4) * np.finfo(dtype).eps / 2 * (np.abs(a).astype(high) @ np.abs(b).astype(high))
    norm_room = _norm_room(dtype, k) * np.sqrt((product ** 2).sum())
    wide = rng.standard_normal((m, n + 2)).astype(dtype)
    for ta in (False, True):
        for tb in (False, True):
            d_a, d_b = _dev(hip, a, ta, ta == tb), _dev(hip, b, tb, ta == tb)
            outs = []
            for _ in range(2):
                d_c = hip.asarray(np.full((m, n), np.nan, dtype))
                assert gemm(d_a, d_b, d_c, 1.0, 0.0).endswith("_fine_splitk")
                outs.append(d_c.asnumpy())
            assert np.array_equal(outs[0], outs[1])
            assert (np.abs(outs[0] - product) <= bound).all(), (ta, tb)
            assert np.sqrt(((outs[0] - product) ** 2).sum()) <= norm_room, (ta, tb)
    d_w = hip.asarray(wide)
    gemm(d_a, d_b, d_w[:, 1:n + 1], 1.5, -0.5)
    got = d_w.asnumpy()
    assert np.array_equal(got[:, 0], wide[:, 0]) and np.array_equal(got[:, n + 1], wide[:, n + 1])
    want = 1.5 * product - 0.5 * wide[:, 1:n + 1].astype(high)
    room = 1.5 * bound + 4 * np.finfo(dtype).eps * (1.5 * np.abs(product) + np.abs(wide[:, 1:n + 1]))
    assert (np.abs(got[:, 1:n + 1] - want) <= room).all()


def test_a_long_k_fills_the_gpu(env):
    """32 x 32 from a million of K: 55 to 68 us in slices on all XCDs, 140 on the
    strided kernel in slices, 350 and more in eight slices on one XCD."""
    import time
    hip, gemm = env
    m = n = 32
    k = 1_000_000
    d_a = hip.asarray(np.ones((k, m), np.float32)).T
    d_b, d_c = hip.asarray(np.ones((k, n), np.float32)), hip.asarray(np.zeros((m, n), np.float32))
    times = []
    for _ in range(20):
        start = time.perf_counter()
        gemm(d_a, d_b, d_c, 1.0, 0.0)
        times.append(time.perf_counter() - start)
    assert (d_c.asnumpy() == k).all()
    assert min(times) < 200e-6


@pytest.mark.parametrize("m,n,k", [(40, 50, 70), (100, 130, 300), (300, 200, 150)])
def test_values_without_a_scaled_form(env, m, n, k):
    """Float32 operands among the largest and the smallest numbers, infinities and
    NaN: what plain float32 arithmetic gives, and a sum among the subnormal numbers
    within one rounding of each wave's part of it."""
    hip, gemm = env
    rng = np.random.default_rng(k)
    a0 = rng.standard_normal((m, k), dtype=np.float32)
    b0 = rng.standard_normal((k, n), dtype=np.float32)
    product = a0.astype(np.float64) @ b0.astype(np.float64)
    bound = (k + 4) * 2.0 ** -24 * (np.abs(a0).astype(np.float64) @ np.abs(b0).astype(np.float64))

    def run(a, b):
        d_c = hip.asarray(np.full((m, n), np.nan, np.float32))
        gemm(hip.asarray(a), hip.asarray(b), d_c, 1.0, 0.0)
        return d_c.asnumpy()

    for ea, eb in ((110, 0), (0, 100), (60, 50), (-70, -66), (-140, 20), (20, -145)):
        a, b = np.ldexp(a0, ea), np.ldexp(b0, eb)
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        error = np.abs(run(a, b) - a64 @ b64)
        room = (k + 4) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
        assert (error <= room + 8 * 2.0 ** -150).all(), (ea, eb)
    a, b = a0.copy(), b0.copy()
    a[3, k - 1], b[0, 5], a[7, 2] = np.inf, np.nan, -np.inf
    got = run(a, b)
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    assert (np.abs(got - product)[fine] <= bound[fine]).all()
