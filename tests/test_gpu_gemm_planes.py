"""GPU parity of float32 products whose operands are split into their bf16 parts
ahead of the product: edges of tiles, of K, of runs of slabs and of shares of K,
every layout, views off the word grid, values that the parts cannot hold."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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


# (rows and columns one more or less than whole tiles of 128; K of one more or less
# than slabs of 16 and runs of 4, 8 and 16; a round not full, of operands on the word
# grid too, whole rounds with a few tiles in shares of one slab and more, several
# rounds)
# (and which of them go in shares)
SHAPES = [(1801, 1300, 433, ""), (3071, 1025, 385, ""), (2047, 2049, 1025, "_even"),
          (3329, 3199, 129, ""), (3201, 3327, 191, ""), (2047, 2177, 3499, "_even"),
          (129, 20001, 700, "_even"), (2055, 2181, 517, "_even"), (1796, 1924, 516, ""), (1153, 3584, 769, "_even"),
          (4481, 4353, 257, ""), (2176, 2045, 256, "")]


@pytest.mark.parametrize("m,n,k,shares", SHAPES)
def test_whole_numbers(hip, m, n, k, shares):
    """Sums below 2^24: exact in any order.  alpha and beta once, nothing written
    beside C, the same bits again."""
    from numba_mlir_amd.mlir import math_runtime, ops
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-9, 9, (m, k), endpoint=True).astype(np.float32)
    b = rng.integers(-9, 9, (k, n), endpoint=True).astype(np.float32)
    product = a @ b
    for ta, tb, off in ((False, False, False), (True, False, False), (False, True, True),
                        (True, True, True)):
        d_a, d_b = _dev(hip, a, ta, off), _dev(hip, b, tb, off)
        d_c = hip.asarray(np.full((m, n), np.nan, np.float32))
        ops.gemm(d_a, d_b, d_c, 1.0, 0.0)
        assert math_runtime.last_kernel() == "sgemm_planes" + shares
        assert np.array_equal(d_c.asnumpy(), product), (ta, tb, off)
    wide = rng.integers(-99, 99, (m, n + 2), endpoint=True).astype(np.float32)
    d_w = hip.asarray(wide)
    ops.gemm(d_a, d_b, d_w[:, 1:n + 1], 3.0, -2.0)
    want = wide.copy()
    want[:, 1:n + 1] = 3 * product - 2 * wide[:, 1:n + 1]
    assert np.array_equal(d_w.asnumpy(), want)
    d_t = hip.asarray(np.ascontiguousarray(wide[:, :n].T)).T      # a column-major C
    ops.gemm(d_a, d_b, d_t, 3.0, -2.0)
    assert np.array_equal(d_t.asnumpy(), 3 * product - 2 * wide[:, :n])


# (of padded 256 x 256 tiles; of 128 x 128 tiles that fill their rounds, two a CU,
# and under eight slabs of a share; shares alone, of operands on the word grid, and
# behind one round for a few tiles; three slices of K; a second round mostly empty)
@pytest.mark.parametrize("m,n,k", [(5163, 2770, 1247), (3599, 4065, 303), (2489, 3108, 168),
                                   (2264, 3380, 848), (2968, 1780, 180), (662, 3332, 3475),
                                   (4840, 507, 3456), (1624, 2528, 2436), (5848, 480, 2820),
                                   (1162, 3222, 1031), (612, 4180, 1876), (4828, 788, 384),
                                   (4635, 822, 608)])
def test_products_that_are_faster_split_beside_the_tiles(hip, m, n, k):
    """0.69 to 0.91 times as fast with parts split ahead."""
    from numba_mlir_amd.mlir import math_runtime, ops
    d_a, d_b = hip.asarray(np.zeros((m, k), np.float32)), hip.asarray(np.zeros((k, n), np.float32))
    ops.gemm(d_a, d_b, hip.asarray(np.zeros((m, n), np.float32)), 1.0, 0.0)
    assert math_runtime.last_kernel().startswith("sgemm_mfma_")


@pytest.mark.parametrize("m,n,k,error", [(1801, 1300, 433, 2.0e-7), (2047, 2049, 1025, 2.9e-7),
                                         (2047, 2177, 3499, 2.9e-7), (3329, 3199, 129, 1.45e-7)])
def test_against_float64(hip, m, n, k, error):
    """Every element within its products' roundings, and the 2-norm of the error
    within a quarter more than measured (1.63, 2.30, 2.33 and 1.15 e-7; over millions
    of elements it repeats to a hundredth.  Without runs of slabs 4.75 at K =
    992 and 8.5 at 3085)."""
    from numba_mlir_amd.mlir import ops
    rng = np.random.default_rng(k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    d_c = hip.asarray(np.full((m, n), np.nan, np.float32))
    outs = []
    for _ in range(2):
        ops.gemm(hip.asarray(a), hip.asarray(b), d_c, 1.0, 0.0)
        outs.append(d_c.asnumpy())
    assert np.array_equal(outs[0], outs[1])
    truth = a.astype(np.float64) @ b.astype(np.float64)
    diff = outs[0] - truth
    bound = (k + 8) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert (np.abs(diff) <= bound).all()
    assert np.linalg.norm(diff) <= error * np.linalg.norm(truth)


def test_every_bit_of_a_permuted_matrix(hip):
    from numba_mlir_amd.mlir import ops
    rng = np.random.default_rng(0)
    m, k = 2049, 1281
    a = np.ldexp(rng.standard_normal((m, k)), rng.integers(-60, 60, (m, k))).astype(np.float32)
    order = rng.permutation(k)
    d_c = hip.asarray(np.zeros((m, k), np.float32))
    ops.gemm(hip.asarray(a), hip.asarray(np.eye(k, dtype=np.float32)[:, order]), d_c, 1.0, 0.0)
    assert np.array_equal(d_c.asnumpy(), a[:, order])


@pytest.mark.parametrize("m,n,k", [(1801, 1300, 433), (2047, 2049, 1025)])
@pytest.mark.parametrize("transposed", [False, True])
def test_values_without_parts(hip, m, n, k, transposed):
    """Infinities, NaN, operands and sums too large for the scaled parts, and values
    near the smallest: what float32 arithmetic gives; a sum among the subnormal
    numbers within a rounding of each of its pieces."""
    from numba_mlir_amd.mlir import ops
    rng = np.random.default_rng(k)
    a0 = rng.standard_normal((m, k), dtype=np.float32)
    b0 = rng.standard_normal((k, n), dtype=np.float32)
    magnitude = np.abs(a0).astype(np.float64) @ np.abs(b0).astype(np.float64)
    product = a0.astype(np.float64) @ b0.astype(np.float64)
    bound = (k + 8) * 2.0 ** -24 * magnitude

    def run(a, b):
        d_c = hip.asarray(np.full((m, n), np.nan, np.float32))
        ops.gemm(_dev(hip, a, transposed, False), _dev(hip, b, transposed, False), d_c, 1.0, 0.0)
        return d_c.asnumpy()

    for ea, eb in ((110, 0), (0, 107), (60, 50), (-70, -64)):
        scale = 2.0 ** (ea + eb)
        got = run(np.ldexp(a0, ea), np.ldexp(b0, eb))
        room = bound * scale + 16 * 2.0 ** -150
        assert (np.abs(got - product * scale) <= room).all(), (ea, eb)
    # a few elements, in the first, the last and a middle tile and slab
    a, b = a0.copy(), b0.copy()
    a[3, k - 1], a[m - 1, 0], b[k // 2, 5], b[k - 1, n - 1] = np.inf, -np.inf, np.nan, np.inf
    got = run(a, b)
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    assert (np.abs(got - product)[fine] <= bound[fine]).all()
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))


@pytest.mark.parametrize("m,n,k", [(1801, 1300, 433), (2047, 2049, 1025), (2176, 2045, 256),
                                   (2047, 2177, 3499)])
@pytest.mark.parametrize("ta,tb,off", [(False, False, False), (True, False, True),
                                       (False, True, True), (True, True, False)])
def test_slabs_without_parts(hip, m, n, k, ta, tb, off):
    """Elements that have no parts, in the first and last rows, columns, slabs and pieces
    of K, in either operand or both: their slabs are added from the operands, once and
    to the rows and columns that they belong to.  Whole numbers times powers of two:
    every sum is exact but those of the large elements, which hide the others."""
    from numba_mlir_amd.mlir import math_runtime, ops
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-9, 9, (m, k), endpoint=True).astype(np.float32)
    b = rng.integers(-9, 9, (k, n), endpoint=True).astype(np.float32)
    rows, columns = [0, 31, 32, 127, 128, m - 130, m - 2, m - 1], [1, 63, 64, 1001, n - 3, n - 1]
    deep = [0, 15, 16, k // 2, k - 17, k - 2, k - 1, k - 3]
    large = np.float32(2.0 ** 110)
    a[rows, deep] = large
    b[deep[:6], columns] = -large
    product = a.astype(np.float64) @ b.astype(np.float64)
    d_c = hip.asarray(np.full((m, n), np.nan, np.float32))
    ops.gemm(_dev(hip, a, ta, off), _dev(hip, b, tb, off), d_c, 1.0, 0.0)
    assert math_runtime.last_kernel().startswith("sgemm_planes")
    got = d_c.asnumpy()
    with np.errstate(over="ignore"):
        want = product.astype(np.float32)         # (large times large: infinite)
    touched = np.zeros((m, n), bool)
    touched[rows], touched[:, columns] = True, True
    assert np.array_equal(got[~touched], want[~touched])
    big = np.isfinite(want) & (np.abs(product) > 2.0 ** 100)
    assert np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert (np.abs(got[big] / want[big] - 1) < 2.0 ** -20).all()
    touched[np.ix_(rows, columns)] = False    # (two large terms may cancel and leave nothing)
    small = touched & (np.abs(product) <= 2.0 ** 100)       # (the large element times zero)
    assert small.any() and np.array_equal(got[small], want[small])


@pytest.mark.parametrize("kind", ["one", "column"])
def test_values_without_parts_cost_what_they_touch(hip, kind):
    """One NaN, or an infinity in every row: the call at 2047 x 2049 x 2051 against that of
    ordinary data.  (1.02 and 1.05 times measured; 2.2 and 2.9 with whole tiles
    computed again.)"""
    import time
    from numba_mlir_amd.mlir import ops
    m, n, k = 2047, 2049, 2051
    rng = np.random.default_rng(3)
    a = rng.standard_normal((m, k), dtype=np.float32)
    d_b = hip.asarray(rng.standard_normal((k, n), dtype=np.float32))
    d_c = hip.asarray(np.zeros((m, n), np.float32))

    def least(d_a):
        times = []
        for _ in range(20):
            start = time.perf_counter()
            ops.gemm(d_a, d_b, d_c, 1.0, 0.0)
            times.append(time.perf_counter() - start)
        return min(times)

    ordinary = least(hip.asarray(a))
    if kind == "one":
        a[1000, 1000] = np.nan
    else:
        a[:, k - 1] = np.inf
    assert least(hip.asarray(a)) < 1.5 * ordinary
