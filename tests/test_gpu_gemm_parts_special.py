"""GPU parity of the float32 products computed from bf16 parts on operands of
extreme values: the smallest floats stay on the bf16 instructions, and what an
infinity or a NaN costs other elements is nothing, not a bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env(hip):
    from numba_mlir_amd.mlir import ops
    return hip, ops


def _product(hip, ops, a, b, ta=False):
    c = hip.asarray(np.full((a.shape[0], b.shape[1]), np.nan, np.float32))
    da = hip.asarray(np.ascontiguousarray(a.T)).T if ta else hip.asarray(a)
    ops.gemm(da, hip.asarray(b), c, 1.0, 0.0)
    return c.asnumpy()


# the 128 x 128 and the 256 x 256 tile; even shares, whole tiles, copies
SHAPES = [(640, 516, 1200), (2048, 2048, 1200), (4096, 3072, 272), (2047, 2049, 515)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("ta", [False, True])
def test_smallest_values_change_nothing(env, m, n, k, ta):
    """A value too small to count beside the others of its row leaves the
    result's bits as a zero there does: the product takes the same path."""
    hip, ops = env
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    a[::5, 7] = 0
    b[3, ::5] = 0
    want = _product(hip, ops, a, b, ta)
    for tiny in (1e-31, 1e-38, 1e-45):
        a[::5, 7] = tiny
        b[3, ::5] = -tiny
        assert np.array_equal(_product(hip, ops, a, b, ta), want)


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("exponent", [-100, -120, -135])
def test_small_operands_keep_every_bit(env, m, n, k, exponent):
    """One operand scaled down to the smallest floats, the other up: where the
    scaled operand is exact, the products are the unscaled ones' bits."""
    hip, ops = env
    rng = np.random.default_rng(k)
    a = rng.integers(-2 ** 13, 2 ** 13, (m, k)).astype(np.float32)  # (14 bits: exact at 2^-149)
    b = rng.standard_normal((k, n), dtype=np.float32)
    want = _product(hip, ops, a, b)
    got = _product(hip, ops, np.ldexp(a, exponent - 13), np.ldexp(b, 80))
    assert np.array_equal(got, np.ldexp(want, exponent - 13 + 80))


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38])
@pytest.mark.parametrize("where", ["left", "right", "both"])
def test_infinities_cost_others_nothing(env, m, n, k, value, where):
    """Elements 32 rows or columns away from one that meets an infinity keep
    their bits; those that meet it are what IEEE says."""
    hip, ops = env
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    want = _product(hip, ops, a, b)
    rows, cols = [], []
    if where != "right":
        a[m // 2 + 3, k - 1] = value
        rows = [m // 2 + 3]
    if where != "left":
        b[k // 2, n - 1] = value
        cols = [n - 1]
    got = _product(hip, ops, a, b)
    far_rows = np.all([abs(np.arange(m) - r) >= 64 for r in rows] or [np.full(m, True)], axis=0)
    far_cols = np.all([abs(np.arange(n) - c) >= 64 for c in cols] or [np.full(n, True)], axis=0)
    assert np.array_equal(got[np.ix_(far_rows, far_cols)], want[np.ix_(far_rows, far_cols)])
    with np.errstate(all="ignore"):
        for r in rows:
            truth = (a[r].astype(np.float64) @ b).astype(np.float32)
            assert np.array_equal(np.isnan(got[r]), np.isnan(truth))
            odd = np.isinf(truth) & (np.abs(b[k - 1]) > 1.2)     # (surely beyond 3.4e38)
            assert np.array_equal(got[r][odd], truth[odd])
        for c in cols:
            truth = (a.astype(np.float64) @ b[:, c]).astype(np.float32)
            assert np.array_equal(np.isnan(got[:, c]), np.isnan(truth))
            odd = np.isinf(truth) & (np.abs(a[:, k // 2]) > 1.2)
            assert np.array_equal(got[:, c][odd], truth[odd])


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_large_results(env, m, n, k):
    """Operands and results beyond what the scaled parts hold (2^112 and 2^96)
    keep float32's accuracy."""
    hip, ops = env
    rng = np.random.default_rng(k)
    a0 = rng.standard_normal((m, k), dtype=np.float32)
    b0 = rng.standard_normal((k, n), dtype=np.float32)
    truth = a0.astype(np.float64) @ b0.astype(np.float64)
    bound = k * 2.0 ** -23 * (np.abs(a0).astype(np.float64) @ np.abs(b0))
    for ea, eb in ((50, 50), (60, 55), (110, -20), (120, -100), (30, 63)):
        got = _product(hip, ops, np.ldexp(a0, ea), np.ldexp(b0, eb)).astype(np.float64)
        assert (np.abs(np.ldexp(got, -ea - eb) - truth) <= bound).all()


@pytest.mark.parametrize("m,n", [(640, 768), (2048, 2047), (4096, 4096)])
def test_one_and_two_products(env, m, n):
    """K = 1: every product rounded to nearest.  K = 2: one rounding of a product
    and one of the sum."""
    hip, ops = env
    rng = np.random.default_rng(m)
    for draw in (rng.standard_normal, rng.random):
        a = draw((m, 2)).astype(np.float32)
        b = draw((2, n)).astype(np.float32)
        got = _product(hip, ops, np.ascontiguousarray(a[:, :1]), np.ascontiguousarray(b[:1]))
        assert np.array_equal(got, a[:, :1] * b[:1])
        truth = a.astype(np.float64) @ b.astype(np.float64)
        larger = np.maximum(np.abs(a[:, :1] * b[:1]), np.abs(a[:, 1:] * b[1:]))
        bound = 2.0 ** -24 * (larger + np.abs(truth)) * 1.000001
        assert (np.abs(_product(hip, ops, a, b) - truth) <= bound).all()


@pytest.mark.parametrize("m,n,k", [(256, 320, 1 << 17), (128, 128, 1 << 18), (500, 512, 1 << 16),
                                   (1100, 1000, 30000), (2048, 1536, 16384)])
def test_long_sums_do_not_lean(env, m, n, k):
    """The matrix core cuts small terms off downwards.  Over a long K that adds
    up to more than all roundings unless the sign of what it adds changes: a
    mean error of 0.4 (2048 x 1536 x 16384) to 0.85 of the errors' root mean
    square then, and of hundredths where errors are as often above as below."""
    hip, ops = env
    rng = np.random.default_rng(17)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    truth = a.astype(np.float64) @ b.astype(np.float64)
    error = _product(hip, ops, a, b) - truth
    assert abs(error.mean()) <= 0.2 * np.sqrt((error ** 2).mean())


@pytest.mark.parametrize("m,n,k", [(640, 516, 80), (640, 516, 2400), (4096, 3072, 100),
                                   (4096, 3072, 1200)])
def test_zero_sums_have_no_sign(env, m, n, k):
    """Sums that are zero, of zeros or of terms that cancel, are +0 as a sum
    that starts from zero is, whatever sign the accumulators had meanwhile."""
    hip, ops = env
    b = np.random.default_rng(k).standard_normal((k, n), dtype=np.float32)
    a = np.zeros((m, k), np.float32)
    a[1] = -0.0
    a[2::2, 1] = 1.0
    a[2::2, k - 3] = -1.0
    b[k - 3] = b[1]
    got = _product(hip, ops, a, b)
    assert not got.any() and not np.signbit(got).any()
