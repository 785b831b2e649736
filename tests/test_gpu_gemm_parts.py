"""GPU parity of the float32 products computed from bf16 parts: accuracy over
the edges of tiles and slabs, exactness, and operands that have no parts."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env(hip):
    from numba_mlir_amd.mlir import ops
    return hip, ops


def _dev(hip, a, transposed):
    return hip.asarray(np.ascontiguousarray(a.T)).T if transposed else hip.asarray(a)


def _product(hip, ops, a, b, ta=False, tb=False):
    c = hip.asarray(np.full((a.shape[0], b.shape[1]), np.nan, np.float32))
    ops.gemm(_dev(hip, a, ta), _dev(hip, b, tb), c, 1.0, 0.0)
    return c.asnumpy()


def _bound(k):
    """|error| / (|a| |b|): three products left out, 2^-24 in all, and for each of
    the six instructions of 16 elements of K two roundings to nearest of the
    accumulator, 2^-24 of it each (what an instruction cuts off besides is under
    2^-24 of a product), six instructions more for a slab that is not whole and
    four roundings of the pieces of a tile.  A bound for every element; it grows
    too fast with K to see a part product missing: the 2-norm below does."""
    return 2.0 ** -24 + 2.0 ** -23 * (6 * (k / 16 + 1) + 4)


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("m,n,k", [
    (512, 512, 16), (512, 512, 32), (512, 512, 48), (512, 640, 64),   # one to four slabs
    (516, 508, 20), (513, 515, 17), (640, 516, 1028),                 # remainders everywhere
    (4096, 3072, 100), (3072, 4096, 16),                              # the 256 x 256 tile
    (2048, 2048, 1040), (3333, 3801, 270),                            # pieces of tiles
])
def test_against_float64(env, m, n, k, ta, tb):
    hip, ops = env
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    got = _product(hip, ops, a, b, ta, tb)
    truth = a.astype(np.float64) @ b.astype(np.float64)
    scale = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - truth) <= _bound(k) * scale).all()


def test_no_less_accurate_than_a_sum_in_float32(env):
    """2-norm of the error against that of float32 multiply-adds in K order,
    on centred and on positive data."""
    hip, ops = env
    rng = np.random.default_rng(3)
    for draw in (rng.standard_normal, rng.random):
        a = draw((512, 2048)).astype(np.float32)
        b = draw((2048, 512)).astype(np.float32)
        truth = a.astype(np.float64) @ b.astype(np.float64)
        plain = np.zeros((512, 512), np.float32)
        for k in range(2048):
            # one rounding a step, as a fused multiply-add has
            plain = (plain + np.multiply.outer(a[:, k].astype(np.float64),
                                               b[k].astype(np.float64))).astype(np.float32)
        got = _product(hip, ops, a, b)
        assert np.linalg.norm(got - truth) <= np.linalg.norm(plain - truth)


@pytest.mark.parametrize("m,n,k", [
    (640, 516, 200), (1024, 1024, 1040), (1500, 1496, 600),   # the 128 x 128 tile: whole, slices, shares
    (4096, 3072, 512), (6144, 3072, 256),                     # the 256 x 256 tile
    (2048, 2048, 1040), (2560, 2304, 2064),                   # its even shares
    (4000, 4000, 530), (2501, 2499, 777),                     # padded copies
])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_two_norm_of_the_error(env, m, n, k, ta, tb):
    """Every part product counts.  A rounding to nearest leaves 2.5e-8 of the
    value (root mean square over its binade); the r-th of 12 k / 16 roundings is
    of a sum of the variance r / (12 k / 16) of the result's, so their errors are
    2.5e-8 sqrt(12 k / 32) of it, and the result's own rounding adds one.  A
    tenth more allowed; h l' or m m' left out would be 2^-18 / 3 = 1.3e-6."""
    hip, ops = env
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    truth = a.astype(np.float64) @ b.astype(np.float64)
    error = np.linalg.norm(_product(hip, ops, a, b, ta, tb) - truth) / np.linalg.norm(truth)
    assert error <= 1.1 * 2.5e-8 * np.sqrt(1 + 12 * k / 32)


@pytest.mark.parametrize("m,k", [(640, 516), (516, 1200), (4096, 3072), (2048, 2048), (2047, 2051)])
@pytest.mark.parametrize("ta", [False, True])
def test_every_bit_of_a_permuted_matrix(env, m, k, ta):
    """A times a permutation with signs: all 24 bits of every value arrive."""
    hip, ops = env
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, k), dtype=np.float32)
    order, signs = rng.permutation(k), rng.choice([-1.0, 1.0], k).astype(np.float32)
    b = np.zeros((k, k), np.float32)
    b[order, np.arange(k)] = signs
    assert np.array_equal(_product(hip, ops, a, b, ta), a[:, order] * signs)


@pytest.mark.parametrize("m,n,k", [(640, 516, 64), (4096, 3072, 64), (2048, 2048, 272)])
def test_products_near_the_smallest_float(env, m, n, k):
    """Products and sums among the subnormal numbers: the bound of others, and
    one rounding to a multiple of 2^-149 of the result or of each piece of it."""
    hip, ops = env
    rng = np.random.default_rng(k)
    a0 = rng.standard_normal((m, k), dtype=np.float32)
    b0 = rng.standard_normal((k, n), dtype=np.float32)
    truth = a0.astype(np.float64) @ b0.astype(np.float64)
    scale = np.abs(a0).astype(np.float64) @ np.abs(b0).astype(np.float64)
    for ea, eb in ((-60, -62), (-66, -64), (-70, -66), (-90, -52)):
        got = _product(hip, ops, np.ldexp(a0, ea), np.ldexp(b0, eb)).astype(np.float64)
        error = np.abs(np.ldexp(got, -ea - eb) - truth)
        assert (error <= _bound(k) * scale + 4 * 2.0 ** (-150 - ea - eb)).all()


def test_whole_numbers_are_exact(env):
    """Products and sums below 2^24 are float32 numbers, and come out as they are."""
    hip, ops = env
    rng = np.random.default_rng(4)
    for high, k in ((511, 60), (4095, 1), (65535, 16)):
        a = rng.integers(-high, high, (600, k), endpoint=True).astype(np.float32)
        b = rng.integers(-2, 2, (k, 520), endpoint=True).astype(np.float32) if high > 511 \
            else rng.integers(-high, high, (k, 520), endpoint=True).astype(np.float32)
        truth = a.astype(np.float64) @ b.astype(np.float64)
        assert np.abs(truth).max() < 2 ** 24
        assert np.array_equal(_product(hip, ops, a, b), truth.astype(np.float32))


@pytest.mark.parametrize("m,n,k", [(640, 516, 1200), (3072, 4096, 1200), (2048, 2048, 1200)])
@pytest.mark.parametrize("ta", [False, True])
def test_operands_without_parts(env, m, n, k, ta):
    """Infinities, NaNs and values that round to infinity in bf16: the float32
    instructions' results.  Values so small that parts of them as they are would
    underflow: float32's accuracy."""
    hip, ops = env
    rng = np.random.default_rng(5)
    a0 = rng.standard_normal((m, k), dtype=np.float32)
    b0 = rng.standard_normal((k, n), dtype=np.float32)
    truth0 = a0.astype(np.float64) @ b0.astype(np.float64)
    scale0 = np.abs(a0).astype(np.float64) @ np.abs(b0).astype(np.float64)
    # (a float32 sum's bound, for pieces that the float32 instructions did)
    tol = k * 2.0 ** -23
    largest = np.finfo(np.float32).max
    for value, at in ((np.inf, (3, 5)), (-np.inf, (m - 1, k - 1)), (np.nan, (7, 1150)),
                      (largest, (m // 2, 17)), (-largest, (0, 0))):
        a = a0.copy()
        a[at] = value
        got = _product(hip, ops, a, b0, ta)
        rest = np.arange(m) != at[0]
        assert (np.abs(got[rest] - truth0[rest]) <= tol * scale0[rest]).all()
        with np.errstate(all="ignore"):
            row = a[at[0]].astype(np.float64) @ b0.astype(np.float64)
            want = row.astype(np.float32)
        if np.isnan(value):
            assert np.isnan(got[at[0]]).all()
        else:
            # (near the largest float32 a sum's order decides what overflows)
            sure = ~(np.abs(np.abs(row) / float(largest) - 1.0) < 1e-3)
            assert np.array_equal(np.isinf(got[at[0]])[sure], np.isinf(want)[sure])
            inf = np.isinf(want) & sure
            assert np.array_equal(got[at[0]][inf], want[inf])
    for exponent in (-101, -110, -120, -126, -140):
        a = np.ldexp(a0, exponent).astype(np.float32)
        b = np.ldexp(b0, 60).astype(np.float32)
        truth = a.astype(np.float64) @ b.astype(np.float64)
        scale = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
        # (products of 2^-80 and above: nothing underflows but the parts)
        assert (np.abs(_product(hip, ops, a, b, ta) - truth) <= tol * scale).all()
    a = a0.copy()
    a[5, 5] = np.float32(1e-42)
    assert (np.abs(_product(hip, ops, a, b0, ta) - a.astype(np.float64) @ b0) <= tol * scale0).all()
