"""GPU parity of reductions along the slow axis read in 128-bit words from any
element: rows that end anywhere, views that begin anywhere, one chunk or many."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [
    (64, 2), (64, 3), (64, 4), (64, 5),          # below, at and above a word
    (65, 7), (127, 17), (96, 129), (200, 257),   # lanes across a row: 2 ... 64
    (2049, 1), (4099, 6), (3001, 515),           # chunks that end anywhere
    (700, 2047), (300, 20003),                   # many strips, short chunks
]


@pytest.mark.parametrize("dtype", [np.int32, np.int64, np.float32, np.float64])
@pytest.mark.parametrize("shape", SHAPES)
def test_columns_of_rows_that_end_anywhere(hip, shape, dtype):
    """Whole numbers: sums are exact in every type, so every element agrees."""
    from numba_mlir_amd.mlir import ops
    rng = np.random.default_rng(shape[0] + shape[1])
    wide = rng.integers(-9, 9, (shape[0], shape[1] + 3), endpoint=True).astype(dtype)
    signs = rng.choice([-1, 1], wide.shape).astype(dtype)
    d, d_signs = hip.asarray(wide), hip.asarray(signs)
    d_t = hip.asarray(np.asfortranarray(wide[:, 1:-2].T))
    views = [(d, wide, d_signs, signs),
             (d[:, 1:-2], wide[:, 1:-2], d_signs[:, 1:-2], signs[:, 1:-2])]
    for x, want, s, want_s in views:
        for _ in range(2):                       # the tickets are zero again
            assert np.array_equal(ops.sum(x, axis=0).asnumpy(), want.sum(axis=0))
        assert np.array_equal(ops.amin(x, axis=0).asnumpy(), want.min(axis=0))
        assert np.array_equal(ops.amax(x, axis=0).asnumpy(), want.max(axis=0))
        assert np.array_equal(ops.prod(s, axis=0).asnumpy(), want_s.prod(axis=0))
    assert np.array_equal(ops.sum(d_t, axis=1).asnumpy(), wide[:, 1:-2].sum(axis=0))


@pytest.mark.parametrize("shape", [(16384, 2047), (5003, 3001), (4096, 40)])
def test_rounding_stays_that_of_short_chains(hip, shape):
    """A lane adds eight rows in pairs, then to its sum; lanes and chunks meet
    behind that: at most `terms` roundings follow one another."""
    from numba_mlir_amd.mlir import ops
    x = np.random.default_rng(2).standard_normal(shape, dtype=np.float32)
    got = ops.sum(hip.asarray(x), axis=0).asnumpy()
    terms = shape[0] / 8 / 4 + 3 + 7 + 8 + 256
    bound = terms * 2.0 ** -24 * np.abs(x).sum(axis=0, dtype=np.float64)
    assert (np.abs(got - x.sum(axis=0, dtype=np.float64)) <= bound).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_nans_lose_and_infinities_pass(hip, dtype):
    from numba_mlir_amd.mlir import ops
    x = np.random.default_rng(3).standard_normal((1000, 67)).astype(dtype)
    x[3, 5] = x[999, 66] = x[:, 9] = np.nan
    x[500, 30], x[501, 31] = np.inf, -np.inf
    d = hip.asarray(x)
    assert np.array_equal(ops.amin(d, axis=0).asnumpy(),
                          np.fmin.reduce(x, axis=0, initial=np.inf))
    assert np.array_equal(ops.amax(d, axis=0).asnumpy(),
                          np.fmax.reduce(x, axis=0, initial=-np.inf))
    with np.errstate(invalid="ignore"):
        sums, want = ops.sum(d, axis=0).asnumpy(), x.sum(axis=0)
    odd = ~np.isfinite(want)
    assert np.array_equal(sums[odd], want[odd], equal_nan=True)
    assert np.isfinite(sums[~odd]).all()


@pytest.mark.parametrize("dtype,cols", [(np.float32, 1048577 + 256), (np.float32, 1048580),
                                        (np.int32, 1048844), (np.float64, 524418)])
def test_more_strips_than_tickets(hip, dtype, cols):
    """Over 4096 strips of columns, in one chunk: words of rows that are whole
    ones, elements of others."""
    from numba_mlir_amd.mlir import ops
    x = np.random.default_rng(cols).integers(-9, 9, (70, cols), endpoint=True).astype(dtype)
    d = hip.asarray(x)
    assert np.array_equal(ops.sum(d, axis=0).asnumpy(), x.sum(axis=0))
    assert np.array_equal(ops.amin(d, axis=0).asnumpy(), x.min(axis=0))
    assert np.array_equal(ops.amax(d[:, 1:], axis=0).asnumpy(), x[:, 1:].max(axis=0))
