"""GPU parity of full reductions, whose result goes straight to host memory:
every type, sizes at the edges of the kernels that serve them, a context that
does not wait, and launches that came before."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("asynchronous", [False, True])
@pytest.mark.parametrize("n", [0, 1, 63, 4095, 4096, 65535, 65536, 1000003])
def test_full_reductions(hip, n, asynchronous):
    from numba_mlir_amd.decorators import njit
    from numba_mlir_amd.mlir import ops
    norm = njit(lambda x: np.sqrt(np.sum(x * x)))
    rng = np.random.default_rng(n)
    ctx = hip.get_context()
    ctx.set_async(asynchronous)
    try:
        for dtype in (np.int32, np.int64, np.float32, np.float64):
            x = rng.integers(-3, 3, n, endpoint=True).astype(dtype)   # exact in every type
            d = hip.asarray(x)
            doubled = ops.add(d, d)          # not waited for in an asynchronous context
            total = ops.sum(doubled)
            assert type(total) is dtype and total == 2 * x.sum(dtype=np.float64)
            if n:
                assert ops.amin(doubled) == 2 * x.min() and ops.amax(doubled) == 2 * x.max()
            if dtype is np.float32:
                got = norm(doubled)
                assert type(got) is np.float32
                assert got == np.sqrt(np.float32(4 * (x.astype(np.float64) ** 2).sum()))
        # int32 sums are held in int64 and come back in the array's own type
        big = hip.asarray(np.full(n, 2 ** 31 - 1, np.int32))
        want = np.int64(n * (2 ** 31 - 1)).astype(np.int32)
        assert ops.sum(big) == want
    finally:
        ctx.set_async(False)
