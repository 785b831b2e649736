"""Host-only checks of the device array front: what it refuses before anything
reaches a device."""

from types import SimpleNamespace

import numpy as np
import pytest

from numba_mlir_amd.mlir import device_array, ops


class _FakeBuffer:
    usm_type = "device"

    def __init__(self, ctx, nbytes, usm_type):
        self.ctx, self.nbytes, self.ptr = ctx, nbytes, 0x1000


@pytest.fixture
def no_device(monkeypatch):
    monkeypatch.setattr(device_array, "_Buffer", _FakeBuffer)
    monkeypatch.setattr(device_array, "get_context",
                        lambda device=None: SimpleNamespace(device=device, handle=None))


@pytest.mark.parametrize("shape", [2 ** 70, (2 ** 64,), (3, 2 ** 63), (2 ** 70, 0), (2 ** 62, 8)])
def test_shapes_beyond_64_bits_are_refused(no_device, shape):
    """(An allocation of the size's low 64 bits would hold none of the elements.)"""
    with pytest.raises(OverflowError):
        device_array.empty(shape, np.float32)


@pytest.mark.parametrize("shape,count", [(5, 5), ((), 1), ((3, 0), 0), ((2, 3, 4), 24),
                                         (np.array([2, 3]), 6), ([np.int32(7), True], 7)])
def test_shapes_that_fit(no_device, shape, count):
    x = device_array.empty(shape, np.float64)
    assert x._buffer.nbytes == 8 * count and x.size == count


@pytest.mark.parametrize("a,b,error", [
    (">f4", ">f4", NotImplementedError),          # (promoted to the native type)
    (">f4", "<f4", NotImplementedError),
    (np.float32, np.float64, NotImplementedError),
    (np.float32, "M8[s]", TypeError),             # no common type
    (np.complex64, np.complex64, TypeError),      # no kernel
])
def test_maps_of_other_types_are_refused_as_before(no_device, a, b, error):
    x, y = device_array.empty(4, a), device_array.empty(4, b)
    with pytest.raises(error):
        ops.add(x, y)
