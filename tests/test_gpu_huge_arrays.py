"""Single-array kernels past the largest launch HIP takes (2**32 work-items):
the grid then strides over the array.  Values at its start, on both sides of
the first stride and at its end, and what lies behind it."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import namitorch_amd as nt
from namitorch_amd import _native

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LARGEST = 2 ** 24 - 1                                     # workgroups of 256 lanes
GUARD = 16


@pytest.fixture
def allocate():
    """DeviceArrays of `count` values, given back to the device afterwards;
    skips where the device has no room for them."""
    made = []

    def make(count, dtype):
        try:
            made.append(nt.DeviceArray.empty((count,), dtype, DEV))
        except RuntimeError as error:
            pytest.skip(f"no room on the device: {error}")
        return made[-1]

    yield make
    made.clear()
    nt.runtime.empty_cache(0)


def _probe(array, start, values):
    array.narrow(start, len(values)).upload(values)


@pytest.mark.parametrize("dtype, tile", [("float16", 2048)])
def test_flat_apply(allocate, dtype, tile):
    edge = tile * LARGEST                                 # the first element of the second stride
    count = edge + tile + 5
    gradient = allocate(count + GUARD, dtype)
    gradient.fill_bits(0)
    values = np.arange(1, 9, dtype=np.float16) * 2
    spots = (0, edge - 8, edge, count - 8)
    for start in spots:
        _probe(gradient, start, values)
    _probe(gradient, count, values)
    xform = _native.GradXform(scale=2.0, unscale=1, clip_coef=1.0)
    backend = nt.get_backend(DEV)
    _native.call("nt_grad_apply_flat", 0, gradient.data_ptr(), gradient.dtype.code, count, ctypes.byref(xform),
                 backend.stream())
    for start in spots:
        np.testing.assert_array_equal(gradient.narrow(start, 8).download(), values / 2)
    np.testing.assert_array_equal(gradient.narrow(count, 8).download(), values)


def test_cast(allocate):
    tile = 1024                                           # with float64 on either side
    edge = tile * LARGEST
    count = edge + tile + 5
    source = allocate(count, "float64")
    target = allocate(count + GUARD, "float16")
    source.fill_bits(0)
    target.fill_bits(0x4700)                              # 7.0
    values = np.arange(1, 9, dtype=np.float64) + 0.25
    spots = (0, edge - 8, edge, count - 8)
    for start in spots:
        _probe(source, start, values)
    target.narrow(0, count).copy_from(source)
    for start in spots:
        np.testing.assert_array_equal(target.narrow(start, 8).download(), values.astype(np.float16))
    assert (target.narrow(8, 100).download() == 0).all()
    assert (target.narrow(count, GUARD).download() == 7).all()
