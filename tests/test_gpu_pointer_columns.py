"""Re-pointing a plan's gradient column (``nt_plan_set_pointers``) at the list
lengths where its launches change: 64 and 448 pointers per kernel."""

from __future__ import annotations

import numpy as np
import pytest

import namitorch_amd as nt
from namitorch_amd import _native

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("count", [1, 63, 64, 65, 447, 448, 449, 896, 897])
def test_update_reaches_every_descriptor(count):
    """The plan zeroes the buffers it was pointed at last, and each queued
    zeroing the ones it was queued with."""
    def buffers():
        flat = nt.DeviceArray.empty((count * 8,), "float32", DEV).upload(np.ones(count * 8, np.float32))
        return flat, [nt.Tensor._from_storage(flat.narrow(8 * k, 8)) for k in range(count)]

    backend = nt.get_backend(DEV)
    flats, sets = zip(*(buffers() for _ in range(3)))
    layout = (_native.NT_DTYPE_NONE, _native.NT_F32, _native.NT_DTYPE_NONE, _native.NT_DTYPE_NONE)
    rows = [(0, 0, 0, 0, 0, 8, 0)] * count
    plan = backend.plan(rows, layout, pointers={1: [t._ptr for t in sets[0]]})
    for k in (1, 2):
        assert backend.plan(rows, layout, pointers={1: [t._ptr for t in sets[k]]}) is plan
        _native.call("nt_grad_zero", plan.handle, backend.stream())
    left = [flat.download() for flat in flats]
    assert (left[0] == 1).all() and (left[1] == 0).all() and (left[2] == 0).all()
