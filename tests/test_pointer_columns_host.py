"""A plan's record of its pointer columns (``HIPBackend._refresh``) when the
library fails or refuses an update, with the library replaced."""

from __future__ import annotations

import threading
from types import SimpleNamespace

import pytest

from namitorch_amd import _native, runtime
from namitorch_amd.backends.hip import HIPBackend


@pytest.fixture
def device(monkeypatch):
    """A backend and a plan over a fake library: `status` is what the next
    updates return, `updates` the pointers they were given."""
    fake = SimpleNamespace(status=_native.NT_OK, updates=[])

    def set_pointers(handle, column, array, count, stream):
        fake.updates.append((column, tuple(array)))
        return fake.status

    library = SimpleNamespace(nt_plan_set_pointers=set_pointers, nt_last_error=lambda: b"a launch failed")
    monkeypatch.setattr(_native, "load", lambda: library)
    backend = HIPBackend.__new__(HIPBackend)
    backend._lock = threading.RLock()
    backend.context = runtime._NoSwitch
    fake.plan = SimpleNamespace(handle=1, columns={1: (16, 32)})
    fake.refresh = lambda values: backend._refresh(fake.plan, {1: values}, 0)
    return fake


def test_a_failed_update_leaves_no_known_pointers(device):
    """Part of the column may hold the new pointers: the old ones are written
    again before the plan is used with them."""
    device.status = _native.NT_ERR_HIP
    with pytest.raises(RuntimeError, match="a launch failed"):
        device.refresh([48, 64])
    device.status = _native.NT_OK
    assert device.refresh([16, 32])
    assert device.updates == [(1, (48, 64)), (1, (16, 32))]
    assert device.refresh([16, 32]) and len(device.updates) == 2


def test_a_refused_update_changes_nothing(device):
    device.status = _native.NT_ERR_VALUE
    assert not device.refresh([48, 65])
    device.status = _native.NT_OK
    assert device.refresh([16, 32]) and device.updates == [(1, (48, 65))]
