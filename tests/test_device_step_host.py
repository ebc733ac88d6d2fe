"""Reading a device-decided step's outcome while its finalize has not run,
with the wait replaced by one that the test ends: no lock is held meanwhile,
and the host mirror returns to its pool once, after the last waiter."""

from __future__ import annotations

import ctypes
import threading
from types import SimpleNamespace

import pytest

from namitorch_amd import _native, amp, runtime
from namitorch_amd.tensor import _settle_lock

TIMEOUT = 20


@pytest.fixture
def waiting(monkeypatch):
    """A step whose norm another thread is waiting for: the step, its mirror,
    the mirrors given back, and a function that ends the wait and returns what
    the thread read."""
    mirror = _native.AmpMirror()
    entered, release, given, read = threading.Event(), threading.Event(), [], []

    def call(name, address, stream):
        assert name == "nt_mirror_wait" and address == ctypes.addressof(mirror)
        entered.set()
        assert release.wait(TIMEOUT)

    monkeypatch.setattr(_native, "call", call)
    monkeypatch.setattr(runtime, "give_mirror", lambda m, launched=True: given.append(ctypes.addressof(m)))
    backend = SimpleNamespace(context=runtime._NoSwitch, stream=lambda: 0)
    step = amp.DeviceStep(backend, None, unscale=False, honor_skip=False, clip_bumps=[], mirror=mirror)
    step.capture()
    reader = threading.Thread(target=lambda: read.append(step.read_norm()))
    reader.start()
    assert entered.wait(TIMEOUT)

    def end():
        release.set()
        reader.join(TIMEOUT)
        return read

    yield SimpleNamespace(step=step, mirror=mirror, given=given, end=end)
    end()


def _finish(mirror, norm):
    ctypes.cast(ctypes.addressof(mirror), ctypes.POINTER(_native.AmpCtrl))[0].norm = norm
    mirror.ready = 1


def test_no_lock_is_held_while_waiting(waiting):
    free = []

    def settle():                                         # another thread's version read
        taken = _settle_lock.acquire(timeout=2)
        free.append(taken)
        if taken:
            _settle_lock.release()

    other = threading.Thread(target=settle)
    other.start()
    other.join(TIMEOUT)
    assert free == [True]
    _finish(waiting.mirror, 3.0)
    assert waiting.end() == [3.0] and len(waiting.given) == 1 and waiting.step.mirror is None


def test_the_mirror_stays_until_the_last_waiter_leaves(waiting):
    _finish(waiting.mirror, 4.0)
    values = []
    other = threading.Thread(target=lambda: values.append(waiting.step.ctrl().norm))
    other.start()
    other.join(2)
    assert values == [4.0] and waiting.given == []       # read, and not yet reused by another step
    assert waiting.end() == [4.0] and len(waiting.given) == 1
