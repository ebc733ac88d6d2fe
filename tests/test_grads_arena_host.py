"""The shared allocations of first gradients (``grads._fresh_gradients``), with
the device allocator replaced by a counter: how much memory one gradient can
keep from reuse, and where the gradients lie."""

from __future__ import annotations

import random
from types import SimpleNamespace

import pytest

from namitorch_amd import grads
from namitorch_amd.array import DeviceArray
from namitorch_amd.device import Device
from namitorch_amd.dtype import normalize_dtype
from namitorch_amd.runtime import _NoSwitch
from namitorch_amd.tensor import Tensor

DEVICE = Device("cuda", 0)
BACKEND = SimpleNamespace(device=DEVICE, context=_NoSwitch)


def _leaf(count, dtype):
    return SimpleNamespace(_dtype=normalize_dtype(dtype), _shape=(count,), _numel=count)


@pytest.fixture
def fresh(monkeypatch):
    """fresh(leaves) -> (the gradients, the allocations behind them)."""
    class Array(DeviceArray):
        __slots__ = ()

        @classmethod
        def empty(cls, shape, dtype, device):
            (count,) = shape
            start = sum(-(-block.nbytes // 4096) * 4096 + 4096 for block in blocks)
            blocks.append(SimpleNamespace(ptr=4096 + start, nbytes=count * dtype.itemsize))
            return DeviceArray._make(blocks[-1], blocks[-1].ptr, shape, dtype, device)

    blocks: list = []
    monkeypatch.setattr(grads, "DeviceArray", Array)
    return lambda leaves: (grads._fresh_gradients(leaves, BACKEND), blocks)


def _check(leaves, gradients, blocks, limit):
    for leaf, gradient in zip(leaves, gradients):
        block = gradient._storage._base
        size = leaf._numel * leaf._dtype.itemsize
        assert gradient._dtype is leaf._dtype and gradient._shape == leaf._shape and gradient._ptr % 16 == 0
        assert block.ptr <= gradient._ptr and gradient._ptr + size <= block.ptr + block.nbytes
        assert block.nbytes <= limit or block.nbytes == size            # at most the limit, or itself
    spans = sorted((g._ptr, g._ptr + g.nbytes) for g in gradients if g.size)
    assert all(end <= start for (_, end), (start, _) in zip(spans, spans[1:]))


def test_a_small_gradient_does_not_keep_a_large_one(fresh):
    """A run of small leaves followed by one larger than the limit."""
    leaves = [_leaf(1000, "bfloat16")] + [_leaf(1 << 20, "bfloat16")] * 31 + [_leaf(103022592, "bfloat16")]
    gradients, blocks = fresh(leaves)
    _check(leaves, gradients, blocks, grads._ARENA_BYTES)
    assert len(blocks) == 2                               # still one allocation for the 32 others


@pytest.mark.parametrize("seed", range(20))
def test_bound_on_any_list(fresh, monkeypatch, seed):
    rng = random.Random(seed)
    monkeypatch.setattr(grads, "_ARENA_BYTES", 1 << 16)
    edges = [0, 1, 255, 256, 257, 8192, 16384, 32767, 32768, 32769, 100000]
    leaves = [_leaf(rng.choice(edges) if rng.random() < 0.3 else int(2 ** rng.uniform(0, 17)),
                    rng.choice(["float32", "float16", "bfloat16", "float64"])) for _ in range(60)]
    gradients, blocks = fresh(leaves)
    _check(leaves, gradients, blocks, 1 << 16)
    # Two neighbours of one dtype that fit together share: at most about twice the fewest allocations.
    total = sum(-(-leaf._numel // 256) * 256 * leaf._dtype.itemsize for leaf in leaves)
    assert len(blocks) <= 2 * (total // (1 << 16)) + 8


def test_views_are_whole_tensors(fresh):
    """``device_views`` fills every slot as the constructor does."""
    (view, _), _ = fresh([_leaf(300, "float16"), _leaf(5, "float16")])
    made = Tensor._from_storage(view._storage)
    for slot in Tensor.__slots__:
        if slot not in ("__weakref__", "_version_counter"):
            assert getattr(view, slot) == getattr(made, slot), slot
    assert view._version_counter.value == 0 and view._version_counter is not made._version_counter
