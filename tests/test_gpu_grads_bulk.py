"""``accumulate_grads`` over a list (checks and allocations for all leaves at
once) against the same leaves one at a time: values, dtypes, versions,
deferred additions, and the memory behind the new gradients."""

from __future__ import annotations

import gc
import weakref

import numpy as np
import pytest

import namitorch_amd as nt
from namitorch_amd import grads as grads_mod

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SHAPES = [(3,), (4096,), (0,), (17, 5), (4097,), (1,), (255,), (256,), (2, 2, 2)]


def _leaves(dtypes):
    return [nt.Parameter(np.zeros(s, np.float64), dtype=d, device=DEV) for s, d in zip(SHAPES, dtypes)]


def _incoming(seed, dtypes):
    rng = np.random.default_rng(seed)
    return [nt.Tensor(rng.standard_normal(s) * 3, dtype=d, device=DEV) for s, d in zip(SHAPES, dtypes)]


def _dtypes(kind):
    if kind == "mixed":
        return [("float32", "float16", "bfloat16", "float64")[k % 4] for k in range(len(SHAPES))]
    return [kind] * len(SHAPES)


@pytest.mark.parametrize("leaf", ["float32", "float16", "bfloat16", "float64", "mixed"])
@pytest.mark.parametrize("source", ["float32", "bfloat16", "mixed"])
@pytest.mark.parametrize("defer", [False, True])
@pytest.mark.parametrize("small_arenas", [False, True])
def test_list_equals_leaf_by_leaf(monkeypatch, leaf, source, defer, small_arenas):
    if small_arenas:                                      # several allocations per call
        monkeypatch.setattr(grads_mod, "_ARENA_BYTES", 4096)
    together, apart = _leaves(_dtypes(leaf)), _leaves(_dtypes(leaf))
    for seed in (1, 2, 3):
        values = _incoming(seed, _dtypes(source)[::-1] if source == "mixed" else _dtypes(source))
        later = defer and seed == 3
        nt.accumulate_grads(together, values, defer=later)
        for p, g in zip(apart, values):
            nt.accumulate_grads([p], [g], defer=later)
    for p, q in zip(together, apart):
        assert (p.grad._incoming is None) == (q.grad._incoming is None)
        assert p.grad._version == q.grad._version and p.grad.dtype is p.dtype and p.grad.shape == p.shape
        assert p.grad.bits().tobytes() == q.grad.bits().tobytes()
    spans = sorted((p.grad._ptr, p.grad._ptr + p.grad.nbytes) for p in together if p.grad.size)
    assert all(end <= start for (_, end), (start, _) in zip(spans, spans[1:])) and all(s % 16 == 0 for s, _ in spans)


def test_a_leaf_that_has_a_gradient_keeps_it():
    """Some leaves with a gradient, some without: the per-leaf path."""
    leaves = _leaves(_dtypes("float32"))
    leaves[1].grad = held = nt.Tensor(np.ones(4096, np.float32), device=DEV)
    nt.accumulate_grads(leaves, _incoming(5, _dtypes("float32")))
    assert leaves[1].grad is held and all(p.grad is not None for p in leaves)


def test_errors_leave_everything_unchanged():
    leaves = _leaves(_dtypes("float32"))
    wrong = _incoming(7, _dtypes("float32"))
    wrong[-1] = nt.Tensor(np.zeros(9, np.float32), device=DEV)
    with pytest.raises(RuntimeError, match="invalid gradient shape"):
        nt.accumulate_grads(leaves, wrong)
    assert all(p.grad is None for p in leaves)
    with pytest.raises(TypeError, match="requires NamiTorch Tensors"):
        nt.accumulate_grads([None, leaves[0]], wrong[:2])


@pytest.mark.parametrize("amp", [False, True])
def test_gradients_of_a_finished_iteration_are_not_kept(amp):
    """Two iterations later nothing refers to an iteration's gradients,
    without a garbage collection."""
    leaves = _leaves(_dtypes("float16"))
    optimizer = nt.optim.AdamW(leaves, master_weights=True)
    scaler = nt.GradScaler(init_scale=1024.0) if amp else None
    refs = []
    gc.collect()
    gc.disable()
    try:
        for seed in range(4):
            if amp:
                scaler.scale(nt.Tensor(np.float32(1), device=DEV))
            nt.accumulate_grads(leaves, _incoming(seed, _dtypes("float16")))
            refs.append([weakref.ref(p.grad) for p in leaves])
            nt.amp.fused_step(optimizer, scaler, max_norm=0.5)
            optimizer.zero_grad()
        assert not any(ref() for ref in refs[0] + refs[1])
    finally:
        gc.enable()
