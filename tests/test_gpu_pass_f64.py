"""The float64 AdamW pass: bits of the oracle at the edges of its 128-element
slices and 4096-element tasks, for tensors that allow 16-byte accesses and
ones that do not, and the same bits for every task size."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import namitorch_amd as nt
from namitorch_amd import _native
from oracle import adam as oadam

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZES = (1, 2, 3, 127, 128, 129, 255, 4095, 4096, 4097, 8191, 20003)
OPTIONS = [dict(), dict(weight_decay=0.0), dict(maximize=True), dict(lr=0.0)]


def _host(seed):
    rng = np.random.default_rng(seed)
    return [[rng.standard_normal(n) * s for s in (0.02, 1e-3, 1e-4)] + [rng.random(n) * 1e-6] for n in SIZES]


@pytest.mark.parametrize("kind", ["AdamW", "Adam"])
@pytest.mark.parametrize("options", OPTIONS)
@pytest.mark.parametrize("offset", [0, 1])
def test_bits_of_the_oracle(kind, options, offset):
    """`offset` 1: every array starts 8 bytes into an allocation."""
    options = {"lr": 3e-4, "weight_decay": 0.1, **options}
    values = _host(5)
    params, states = [], []
    for host in values:
        arrays = []
        for array in host:
            flat = nt.DeviceArray.empty((array.size + offset,), "float64", DEV).upload(
                np.concatenate([np.full(offset, 7.0), array]))
            arrays.append(flat.narrow(offset, array.size))
        parameter = nt.Parameter.__new__(nt.Parameter)
        nt.Tensor._initialize(parameter, arrays[0], True)
        parameter.grad = nt.Tensor._from_storage(arrays[1])
        params.append(parameter)
        states.append([nt.Tensor._from_storage(array) for array in arrays[2:]])
    optimizer = getattr(nt.optim, kind)(params, betas=(0.9, 0.999), eps=1e-8, **options)
    for parameter, (first, second) in zip(params, states):
        optimizer.state[id(parameter)] = {"step": 4, "exp_avg": first, "exp_avg_sq": second}
    optimizer.step()
    for parameter, (first, second), (p, g, m, v) in zip(params, states, values):
        oadam.adam_step(p, g, m, v, 5, betas=(0.9, 0.999), eps=1e-8, decoupled=kind == "AdamW", **options)
        for got, want in ((parameter, p), (first, m), (second, v)):
            assert np.array_equal(got.numpy().view(np.uint64), want.view(np.uint64)), p.size


@pytest.mark.parametrize("chunk", [2048, 6144, 8192, 65536])
def test_task_sizes_give_the_same_bits(chunk):
    """8192 is the largest task that splits; 6144 and 65536 run whole."""
    layout = (_native.NT_F64, _native.NT_F64, _native.NT_F64, _native.NT_DTYPE_NONE)
    coefs = (_native.AdamWCoefs64 * 1)(_native.AdamWCoefs64(3e-4, 0.9, 0.999, 0.1, 0.001, 1e-8, 0.1, 1 - 3e-5, 0.4,
                                                            0.005, 0, 1, 0, 0))
    xform = _native.GradXform(scale=3.0, unscale=1, clip=1, clip_coef=0.7)
    backend = nt.get_backend(DEV)
    results = []
    for size in (0, chunk):
        tensors = [[nt.Tensor(array, device=DEV) for array in host] for host in _host(9)]
        rows = [tuple(t._ptr for t in four) + (0, four[0].size, 0) for four in tensors]
        backend.adamw_multi(backend.plan(rows, layout, chunk=size), coefs, xform)
        results.append([t.numpy().tobytes() for four in tensors for t in four])
    assert results[0] == results[1]
