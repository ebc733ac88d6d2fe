"""``nt_grad_apply_flat`` (the read of one transformed gradient) against the
plan's ``nt_grad_apply``, bit for bit: tile edges, tails, unaligned starts,
host-known transforms and a control block's."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import namitorch_amd as nt
from namitorch_amd import _native
from oracle import lowp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("offset", [0, 1, 2])
@pytest.mark.parametrize("count", [1, 3, 4, 255, 1023, 1024, 1025, 2047, 2048, 2049, 70001])
def test_flat_equals_plan(dtype, offset, count):
    rng = np.random.default_rng(count + offset)
    values = lowp.round_to(dtype, rng.standard_normal(count + offset) * 300)
    backend = nt.get_backend(DEV)
    ctrl = backend.new_ctrl(1024.0)
    block = backend.read_ctrl(ctrl)
    block.scale_used, block.clip, block.clip_coef = 1024.0, 1, 0.37
    _native.call("nt_memcpy_h2d", ctrl.data_ptr(), ctypes.addressof(block), ctypes.sizeof(block), backend.stream())
    for transform in (dict(scale=3.0, unscale=1), dict(scale=65536.0, unscale=1, clip=1, clip_coef=0.123456789),
                      dict(clip=1, clip_coef=1e-3), dict(unscale=1, ctrl=ctrl.data_ptr()), {}):
        xform = _native.GradXform(**{**dict(scale=1.0, clip_coef=1.0), **transform})
        results = []
        for flat in (False, True):
            whole = nt.Tensor(values, dtype=dtype, device=DEV)
            kind = whole.dtype
            part = whole._storage.narrow(offset, count)
            if flat:
                _native.call("nt_grad_apply_flat", 0, part.data_ptr(), kind.code, count, ctypes.byref(xform),
                             backend.stream())
            else:
                plan = backend.plan([(0, 0, 0, 0, 0, count, 0)], (_native.NT_DTYPE_NONE, kind.code,
                                    _native.NT_DTYPE_NONE, _native.NT_DTYPE_NONE), pointers={1: [part.data_ptr()]})
                backend.grad_apply(plan, xform)
            results.append(whole.bits().tobytes())
        assert results[0] == results[1], transform
    assert whole.bits().tobytes() == nt.Tensor(values, dtype=dtype, device=DEV).bits().tobytes()   # {}: nothing applied


def test_arguments_are_checked():
    xform = _native.GradXform(scale=2.0, unscale=1, clip_coef=1.0)
    with pytest.raises(TypeError, match="float32, float16 or bfloat16"):
        _native.call("nt_grad_apply_flat", 0, None, _native.NT_F64, 4, ctypes.byref(xform), None)
    with pytest.raises(ValueError, match="NULL gradient"):
        _native.call("nt_grad_apply_flat", 0, None, _native.NT_F32, 4, ctypes.byref(xform), None)
    with pytest.raises(ValueError, match="not aligned"):
        _native.call("nt_grad_apply_flat", 0, 6, _native.NT_F32, 4, ctypes.byref(xform), None)
    _native.call("nt_grad_apply_flat", 0, None, _native.NT_F32, 0, ctypes.byref(xform), None)
