"""The float16 AdamW pass on whole aligned slices (packed float16 arithmetic,
short division and root sequences) against NumPy's float16 arithmetic and
against the general loop, which whole-task plans run: the same bits."""

from __future__ import annotations

import numpy as np
import pytest

import namitorch_amd as nt
from namitorch_amd import _native
from oracle import adam as oadam

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZES = (1, 511, 512, 513, 2047, 2048, 2049, 4096, 70001)
F16, NONE = _native.NT_F16, _native.NT_DTYPE_NONE


def _host(seed, wide=False):
    """Ordinary values, or (`wide`) every kind of float16: all exponents,
    subnormals, zeros of both signs, infinities and NaN."""
    rng = np.random.default_rng(seed)
    values = []
    for n in SIZES:
        if wide:
            four = [rng.integers(0, 1 << 16, n, dtype=np.uint16).view(np.float16) for _ in range(4)]
            four[3] = np.abs(four[3])
        else:
            four = [(rng.standard_normal(n) * s).astype(np.float16) for s in (0.02, 0.1, 0.03)]
            four.append((rng.standard_normal(n) ** 2 * 0.01).astype(np.float16))
        values.append(four)
    return values


def _same(got, want) -> bool:
    return bool(((got.view(np.uint16) == want.view(np.uint16)) | (np.isnan(got) & np.isnan(want))).all())


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("step", [1, 5, 3000])
@pytest.mark.parametrize("weight_decay", [0.0, 0.1])
def test_bits_of_numpy(wide, step, weight_decay):
    values = _host(3, wide)
    params = [nt.Parameter(four[0], device=DEV) for four in values]
    optimizer = nt.optim.AdamW(params, lr=1e-3, betas=(0.9, 0.999), eps=1e-4, weight_decay=weight_decay)
    for parameter, (_, g, m, v) in zip(params, values):
        parameter.grad = nt.Tensor(g, device=DEV)
        first, second = nt.Tensor(m, device=DEV), nt.Tensor(v, device=DEV)
        optimizer.state[id(parameter)] = {"step": step - 1, "exp_avg": first, "exp_avg_sq": second}
    optimizer.step()
    for parameter, (p, g, m, v) in zip(params, values):
        with np.errstate(all="ignore"):
            oadam.adam_step(p, g, m, v, step, lr=1e-3, betas=(0.9, 0.999), eps=1e-4, weight_decay=weight_decay)
        state = optimizer.state[id(parameter)]
        for got, want in ((parameter, p), (state["exp_avg"], m), (state["exp_avg_sq"], v)):
            assert _same(got.numpy(), want), p.size


# The first record is the optimizer's kind (float16 values); the others keep
# the general loop: a learning rate that is no float16 value, a zero bias
# correction, maximize, coupled decay, no parameter update.
RECORDS = [(0.001, 1.0, 0, 1, 0), (0.0003, 1.0, 0, 1, 0), (0.001, 0.0, 0, 1, 0), (0.001, 1.0, 1, 1, 0),
           (0.001, 1.0, 0, 1, 1), (0.001, 1.0, 0, 0, 0)]


@pytest.mark.parametrize("record", range(len(RECORDS)))
@pytest.mark.parametrize("transform", [None, dict(scale=1024.0, unscale=1), dict(scale=3.0, unscale=1, clip=1, clip_coef=0.37)])
@pytest.mark.parametrize("misaligned", [False, True])
def test_split_equals_whole_tasks(record, transform, misaligned):
    half = lambda x: float(np.float16(x))  # noqa: E731
    lr, corrected, *flags = RECORDS[record]
    coefs = (_native.AdamWCoefs * 1)(_native.AdamWCoefs(
        half(lr) if record else half(0.001), half(0.9), half(0.999), half(0.1), half(0.001), half(1e-4), half(0.1),
        half(1 - 1e-4), half(0.41) * corrected, half(0.005) * corrected, *flags, 0))
    if record == 1:
        coefs[0].lr = 0.0003
    xform = None if transform is None else _native.GradXform(**{**dict(scale=1.0, clip_coef=1.0), **transform})
    backend = nt.get_backend(DEV)
    results = []
    for chunk in (2048, 8192, 6144, 65536):              # the last two run whole tasks
        tensors = [[nt.Tensor(np.concatenate([array, np.zeros(1, np.float16)]), device=DEV) for array in four]
                   for four in _host(11, wide=record == 0)]
        shift = 2 if misaligned else 0
        rows = [tuple(t._ptr + shift * (k == 4) for t in four) + (0, four[0].size - 1, 0)
                for k, four in enumerate(tensors)]
        backend.adamw_multi(backend.plan(rows, (F16, F16, F16, NONE), chunk=chunk), coefs, xform)
        results.append([t.numpy() for four in tensors for t in four])
    for other in results[1:]:
        assert all(_same(a, b) for a, b in zip(results[0], other)), record
