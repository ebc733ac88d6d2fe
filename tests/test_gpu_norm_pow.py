"""The general p-norm's second pass (``nt_grad_norm_pow``) against the oracle.

``get_grad_norm`` leaves every finite norm type on the device for 16- and
32-bit gradients; ``clip_grad_norm_`` and float64 gradients read the sums
back.  Exponents 1, 2 and 3 sum products under a power-of-two prescale, the
others ``pow`` under the prescale max|g|.

Tolerance: the sum of n nonnegative float64 terms carries at most
n * 2**-53 relative error in any order, a term at most 4 * 2**-53 and the
root and the rescaling as much again: (n + 16) * 2**-53, below 1e-11 here.
"""

from __future__ import annotations

import numpy as np
import pytest

import namitorch_amd as nt
from oracle import clip as oclip
from oracle import lowp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZES = {
    "one": [1],
    "edges": [3, 4, 1023, 4095, 4096, 4097, 0, 2 * 4096 + 5],
    "many": [4096 * 9 + 1] * 3 + [17] * 40,
}


def _bound(grads) -> float:
    return (sum(g.size for g in grads) + 16) * 2.0 ** -53


def _params(grads, dtype):
    params = [nt.Parameter(np.zeros(g.shape), dtype=dtype, device=DEV) for g in grads]
    for p, g in zip(params, grads):
        p.grad = nt.Tensor(g, dtype=dtype, device=DEV)
    return params


def _grads(sizes, dtype, sigma=1e-2):
    rng = np.random.default_rng(41)
    values = [rng.standard_normal(n) * sigma for n in sizes]
    return values if dtype == "float64" else [lowp.round_to(dtype, v) for v in values]


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16", "float64"])
@pytest.mark.parametrize("norm_type", [1, 3, 0.5, 2.5, 4.0])
@pytest.mark.parametrize("sizes", sorted(SIZES))
def test_norm_types(sizes, norm_type, dtype):
    grads = _grads(SIZES[sizes], dtype)
    wide = [g.astype(np.float64) for g in grads]
    want = oclip.total_norm(wide, norm_type)
    got = nt.optim.get_grad_norm(_params(grads, dtype), norm_type=norm_type)
    assert got.dtype is nt.float64 and got.shape == ()
    assert abs(got.item() - want) <= _bound(grads) * want
    # The host path: the sums of two dtypes, combined under the larger max|g|.
    mixed = _params(grads, dtype) + _params(_grads([5000], "float32", 3e-2), "float32")
    want = oclip.total_norm(wide + [g.astype(np.float64) for g in _grads([5000], "float32", 3e-2)], norm_type)
    norm = nt.optim.clip_grad_norm_(mixed, 1e300, norm_type=norm_type).item()
    assert abs(norm - want) <= (_bound(grads) + 6000 * 2.0 ** -53) * want


@pytest.mark.parametrize("norm_type", [1, 2, 3, 1.5, 500.0])
@pytest.mark.parametrize("magnitude", [1e-310, 1e-200, 1.0, 1e200, 1e307])
def test_float64_range(magnitude, norm_type):
    """Magnitudes whose powers leave the float64 range: the prescale holds them."""
    grads = [g * magnitude for g in _grads([1, 4097, 33], "float64", 0.3)]
    want = oclip.total_norm(grads, norm_type)
    got = nt.optim.get_grad_norm(_params(grads, "float64"), norm_type=norm_type).item()
    # Subnormal results have a coarser spacing than the relative bound.
    assert abs(got - want) <= max(2 * _bound(grads) * want, 2 * np.nextafter(0, 1)) or (np.isinf(got) and np.isinf(want))


@pytest.mark.parametrize("bad", ["inf", "nan"])
def test_nonfinite_and_zero(bad):
    grads = _grads([4097, 5], "float32")
    grads[1][2] = float(bad)
    got = nt.optim.get_grad_norm(_params(grads, "float32"), norm_type=3).item()
    assert np.isnan(got) if bad == "nan" else np.isinf(got)
    assert nt.optim.get_grad_norm(_params([np.zeros(7, np.float32)], "float32"), norm_type=1).item() == 0.0


@pytest.mark.parametrize("norm_type", [1, 3, 2.5])
def test_deferred_addend_counts(norm_type):
    """Added in the pass (1, 3) or written back before it."""
    grads, more = _grads([4096, 9], "float32"), _grads([9, 4096], "float32")[::-1]
    params = _params(grads, "float32")
    nt.accumulate_grads(params, [nt.Tensor(g, device=DEV) for g in more], defer=True)
    want = oclip.total_norm([(a + b).astype(np.float64) for a, b in zip(grads, more)], norm_type)
    assert abs(nt.optim.get_grad_norm(params, norm_type=norm_type).item() - want) <= _bound(grads) * want


@pytest.mark.parametrize("dtype, value", [("float32", 3.4e38), ("float32", 1e-45), ("float16", 65504.0),
                                          ("float16", 6e-8), ("bfloat16", 3.3e38), ("bfloat16", 1e-40)])
@pytest.mark.parametrize("norm_type", [1, 3])
def test_extremes_of_the_narrow_types(dtype, value, norm_type):
    """No prescale is needed: the largest and smallest values' powers stay in float64."""
    grads = [lowp.round_to(dtype, np.full(n, value)) for n in (1, 4099)]
    want = oclip.total_norm([g.astype(np.float64) for g in grads], norm_type)
    got = nt.optim.get_grad_norm(_params(grads, dtype), norm_type=norm_type).item()
    assert want > 0 and abs(got - want) <= _bound(grads) * want


def test_many_partials_take_the_second_stage():
    """Over 4096 workgroups of the pass."""
    flat = nt.Tensor(np.full(4096 * 8 * 4097 + 5, 0.5, np.float16), device=DEV)
    parameter = nt.Parameter(np.zeros(flat.shape, np.float16), device=DEV)
    parameter.grad = flat
    assert nt.optim.get_grad_norm([parameter], norm_type=1).item() == 0.5 * flat.size


@pytest.mark.parametrize("norm_type", [1, 2, 3, 2.5, np.inf])
@pytest.mark.parametrize("kind", ["finite", "zero", "inf", "nan"])
@pytest.mark.parametrize("clip", [False, True])
def test_item_is_the_device_scalar(norm_type, kind, clip):
    """``.item()`` of a norm, a view of its control block or the host copy of it: the bits
    a copy from the device gives, also again, and not after a write."""
    grads = _grads([4097, 5], "float32")
    if kind == "zero":
        grads = [g * 0 for g in grads]
    elif kind != "finite":
        grads[0][7] = float(kind)
    params = _params(grads, "float32")
    norm = (nt.optim.clip_grad_norm_(params, 1e3, norm_type=norm_type) if clip
            else nt.optim.get_grad_norm(params, norm_type=norm_type))
    first, copied, again = norm.item(), norm.numpy(), norm.item()
    assert type(first) is float and copied.shape == ()
    assert np.float64(first).tobytes() == copied.tobytes() == np.float64(again).tobytes()
    norm.fill_(7.0)
    assert norm.item() == 7.0
