"""The accumulation kernel's groups of 16 bytes and its temporal stores.

Between 16-bit types a lane moves eight elements at once, otherwise four; the
last 320 MiB of a list are stored with temporal accesses.  Results are exact:
one rounding of the incoming value to the stored type, one of the float32 sum.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import namitorch_amd as nt

pytestmark = pytest.mark.gpu
TORCH = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
# A group, a wave, a slice and a task of 4096 elements, and what is left beside them.
SIZES = [1, 7, 8, 9, 511, 513, 2047, 2048, 2049, 2055, 2056, 4096, 4103, 3 * 4096 + 12, 20483]


def _wrap(view):
    return nt.Tensor._from_storage(nt.DeviceArray.wrap(view))


def _check(sizes, stored, incoming, offset):
    """Gradients as views of one buffer that start `offset` elements past a multiple of 64."""
    generator = torch.Generator(device="cuda").manual_seed(9)
    starts = np.concatenate([[0], np.cumsum([-(-n // 64) * 64 + 64 for n in sizes])]) + offset
    flats = [torch.randn(int(starts[-1]), generator=generator, device="cuda").mul_(3).to(TORCH[d])
             for d in (incoming, incoming)]
    kept = torch.full((int(starts[-1]),), 7.0, dtype=TORCH[stored], device="cuda")
    views = [[flat[a:a + n] for a, n in zip(starts.tolist(), sizes)] for flat in flats]
    grads = [kept[a:a + n] for a, n in zip(starts.tolist(), sizes)]
    params = []
    for grad in grads:
        grad.zero_()
        parameter = nt.Parameter.__new__(nt.Parameter)
        nt.Tensor._initialize(parameter, nt.DeviceArray.wrap(torch.zeros_like(grad)), True)
        parameter.grad = _wrap(grad)
        params.append(parameter)
    torch.cuda.synchronize()
    for batch in views:
        nt.accumulate_grads(params, [_wrap(view) for view in batch])
    torch.cuda.synchronize()
    for k, grad in enumerate(grads):
        first, second = (batch[k].to(TORCH[stored]) for batch in views)
        want = (first.float() + second.float()).to(TORCH[stored])
        assert torch.equal(grad, want), sizes[k]
    for a, n, b in zip(starts.tolist(), sizes, starts.tolist()[1:]):        # nothing past an end
        assert bool((kept[a + n:b] == 7.0).all())
    # The first gradient of a leaf is the incoming one, cast.
    for parameter in params:
        parameter.grad = None
    nt.accumulate_grads(params, [_wrap(view) for view in views[0]])
    for k, parameter in enumerate(params):
        got = parameter.grad.bits()
        want = views[0][k].to(TORCH[stored]).view(torch.int16 if stored != "float32" else torch.int32)
        assert got.tobytes() == want.cpu().numpy().tobytes(), sizes[k]


@pytest.mark.parametrize("stored, incoming", [("float16", "float16"), ("bfloat16", "bfloat16"), ("float16", "bfloat16"),
                                              ("bfloat16", "float32"), ("float32", "bfloat16"),
                                              ("float32", "float32")])
@pytest.mark.parametrize("offset", [0, 4, 1])
def test_group_edges(stored, incoming, offset):
    _check(SIZES, stored, incoming, offset)


def test_longer_than_the_kept_window():
    """The line between bypassing and temporal stores lies inside the list."""
    _check([3 * 4096 + 5, (320 << 20) // 2 + 5 * 4096 + 13], "bfloat16", "bfloat16", 0)
