"""``nt_cast`` at the edges of its tiles (1024 elements with float64 on either
side, 2048 with float32, 4096 between 16-bit types), for tails and for arrays
that do not allow 16-byte accesses: NumPy's cast with one rounding, special
values included."""

from __future__ import annotations

import numpy as np
import pytest

import namitorch_amd as nt
from oracle import lowp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TYPES = ["float32", "float16", "bfloat16", "float64"]
SPECIAL = [0.0, -0.0, 1.0, -1.0, 65504.0, 65520.0, 3.4e38, 1e-8, -1e-45, 6e-8, np.inf, -np.inf, np.nan,
           1.00390625, 1.01171875, 1.00048828125, 1.00146484375, 2.0 ** -14, 2.0 ** -24, 2.0 ** -133]


@pytest.mark.parametrize("source", TYPES)
@pytest.mark.parametrize("target", TYPES)
def test_values_and_tile_edges(source, target):
    if source == target:
        pytest.skip("a copy")
    for count in (1, 20, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 12289):
        rng = np.random.default_rng(count)
        host = rng.standard_normal(count + 3) * np.exp2(rng.integers(-30, 17, count + 3))
        host[:min(count, 20)] = SPECIAL[:min(count, 20)]
        with np.errstate(over="ignore"):
            values = host if source == "float64" else lowp.round_to(source, host)
            want = values.astype(np.float64) if target == "float64" else lowp.round_to(target, values.astype(np.float64))
        whole = nt.Tensor(values, dtype=source, device=DEV)
        for start in (0, 1, 3):                           # 1 and 3: unaligned input, output, or both
            out = nt.Tensor(np.full(count + 3, 7.0), dtype=target, device=DEV)
            into = out._storage.narrow(start if start == 1 else 0, count)
            into.copy_from(whole._storage.narrow(start, count))
            got = out.numpy()
            first = start if start == 1 else 0
            np.testing.assert_array_equal(got[first:first + count], want[start:start + count])
            assert (np.signbit(got[first:first + count]) == np.signbit(want[start:start + count]))[
                ~np.isnan(want[start:start + count])].all()
            assert (got[:first] == 7).all() and (got[first + count:] == 7).all()


@pytest.mark.parametrize("bits, source, view", [(0x7F81, "bfloat16", np.uint16), (0x7C01, "float16", np.uint16),
                                                 (0x7F800001, "float32", np.uint32)])
@pytest.mark.parametrize("target", TYPES)
def test_signaling_nan_comes_out_quiet(bits, source, view, target):
    if source == target:
        pytest.skip("a copy")
    raw = nt.DeviceArray.empty((600,), source, DEV).upload(np.full(600, bits, view))
    out = nt.DeviceArray.empty((600,), target, DEV).copy_from(raw).raw_bits()
    quiet = {"float32": 1 << 22, "float16": 1 << 9, "bfloat16": 1 << 6, "float64": 1 << 51}[target]
    assert (out & type(out[0])(quiet)).all()
