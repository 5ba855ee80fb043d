"""Radius-1 iterations in registers against the oracle, bit for bit: both window
widths at tile remainders, and cells that leave the two-operation division
(tiny, negative, signed zeros, infinite, NaN, huge)."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


def _check(x, nv, iters):
    rows, cols = x.shape
    a, b = DeviceArray.from_host(x), DeviceArray(x.shape, np.float32)
    inb = C.c_int()
    call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, rows, cols, 1, nv, iters, C.byref(inb))
    ref = x
    for _ in range(iters):
        ref = R.stencil2d_mean_f32(ref, 1, nv)
    got = (b if inb.value else a).to_host()
    np.testing.assert_array_equal(got, ref)
    keep = ~np.isnan(ref)
    np.testing.assert_array_equal(got.view(np.uint32)[keep], ref.view(np.uint32)[keep])


@pytest.mark.parametrize("shape", [(52, 52), (53, 53), (104, 105), (1, 200), (1660, 1857), (1664, 2089)])
@pytest.mark.parametrize("iters", [2, 6, 7, 8])
def test_mean3_windows(shape, iters):
    print(f"[case] mean3 {shape} x{iters}", flush=True)
    hip.init(0)
    _check(R.fill_uniform_f32(shape[0] * shape[1], 5).reshape(shape), 3.5, iters)


@pytest.mark.parametrize("shape", [(120, 130), (1660, 1857)])
def test_mean3_cells_outside_the_short_division(shape):
    print(f"[case] mean3 special values {shape}", flush=True)
    hip.init(0)
    rng = np.random.default_rng(2)
    base = rng.uniform(0.0, 255.0, shape).astype(np.float32)
    for v in (2.0**-61, 2.0**-149, -0.0, -7.25, 2.0**101, np.finfo(np.float32).max, np.inf, -np.inf, np.nan):
        x = base.copy()
        x.ravel()[rng.integers(0, x.size, 5)] = v
        _check(x, 0.0, 6)
    _check((base * np.float32(1e-44)).astype(np.float32), 0.0, 6)
    _check(base, -0.0, 6)
