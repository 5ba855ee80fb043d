"""Thin cubes and grids, which leave most of a tile empty, run the marches:
the kernel chosen on both sides of each rule, and its results bit for bit."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


# Shapes are (nz, ny, nx).  Up to 4.2 million cells: one generation per launch
# (the march) or several (tiles).
@pytest.mark.parametrize("shape,gens", [((1, 500, 1000), 1), ((3, 700, 900), 1), ((700, 1, 900), 1), ((1900, 3, 700), 1),
                                        ((1, 1, 300000), 1), ((1, 60, 70), 4), ((300, 8, 300), 3), ((8, 300, 300), 3)])
@pytest.mark.parametrize("every", [0, 1, 3])
def test_heat_thin_cubes(shape, gens, every):
    print(f"[case] heat thin {shape} every {every}", flush=True)
    hip.init(0)
    nz, ny, nx = shape
    iters = 6
    plan = hip.heat_iterate_plan(nx, ny, nz, iters, 0)
    assert max(plan) == min(gens, 3) if gens > 1 else plan == [1] * iters, plan
    _heat(shape, iters, every)


# Above 4.2 million cells: the two-generation march from 64 MiB on, with
# ordinary and (above 128 MiB) non-temporal stores, residuals in both.
@pytest.mark.parametrize("shape", [(1300, 4, 900), (1700, 10, 1000), (1, 4200, 4100), (2200, 500, 16), (3400, 10, 1010),
                                   (2, 4200, 4101)])
def test_heat_thin_large_cubes(shape):
    print(f"[case] heat thin large {shape}", flush=True)
    hip.init(0)
    nz, ny, nx = shape
    small = nx * ny * nz * 4 <= 64 << 20
    assert max(hip.heat_iterate_plan(nx, ny, nz, 5, 0)) == (1 if small else 2)
    _heat(shape, 5, 0)
    _heat(shape, 4, 2)


def _heat(shape, iters, every):
    nz, ny, nx = shape
    host = R.fill_uniform_f32(nx * ny * nz, 9, R.SCALE_UNIT).reshape(shape)
    a, b = DeviceArray.from_host(host), DeviceArray(shape, np.float32)
    res = (C.c_float * max(iters, 1))()
    inb = C.c_int()
    call("msl_heat7_iterate_f32", a.ptr, b.ptr, nx, ny, nz, 0.25, iters, every, res if every else None, C.byref(inb))
    want_res = []
    for it in range(iters):
        if every and (it + 1) % every == 0:
            host, m = R.heat7_residual_f32(host, 0.25)
            want_res.append(m)
        else:
            host = R.heat7_f32(host, 0.25)
    got = (b if inb.value else a).to_host()
    np.testing.assert_array_equal(got.view(np.uint32), host.view(np.uint32))
    assert list(res)[: len(want_res)] == want_res
