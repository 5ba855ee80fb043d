"""The marches on the sizes where they are the default, with the kernel asserted:
one generation (aligned and unaligned rows, rows of fewer than four cells) and two
generations, against the oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


# Above 26 million cells at any row alignment, ordinary and (above 128 MiB)
# non-temporal stores; r = 10 on aligned rows from 13.6 million cells; radii 2 to 4
# above 3 million.
@pytest.mark.parametrize("r,shape", [(7, (5200, 5201)), (7, (5200, 5204)), (12, (5200, 5201)), (12, (5200, 5204)),
                                     (16, (5200, 5201)), (16, (5200, 5204)), (9, (6000, 6000)), (10, (3700, 3700)),
                                     (10, (6000, 6000)), (11, (5900, 5801)),
                                     (8, (9000000, 3)), (15, (9000000, 3)), (2, (2000, 1700)), (3, (2001, 1703)), (4, (2000, 1701))])
def test_single_steps_that_march(r, shape):
    print(f"[case] march r={r} {shape}", flush=True)
    hip.init(0)
    rows, cols = shape
    x = R.fill_uniform_f32(rows * cols, 20 + r).reshape(shape)
    a, b = DeviceArray.from_host(x), DeviceArray(shape, np.float32)
    assert hip.mean_iterate_kernels(a.ptr, b.ptr, rows, cols, r, 1) == ["march"]
    call("msl_stencil2d_mean_f32", b.ptr, a.ptr, rows, cols, r, 3.5)
    np.testing.assert_array_equal(b.to_host(), R.stencil2d_mean_f32(x, r, 3.5))


@pytest.mark.parametrize("r,shape", [(4, (4200, 4100)), (4, (4101, 4203)), (5, (5900, 5800)), (7, (5801, 5903))])
def test_iterations_in_pairs(r, shape):
    print(f"[case] pairs r={r} {shape}", flush=True)
    hip.init(0)
    rows, cols = shape
    x = R.fill_uniform_f32(rows * cols, 30 + r).reshape(shape)
    a, b = DeviceArray.from_host(x), DeviceArray(shape, np.float32)
    kernels = hip.mean_iterate_kernels(a.ptr, b.ptr, rows, cols, r, 5)
    assert kernels.count("pair") == 2 and kernels.count("march") == 1
    inb = C.c_int()
    call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, rows, cols, r, 3.5, 5, C.byref(inb))
    for _ in range(5):
        x = R.stencil2d_mean_f32(x, r, 3.5)
    np.testing.assert_array_equal(b.to_host(), x)
