"""Environment overrides of the kernel choice: results stay bit-identical to
the oracle under each of them."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


# Only 1 and 2 force a count of generations per launch; any other value is as
# if the variable were unset.
@pytest.mark.parametrize("value", ["-1", "0", "3", "8", "x"])
def test_generation_overrides_other_than_1_and_2(value, monkeypatch):
    print(f"[case] generations forced to {value}", flush=True)
    hip.init(0)
    nx, ny, nz, iters = 40, 30, 20, 7
    host = R.fill_uniform_f32(nx * ny * nz, 6, R.SCALE_UNIT).reshape(nz, ny, nx)
    want = host
    for _ in range(iters):
        want = R.heat7_f32(want, 0.25)
    plans = [hip.heat_iterate_plan(nx, ny, nz, iters, 0), hip.mean_iterate_plan(None, None, 90, 130, 3, iters)]
    monkeypatch.setenv("MSL_HEAT_GENS", value)
    monkeypatch.setenv("MSL_MEAN_GENS", value)
    a, b = DeviceArray.from_host(host), DeviceArray(host.shape, np.float32)
    inb = C.c_int()
    call("msl_heat7_iterate_f32", a.ptr, b.ptr, nx, ny, nz, 0.25, iters, 0, None, C.byref(inb))
    np.testing.assert_array_equal((b if inb.value else a).to_host(), want)

    host = R.fill_uniform_f32(90 * 130, 7).reshape(90, 130)
    want = host
    for _ in range(iters):
        want = R.stencil2d_mean_f32(want, 3, 0.5)
    a, b = DeviceArray.from_host(host), DeviceArray(host.shape, np.float32)
    call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, 90, 130, 3, 0.5, iters, C.byref(inb))
    np.testing.assert_array_equal((b if inb.value else a).to_host(), want)
    assert [hip.heat_iterate_plan(nx, ny, nz, iters, 0),
            hip.mean_iterate_plan(None, None, 90, 130, 3, iters)] == plans


MARCH = r"""
import numpy as np
from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R
import ctypes as C
hip.init(0)
for r in (1, 2, 3, 5, 7, 9, 10, 12, 16):
    for shape in [(200, 301), (130, 260), (333, 3), (1, 700), (70, 1028)]:
        n = shape[0] * shape[1]
        x = R.fill_uniform_f32(n, 3 + r).reshape(shape)
        a, b = DeviceArray.from_host(x), DeviceArray(shape, np.float32)
        assert hip.mean_iterate_kernels(a.ptr, b.ptr, *shape, r, 1) == ["march"], (shape, r)
        call("msl_stencil2d_mean_f32", b.ptr, a.ptr, *shape, r, 1.5)
        np.testing.assert_array_equal(b.to_host(), R.stencil2d_mean_f32(x, r, 1.5), err_msg=f"{shape} r={r}")
        inb = C.c_int()
        call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, *shape, r, 1.5, 3, C.byref(inb))
        want = x
        for _ in range(3):
            want = R.stencil2d_mean_f32(want, r, 1.5)
        np.testing.assert_array_equal(b.to_host(), want, err_msg=f"{shape} r={r} x3")
"""


# The overrides of the march's shape (read once per process) march at every
# size: every radius and row mode of it, with both strip widths.
@pytest.mark.parametrize("env", [{"MSL_STRIP_SEG": "24"}, {"MSL_STRIP_C": "4"}, {"MSL_STRIP_C": "1"},
                                 {"MSL_STRIP_C": "1", "MSL_STRIP_SEG": "7"}])
def test_march_shape_overrides(env):
    print(f"[case] march with {env}", flush=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", MARCH], cwd=root, env={**os.environ, **env}, stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=100)
    assert res.returncode == 0, res.stdout
