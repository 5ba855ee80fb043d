"""Heat steps in LDS (3-D tiles on small cubes, the two-generation plane march
on larger ones) against the oracle, bit for bit, residuals included: tile and
vector remainders, cubes narrower than a vector, launch plans around residuals,
an unaligned base pointer, and sums whose division needs the full form
(subnormal, infinite and NaN cells, signed zeros)."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


def _check(x, nv, iters, every, shift=0):
    nz, ny, nx = x.shape
    n = x.size
    a = DeviceArray.from_host(np.concatenate([np.zeros(shift, np.float32), x.ravel()]))
    b = DeviceArray(n + shift, np.float32)
    nres = iters // every if every else 0
    res = (C.c_float * max(nres, 1))()
    inb = C.c_int()
    call("msl_heat7_iterate_f32", a.ptr + 4 * shift, b.ptr + 4 * shift, nx, ny, nz, nv, iters, every,
         res if nres else None, C.byref(inb))
    assert inb.value == (iters & 1)
    ref, ref_res = x, []
    for it in range(iters):
        if every and (it + 1) % every == 0:
            ref, m = R.heat7_residual_f32(ref, nv)
            ref_res.append(m)
        else:
            ref = R.heat7_f32(ref, nv)
    got = (b if inb.value else a).to_host()[shift:].reshape(x.shape)
    np.testing.assert_array_equal(got, ref)
    fin = np.isfinite(x).all()
    if fin:
        np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))
        assert list(res)[:nres] == ref_res


def _cube(shape, seed):
    n = int(np.prod(shape))
    return R.fill_uniform_f32(n, seed, R.SCALE_UNIT).reshape(shape)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 5), (12, 16, 3), (11, 17, 33), (13, 9, 64), (30, 31, 67),
                                   (60, 70, 80), (110, 90, 129)])
@pytest.mark.parametrize("iters,every", [(1, 0), (2, 0), (3, 0), (7, 0), (12, 0), (3, 1), (6, 3), (11, 5)])
def test_heat_tiles(shape, iters, every):
    print(f"[case] heat tiles {shape} x{iters} every {every}", flush=True)
    hip.init(0)
    _check(_cube(shape, 3 + iters), 0.25, iters, every, shift=iters & 1)


# above 4.2 million cells: both tilings of the plane march, aligned and odd rows
@pytest.mark.parametrize("shape", [(170, 165, 164), (101, 300, 163), (40, 210, 514), (300, 130, 129), (9, 700, 701)])
@pytest.mark.parametrize("iters,every", [(4, 2), (5, 0)])
def test_heat_pairs(shape, iters, every):
    print(f"[case] heat pairs {shape} x{iters} every {every}", flush=True)
    hip.init(0)
    assert max(hip.heat_iterate_plan(shape[2], shape[1], shape[0], iters, every)) == 2
    _check(_cube(shape, 8), 0.25, iters, every, shift=iters & 1)


@pytest.mark.parametrize("shape", [(20, 30, 50), (170, 165, 164)])
def test_heat_special_values(shape):
    print(f"[case] heat special values {shape}", flush=True)
    hip.init(0)
    rng = np.random.default_rng(4)
    for kind in ("subnormal", "zeros", "inf", "nan", "large"):
        if kind == "subnormal":
            x = (rng.integers(-40, 40, shape) * np.float64(2.0**-149)).astype(np.float32)
        elif kind == "zeros":
            x = np.where(rng.random(shape) < 0.01, 1.0, -0.0).astype(np.float32)
        else:
            x = rng.uniform(-1.0, 1.0, shape).astype(np.float32)
            x.ravel()[rng.integers(0, x.size, 9)] = {"inf": np.inf, "nan": np.nan,
                                                    "large": np.finfo(np.float32).max}[kind]
        _check(x, -0.0, 4, 0)
