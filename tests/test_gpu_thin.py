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


# Grids of few rows: the widths on both sides of the rules (for 256 CUs), by
# the kernel that a single step and an iteration run.
@pytest.mark.parametrize("r,shape,step,iterate", [
    (2, (1, 122881), "march", "tile"), (2, (1, 122700), "tile", "tile"),
    (2, (8, 245761), "march", "march"), (2, (9, 245761), "march", "tile"),
    (2, (16, 983041), "march", "pair"), (3, (17, 983041), "march", "tile"),
    (5, (16, 110600), "march", "tile"), (8, (12, 196609), "march", "march"), (8, (13, 196609), "march", "march"),
    (10, (2, 90113), "march", "march"), (13, (8, 208897), "march", "march"), (13, (9, 208897), "tile", "tile"),
    (16, (3, 196609), "march", "march"), (4, (5, 1000003), "march", "march"),
])
def test_mean_thin_grids(r, shape, step, iterate):
    print(f"[case] mean r={r} thin {shape}", flush=True)
    hip.init(0)
    rows, cols = shape
    x = R.fill_uniform_f32(rows * cols, 4).reshape(shape)
    a, b = DeviceArray.from_host(x), DeviceArray(shape, np.float32)
    assert hip.mean_iterate_kernels(a.ptr, b.ptr, rows, cols, r, 1) == [step]
    assert hip.mean_iterate_kernels(a.ptr, b.ptr, rows, cols, r, 4)[0] == iterate
    inb = C.c_int()
    for iters in (1, 4):
        a = DeviceArray.from_host(x)
        call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, rows, cols, r, 1.5, iters, C.byref(inb))
        want = x
        for _ in range(iters):
            want = R.stencil2d_mean_f32(want, r, 1.5)
        np.testing.assert_array_equal((b if inb.value else a).to_host(), want)


# Narrow grids: rows that one strip of the two-generation march holds, and
# tile plans with launches of one generation.
@pytest.mark.parametrize("r,shape,kernel", [(2, (70000, 160), "pair"), (2, (70000, 191), "tile"), (3, (40000, 240), "pair"),
                                            (3, (40000, 250), "tile"), (3, (160000, 56), "tile"), (2, (150000, 60), "tile")])
@pytest.mark.parametrize("iters", [2, 6])
def test_mean_narrow_grids(r, shape, kernel, iters):
    print(f"[case] mean r={r} narrow {shape} x{iters}", flush=True)
    hip.init(0)
    rows, cols = shape
    x = R.fill_uniform_f32(rows * cols, 6).reshape(shape)
    a, b = DeviceArray.from_host(x), DeviceArray(shape, np.float32)
    if iters > 2:
        assert set(hip.mean_iterate_kernels(a.ptr, b.ptr, rows, cols, r, iters)) <= {kernel, "march" if kernel == "pair" else kernel}
    inb = C.c_int()
    call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, rows, cols, r, 1.5, iters, C.byref(inb))
    for _ in range(iters):
        x = R.stencil2d_mean_f32(x, r, 1.5)
    np.testing.assert_array_equal((b if inb.value else a).to_host(), x)


# Radius-1 windows over the grid's edge: every window shape on narrow and flat
# grids, odd widths, waves without rows in the grid, cells of either sign and
# neutral values that are no ordinary number.
@pytest.mark.parametrize("shape", [(13400, 60), (27000, 52), (27000, 104), (27000, 105), (9000, 117), (1, 30000), (7, 20001),
                                   (53, 9000), (70000, 1), (40000, 3), (200, 64), (1700, 1801)])
def test_mean3_edge_windows(shape):
    print(f"[case] mean3 edges {shape}", flush=True)
    hip.init(0)
    rows, cols = shape
    x = R.fill_uniform_f32(rows * cols, 8).reshape(shape)
    for data, nv in ((x, 3.5), (x - np.float32(127.5), 0.0), (x, -np.inf), (x, np.nan)):
        for iters in (3, 6):
            a, b = DeviceArray.from_host(data), DeviceArray(shape, np.float32)
            assert hip.mean_iterate_kernels(a.ptr, b.ptr, rows, cols, 1, iters)[0] == "window"
            inb = C.c_int()
            call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, rows, cols, 1, nv, iters, C.byref(inb))
            want = data
            for _ in range(iters):
                want = R.stencil2d_mean_f32(want, 1, nv)
            got = (b if inb.value else a).to_host()
            np.testing.assert_array_equal(got, want)
            keep = ~np.isnan(want)
            np.testing.assert_array_equal(got.view(np.uint32)[keep], want.view(np.uint32)[keep])
