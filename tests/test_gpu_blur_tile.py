"""Tile kernel of the mean blur against the oracle, bit for bit: single steps
of radius 5 and above and iterations of radius 2 and above on grids up to a
few million cells, at tile and vector remainders, in every tile kind (the
shapes grow from one tile to thousands), with neutral values, a base pointer
that is not 16-byte aligned, signed zeros, infinities and NaN."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (5, 3), (33, 31), (65, 41), (64, 128), (130, 523)]


def _iterate(x, r, nv, iters, shift=0):
    """The library's result of `iters` iterations from a buffer that starts
    `shift` floats into its allocation, and the oracle's."""
    rows, cols = x.shape
    n = rows * cols
    a = DeviceArray.from_host(np.concatenate([np.zeros(shift, np.float32), x.ravel()]))
    b = DeviceArray(n + shift, np.float32)
    inb = C.c_int()
    call("msl_stencil2d_mean_iterate_f32", a.ptr + 4 * shift, b.ptr + 4 * shift, rows, cols, r, nv, iters,
         C.byref(inb))
    assert inb.value == (iters & 1)
    ref = x
    for _ in range(iters):
        ref = R.stencil2d_mean_f32(ref, r, nv)
    return (b if inb.value else a).to_host()[shift:].reshape(rows, cols), ref


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("r", [2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 16])
@pytest.mark.parametrize("iters", [1, 2, 5, 12])
def test_blur_tile_edges(shape, r, iters):
    print(f"[case] blur tile {shape} r={r} x{iters}", flush=True)
    hip.init(0)
    x = R.fill_uniform_f32(shape[0] * shape[1], 7 + r).reshape(shape)
    got, ref = _iterate(x, r, 2.5, iters, shift=r & 1)
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("shape", [(517, 1031), (1024, 1024), (1100, 2050)])
@pytest.mark.parametrize("r", [2, 5, 8, 10])
def test_blur_tile_larger_grids(shape, r):
    print(f"[case] blur tile {shape} r={r}", flush=True)
    hip.init(0)
    x = R.fill_uniform_f32(shape[0] * shape[1], 3).reshape(shape)
    for iters in (1, 6):
        got, ref = _iterate(x, r, 0.0, iters)
        np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("r", [2, 5, 10])
@pytest.mark.parametrize("iters", [1, 4])
def test_blur_tile_special_values(r, iters):
    print(f"[case] blur tile special values r={r} x{iters}", flush=True)
    hip.init(0)
    rng = np.random.default_rng(r)
    x = np.full((150, 260), -0.0, np.float32)
    x[:, 130:] = rng.normal(0.0, 1e-42, (150, 130)).astype(np.float32)  # subnormal
    got, ref = _iterate(x, r, -0.0, iters)
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))
    for v in (np.inf, -np.inf, np.nan, np.finfo(np.float32).max):
        y = rng.uniform(-1.0, 1.0, (150, 260)).astype(np.float32)
        y[rng.integers(0, 150, 6), rng.integers(0, 260, 6)] = v
        got, ref = _iterate(y, r, 0.0, iters)
        np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("shape,r", [((2200, 2201), 5), ((2200, 2201), 10), ((2201, 2204), 9), ((1030, 4099), 12)])
def test_blur_tile_wide_single_steps(shape, r):
    """Single steps in 128-column tiles: grids above 4.7 million cells, and
    radii above 10 from four 64-column tiles per CU."""
    print(f"[case] blur tile wide {shape} r={r}", flush=True)
    hip.init(0)
    x = R.fill_uniform_f32(shape[0] * shape[1], 11).reshape(shape)
    got, ref = _iterate(x, r, 1.5, 1, shift=1)
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))
