"""Short Game of Life iterations and single columns, in windows of int cells:
bit-exact against the oracle, and odd counts of one launch leave their input
as it was."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import DeviceArray, call
from oracle import refcpu as R

pytestmark = pytest.mark.gpu


def _iterate(grid, iters):
    rows, cols = grid.shape
    a, b = DeviceArray.from_host(grid), DeviceArray((rows, cols), np.int32)
    inb = C.c_int()
    call("msl_gol_iterate_i32", a.ptr, b.ptr, rows, cols, iters, C.byref(inb))
    assert inb.value == (iters & 1)
    ref = grid
    for _ in range(iters):
        ref = R.gol_i32(ref)
    np.testing.assert_array_equal((b if inb.value else a).to_host(), ref)
    return a.to_host()


@pytest.mark.parametrize("shape,counts", [((1, 2), (1, 3, 7)), ((48, 48), (3, 5, 7)), ((49, 97), (1, 3, 5, 7)),
                                          ((1024, 1024), (3, 7)), ((1025, 1024), (1, 3)), ((1300, 1111), (3,))])
@pytest.mark.parametrize("low,high", [(0, 2), (-2, 4)])
def test_odd_counts_of_one_launch_leave_the_input(shape, counts, low, high):
    hip.init(0)
    grid = np.random.default_rng(7).integers(low, high, shape).astype(np.int32)
    for iters in counts:
        print(f"[case] gol windows {shape} x{iters}", flush=True)
        np.testing.assert_array_equal(_iterate(grid, iters), grid)


@pytest.mark.parametrize("rows", [1, 47, 48, 49, 5000])
@pytest.mark.parametrize("iters", [2, 3, 8, 9, 16, 21])
def test_single_column(rows, iters):
    print(f"[case] gol column of {rows} x{iters}", flush=True)
    hip.init(0)
    _iterate(np.random.default_rng(rows).integers(0, 2, (rows, 1)).astype(np.int32), iters)
