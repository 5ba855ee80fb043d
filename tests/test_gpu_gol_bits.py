"""Bit-packed Game of Life iterations against the oracle (bit-exact): edges of
the packed words (32 columns) and windows (64 columns x 32 rows stored), the
launch plans around the 16 generations of one launch for both result buffers,
and cells other than 0 and 1 in the input."""
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


@pytest.mark.parametrize("shape", [(1, 2), (31, 31), (32, 32), (33, 65), (63, 64), (65, 127), (96, 97), (129, 160)])
@pytest.mark.parametrize("iters", [2, 3, 16, 17, 18, 33, 34, 50])
def test_gol_bits_edges(shape, iters):
    print(f"[case] gol bits {shape} x{iters}", flush=True)
    hip.init(0)
    rows, cols = shape
    _iterate(R.fill_bernoulli_i32(rows * cols, 5 + iters).reshape(rows, cols), iters)


@pytest.mark.parametrize("iters", [1, 2, 3, 20])
def test_gol_bits_cells_other_than_0_and_1(iters):
    print(f"[case] gol bits, other cells x{iters}", flush=True)
    hip.init(0)
    _iterate(np.random.default_rng(9).integers(-3, 5, (70, 130)).astype(np.int32), iters)
