"""Narrow grids of a batch in LDS tiles: folds as exact as those of the strip
items, whatever the grid's size."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import BatchGrid, DeviceArray, call

pytestmark = pytest.mark.gpu

# A lane adds 64 cells to its compensated pair and six merges follow: the
# correction term is off by at most (n u)^2 of the sum of magnitudes.
FOLD_TOL = (70 * 2.0**-24) ** 2


class Grids:
    """A batch over host arrays, state a in them."""

    def __init__(self, arrays, radii, nv):
        self.a = [DeviceArray.from_host(x) for x in arrays]
        self.b = [DeviceArray(x.shape, np.float32) for x in arrays]
        self.sums = DeviceArray(len(arrays), np.float64)
        g = (BatchGrid * len(arrays))()
        for k, x in enumerate(arrays):
            g[k] = BatchGrid(self.a[k].ptr, self.b[k].ptr, x.shape[0], x.shape[1], radii[k], nv)
        h = C.c_void_p()
        call("msl_batch_create", g, len(arrays), C.byref(h))
        self.handle = h.value

    def run(self, iters):
        inb = C.c_int()
        call("msl_batch_run", self.handle, iters, self.sums.ptr, C.byref(inb))
        return [x.to_host() for x in (self.b if inb.value else self.a)], self.sums.to_host()

    def close(self):
        call("msl_batch_destroy", self.handle)


@pytest.mark.parametrize("iters", [3, 6])
def test_fold_of_tile_grids_keeps_its_precision(iters):
    """Constant grids: every addition of a lane rounds the same way, so an
    error of the correction term adds up."""
    hip.init(0)
    shapes = [(30000, 190), (4096, 1), (4097, 1), (63, 65), (1, 3), (333, 41)]
    radii = [3, 1, 8, 2, 5, 7]
    print(f"[case] batch fold precision x{iters}", flush=True)
    b = Grids([np.full(s, 0.1, np.float32) for s in shapes], radii, 0.1)
    states, sums = b.run(iters)
    b.close()
    for x, s, shape in zip(states, sums, shapes):
        ref = float(np.sum(x.astype(np.float64)))
        assert abs(s - ref) <= FOLD_TOL * float(np.sum(np.abs(x.astype(np.float64)))), (shape, s, ref)
