"""Narrow grids of a batch in LDS tiles: which grids run there, and folds as
exact as those of the strip items, whatever the grid's size."""
import ctypes as C

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.hip import BatchGrid, DeviceArray, call
from oracle import refcpu as R

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

    def rounds(self, iters):
        n = C.c_int()
        call("msl_batch_run_plan", self.handle, iters, 1, C.byref(n), None, None, None)
        return n.value

    def set_columns(self, c):
        for r in range(1, 11):
            for wc in range(4):
                call("msl_batch_set_tile", self.handle, r, wc, c, 64)

    def close(self):
        call("msl_batch_destroy", self.handle)


def _uniform(shapes, seed=3):
    return [R.fill_uniform_f32(s[0] * s[1], seed + k).reshape(s) for k, s in enumerate(shapes)]


def _oracle(x, r, nv, iters):
    for _ in range(iters):
        x = R.stencil2d_mean_f32(x, r, nv)
    return x


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


def test_narrow_grids_run_in_tiles_whatever_their_strips(tmp_path):
    """The columns per lane of a narrow class shape its one-generation rounds
    only, also when they come from a saved table."""
    print("[case] batch narrow grids with either strip width", flush=True)
    hip.init(0)
    shapes, radii, iters = [(70, 40), (33, 95), (120, 100), (65, 191), (9, 5)], [1, 2, 4, 3, 5], 12
    grids = _uniform(shapes)
    b = Grids(grids, radii, 0.5)
    rounds = b.rounds(iters)
    assert rounds == 4  # three generations a round at r = 2..5 (in strips: six pairs)
    for c in (1, 4):
        b.set_columns(c)
        assert b.rounds(iters) == rounds
    table = tmp_path / "tiles.txt"
    n = C.c_int()
    call("msl_batch_autotune", b.handle, str(table).encode(), C.byref(n))
    assert n.value == len(radii)
    lines = [ln.split() for ln in table.read_text().splitlines()]
    for ln in lines:
        if ln[0] == "tile":
            ln[3] = "4"
    table.write_text("".join(" ".join(ln) + "\n" for ln in lines))
    call("msl_batch_autotune", b.handle, str(table).encode(), C.byref(n))
    assert n.value < 0  # loaded
    assert b.rounds(iters) == rounds
    states, _ = b.run(iters)
    b.close()
    for x, got, r in zip(grids, states, radii):
        np.testing.assert_array_equal(got, _oracle(x, r, 0.5, iters), err_msg=f"r={r}")


@pytest.mark.parametrize("iters", [8, 11, 12])
def test_tiles_of_every_generation_count(iters):
    """Rounds of six generations at r = 1 (12 steps), four at r = 2 and 3 (8),
    three at r = 4 and 5, two above; widths at the edges of both tile widths."""
    print(f"[case] batch tiles x{iters}", flush=True)
    hip.init(0)
    widths = [1, 3, 5, 28, 29, 52, 53, 96, 97, 116, 117, 191]
    shapes = [(40 + 13 * (k % 5), w) for k, w in enumerate(widths)]
    for r in range(1, 9):
        grids = _uniform(shapes, seed=10 * r)
        b = Grids(grids, [r] * len(shapes), 2.5)
        states, sums = b.run(iters)
        b.close()
        for x, got, s in zip(grids, states, sums):
            want = _oracle(x, r, 2.5, iters)
            np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32), err_msg=f"r={r} {x.shape}")
            ref = want.astype(np.float64)
            assert abs(s - np.sum(ref)) <= FOLD_TOL * np.sum(np.abs(ref)), (r, x.shape)


@pytest.mark.parametrize("nv", [0.0, -0.0, np.inf, np.nan])
def test_tiles_with_special_values(nv):
    print(f"[case] batch tiles, special values, nv={nv}", flush=True)
    hip.init(0)
    rng = np.random.default_rng(3)
    grids, radii = [], []
    for r in range(1, 9):
        for v in (np.inf, -np.inf, np.nan, np.finfo(np.float32).max, 2.0**-149):
            x = rng.uniform(-1.0, 1.0, (60, 70)).astype(np.float32)
            x[rng.integers(0, 60, 4), rng.integers(0, 70, 4)] = v
            grids.append(x)
            radii.append(r)
        grids.append(np.full((60, 70), -0.0, np.float32))
        radii.append(r)
    b = Grids(grids, radii, nv)
    states, _ = b.run(4)
    b.close()
    for x, got, r in zip(grids, states, radii):
        want = _oracle(x, r, nv, 4)
        np.testing.assert_array_equal(got, want, err_msg=f"r={r}")
        keep = ~np.isnan(want)
        np.testing.assert_array_equal(got.view(np.uint32)[keep], want.view(np.uint32)[keep], err_msg=f"r={r}")
