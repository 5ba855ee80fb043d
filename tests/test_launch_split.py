"""Launches of kernels whose grid grows with the data: split where one launch
would take 2^32 threads or more.  The arithmetic on the CPU; on the GPU every such
kernel in several launches (a lowered bound, read once per process), bit for bit."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from muesli4_amd import hip
from muesli4_amd.hip import call

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _split(blocks, threads):
    n, most = C.c_int(), C.c_int64()
    call("msl_selftest_launch_split", blocks, threads, C.byref(n), C.byref(most))
    return n.value, most.value


# 11.4 million blur tiles: a job of 10^9 rows of one column, r = 10; 10.4
# million: 5 * 10^8 rows of four, r = 2; 1.25 * 10^8 waves: 10^9 x 2 cells of Life.
@pytest.mark.parametrize("blocks,threads,launches", [
    (0, 512, 0), (1, 1024, 1), (11363637, 512, 2), (10416667, 512, 2), (125000000, 64, 2), (8388607, 512, 1), (8388608, 512, 2),
    (67108863, 64, 1), (67108864, 64, 2), (4194303, 1024, 1), (2**31 - 1, 1024, 513)])
def test_launches_stay_below_the_thread_limit(blocks, threads, launches):
    n, most = _split(blocks, threads)
    assert n == launches and most < 2**32
    assert most == min(blocks, (2**32 - 1) // threads) * threads


def test_more_workgroups_than_an_int_holds_are_refused():
    with pytest.raises(hip.MslError):
        _split(2**31, 64)


KERNELS = r"""
import ctypes as C
import numpy as np
from muesli4_amd import hip
from muesli4_amd.batch import BatchArena
from muesli4_amd.hip import DeviceArray, call
from muesli4_amd.serve import Server
from oracle import refcpu as R
hip.init(0)
inb = C.c_int()

def check(name, got, want):
    print("[case]", name, flush=True)
    np.testing.assert_array_equal(got, want, err_msg=name)

for r, shape in ((1, (300, 500)), (1, (20000, 30)), (1, (27000, 104)), (3, (500, 517)), (10, (300, 200))):
    x = R.fill_uniform_f32(shape[0] * shape[1], r).reshape(shape)
    a, b = DeviceArray.from_host(x), DeviceArray(shape, np.float32)
    call("msl_stencil2d_mean_iterate_f32", a.ptr, b.ptr, *shape, r, 0.5, 7, C.byref(inb))
    for _ in range(7):
        x = R.stencil2d_mean_f32(x, r, 0.5)
    check(f"mean r={r} {shape}", b.to_host(), x)

for shape, iters in (((300, 500), 3), ((300, 500), 40), ((5000, 1), 9)):
    g = R.fill_bernoulli_i32(shape[0] * shape[1], 3).reshape(shape)
    a, b = DeviceArray.from_host(g), DeviceArray(shape, np.int32)
    call("msl_gol_iterate_i32", a.ptr, b.ptr, *shape, iters, C.byref(inb))
    for _ in range(iters):
        g = R.gol_i32(g)
    check(f"gol {shape} x{iters}", (b if inb.value else a).to_host(), g)

batch = BatchArena([200, 90, 333], [100, 60, 190], [3, 1, 8], nv=0.5, seed=4)
init = batch.state("a")
batch.run(6)
out = batch.state("a")
for g in range(3):
    x = batch.grid(init, g)
    for _ in range(6):
        x = R.stencil2d_mean_f32(x, int(batch.radii[g]), 0.5)
    check(f"batch grid {g}", batch.grid(out, g), x)
batch.close()

srv = Server(1 << 28, 16)
jobs = [dict(kind=1, d0=500, d1=300, r=4, steps=9, seed=5, nv=0.5), dict(kind=2, d0=70, d1=50, d2=40, steps=5, seed=6, nv=0.25)]
ids = [srv.submit(d, keep_final=True) for d in jobs]
srv.drain()
x = R.fill_uniform_f32(500 * 300, 5).reshape(500, 300)
for _ in range(9):
    x = R.stencil2d_mean_f32(x, 4, 0.5)
check("served blur", srv.poll(ids[0], jobs[0])["final"], x)
h = R.fill_uniform_f32(70 * 50 * 40, 6, R.SCALE_UNIT).reshape(40, 50, 70)
for _ in range(5):
    h = R.heat7_f32(h, 0.25)
check("served heat", srv.poll(ids[1], jobs[1])["final"], h)
srv.close()
"""


@pytest.mark.gpu
@pytest.mark.parametrize("threads", ["1", "2500", "20000"])
def test_kernels_in_several_launches(threads):
    print(f"[case] at most {threads} threads a launch", flush=True)
    res = subprocess.run([sys.executable, "-c", KERNELS], cwd=ROOT, env={**os.environ, "MSL_LAUNCH_THREADS": threads},
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert res.returncode == 0, res.stdout
