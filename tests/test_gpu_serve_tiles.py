"""Served blur jobs in the tiles for load (128 columns) and for light load (64):
final states bit-identical to the oracle and to the same job alone, with the
tiling that ran asserted."""
import math

import numpy as np
import pytest

from muesli4_amd import hip
from muesli4_amd.serve import Server
from muesli4_amd.workloads import JOB_BLUR2D, JOB_HEAT3D
from oracle import refcpu as R

pytestmark = pytest.mark.gpu

# A lane adds 128 cells of a chunk to its compensated pair and six merges
# follow: the correction term is off by at most (n u)^2 of the sum.
FOLD_TOL = (134 * 2.0**-24) ** 2


def _serve(jobs):
    srv = Server(1 << 30, 64)
    ids = [srv.submit(d, keep_final=True) for d in jobs]
    srv.drain()
    out = [srv.poll(i, d) for i, d in zip(ids, jobs)]
    rounds = srv.blur_rounds()
    srv.close()
    return out, rounds


def _blur(rows, cols, r, steps, seed, nv):
    return dict(kind=JOB_BLUR2D, d0=rows, d1=cols, r=r, steps=steps, seed=seed, nv=nv)


def _oracle(d):
    x = R.fill_uniform_f32(d["d0"] * d["d1"], d["seed"]).reshape(d["d0"], d["d1"])
    for _ in range(d["steps"]):
        x = R.stencil2d_mean_f32(x, d["r"], d["nv"])
    return x


def _check(d, res):
    want = _oracle(d)
    np.testing.assert_array_equal(res["final"], want, err_msg=str(d))
    ref = math.fsum(want.astype(np.float64).ravel())
    if math.isfinite(ref):
        assert abs(res["sum"] - ref) <= FOLD_TOL * ref, (d, res["sum"], ref)


# Step counts that leave a short last launch (and a single step): under load a
# job takes 6, 4, 4, 3, 3, 2, ... generations per launch by its radius.
@pytest.mark.parametrize("r", range(1, 11))
def test_job_under_load_equals_oracle_and_alone(r):
    print(f"[case] served blur r={r} under load", flush=True)
    hip.init(0)
    job = _blur(301, 517, r, 11, 40 + r, 0.5)
    others = [_blur(1400, 1300, 1 + (r + 3 * k) % 10, 13, 60 + k, 0.0) for k in range(2)]
    mix, rounds = _serve(others + [job, _blur(33, 120, r, 1, 7, 2.5)])
    assert rounds["loaded"] >= 1
    alone, rounds = _serve([job])
    assert rounds["loaded"] == 0 and rounds["light"] >= 1
    _check(job, mix[2])
    _check(_blur(33, 120, r, 1, 7, 2.5), mix[3])
    np.testing.assert_array_equal(alone[0]["final"], mix[2]["final"])
    assert alone[0]["sum"] == mix[2]["sum"]
    if r in (1, 6):
        for d, res in zip(others, mix):
            _check(d, res)


@pytest.mark.parametrize("nv", [-0.0, np.inf, -np.inf, np.nan])
def test_neutral_values_that_are_no_ordinary_number(nv):
    print(f"[case] served jobs nv={nv}", flush=True)
    hip.init(0)
    jobs = [_blur(97, 130, r, 7, r, nv) for r in range(1, 11)] + [_blur(1500, 1400, 4, 7, 77, nv)] * 2
    heat = dict(kind=JOB_HEAT3D, d0=70, d1=33, d2=20, steps=5, seed=3, nv=nv)
    out, rounds = _serve(jobs + [heat])
    assert rounds["loaded"] >= 1
    for d, res in zip(jobs, out):
        _check(d, res)
    x = R.fill_uniform_f32(70 * 33 * 20, 3, R.SCALE_UNIT).reshape(20, 33, 70)
    for _ in range(5):
        x = R.heat7_f32(x, nv)
    np.testing.assert_array_equal(out[-1]["final"], x)
