"""Measured cases of the skeleton library: what a program that uses it does.

Each case is one pass through the C ABI (muesli4_amd.hip.call, declared in
include/msl_hip.h) or through the serving front end, on device buffers that
the program holds.  Kinds:

  da     containers of floats or uint32: map, zip, mapIndex, fold, one call
         after the other, each result kept (the small one is bound by launches
         and the fold's way to the host, the large one by HBM)
  blur1  one mean-blur mapStencil call on an image
  blur   `iters` ping-pong mean-blur iterations on one grid
  gol    `iters` Game of Life generations and the count of live cells
  heat   `iters` 7-point heat steps on a cube with a residual every `every`
  batch  `iters` mean-blur steps on many grids of different shapes and radii,
         with a fold of each
  serve  a queue of blur, heat and map+fold jobs, all there at the start,
         run to the end by the serving engine
"""
import ctypes as C
import math

import numpy as np
import torch

from muesli4_amd import hip
from muesli4_amd.hip import BatchGrid, call
from muesli4_amd.serve import Server
from muesli4_amd.workloads import JOB_BLUR2D, JOB_HEAT3D, arena_offsets, batch_shapes, serve_trace

SERVE_BUDGET = 16 << 30


def listed():
    return [
        # a small container: three calls and a scalar back on the host
        {"name": "da_small", "kind": "da", "dtype": "f32", "rows": 1, "cols": 10007},
        # the benchmark's matrix: 8192 x 8192 floats
        {"name": "dm_8192", "kind": "da", "dtype": "f32", "rows": 8192, "cols": 8192},
        # one filter call on an image of odd width
        {"name": "blur1_photo_r7", "kind": "blur1", "rows": 1201, "cols": 1999, "r": 7, "nv": 0.0},
        # a small grid iterated: many short launches
        {"name": "blur_small_r3", "kind": "blur", "rows": 500, "cols": 517, "r": 3, "nv": 0.0, "iters": 20},
        # a grid that fits the caches, the widest radius of the benchmark
        {"name": "blur_2048_r10", "kind": "blur", "rows": 2048, "cols": 2048, "r": 10, "nv": 0.0, "iters": 20},
        # the benchmark's headline: 8192 x 8192, radii 1, 5 and 10, 20 iterations each
        {"name": "blur_8192_r1", "kind": "blur", "rows": 8192, "cols": 8192, "r": 1, "nv": 0.0, "iters": 20},
        {"name": "blur_8192_r5", "kind": "blur", "rows": 8192, "cols": 8192, "r": 5, "nv": 0.0, "iters": 20},
        {"name": "blur_8192_r10", "kind": "blur", "rows": 8192, "cols": 8192, "r": 10, "nv": 0.0, "iters": 20},
        # the benchmark's Game of Life
        {"name": "gol_1024", "kind": "gol", "rows": 1024, "cols": 1024, "iters": 100},
        # the benchmark's heat run
        {"name": "heat_512", "kind": "heat", "nx": 512, "ny": 512, "nz": 512, "nv": 0.0, "iters": 200, "every": 10},
        # the benchmark's batch: 4096 grids, 10 steps, a fold of each
        {"name": "batch_4096", "kind": "batch", "shapes": 2024, "grids": 4096, "iters": 10},
        # a queue of the benchmark's job mix
        {"name": "serve_128", "kind": "serve", "trace": 2025, "jobs": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["da", "blur1", "blur", "blur", "gol", "heat", "batch", "serve"])
    if kind == "da":
        return {"kind": kind, "dtype": rng.choice(["f32", "u32"]), "rows": _log(rng, 1, 8192), "cols": _log(rng, 1000, 8192)}
    if kind in ("blur1", "blur"):
        c = {"kind": kind, "rows": _log(rng, 64, 8192), "cols": _log(rng, 64, 8192), "r": rng.randint(1, 10),
             "nv": rng.choice([0.0, 0.0, 127.5])}
        if kind == "blur":
            c["iters"] = rng.randint(2, 20)
        return c
    if kind == "gol":
        return {"kind": kind, "rows": _log(rng, 64, 4096), "cols": _log(rng, 64, 4096), "iters": rng.randint(10, 100)}
    if kind == "heat":
        return {"kind": kind, "nx": _log(rng, 32, 512), "ny": _log(rng, 32, 512), "nz": _log(rng, 32, 512),
                "nv": rng.choice([0.0, 0.25]), "iters": rng.randint(10, 200), "every": rng.choice([0, 10])}
    if kind == "batch":
        return {"kind": kind, "shapes": rng.randrange(1 << 20), "grids": _log(rng, 64, 4096),
                "iters": 2 * rng.randint(1, 5)}
    return {"kind": kind, "trace": rng.randrange(1 << 20), "jobs": _log(rng, 4, 128)}


# ---- inputs ---------------------------------------------------------------
def _uniform(shape, seed, scale):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * scale


def _bits(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(-(1 << 31), 1 << 31, (n,), generator=g, device="cuda", dtype=torch.int32)


def _inputs(case, seed):
    """The program's data: tensors on the GPU, made from the seed."""
    kind = case["kind"]
    if kind == "da":
        n = case["rows"] * case["cols"]
        if case["dtype"] == "u32":
            return {"a": _bits(n, seed)}
        return {"a": _uniform(n, seed, 255.0), "b": _uniform(n, seed + 7919, 255.0)}
    if kind in ("blur1", "blur"):
        return {"a": _uniform((case["rows"], case["cols"]), seed, 255.0)}
    if kind == "gol":
        return {"a": (_uniform((case["rows"], case["cols"]), seed, 1.0) < 0.3).to(torch.int32)}
    if kind == "heat":
        return {"a": _uniform((case["nz"], case["ny"], case["nx"]), seed, 1.0)}
    if kind == "batch":
        rows, cols, radii = batch_shapes(case["grids"], case["shapes"])
        offsets, total = arena_offsets(rows, cols)
        return {"a": _uniform(total, seed, 255.0), "rows": rows, "cols": cols, "radii": radii, "offsets": offsets}
    jobs, arrivals = serve_trace(case["jobs"], case["trace"], 0.0)
    for j in jobs:  # the trace gives the shapes, the seed the states
        j["seed"] = (j["seed"] + seed) % (1 << 64)
    return {"jobs": jobs, "arrivals": arrivals}


class _Batch:
    """Handle of a batch over two arenas (state a and state b)."""

    def __init__(self, s):
        grids = (BatchGrid * len(s["rows"]))()
        for g in range(len(s["rows"])):
            off = 4 * int(s["offsets"][g])
            grids[g] = BatchGrid(s["a"].data_ptr() + off, s["b"].data_ptr() + off, int(s["rows"][g]),
                                 int(s["cols"][g]), int(s["radii"][g]), 0.0)
        h = C.c_void_p()
        call("msl_batch_create", grids, len(grids), C.byref(h))
        self.handle = h.value
        self.keep = (s["a"], s["b"])

    def __del__(self):
        if getattr(self, "handle", None):
            hip.lib().msl_batch_destroy(self.handle)
            self.handle = None


def prepare(case, seed):
    hip.init(0)
    s = dict(_inputs(case, seed), case=case)
    kind = case["kind"]
    if kind == "da":
        s["m"] = torch.empty_like(s["a"])
        if case["dtype"] == "f32":
            s["z"], s["i"] = torch.empty_like(s["a"]), torch.empty_like(s["a"])
    elif kind == "serve":
        s["server"] = Server(SERVE_BUDGET, 1024)
    else:
        s["b"] = torch.zeros_like(s["a"])
    if kind == "batch":
        s["sums"] = torch.zeros(case["grids"], device="cuda", dtype=torch.float64)
        s["batch"] = _Batch(s)
    torch.cuda.synchronize()
    return s


# ---- one pass -------------------------------------------------------------
def _result(s, in_b):
    """The grid that holds the result; the next pass goes on from it."""
    if in_b:
        s["a"], s["b"] = s["b"], s["a"]
    return s["a"]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "da":
        n = case["rows"] * case["cols"]
        if case["dtype"] == "u32":
            u = C.c_uint32()
            call("msl_map_affine_u32", s["m"].data_ptr(), s["a"].data_ptr(), n, 3, 1)
            call("msl_fold_sum_u32_host", s["m"].data_ptr(), n, C.byref(u))
            return {"map": s["m"], "sum": u.value}
        total, top = C.c_double(), C.c_float()
        call("msl_map_affine_f32", s["m"].data_ptr(), s["a"].data_ptr(), n, 1.5, 3.0)
        call("msl_zip_add_f32", s["z"].data_ptr(), s["m"].data_ptr(), s["b"].data_ptr(), n)
        call("msl_mapindex_lin_f32", s["i"].data_ptr(), case["rows"], case["cols"])
        call("msl_fold_sum_f32_host", s["z"].data_ptr(), n, C.byref(total), None)
        call("msl_fold_max_f32_host", s["z"].data_ptr(), n, C.byref(top))
        return {"map": s["m"], "zip": s["z"], "index": s["i"], "sum": total.value, "max": np.float32(top.value)}
    if kind == "blur1":
        call("msl_stencil2d_mean_f32", s["b"].data_ptr(), s["a"].data_ptr(), case["rows"], case["cols"], case["r"],
             case["nv"])
        return s["b"]
    in_b = C.c_int()
    if kind == "blur":
        call("msl_stencil2d_mean_iterate_f32", s["a"].data_ptr(), s["b"].data_ptr(), case["rows"], case["cols"],
             case["r"], case["nv"], case["iters"], C.byref(in_b))
        return _result(s, in_b.value)
    if kind == "gol":
        live = C.c_int64()
        call("msl_gol_iterate_i32", s["a"].data_ptr(), s["b"].data_ptr(), case["rows"], case["cols"], case["iters"],
             C.byref(in_b))
        grid = _result(s, in_b.value)
        call("msl_fold_sum_i32_host", grid.data_ptr(), case["rows"] * case["cols"], C.byref(live))
        return {"grid": grid, "live": live.value}
    if kind == "heat":
        res = np.zeros(case["iters"] // case["every"] if case["every"] else 0, np.float32)
        call("msl_heat7_iterate_f32", s["a"].data_ptr(), s["b"].data_ptr(), case["nx"], case["ny"], case["nz"],
             case["nv"], case["iters"], case["every"],
             res.ctypes.data_as(C.POINTER(C.c_float)) if len(res) else None, C.byref(in_b))
        grid = _result(s, in_b.value)
        return {"grid": grid, "residuals": res} if len(res) else {"grid": grid}
    if kind == "batch":
        # the batch is bound to its arenas: with an even count the next pass goes on from state a
        call("msl_batch_run", s["batch"].handle, case["iters"], s["sums"].data_ptr(), C.byref(in_b))
        return {"states": s["b"] if in_b.value else s["a"], "sums": s["sums"]}
    res = s["server"].run_trace(s["jobs"], s["arrivals"])
    return {"sum": np.array([r["sum"] for r in res], np.float64),
            "sum_u32": np.array([r["sum_u32"] for r in res], np.int64)}


# ---- the same in 64 bits --------------------------------------------------
def _mean64(x, r, nv):
    """One mean-blur step of a 2-D float64 tensor."""
    p = torch.nn.functional.pad(x, (r, r, r, r), value=nv)
    h = p[:, :x.shape[1]].clone()
    for d in range(1, 2 * r + 1):
        h += p[:, d:d + x.shape[1]]
    v = h[:x.shape[0]].clone()
    for d in range(1, 2 * r + 1):
        v += h[d:d + x.shape[0]]
    return v.div_((2 * r + 1) ** 2)


def _heat64(x, nv):
    """One 7-point heat step of a float64 cube (z, y, x)."""
    p = torch.nn.functional.pad(x, (1, 1, 1, 1, 1, 1), value=nv)
    v = p[1:-1, 1:-1, :-2] + p[1:-1, 1:-1, 2:]
    for q in (p[1:-1, :-2, 1:-1], p[1:-1, 2:, 1:-1], p[:-2, 1:-1, 1:-1], p[2:, 1:-1, 1:-1]):
        v += q
    return v.div_(6.0)


def _s64(v):
    return v - (1 << 64) if v >> 63 else v


def _hash64(seed, n):
    """SplitMix64 of (seed, 0 .. n-1), the generator of served jobs' states (int64 bit patterns)."""
    def shr(z, k):
        return (z >> k) & ((1 << (64 - k)) - 1)
    z = torch.arange(1, n + 1, device="cuda", dtype=torch.int64) * _s64(0x9E3779B97F4A7C15) + _s64(seed)
    z = (z ^ shr(z, 30)) * _s64(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * _s64(0x94D049BB133111EB)
    return z ^ shr(z, 31)


def _served64(job):
    """(sum, wrapping sum) of a served job."""
    if job["kind"] not in (JOB_BLUR2D, JOB_HEAT3D):
        v = ((_hash64(job["seed"], job["n"]) >> 32) & 0xFFFFFFFF) * job["mul"] + job["add"]
        return 0.0, int((v & 0xFFFFFFFF).sum()) & 0xFFFFFFFF
    blur = job["kind"] == JOB_BLUR2D
    shape = (job["d0"], job["d1"]) if blur else (job["d2"], job["d1"], job["d0"])
    scale = np.float32(255.0 / 16777216.0) if blur else np.float32(1.0 / 16777216.0)
    u = (_hash64(job["seed"], math.prod(shape)) >> 40) & 0xFFFFFF
    x = (u.to(torch.float32) * float(scale)).double().view(shape)
    for _ in range(job["steps"]):
        x = _mean64(x, job["r"], 0.0) if blur else _heat64(x, 0.0)
    return float(x.sum()), 0


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "da":
        if case["dtype"] == "u32":
            m = (s["a"].to(torch.int64) * 3 + 1) & 0xFFFFFFFF
            return {"map": torch.where(m >= 1 << 31, m - (1 << 32), m), "sum": int(m.sum()) & 0xFFFFFFFF}
        m = s["a"].double() * 1.5 + 3.0
        z = m + s["b"].double()
        return {"map": m, "zip": z, "index": torch.arange(z.numel(), device="cuda", dtype=torch.float64),
                "sum": float(z.sum()), "max": np.float64(float(z.max()))}
    if kind in ("blur1", "blur"):
        x = s["a"].double()
        for _ in range(case.get("iters", 1)):
            x = _mean64(x, case["r"], case["nv"])
        return x
    if kind == "gol":
        return None  # whole numbers: they stay equal
    if kind == "heat":
        x, res = s["a"].double(), []
        for k in range(1, case["iters"] + 1):
            y = _heat64(x, case["nv"])
            if case["every"] and k % case["every"] == 0:
                res.append(float((y - x).abs().max()))
            x = y
        return {"grid": x, "residuals": np.array(res, np.float64)} if res else {"grid": x}
    if kind == "batch":
        out = torch.zeros(s["a"].numel(), device="cuda", dtype=torch.float64)
        if case["iters"] % 2 == 0:
            out.copy_(s["a"])  # the gaps between the grids keep what state a held
        sums = []
        for g in range(case["grids"]):
            rows, cols, off = int(s["rows"][g]), int(s["cols"][g]), int(s["offsets"][g])
            x = s["a"][off:off + rows * cols].view(rows, cols).double()
            for _ in range(case["iters"]):
                x = _mean64(x, int(s["radii"][g]), 0.0)
            out[off:off + rows * cols] = x.reshape(-1)
            sums.append(x.sum())
        return {"states": out, "sums": torch.stack(sums)}
    got = [_served64(j) for j in s["jobs"]]
    return {"sum": np.array([g[0] for g in got], np.float64), "sum_u32": np.array([g[1] for g in got], np.int64)}


# ---- what one pass cannot do without --------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "da":
        n = case["rows"] * case["cols"]
        if case["dtype"] == "u32":
            return {"bytes": 12 * n, "flops": 3 * n}  # map 8, fold 4
        return {"bytes": 32 * n, "flops": 6 * n}  # map 8, zip 12, mapIndex 4, two folds 4 each
    if kind in ("blur1", "blur"):
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n, "flops": case.get("iters", 1) * n * (2 * (2 * case["r"] + 1) - 1)}
    if kind == "gol":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n, "flops": 8 * n * case["iters"]}
    if kind == "heat":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 8 * n, "flops": 6 * n * case["iters"]}
    if kind == "batch":
        rows, cols, radii = batch_shapes(case["grids"], case["shapes"])
        n = rows * cols
        return {"bytes": int(8 * n.sum()), "flops": int(case["iters"] * (n * (4 * radii + 1)).sum() + n.sum())}
    total_bytes = flops = 0
    for j in serve_trace(case["jobs"], case["trace"], 0.0)[0]:
        if j["kind"] == JOB_BLUR2D:
            n = j["d0"] * j["d1"]
            flops += j["steps"] * n * (4 * j["r"] + 1)
        elif j["kind"] == JOB_HEAT3D:
            n = j["d0"] * j["d1"] * j["d2"]
            flops += j["steps"] * n * 6
        else:
            n = j["n"]
            flops += 3 * n
        total_bytes += 4 * n
    return {"bytes": total_bytes, "flops": flops}
