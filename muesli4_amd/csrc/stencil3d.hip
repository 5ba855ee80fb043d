// 3-D 7-point heat step on an nx x ny x nz cube (x fastest).
//
// Reference: DC::mapStencil<heat3D> runs one thread per cell with seven
// bounds-checked reads through PLCube::operator() and no reuse
// (include/detail/map_kernels.cuh:140-149, include/plcube.h:105-119,
// functor examples/heatdiffusion.cpp:55-65).
//
// Here one wavefront owns a 64 x 8 column of the cube and marches a segment
// of z-planes with all neighbours in registers (heat7_march): each cell is
// read from HBM once and written once (8 bytes per cell per step), in the
// reference functor's operation order.  Small cubes and iterations run other
// kernels (heat_tile.hip, heat_pair.hip; see heat_way).  The optional fused residual folds
// max |v - in| into one device scalar with an integer atomic max (the bit
// patterns of non-negative floats order like unsigned integers).
#include <cstdlib>
#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "heat.hpp"
#include "heat_tile.hpp"

namespace mslhip {

// One wave per (64 x kTY column tile, z-segment), or per kT2X x kT2Y tile of
// two generations (kPair); four independent waves per workgroup, no LDS and no
// barrier.
template <bool kPair, bool kResidual, bool NT>
__global__ __launch_bounds__(256) void heat7_kernel(float *__restrict__ out, const float *__restrict__ in, int nx,
                                                    int ny, int nz, float nv, int zseg, int xtiles, int ytiles,
                                                    int nitems, float *__restrict__ maxdiff) {
    const int lane = threadIdx.x & 63;
    const int item = __builtin_amdgcn_readfirstlane((int)xcd_tile(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6));
    float dmax = 0.0f;
    if (item < nitems) {
        const int xt = item % xtiles;
        const int rest = item / xtiles;
        const int yt = rest % ytiles;
        const int zs = rest / ytiles;
        const int z0 = zs * zseg;
        const int z1 = min(z0 + zseg, nz);
        if constexpr (kPair)
            heat7x2_march<false, true, kResidual, NT>(out, in, nx, ny, nz, nv, xt * kT2X, yt * kT2Y, z0, z1, &dmax);
        else
            heat7_march<kResidual, NT>(out, in, nx, ny, nz, nv, xt * kTX, yt * kTY, z0, z1, &dmax);
    }
    if (kResidual) {
        __shared__ float wmax[4];
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            const float o = __shfl_xor(dmax, m);
            dmax = o > dmax ? o : dmax;
        }
        if (lane == 0) wmax[threadIdx.x >> 6] = dmax;
        __syncthreads();
        if (threadIdx.x == 0) {
            const float m = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
            atomicMax(reinterpret_cast<unsigned int *>(maxdiff), __float_as_uint(m));
        }
    }
}

struct HeatShape {
    int zseg, xtiles, ytiles, zsegs, nitems;
};

inline HeatShape heat_shape(int nx, int ny, int nz, bool pair) {
    HeatShape s;
    s.xtiles = (nx + kTX - 1) / kTX;
    s.ytiles = (ny + kTY - 1) / kTY;
    const long cols = (long)s.xtiles * s.ytiles;
    const long target = (long)ctx().num_cus * 32;  // waves wanted
    long zsegs = (target + cols - 1) / cols;
    if (zsegs < 1) zsegs = 1;
    int zseg = (int)((nz + zsegs - 1) / zsegs);
    zseg = (zseg + kP - 1) / kP * kP;  // whole blocks of the plane ring
    if (zseg < 16) zseg = 16;
    if (int z = tune_int("MSL_HEAT_ZSEG", 0)) zseg = z;
    s.zseg = zseg;
    s.zsegs = (nz + zseg - 1) / zseg;
    if (pair) {
        s.xtiles = (nx + kT2X - 1) / kT2X;
        s.ytiles = (ny + kT2Y - 1) / kT2Y;
    }
    s.nitems = s.xtiles * s.ytiles * s.zsegs;
    return s;
}

template <bool kPair>
static int launch_heat_march(float *out, const float *in, int nx, int ny, int nz, float nv, float *maxdiff) {
    const HeatShape s = heat_shape(nx, ny, nz, kPair);
    const bool nt = stream_stores((size_t)nx * ny * nz * sizeof(float));
    const int blocks = (s.nitems + 3) / 4;
    if (maxdiff && nt)
        heat7_kernel<kPair, true, true><<<blocks, 256, 0, ctx().stream>>>(out, in, nx, ny, nz, nv, s.zseg, s.xtiles,
                                                                          s.ytiles, s.nitems, maxdiff);
    else if (maxdiff)
        heat7_kernel<kPair, true, false><<<blocks, 256, 0, ctx().stream>>>(out, in, nx, ny, nz, nv, s.zseg, s.xtiles,
                                                                           s.ytiles, s.nitems, maxdiff);
    else if (nt)
        heat7_kernel<kPair, false, true><<<blocks, 256, 0, ctx().stream>>>(out, in, nx, ny, nz, nv, s.zseg, s.xtiles,
                                                                           s.ytiles, s.nitems, nullptr);
    else
        heat7_kernel<kPair, false, false><<<blocks, 256, 0, ctx().stream>>>(out, in, nx, ny, nz, nv, s.zseg, s.xtiles,
                                                                            s.ytiles, s.nitems, nullptr);
    return check_launch("msl_heat7_f32");
}

// Times of a launch in us, fitted to 340 cubes of 0.2 to 4.2 million cells with
// an extent of 1 to 24 (both within 12 % on average): a tile costs the same
// however few of its planes or rows lie in the cube, the march only the planes
// and rows that do.
static double heat_march_us(int nx, int ny, int nz) {
    const HeatShape s = heat_shape(nx, ny, nz, false);
    auto whole = [](int planes) { return (planes + kP - 1) / kP * kP; };
    const double chain = whole(std::min(s.zseg, nz));
    const double planes = (double)(s.zsegs - 1) * whole(s.zseg) + whole(nz - (s.zsegs - 1) * s.zseg);
    return 3.74 + std::max(0.566 * chain, 3.22e-4 * s.xtiles * s.ytiles * planes);
}
static double heat_tile_us(int nx, int ny, int nz, int gens, bool small, bool residual) {
    const double blocks = (double)heat_tile_blocks(nx, ny, nz, gens, small);
    const double each = (small ? 0.00582 : 0.0105) * (1.0 + 0.5 * (gens - 1)) + (residual ? (small ? 0.010 : 0.006) : 0.0);
    return (small ? 3.48 : 6.64) + each * blocks;
}

// How a cube's iterations run.  us per generation, one-step march / small
// tiles / large tiles / pair kernel: 32^3 12.5 / 1.6 / 3.0 / 5.1, 64^3 12.9 /
// 1.7 / 3.0 / 4.7, 80^3 13.1 / 2.7 / 3.3 / 4.8, 100^3 13.4 / 3.8 / 3.7 / 5.6,
// 128^3 14.1 / 5.2 / 5.4 / 5.4, 150^3 14.6 / 8.5 / 6.9 / 8.7, 200^3 17.8 / 14.9
// / 11.1 / 10.8, 256^3 22.6 / 27.6 / 18.4 / 14.0, 512^3 215 / 242 / 138 / 106
// (tiles at the generations per launch given here).
// Thin cubes leave most of a tile or of the pair kernel's planes empty: up to
// 4.2 million cells they march wherever that is modelled as faster (2000 x
// 2000 x 1, tiles / march: 47 / 15; 1000 x 1000 x 3 14 / 9), and larger ones run
// the march of one wave per tile, two generations per launch where the cube
// exceeds 64 MiB (pair kernel / that march, 25 million cells: 5000 x 1 x 5000
// 235 / 74, 2000 x 10 x 1250 33 / 29, 2000 x 12 x 1041 29 / 29; 16 x 300 x 5208 63 /
// 60, 32 x 300 x 2604 35 / 36; 2000 x 6250 x 2 36 / 31, 2000 x 3125 x 4 25 / 27).
enum HeatKernel { kHeatMarch, kHeatSmallTile, kHeatTile, kHeatPair, kHeatMarchPair };
struct HeatWay {
    int gens;  // most generations per launch
    HeatKernel kernel;
};
constexpr size_t kHeatTileCells = 4200000, kHeatSmallTileCells = 900000;
constexpr size_t kHeatMarchPairMinBytes = (size_t)64 << 20;

static HeatWay heat_way(int nx, int ny, int nz) {
    const size_t cells = (size_t)nx * ny * nz;
    if (cells <= kHeatTileCells) {
        const bool small = cells <= kHeatSmallTileCells;
        const int gens = cells <= 350000 ? 4 : 3;
        if (heat_tile_us(nx, ny, nz, gens, small, false) < gens * heat_march_us(nx, ny, nz))
            return HeatWay{gens, small ? kHeatSmallTile : kHeatTile};
        return HeatWay{1, kHeatMarch};
    }
    if (nx < 32 || ny <= 10 || nz <= 2)
        return cells * sizeof(float) > kHeatMarchPairMinBytes ? HeatWay{2, kHeatMarchPair} : HeatWay{1, kHeatMarch};
    return HeatWay{2, kHeatPair};
}

int heat_step(float *out, const float *in, int nx, int ny, int nz, float nv, float *maxdiff) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(nx >= 0 && ny >= 0 && nz >= 0, "msl_heat7_f32: negative shape");
    MSL_REQUIRE((int64_t)nx * ny * nz <= ((int64_t)1 << 40), "msl_heat7_f32: cube too large");
    MSL_REQUIRE((int64_t)nx * ny < ((int64_t)1 << 30), "msl_heat7_f32: plane of 2^30 cells or more");
    if (nx == 0 || ny == 0 || nz == 0) return MSL_OK;
    MSL_REQUIRE(out && in && out != in, "msl_heat7_f32: null or aliased buffers");
    const size_t cells = (size_t)nx * ny * nz;
    const bool small = cells <= kHeatSmallTileCells;
    if (cells <= kHeatTileCells &&
        1.05 * heat_tile_us(nx, ny, nz, 1, small, maxdiff != nullptr) < heat_march_us(nx, ny, nz))
        return heat_tile_step(out, in, nx, ny, nz, nv, 1, small, maxdiff);
    return launch_heat_march<false>(out, in, nx, ny, nz, nv, maxdiff);
}

// Small fill used instead of hipMemsetAsync so that captured graphs contain
// kernel nodes only.
__global__ void zero_f32_kernel(float *p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// Generations per launch of msl_heat7_iterate_f32, in launch order: the steps
// up to each residual are dealt evenly to as few launches as heat_way allows
// (a residual generation is the last of its launch; MSL_HEAT_GENS = 1 or 2
// forces that many at most, through the one-step or the pair kernel, read on
// every call so a process can compare both).  The number of launches must have
// the parity of iters (the result ends in b exactly when iters is odd, as with
// one launch per generation); when it does not, one launch is split in two.
static int heat_gens_env() {  // 0: not forced (unset, or any other value)
    const char *ge = getenv("MSL_HEAT_GENS");
    const int gens = ge ? atoi(ge) : 0;
    return gens == 1 || gens == 2 ? gens : 0;
}

static std::vector<int> heat_iterate_plan(int nx, int ny, int nz, int iters, int residual_every) {
    const int env = heat_gens_env();
    const int most = env ? env : heat_way(nx, ny, nz).gens;
    std::vector<int> plan;
    for (int it = 0; it < iters;) {
        int seg = iters - it;
        if (residual_every > 0) seg = std::min(seg, residual_every - it % residual_every);
        it += seg;
        for (int left = (seg + most - 1) / most; left > 0; left--) {
            plan.push_back((seg + left - 1) / left);
            seg -= plan.back();
        }
    }
    if ((int)(plan.size() & 1) != (iters & 1)) {
        for (size_t j = plan.size(); j-- > 0;)
            if (plan[j] >= 2) {
                const int first = plan[j] / 2;
                plan.insert(plan.begin() + j + 1, plan[j] - first);
                plan[j] = first;
                break;
            }
    }
    return plan;
}

struct HeatGraph {
    hipGraphExec_t exec = nullptr;
    float *d_res = nullptr;  // residual slots owned by this graph
};
struct HeatGraphs {
    std::mutex mu;
    std::map<std::string, HeatGraph> graphs;
};
static HeatGraphs g_heat_graphs;

}  // namespace mslhip

using namespace mslhip;

extern "C" {

int msl_heat7_f32(float *d_out, const float *d_in, int nx, int ny, int nz, float nv) {
    return heat_step(d_out, d_in, nx, ny, nz, nv, nullptr);
}

int msl_heat7_residual_f32(float *d_out, const float *d_in, int nx, int ny, int nz, float nv, float *d_maxdiff) {
    MSL_REQUIRE(d_maxdiff != nullptr, "msl_heat7_residual_f32: null residual pointer");
    return heat_step(d_out, d_in, nx, ny, nz, nv, d_maxdiff);
}

int msl_heat7_iterate_f32(float *d_a, float *d_b, int nx, int ny, int nz, float nv, int iters, int residual_every,
                          float *h_residuals, int *h_result_in_b) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(iters >= 0 && residual_every >= 0, "msl_heat7_iterate_f32: negative count");
    MSL_REQUIRE(nx >= 0 && ny >= 0 && nz >= 0, "msl_heat7_iterate_f32: negative shape");
    MSL_REQUIRE((int64_t)nx * ny < ((int64_t)1 << 30) && (int64_t)nx * ny * nz <= ((int64_t)1 << 40),
                "msl_heat7_iterate_f32: cube too large");
    const int nres = residual_every > 0 ? iters / residual_every : 0;
    MSL_REQUIRE(nres == 0 || h_residuals != nullptr, "msl_heat7_iterate_f32: residual output required");
    if (h_result_in_b) *h_result_in_b = iters & 1;
    if (iters == 0 || nx == 0 || ny == 0 || nz == 0) return MSL_OK;
    const int env = heat_gens_env();
    char keybuf[256];
    snprintf(keybuf, sizeof keybuf, "heat7|%p|%p|%d|%d|%d|%08x|%d|%d|%d", (void *)d_a, (void *)d_b, nx, ny, nz,
             __builtin_bit_cast(unsigned, nv), iters, residual_every, env);
    std::string key(keybuf);
    HeatGraph hg;
    {
        std::lock_guard<std::mutex> lock(g_heat_graphs.mu);
        auto it = g_heat_graphs.graphs.find(key);
        if (it != g_heat_graphs.graphs.end()) hg = it->second;
    }
    if (!hg.exec) {
        if (nres > 0) MSL_HIP_TRY(hipMalloc(&hg.d_res, (size_t)nres * sizeof(float)));
        float *d_res = hg.d_res;
        rc = msl_graph_begin();
        if (rc) {
            if (hg.d_res) hipFree(hg.d_res);
            return rc;
        }
        int brc = MSL_OK;
        if (nres > 0) {
            zero_f32_kernel<<<(nres + 255) / 256, 256, 0, ctx().stream>>>(d_res, nres);
            brc = check_launch("zero residuals");
        }
        auto is_res = [&](int it) { return residual_every > 0 && ((it + 1) % residual_every == 0); };
        const std::vector<int> plan = heat_iterate_plan(nx, ny, nz, iters, residual_every);
        const HeatKernel kernel = env ? kHeatPair : heat_way(nx, ny, nz).kernel;
        int k = 0, it = 0;
        for (size_t j = 0; j < plan.size() && brc == MSL_OK; j++) {
            float *src = (j & 1) ? d_b : d_a;
            float *dst = (j & 1) ? d_a : d_b;
            it += plan[j];
            const bool res = is_res(it - 1);
            float *maxdiff = res ? d_res + (k++) : nullptr;
            if (plan[j] == 1)
                brc = heat_step(dst, src, nx, ny, nz, nv, maxdiff);
            else if (kernel == kHeatPair)
                brc = heat_pair_step(dst, src, nx, ny, nz, nv, maxdiff);
            else if (kernel == kHeatMarchPair)
                brc = launch_heat_march<true>(dst, src, nx, ny, nz, nv, maxdiff);
            else
                brc = heat_tile_step(dst, src, nx, ny, nz, nv, plan[j], kernel == kHeatSmallTile, maxdiff);
        }
        void *g = nullptr;
        int erc = msl_graph_end(&g);
        if (brc || erc) {
            if (g) msl_graph_destroy(g);
            if (hg.d_res) hipFree(hg.d_res);
            return brc ? brc : erc;
        }
        hg.exec = (hipGraphExec_t)g;
        std::lock_guard<std::mutex> lock(g_heat_graphs.mu);
        if (g_heat_graphs.graphs.size() > 32) {
            hipStreamSynchronize(ctx().stream);
            for (auto &kv : g_heat_graphs.graphs) {
                hipGraphExecDestroy(kv.second.exec);
                if (kv.second.d_res) hipFree(kv.second.d_res);
            }
            g_heat_graphs.graphs.clear();
        }
        g_heat_graphs.graphs[key] = hg;
    }
    hipGraphExec_t exec = hg.exec;
    float *d_res = hg.d_res;
    MSL_HIP_TRY(hipGraphLaunch(exec, ctx().stream));
    if (nres > 0) {
        MSL_HIP_TRY(hipMemcpyAsync(h_residuals, d_res, (size_t)nres * sizeof(float), hipMemcpyDeviceToHost,
                                   ctx().stream));
        MSL_HIP_TRY(hipStreamSynchronize(ctx().stream));
    }
    return MSL_OK;
}

int msl_heat7_iterate_plan(int nx, int ny, int nz, int iters, int residual_every, int *h_gens, int capacity,
                           int *h_launches) {
    MSL_REQUIRE(iters >= 0 && residual_every >= 0 && nx >= 0 && ny >= 0 && nz >= 0,
                "msl_heat7_iterate_plan: negative argument");
    MSL_REQUIRE(h_launches != nullptr && capacity >= 0, "msl_heat7_iterate_plan: bad output arguments");
    std::vector<int> plan;
    if (iters > 0 && nx > 0 && ny > 0 && nz > 0) plan = heat_iterate_plan(nx, ny, nz, iters, residual_every);
    *h_launches = (int)plan.size();
    MSL_REQUIRE(h_gens != nullptr || plan.empty() || capacity == 0, "msl_heat7_iterate_plan: null output");
    for (size_t k = 0; k < plan.size() && (int)k < capacity; k++) h_gens[k] = plan[k];
    return MSL_OK;
}

}  // extern "C"
