// Two 7-point heat generations per launch on large cubes: a workgroup marches
// a 128 x 26 column tile through a z-segment.
//
// A wave-wide march (heat7x2_march) reads 9 rows for 5 and lines that straddle
// its 60-column tiles: 14.6 bytes per cell and launch from beyond the L2 where
// 8 are needed, which bounded it (512^3: 154 us per generation whatever the
// arithmetic cost).  Here 34 x 30 threads own one quad each of a 136 x 30
// plane: the quad's z neighbours stay in registers, its x and y neighbours
// come from LDS, so the region is read once: (136 x 30) / (128 x 26) = 1.23
// of the cells, and whole lines.  Step zi forms generation 1 of plane zi and
// generation 2 of plane zi - 1; both need planes that were staged in the step
// before, so one LDS-only barrier per step suffices, and the loads of plane
// zi + 3 stay in flight across it.  64 VGPRs (the residual form spills six of
// them: 237 us per launch on 512^3 against 214) and 65 KB: two workgroups per
// CU.  Same order per cell as two single steps (cells outside the cube are nv
// in both generations): bit-identical.
#include <algorithm>

#include "heat.hpp"
#include "heat_tile.hpp"

namespace mslhip {

constexpr int kPairThreads = 1024;

// Region of kPQ quads x kPY rows, a thread per quad.
template <int kPQ, int kPY, bool kResidual, bool NT>
__global__ __launch_bounds__(kPairThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void heat_pair_kernel(
    float *__restrict__ out, const float *__restrict__ in, int nx, int ny, int nz, float nv, int zseg, int tiles_x,
    int tiles_y, float *__restrict__ maxdiff) {
    static_assert(kPQ * kPY <= kPairThreads, "a thread per quad");
    constexpr int kPX = 4 * kPQ;                 // columns of the region
    constexpr int kPW = kPX - 8, kPH = kPY - 4;  // cells stored per plane
    typedef NativeVecN<float, 4>::type V;
    typedef VecN<float, 4> Q;
    constexpr int kBuf = kPX * kPY + 8;
    __shared__ __attribute__((aligned(16))) float lds[4][kBuf];  // input planes 0 / 1, generation-1 planes 2 / 3

    const int tile = (int)xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = (tile / tiles_x) % tiles_y, zs = tile / (tiles_x * tiles_y);
    const int t = threadIdx.x;
    const bool owner = t < kPQ * kPY;
    const int q = owner ? t % kPQ : 0, y = owner ? t / kPQ : 0;
    const int gx = tx * kPW - 4 + 4 * q, gy = ty * kPH - 2 + y;
    const int z0 = zs * zseg, z1 = min(z0 + zseg, nz);
    const size_t plane = (size_t)nx * ny;
    // workgroup-uniform: the region's columns and rows lie in the cube
    const bool inside = tx > 0 && tx * kPW - 4 + kPX <= nx && ty > 0 && ty * kPH - 2 + kPY <= ny;
    const bool rowok = (unsigned)gy < (unsigned)ny;
    const int yc = min(max(gy, 0), ny - 1);
    const bool wide = nx >= 4;
    const unsigned off = (unsigned)(yc * nx + (wide ? min(max(gx, 0), nx - 4) : 0)) * (unsigned)sizeof(float);
    // raw cells of the thread's quad in plane zz (the plane clamped into the cube)
    auto load = [&](int zz) -> Q {
        const char *p = reinterpret_cast<const char *>(in + (size_t)min(max(zz, 0), nz - 1) * plane);
        if (wide) return load_dword_aligned<float, 4>(reinterpret_cast<const float *>(p + off));
        Q v;
#pragma unroll
        for (int k = 0; k < 4; k++)
            v.v[k] = reinterpret_cast<const float *>(p + off)[min(max(gx + k, 0), nx - 1)];
        return v;
    };
    auto fix = [&](const Q &v, int zz) -> Q {
        const bool zok = (unsigned)zz < (unsigned)nz;
        if (inside && zok) return v;
        const int ok = rowok && zok ? 0 : -1;
        return wide ? fix_vec<float, 4, kUnaligned>(v, ok, gx, 1, nx, nv)
                    : fix_vec<float, 4, kScalar>(v, ok, gx, 1, nx, nv);
    };
    const int base = 4 + y * kPX + 4 * q;
    const int dym = y > 0 ? -kPX : 0, dyp = y < kPY - 1 ? kPX : 0;
    // one generation of the quad c (its plane staged in buf) between the
    // quads below and above it
    auto step = [&](const float *buf, const Q &c, const Q &below, const Q &above) -> Q {
        const float *p = buf + base;
        const Q ym = to_vecn<float, 4>(*reinterpret_cast<const V *>(p + dym));
        const Q yp = to_vecn<float, 4>(*reinterpret_cast<const V *>(p + dyp));
        const float xs[6] = {p[-1], c.v[0], c.v[1], c.v[2], c.v[3], p[4]};
        Q sum, r;
        bool suspect = false;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float a = __fadd_rn(xs[k], xs[k + 2]);  // the leading "0 +" is in the division
            a = __fadd_rn(a, ym.v[k]);
            a = __fadd_rn(a, yp.v[k]);
            a = __fadd_rn(a, below.v[k]);
            a = __fadd_rn(a, above.v[k]);
            sum.v[k] = a;
            r.v[k] = div6_fast(a);
            suspect |= div6_suspect(r.v[k]);
        }
        if (suspect) {
#pragma unroll
            for (int k = 0; k < 4; k++) r.v[k] = div6_plus0(sum.v[k]);
        }
        return r;
    };
    const bool stores = owner && q >= 1 && q <= kPQ - 2 && y >= 2 && y < kPY - 2 && gy < ny && gx < nx;
    const bool aligned = ((nx & 3) == 0) && ((reinterpret_cast<uintptr_t>(out) & 15u) == 0);

    if (t < 4) {  // the cells before the first and after the last quad
#pragma unroll
        for (int k = 0; k < 4; k++) {
            lds[k][t] = 0.0f;
            lds[k][kBuf - 1 - t] = 0.0f;
        }
    }
    Q zm = fix(load(z0 - 2), z0 - 2), zc = fix(load(z0 - 1), z0 - 1), zp = fix(load(z0), z0);
    Q pre = load(z0 + 1);
    Q gm = zc, gc = zc;  // read (unstored) by the first steps
    if (owner) *reinterpret_cast<V *>(&lds[0][base]) = to_native<float, 4>(zc);
    lds_barrier();

    float dmax = 0.0f;
    int cur = 0;
    for (int zi = z0 - 1; zi <= z1; zi++) {
        const Q next = load(zi + 3);
        Q g = step(lds[cur], zc, zm, zp);  // generation 1 of plane zi
        const bool zok = (unsigned)zi < (unsigned)nz;
        if (!inside || !zok) {
#pragma unroll
            for (int k = 0; k < 4; k++) g.v[k] = zok && rowok && (unsigned)(gx + k) < (unsigned)nx ? g.v[k] : nv;
        }
        if (zi > z0) {  // generation 2 of plane zi - 1
            const Q w = step(lds[2 + cur], gc, gm, g);
            if (stores) {
                float *o = reinterpret_cast<float *>(reinterpret_cast<char *>(out + (size_t)(zi - 1) * plane) +
                                                     (unsigned)(gy * nx + gx) * (unsigned)sizeof(float));
                if (aligned) {
                    if constexpr (NT)
                        __builtin_nontemporal_store(to_native<float, 4>(w), reinterpret_cast<V *>(o));
                    else
                        *reinterpret_cast<V *>(o) = to_native<float, 4>(w);
                } else if (gx + 4 <= nx) {
                    const V v = to_native<float, 4>(w);
                    __builtin_memcpy(o, &v, sizeof(v));
                } else {
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        if (gx + k < nx) o[k] = w.v[k];
                }
                if constexpr (kResidual) {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float d = fabsf(__fsub_rn(w.v[k], gc.v[k]));
                        if (gx + k < nx) dmax = d > dmax ? d : dmax;
                    }
                }
            }
        }
        if (owner) {
            *reinterpret_cast<V *>(&lds[cur ^ 1][base]) = to_native<float, 4>(zp);
            *reinterpret_cast<V *>(&lds[2 + (cur ^ 1)][base]) = to_native<float, 4>(g);
        }
        zm = zc;
        zc = zp;
        zp = fix(pre, zi + 2);
        pre = next;
        gm = gc;
        gc = g;
        cur ^= 1;
        lds_barrier();
    }
    if constexpr (kResidual) {
        __shared__ float wmax[kPairThreads / 64];
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            const float o = __shfl_xor(dmax, m);
            dmax = o > dmax ? o : dmax;
        }
        if ((t & 63) == 0) wmax[t >> 6] = dmax;
        __syncthreads();
        if (t == 0) {
            for (int w = 1; w < kPairThreads / 64; w++) dmax = wmax[w] > dmax ? wmax[w] : dmax;
            atomicMax(reinterpret_cast<unsigned int *>(maxdiff), __float_as_uint(dmax));
        }
    }
}

// z-segments of a tiling: the workgroups run in rounds of two per CU, each
// marching zseg + 3 planes, so the count of segments that minimises rounds x
// (zseg + 3) is taken (512^3: 6 segments of 86 planes 106 us per generation,
// 12 of 43 112, 4 of 128 128).
struct PairShape {
    int tiles_x, tiles_y, zseg;
    long steps;
};

static PairShape pair_shape(int nx, int ny, int nz, int w, int h) {
    PairShape s{(nx + w - 1) / w, (ny + h - 1) / h, nz, 0};
    const long tiles = (long)s.tiles_x * s.tiles_y, slots = 2L * ctx().num_cus;
    s.steps = (tiles + slots - 1) / slots * (nz + 3L);
    for (int segs = 2; segs <= 256 && nz / segs >= 4; segs++) {
        const int zseg = (nz + segs - 1) / segs;
        const long steps = (tiles * segs + slots - 1) / slots * (zseg + 3L);
        if (steps < s.steps) {
            s.steps = steps;
            s.zseg = zseg;
        }
    }
    return s;
}

template <int kPQ, int kPY>
static int launch_heat_pair(float *out, const float *in, int nx, int ny, int nz, float nv, const PairShape &s,
                            float *maxdiff) {
    const long blocks = (long)s.tiles_x * s.tiles_y * ((nz + s.zseg - 1) / s.zseg);
    // (planes of fewer than 2^30 cells, 32 columns and 11 rows or more, which
    // heat_way asks for here, have at most 1.3 million tiles, in one segment each)
    MSL_REQUIRE(blocks <= launch_limit(kPairThreads), "msl_heat7_iterate_f32: cube too large");
    const bool nt = stream_stores((size_t)nx * ny * nz * sizeof(float));
    const dim3 grid((unsigned)blocks), threads(kPairThreads);
    hipStream_t st = ctx().stream;
    if (maxdiff && nt)
        heat_pair_kernel<kPQ, kPY, true, true>
            <<<grid, threads, 0, st>>>(out, in, nx, ny, nz, nv, s.zseg, s.tiles_x, s.tiles_y, maxdiff);
    else if (maxdiff)
        heat_pair_kernel<kPQ, kPY, true, false>
            <<<grid, threads, 0, st>>>(out, in, nx, ny, nz, nv, s.zseg, s.tiles_x, s.tiles_y, maxdiff);
    else if (nt)
        heat_pair_kernel<kPQ, kPY, false, true>
            <<<grid, threads, 0, st>>>(out, in, nx, ny, nz, nv, s.zseg, s.tiles_x, s.tiles_y, nullptr);
    else
        heat_pair_kernel<kPQ, kPY, false, false>
            <<<grid, threads, 0, st>>>(out, in, nx, ny, nz, nv, s.zseg, s.tiles_x, s.tiles_y, nullptr);
    return check_launch("msl_heat7_iterate_f32");
}

// 128 x 26 tiles (34 x 30 quads), or 80 x 42 ones (22 x 46) where they take
// fewer plane steps: us per generation 128 x 26 / 80 x 42: 512^3 106 / 124,
// 320^3 31 / 23, 300^3 24.0 / 21.9, 600 x 500 x 400 118 / 123 (96 x 35 and
// 64 x 52 tiles won nowhere).
int heat_pair_step(float *out, const float *in, int nx, int ny, int nz, float nv, float *maxdiff) {
    const PairShape wide = pair_shape(nx, ny, nz, 128, 26), tall = pair_shape(nx, ny, nz, 80, 42);
    return tall.steps < wide.steps ? launch_heat_pair<22, 46>(out, in, nx, ny, nz, nv, tall, maxdiff)
                                   : launch_heat_pair<34, 30>(out, in, nx, ny, nz, nv, wide, maxdiff);
}

}  // namespace mslhip
