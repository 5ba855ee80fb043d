// 7-point heat steps of small and medium cubes: one workgroup per 3-D tile,
// one or more generations per launch in LDS.
//
// The march (heat.hpp) keeps one plane in flight per wave and runs at least 16
// planes one after another: 13 us per step on a 32^3 cube.  Here a workgroup
// loads a 40 x 24 x 20 region (all loads at once) and applies `steps`
// generations to it in LDS, the exact part shrinking by one cell on each side
// per generation; the inner (40 - 2 steps) x (24 - 2 steps) x (20 - 2 steps)
// cells are stored.  A thread owns four x-adjacent cells of five planes: their
// z neighbours stay in registers, x and y neighbours are LDS reads (15.6
// bytes per cell and generation), and the results are held in registers until
// every thread has read, so one buffer of 77 KB suffices and two workgroups
// fit a CU.  Each cell is computed in the one-step order (cells outside the
// cube are nv in every generation): bit-identical to the march.
#include "heat.hpp"
#include "heat_tile.hpp"

namespace mslhip {

constexpr int kHX = 40;             // region columns
constexpr int kHQ = kHX / 4;        // quads per row
constexpr int kHeatThreads = 1024;  // 960 of them own cells

// Region of kHX x kHY x kHZ cells, kHZP planes per thread: 24 x 20 x 5 planes,
// or 16 x 12 x 2 for cubes of few tiles.
template <int kHY, int kHZ, int kHZP, bool kResidual>
__global__ __launch_bounds__(kHeatThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void heat_tile_kernel(
    float *__restrict__ out, const float *__restrict__ in, int nx, int ny, int nz, float nv, int steps, int tiles_x,
    int tiles_y, float *__restrict__ maxdiff) {
    static_assert(kHQ * kHY * (kHZ / kHZP) <= kHeatThreads, "a thread per quad and plane group");
    typedef NativeVecN<float, 4>::type V;
    __shared__ __attribute__((aligned(16))) float region[kHX * kHY * kHZ + 8];
    float *lds = region + 4;  // the reads at x - 1 and x + 4 of the first and last quad stay inside

    const int tile = (int)xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = (tile / tiles_x) % tiles_y, tz = tile / (tiles_x * tiles_y);
    const int t = threadIdx.x;
    const bool owner = t < kHQ * kHY * (kHZ / kHZP);
    const int q = t % kHQ, y = (t / kHQ) % kHY, z = owner ? t / (kHQ * kHY) * kHZP : 0;  // region cell of the thread
    // grid cell of the thread's first cell
    const int gx = tx * (kHX - 2 * steps) - steps + 4 * q;
    const int gy = ty * (kHY - 2 * steps) - steps + y;
    const int gz = tz * (kHZ - 2 * steps) - steps + z;
    const size_t plane = (size_t)nx * ny;
    // wave-uniform: whether the whole region lies in the cube
    const int rx = tx * (kHX - 2 * steps) - steps, ry = ty * (kHY - 2 * steps) - steps,
              rz = tz * (kHZ - 2 * steps) - steps;
    const bool inside =
        rx >= 0 && rx + kHX <= nx && ry >= 0 && ry + kHY <= ny && rz >= 0 && rz + kHZ <= nz;
    float *cell = lds + (z * kHY + y) * kHX + 4 * q;
    constexpr int kPlane = kHX * kHY;

    if (owner) {
        VecN<float, 4> v[kHZP];
        if (inside) {
            const float *p = in + ((size_t)gz * ny + gy) * nx + gx;
#pragma unroll
            for (int i = 0; i < kHZP; i++) v[i] = load_dword_aligned<float, 4>(p + i * plane);
        } else if (nx >= 4) {
            // a clamped quad per plane; columns pick their cell by the shift
            const int yc = min(max(gy, 0), ny - 1), xc = min(max(gx, 0), nx - 4);
#pragma unroll
            for (int i = 0; i < kHZP; i++)
                v[i] = load_dword_aligned<float, 4>(in + ((size_t)min(max(gz + i, 0), nz - 1) * ny + yc) * nx + xc);
#pragma unroll
            for (int i = 0; i < kHZP; i++) {
                const bool rowok = (unsigned)gy < (unsigned)ny && (unsigned)(gz + i) < (unsigned)nz;
                v[i] = fix_vec<float, 4, kUnaligned>(v[i], rowok ? 0 : -1, gx, 1, nx, nv);
            }
        } else {
            const int yc = min(max(gy, 0), ny - 1);
            const bool yok = (unsigned)gy < (unsigned)ny;
#pragma unroll
            for (int i = 0; i < kHZP; i++) {
                const float *row = in + ((size_t)min(max(gz + i, 0), nz - 1) * ny + yc) * nx;
                const bool ok = yok && (unsigned)(gz + i) < (unsigned)nz;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float f = row[min(max(gx + c, 0), nx - 1)];
                    v[i].v[c] = ok && (unsigned)(gx + c) < (unsigned)nx ? f : nv;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kHZP; i++) *reinterpret_cast<V *>(cell + i * kPlane) = to_native<float, 4>(v[i]);
    }
    __syncthreads();

    // offsets of the y and z neighbours, clamped at the region's faces (those
    // results are not exact and never stored)
    const int dym = y > 0 ? -kHX : 0, dyp = y < kHY - 1 ? kHX : 0;
    const int dzm = z > 0 ? -kPlane : 0, dzp = z + kHZP < kHZ ? kHZP * kPlane : (kHZP - 1) * kPlane;
    float dmax = 0.0f;
    for (int s = 1; s <= steps; s++) {
        VecN<float, 4> o[kHZP];
        if (owner) {
            VecN<float, 4> below = to_vecn<float, 4>(*reinterpret_cast<const V *>(cell + dzm));
            VecN<float, 4> c = to_vecn<float, 4>(*reinterpret_cast<const V *>(cell));
#pragma unroll
            for (int i = 0; i < kHZP; i++) {
                const float *p = cell + i * kPlane;
                const VecN<float, 4> above =
                    to_vecn<float, 4>(*reinterpret_cast<const V *>(i + 1 < kHZP ? p + kPlane : cell + dzp));
                const VecN<float, 4> ym = to_vecn<float, 4>(*reinterpret_cast<const V *>(p + dym));
                const VecN<float, 4> yp = to_vecn<float, 4>(*reinterpret_cast<const V *>(p + dyp));
                // planes that no later generation and no store needs keep
                // their old cells (a whole group of planes for most waves)
                const bool needed = kHZP > 2 || (z + i >= s && z + i < kHZ - s && (unsigned)(gz + i) < (unsigned)nz);
                if constexpr (kHZP <= 2) o[i] = c;
                if (needed) {
                float sum[4];
                const float xs[6] = {p[-1], c.v[0], c.v[1], c.v[2], c.v[3], p[4]};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    float a = __fadd_rn(xs[k], xs[k + 2]);  // the leading "0 +" is in div6_plus0
                    a = __fadd_rn(a, ym.v[k]);
                    a = __fadd_rn(a, yp.v[k]);
                    a = __fadd_rn(a, below.v[k]);
                    a = __fadd_rn(a, above.v[k]);
                    sum[k] = a;
                }
                bool suspect = false;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    o[i].v[k] = div6_fast(sum[k]);
                    suspect |= div6_suspect(o[i].v[k]);
                }
                if (suspect) {
#pragma unroll
                    for (int k = 0; k < 4; k++) o[i].v[k] = div6_plus0(sum[k]);
                }
                if (kResidual && s == steps) {
                    const bool rowok = y >= steps && y < kHY - steps && z + i >= steps && z + i < kHZ - steps &&
                                       gy < ny && gz + i < nz;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float d = fabsf(__fsub_rn(o[i].v[k], c.v[k]));
                        const int x = 4 * q + k;
                        if (rowok && x >= steps && x < kHX - steps && gx + k < nx) dmax = d > dmax ? d : dmax;
                    }
                }
                }
                below = c;
                c = above;
            }
        }
        if (s == steps) {
            if (owner && y >= steps && y < kHY - steps && gy < ny) {
#pragma unroll
                for (int i = 0; i < kHZP; i++) {
                    if (z + i < steps || z + i >= kHZ - steps || gz + i >= nz) continue;
                    float *p = out + ((size_t)(gz + i) * ny + gy) * nx + gx;
                    if (4 * q >= steps && 4 * q + 4 <= kHX - steps && gx + 4 <= nx) {
                        const V v = to_native<float, 4>(o[i]);
                        __builtin_memcpy(p, &v, sizeof(v));
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            if (4 * q + k >= steps && 4 * q + k < kHX - steps && gx + k < nx) p[k] = o[i].v[k];
                    }
                }
            }
        } else {
            if (!inside) {
                const bool yok = (unsigned)gy < (unsigned)ny;
#pragma unroll
                for (int i = 0; i < kHZP; i++) {
                    const bool ok = yok && (unsigned)(gz + i) < (unsigned)nz;
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        o[i].v[k] = ok && (unsigned)(gx + k) < (unsigned)nx ? o[i].v[k] : nv;
                }
            }
            __syncthreads();
            if (owner) {
#pragma unroll
                for (int i = 0; i < kHZP; i++) *reinterpret_cast<V *>(cell + i * kPlane) = to_native<float, 4>(o[i]);
            }
            __syncthreads();
        }
    }
    if (kResidual) {
        __shared__ float wmax[kHeatThreads / 64];
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            const float o = __shfl_xor(dmax, m);
            dmax = o > dmax ? o : dmax;
        }
        if ((t & 63) == 0) wmax[t >> 6] = dmax;
        __syncthreads();
        if (t == 0) {
            for (int w = 1; w < kHeatThreads / 64; w++) dmax = wmax[w] > dmax ? wmax[w] : dmax;
            atomicMax(reinterpret_cast<unsigned int *>(maxdiff), __float_as_uint(dmax));
        }
    }
}

template <int kHY, int kHZ>
static long tile_blocks(int nx, int ny, int nz, int steps) {
    const int tx = kHX - 2 * steps, ty = kHY - 2 * steps, tz = kHZ - 2 * steps;
    return (long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty) * ((nz + tz - 1) / tz);
}

long heat_tile_blocks(int nx, int ny, int nz, int steps, bool small) {
    return small ? tile_blocks<16, 12>(nx, ny, nz, steps) : tile_blocks<24, 20>(nx, ny, nz, steps);
}

template <int kHY, int kHZ, int kHZP>
static int launch_heat_tile(float *out, const float *in, int nx, int ny, int nz, float nv, int steps, float *maxdiff) {
    const int tx = kHX - 2 * steps, ty = kHY - 2 * steps, tz = kHZ - 2 * steps;
    MSL_REQUIRE(steps >= 1 && tz >= 1, "msl_heat7_f32: generations per launch out of range");
    const int tiles_x = (nx + tx - 1) / tx, tiles_y = (ny + ty - 1) / ty;
    const long blocks = tile_blocks<kHY, kHZ>(nx, ny, nz, steps);
    MSL_REQUIRE(blocks <= INT32_MAX, "msl_heat7_f32: cube too large");
    if (maxdiff)
        heat_tile_kernel<kHY, kHZ, kHZP, true><<<(int)blocks, kHeatThreads, 0, ctx().stream>>>(
            out, in, nx, ny, nz, nv, steps, tiles_x, tiles_y, maxdiff);
    else
        heat_tile_kernel<kHY, kHZ, kHZP, false><<<(int)blocks, kHeatThreads, 0, ctx().stream>>>(
            out, in, nx, ny, nz, nv, steps, tiles_x, tiles_y, nullptr);
    return check_launch("msl_heat7_f32");
}

int heat_tile_step(float *out, const float *in, int nx, int ny, int nz, float nv, int steps, bool small,
                   float *maxdiff) {
    return small ? launch_heat_tile<16, 12, 2>(out, in, nx, ny, nz, nv, steps, maxdiff)
                 : launch_heat_tile<24, 20, 5>(out, in, nx, ny, nz, nv, steps, maxdiff);
}

}  // namespace mslhip
