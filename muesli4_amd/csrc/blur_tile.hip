// Mean blur of small and medium grids: one workgroup per tile, one or more
// generations per launch in LDS.
//
// The strip march (strip.hpp) keeps one row per step in flight and repeats
// 2R warm-up rows per segment; on grids of a few million cells its waves run
// short segments one after another, bound by the latency of that chain.  Here
// a workgroup of 4 W threads loads a whole tile (W columns, up to 64 + 2R
// rows, all loads at once), forms every row sum of the tile in place (four
// outputs per thread from a register window), then the column sums (4 x 4
// outputs per thread), and repeats that for `steps` generations, the valid
// region shrinking by R on each side.  Every output has the operation order
// of the strip march (row sums dx ascending, column sums dy ascending, the
// exact division; cells outside the grid are nv in every generation), so the
// results are bit-identical to it.
#include <algorithm>
#include <cmath>

#include "blur_tile.hpp"
#include "strip.hpp"

namespace mslhip {

constexpr int kTileRows = 64;  // most output rows of a tile's first generation

// Row pass: a row's quads sit in one wave (16 or 32 lanes), whose lanes all
// read their windows before any of them stores, so the sums replace the row.
// Reads past the valid columns feed only sums that no output uses.
// Read: M rows per thread of the column pass, 64 / M rows per round of all
// threads.  1 on grids of few tiles (16 waves per tile, the shortest chain),
// 4 on many (fewest LDS reads per output).
template <int R, int W, int M>
__global__ __launch_bounds__(16 * W / M) void blur_tile_kernel(float *__restrict__ out, const float *__restrict__ in,
                                                          int rows, int cols, float nv, int steps, int tile_w,
                                                          int tile_h, int tiles_x, float denom, float rcp) {
    constexpr int QW = W / 4;                           // quads per LDS row
    constexpr int RPR = kTileRows / M;                  // rows per pass of all threads
    constexpr int ROUNDS = (kTileRows + 2 * R + RPR - 1) / RPR;
    constexpr int NQ = (2 * R + 4 + 3) / 4;             // quads of a four-output window
    extern __shared__ __attribute__((aligned(16))) float lds[];
    typedef NativeVecN<float, 4>::type V;

    const int tile = (int)xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const int q = threadIdx.x % QW, rr = threadIdx.x / QW;
    const int ox = tx * tile_w, oy = ty * tile_h;       // first output cell of the tile
    const int th = min(tile_h, rows - oy);
    int h = th + 2 * R * steps;
    int x0 = ox - R * steps, y0 = oy - R * steps;       // grid cell of LDS (0, 0)
    const bool inside = x0 >= 0 && x0 + W <= cols && y0 >= 0 && y0 + h <= rows;

    {
        const int c0 = x0 + 4 * q;
        VecN<float, 4> v[ROUNDS];
#pragma unroll
        for (int i = 0; i < ROUNDS; i++) {
            const int y = y0 + min(rr + RPR * i, h - 1);
            if (inside) {
                v[i] = load_dword_aligned<float, 4>(in + (size_t)y * cols + c0);
            } else {
                const float *row = in + (size_t)min(max(y, 0), rows - 1) * cols;
#pragma unroll
                for (int k = 0; k < 4; k++) v[i].v[k] = row[min(max(c0 + k, 0), cols - 1)];
            }
        }
#pragma unroll
        for (int i = 0; i < ROUNDS; i++) {
            const int row = rr + RPR * i;
            if (!inside) {
                const bool rowok = (unsigned)(y0 + row) < (unsigned)rows;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    v[i].v[k] = rowok && (unsigned)(c0 + k) < (unsigned)cols ? v[i].v[k] : nv;
            }
            if (row < h) *reinterpret_cast<V *>(lds + row * W + 4 * q) = to_native<float, 4>(v[i]);
        }
    }
    __syncthreads();

    for (int s = 0; s < steps; s++) {
#pragma unroll
        for (int i = 0; i < ROUNDS; i++) {
            const int row = rr + RPR * i;
            if (row < h) {
                float *p = lds + row * W + 4 * q;
                float w[4 * NQ];
#pragma unroll
                for (int k = 0; k < NQ; k++) {
                    const VecN<float, 4> t = to_vecn<float, 4>(*reinterpret_cast<const V *>(p + 4 * k));
#pragma unroll
                    for (int c = 0; c < 4; c++) w[4 * k + c] = t.v[c];
                }
                VecN<float, 4> o;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    float a = w[c];
#pragma unroll
                    for (int d = 1; d <= 2 * R; d++) a = __fadd_rn(a, w[c + d]);
                    o.v[c] = a;
                }
                wave_lds_sync();
                *reinterpret_cast<V *>(p) = to_native<float, 4>(o);
            }
        }
        __syncthreads();
        h -= 2 * R;
        x0 += R;
        y0 += R;
        const bool active = M * rr < h;
        VecN<float, 4> o[M];
        if (active) {
            const float *p = lds + M * rr * W + 4 * q;
#pragma unroll
            for (int k = 0; k < 2 * R + M; k++) {
                const VecN<float, 4> t = to_vecn<float, 4>(*reinterpret_cast<const V *>(p + k * W));
#pragma unroll
                for (int m = 0; m < M; m++)
                    if (k >= m && k <= m + 2 * R) {
#pragma unroll
                        for (int c = 0; c < 4; c++) o[m].v[c] = k == m ? t.v[c] : __fadd_rn(o[m].v[c], t.v[c]);
                    }
            }
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int c = 0; c < 4; c++) o[m].v[c] = div_plus0(o[m].v[c], denom, rcp);
        }
        if (s + 1 == steps) {
            if (active && 4 * q < tile_w) {
#pragma unroll
                for (int m = 0; m < M; m++)
                    if (M * rr + m < h)
                        write_vec<float, 4, kUnaligned, false>(out + (size_t)(y0 + M * rr + m) * cols, x0 + 4 * q, cols,
                                                               o[m]);
            }
        } else {
            if (!inside && active) {
#pragma unroll
                for (int m = 0; m < M; m++) {
                    const bool rowok = (unsigned)(y0 + M * rr + m) < (unsigned)rows;
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        o[m].v[c] = rowok && (unsigned)(x0 + 4 * q + c) < (unsigned)cols ? o[m].v[c] : nv;
                }
            }
            __syncthreads();
            if (active) {
#pragma unroll
                for (int m = 0; m < M; m++)
                    *reinterpret_cast<V *>(lds + (M * rr + m) * W + 4 * q) = to_native<float, 4>(o[m]);
            }
            __syncthreads();
        }
    }
}

template <int R, int W, int M>
static int launch_tile_rw(float *out, const float *in, int rows, int cols, float nv, int steps, int tile_h) {
    const int tile_w = (W - 2 * R * steps) / 4 * 4;
    MSL_REQUIRE(tile_w >= 4 && tile_h >= 1 && tile_h + 2 * R * (steps - 1) <= kTileRows,
                "msl_stencil2d_mean_f32: tile out of range");
    const int tiles_x = (cols + tile_w - 1) / tile_w;
    const long blocks = (long)tiles_x * ((rows + tile_h - 1) / tile_h);
    MSL_REQUIRE(blocks <= INT32_MAX, "msl_stencil2d_mean_f32: grid too large");
    // rows of the tile, three more that a partial group of four reads, and
    // the window of the last quad
    const size_t lds = sizeof(float) * ((size_t)(tile_h + 2 * R * steps + 3) * W + 2 * R + 8);
    const MeanPolicy<R> pol = MeanPolicy<R>::make();
    blur_tile_kernel<R, W, M><<<(int)blocks, 16 * W / M, lds, ctx().stream>>>(out, in, rows, cols, nv, steps, tile_w, tile_h,
                                                                       tiles_x, pol.denom, pol.rcp);
    return check_launch("msl_stencil2d_mean_f32");
}

template <int R>
static int launch_tile_r(float *out, const float *in, int rows, int cols, float nv, int steps, const TileShape &t) {
    if (t.w == 64)
        return t.m == 1 ? launch_tile_rw<R, 64, 1>(out, in, rows, cols, nv, steps, t.tile_h)
                        : launch_tile_rw<R, 64, 2>(out, in, rows, cols, nv, steps, t.tile_h);
    return t.m == 2 ? launch_tile_rw<R, 128, 2>(out, in, rows, cols, nv, steps, t.tile_h)
                    : launch_tile_rw<R, 128, 4>(out, in, rows, cols, nv, steps, t.tile_h);
}

int blur_tile_step(float *out, const float *in, int rows, int cols, int r, float nv, int steps, const TileShape &t) {
    typedef int (*Launcher)(float *, const float *, int, int, float, int, const TileShape &);
    static const Launcher kLaunch[] = {nullptr,           nullptr,           launch_tile_r<2>,  launch_tile_r<3>,
                                       launch_tile_r<4>,  launch_tile_r<5>,  launch_tile_r<6>,  launch_tile_r<7>,
                                       launch_tile_r<8>,  launch_tile_r<9>,  launch_tile_r<10>, launch_tile_r<11>,
                                       launch_tile_r<12>, launch_tile_r<13>, launch_tile_r<14>, launch_tile_r<15>,
                                       launch_tile_r<16>};
    MSL_REQUIRE(r >= 2 && r <= 16 && steps >= 1, "msl_stencil2d_mean_f32: tile out of range");
    return kLaunch[r](out, in, rows, cols, nv, steps, t);
}

// Tile of a launch of `steps` generations: columns, rows per thread of the
// column pass (the workgroup has 16 w / m threads) and output rows, by the
// smallest modelled time.  The model is the kernel's structure with six
// coefficients fitted to 9000 timings (64^2 .. 4096^2, r = 1 .. 10, 1 .. 6
// generations; its choice is 3 % slower than the best shape on average, 22 %
// at worst):
//   3.1 us         per launch (drain, launch, first load, last store)
//   0.6 us         per generation (two barriers)
//   lat            the dependent chain of one wave: its rounds of row sums
//                  and its column sums
//   B (vw, mem, w) work of a CU: lane operations, LDS cells loaded, waves,
//                  for B tiles per CU (half of a partial round counts whole)
TileShape tile_shape(int rows, int cols, int r, int steps) {
    static const TileShape kKinds[] = {{64, 1, 0, 0.0}, {64, 2, 0, 0.0}, {128, 2, 0, 0.0}, {128, 4, 0, 0.0}};
    static const int kHeights[] = {8, 16, 24, 32, 40, 48, 64};
    TileShape best{0, 0, 0, 1e30};
    const double cus = ctx().num_cus;
    for (const TileShape &kind : kKinds) {
        const int w = kind.w, m = kind.m, rpr = kTileRows / m;
        const int tile_w = (w - 2 * r * steps) / 4 * 4;
        if (tile_w < 16) continue;
        for (int th : kHeights) {
            if (th + 2 * r * (steps - 1) > kTileRows) break;
            double vw = 0.0, lat = 0.0;
            for (int s = 0; s < steps; s++) {
                const int hi = th + 2 * r * (steps - s), ho = hi - 2 * r;
                vw += (double)hi * w * (2 * r + 6) + (double)((ho + m - 1) / m * m) * w * (2 * r + 8);
                lat += (hi + rpr - 1) / rpr * (2 * r + 8) + m * (2 * r + 6);
            }
            const double tiles =
                (double)((cols + tile_w - 1) / tile_w) * (double)((rows + th - 1) / th) / cus;
            const double b = tiles <= 1.0 ? 1.0 : 0.5 * (std::ceil(tiles) + tiles);
            const double us = 3.14 + 0.592 * steps + 0.00938 * lat +
                              b * (1.31e-6 * vw + 2.19e-4 * (th + 2 * r * steps) * w + 0.0163 * steps * (w / (4 * m)));
            if (us < best.us) best = TileShape{w, m, th, us};
        }
    }
    return best;
}

}  // namespace mslhip
