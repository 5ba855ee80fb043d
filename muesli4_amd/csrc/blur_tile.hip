// Mean blur of small and medium grids: one workgroup per tile, one or more
// generations per launch in LDS (blur_tile.hpp).
//
// The strip march (strip.hpp) keeps one row per step in flight and repeats
// 2R warm-up rows per segment; on grids of a few million cells its waves run
// short segments one after another, bound by the latency of that chain.  A
// tile's loads are all in flight at once and its row sums are formed once per
// workgroup.
#include <algorithm>
#include <cmath>

#include "blur_tile.hpp"

namespace mslhip {

template <int R, int W, int M>
__global__ __launch_bounds__(16 * W / M) void blur_tile_kernel(float *__restrict__ out, const float *__restrict__ in,
                                                               int rows, int cols, float nv, int steps, int tile_w,
                                                               int tile_h, int tiles_x, int tile0) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tile = tile0 + (int)xcd_tile(blockIdx.x, gridDim.x);
    blur_tile<R, W, M>(out, in, rows, cols, nv, steps, tile_w, tile_h, tile % tiles_x, tile / tiles_x, lds);
}

template <int R, int W, int M>
static int launch_tile_rw(float *out, const float *in, int rows, int cols, float nv, int steps, int tile_h) {
    const int tile_w = (W - 2 * R * steps) / 4 * 4;
    MSL_REQUIRE(tile_w >= 4 && tile_h >= 1 && tile_h + 2 * R * (steps - 1) <= kTileRows,
                "msl_stencil2d_mean_f32: tile out of range");
    const int tiles_x = (cols + tile_w - 1) / tile_w;
    const long blocks = (long)tiles_x * (((long)rows + tile_h - 1) / tile_h);
    return launch_split(blocks, 16 * W / M, "msl_stencil2d_mean_f32", [&](int first, int count) {
        blur_tile_kernel<R, W, M><<<count, 16 * W / M, blur_tile_lds(R, W, tile_h, steps), ctx().stream>>>(
            out, in, rows, cols, nv, steps, tile_w, tile_h, tiles_x, first);
    });
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
// coefficients fitted to 8000 timings (64^2 .. 4096^2, r = 2 .. 13, 1 .. 6
// generations; its choice is 1 % slower than the best shape on average, 14 %
// at worst):
//   1.9 us         per launch (drain, launch, first load, last store)
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
                (double)((cols + tile_w - 1) / tile_w) * (double)(((long)rows + th - 1) / th) / cus;
            const double b = tiles <= 1.0 ? 1.0 : 0.5 * (std::ceil(tiles) + tiles);
            const double us = 1.90 + 0.613 * steps + 0.00719 * lat +
                              b * (2.12e-6 * vw + 1.70e-4 * (th + 2 * r * steps) * w + 0.0145 * steps * (w / (4 * m)));
            if (us < best.us) best = TileShape{w, m, th, us};
        }
    }
    return best;
}

}  // namespace mslhip
