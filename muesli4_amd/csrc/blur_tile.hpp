// Tile form of the mean blur: one workgroup per tile, one or more generations
// in LDS (blur_tile.hip, and the serving engine's items).
//
// A workgroup of 16 W / M threads loads a whole tile (W columns, up to 64 + 2R
// rows, all loads at once), forms every row sum of the tile in place (four
// outputs per thread from a register window), then the column sums (4 x M
// outputs per thread), and repeats that for `steps` generations, the valid
// region shrinking by R on each side.  Every output has the operation order
// of the strip march (row sums dx ascending, column sums dy ascending, the
// exact division; cells outside the grid are nv in every generation), so the
// results are bit-identical to it.
#pragma once

#include "strip.hpp"

namespace mslhip {

constexpr int kTileRows = 64;  // most output rows of a tile's first generation

// Generations per launch, by radius, of the batch's and the serving engine's
// 128-column tiles.  Measured at r = 3, 5, 7 and 10 (us per generation of 2048^2 at
// 1 / 2 / 3 / 4 generations, M = 4: 10.6 / 7.3 / 6.8 / 6.1, 11.1 / 9.1 / 8.4 / 8.5,
// 12.0 / 10.4 / 11.0, 13.6 / 13.4 / 19.6); the radii between take the count of the
// next larger one that was measured, r = 1 the most there are.
constexpr int kTileGens[11] = {0, 6, 4, 4, 3, 3, 2, 2, 2, 2, 2};

// Row pass: a row's quads sit in one wave (16 or 32 lanes), whose lanes all
// read their windows before any of them stores, so the sums replace the row.
// Reads past the valid columns feed only sums that no output uses.
// M is the rows per thread of the column pass (all threads cover 64 / M rows at a
// time): 1 on grids of few tiles (16 waves per tile, the shortest chain), 4 on
// many (fewest LDS reads per output).
template <int R, int W, int M>
__device__ __forceinline__ void blur_tile(float *__restrict__ out, const float *__restrict__ in, int rows, int cols,
                                          float nv, int steps, int tile_w, int tile_h, int tx, int ty, float *lds) {
    const MeanPolicy<R> pol = MeanPolicy<R>::make();
    constexpr int QW = W / 4;                           // quads per LDS row
    constexpr int RPR = kTileRows / M;                  // rows per pass of all threads
    constexpr int ROUNDS = (kTileRows + 2 * R + RPR - 1) / RPR;
    constexpr int NQ = (2 * R + 4 + 3) / 4;             // quads of a four-output window
    typedef NativeVecN<float, 4>::type V;

    const int q = threadIdx.x % QW, rr = threadIdx.x / QW;
    const int ox = tx * tile_w, oy = ty * tile_h;       // first output cell of the tile
    const int th = min(tile_h, rows - oy);
    int h = th + 2 * R * steps;
    int x0 = ox - R * steps, y0 = oy - R * steps;       // grid cell of LDS (0, 0)
    const bool inside = x0 >= 0 && x0 + W <= cols && y0 >= 0 && y0 + h <= rows;

    // The tile's cells, all loads at once.  Tiles over the grid's edge are
    // filled with nv first, and each quad that overlaps the grid is loaded and
    // stored shifted to lie in it (overlapping quads store equal values):
    // cheaper than selecting per cell, and most tiles of small grids are such.
    if (inside || cols >= 4) {
        const int c0 = x0 + 4 * q, cc = min(max(c0, 0), cols - 4);
        VecN<float, 4> v[ROUNDS];
#pragma unroll
        for (int i = 0; i < ROUNDS; i++) {
            const int y = min(max(y0 + min(rr + RPR * i, h - 1), 0), rows - 1);
            v[i] = load_dword_aligned<float, 4>(in + (size_t)y * cols + cc);
        }
        if (inside) {
#pragma unroll
            for (int i = 0; i < ROUNDS; i++)
                if (rr + RPR * i < h)
                    *reinterpret_cast<V *>(lds + (rr + RPR * i) * W + 4 * q) = to_native<float, 4>(v[i]);
        } else {
            for (int row = rr; row < h; row += RPR) *reinterpret_cast<V *>(lds + row * W + 4 * q) = V{nv, nv, nv, nv};
            __syncthreads();
            const int p = cc - x0;
            if (c0 < cols && c0 + 4 > 0) {
#pragma unroll
                for (int i = 0; i < ROUNDS; i++) {
                    const int row = rr + RPR * i;
                    if (row < h && (unsigned)(y0 + row) < (unsigned)rows) {
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            if (p + k >= 0) lds[row * W + p + k] = v[i].v[k];
                    }
                }
            }
        }
    } else {
        const int c0 = x0 + 4 * q;
        for (int row = rr; row < h; row += RPR) {
            const bool rowok = (unsigned)(y0 + row) < (unsigned)rows;
            const float *src = in + (size_t)min(max(y0 + row, 0), rows - 1) * cols;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float f = src[min(max(c0 + k, 0), cols - 1)];
                lds[row * W + 4 * q + k] = rowok && (unsigned)(c0 + k) < (unsigned)cols ? f : nv;
            }
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
                for (int c = 0; c < 4; c++) o[m].v[c] = div_plus0(o[m].v[c], pol.denom, pol.rcp);
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


// LDS bytes of a tile of tile_h output rows: its input rows, three more that
// a partial group of M <= 4 reads, and the window of the last quad.
constexpr size_t blur_tile_lds(int r, int w, int tile_h, int steps) {
    return sizeof(float) * ((size_t)(tile_h + 2 * r * steps + 3) * w + 2 * r + 8);
}

struct TileShape {
    int w, m, tile_h;  // LDS columns, rows per thread of the column pass, output rows; w = 0: none fits
    double us;         // modelled time of the launch
};
TileShape tile_shape(int rows, int cols, int r, int steps);
int blur_tile_step(float *out, const float *in, int rows, int cols, int r, float nv, int steps, const TileShape &t);

}  // namespace mslhip
