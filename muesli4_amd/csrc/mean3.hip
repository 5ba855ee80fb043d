// Mean blur of radius 1, up to six generations per launch in registers.
#include <type_traits>

#include "strip.hpp"

namespace mslhip {

// Whole-wave lane shifts with the vacated lane reading 0 (bound_ctrl): no
// 'old' operand to materialise, so the compiler folds the shift into the
// add that consumes it (v_add_f32_dpp).
__device__ __forceinline__ float lane_from_left(float v) {  // lane l gets lane l-1 (lane 0: 0)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xF, 0xF, true));
}
__device__ __forceinline__ float lane_from_right(float v) {  // lane l gets lane l+1 (lane 63: 0)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xF, 0xF, true));
}

// A block owns a window of 64 NC columns x NW RPW rows: lane l holds columns
// NC l .. NC l + NC - 1, wave w rows [w RPW, (w + 1) RPW) in registers.  The
// window edges lack neighbours, so after s generations only cells at least s
// from every window edge are exact; the block stores the window without K
// cells on each side, exact after up to K generations.  Row sums
// ((0 + left) + centre) + right with the side cells by DPP, column sums
// ((0 + above) + row) + below with the wave edge rows through LDS, then the
// exact division by 9 -- the operation order of the one-step kernel (the
// leading "0 +" of both sums folded into the division), so every generation
// is bit-identical to it.  Cells outside the grid hold nv at every generation.
//
// Windows of 128 x 64 (NC = 2) compute 1.36 cells per stored one where 64 x 64
// ones compute 1.51, and whole windows of non-negative cells of ordinary size
// divide in two operations instead of four (div_pair; the block votes once
// per launch): 6.2 VALU operations per cell and generation of a window, 9.1
// before.  8 rows per wave keep 62 VGPRs, eight waves per SIMD (16 rows: 104).
// 8192^2 x 20: 653 -> 533 us (500 with every XCD on a contiguous range; 527 with
// cells of either sign, whose windows divide in four operations), of which 4
// passes over HBM take 370 at the rate of the map and the VALU issue 373; with the
// next window's cells loaded ahead by persistent blocks 685 (99 VGPRs).  Windows
// over the grid's edge keep the cells outside at nv by bits and leave out waves
// without rows in it (20 iterations, with a select per cell, which became a
// branch around each division / now: 4096^2 135 / 122 us, 20000 x 250 93 / 61).
template <int K, int RPW, int NW, int NC>
__global__ __launch_bounds__(64 * NW) void mean3_multi_kernel(float *__restrict__ out, const float *__restrict__ in,
                                                              int rows, int cols, float nv, int steps, int tiles_x,
                                                              int tile0, float denom, float rcp, RcpPair pair) {
    constexpr int W = 64 * NC, H = NW * RPW, TW = W - 2 * K, TH = H - 2 * K;
    static_assert(K % NC == 0, "a lane's columns are stored together");
    __shared__ float edge[2][NW][2][W];  // double-buffered: one barrier per generation
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int tile = tile0 + (int)xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const int wx = tx * TW - K, wy = ty * TH - K;  // window origin
    const int gx = wx + NC * lane, gy0 = wy + wave * RPW;
    const bool inside = wx >= 0 && wx + W <= cols && wy >= 0 && wy + H <= rows;
    float c[RPW][NC];
    if (inside) {
        const float *p = in + (size_t)gy0 * cols + gx;
#pragma unroll
        for (int i = 0; i < RPW; i++) __builtin_memcpy(c[i], p + (size_t)i * cols, sizeof(c[i]));
    } else {
#pragma unroll
        for (int i = 0; i < RPW; i++)
#pragma unroll
            for (int k = 0; k < NC; k++) c[i][k] = nv;
        const float *p = in + (ptrdiff_t)gy0 * cols + gx;
        if (gx >= 0 && gx + NC <= cols) {
#pragma unroll
            for (int i = 0; i < RPW; i++)
                if ((unsigned)(gy0 + i) < (unsigned)rows)  // wave-uniform
                    __builtin_memcpy(c[i], p + (ptrdiff_t)i * cols, sizeof(c[i]));
        } else if (NC > 1 && gx + NC > 0 && gx < cols) {
#pragma unroll
            for (int i = 0; i < RPW; i++)
#pragma unroll
                for (int k = 0; k < NC; k++)
                    if ((unsigned)(gy0 + i) < (unsigned)rows && (unsigned)(gx + k) < (unsigned)cols)
                        c[i][k] = p[(ptrdiff_t)i * cols + k];
        }
    }
    // waves whose rows all lie outside the grid only hand on their edge rows
    const bool live = gy0 < rows && gy0 + RPW > 0, rows_in = gy0 >= 0 && gy0 + RPW <= rows;
    // columns outside the grid by bits: as selects they became a branch around
    // each cell's division
    uint32_t colmask[NC], nvcol[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) {
        colmask[k] = (unsigned)(gx + k) < (unsigned)cols ? ~0u : 0u;
        nvcol[k] = ~colmask[k] & __float_as_uint(nv);
    }
    PairDomain domain;
    domain.push(nv);
#pragma unroll
    for (int i = 0; i < RPW; i++)
#pragma unroll
        for (int k = 0; k < NC; k++) domain.push(c[i][k]);

    // row sum of row i of the window (no leading +0: the column sum below
    // is finished as if it started at +0, which makes a -0 row sum and a
    // +0 one give the same result)
    auto rowsum = [&](int i, float(&s)[NC]) __attribute__((always_inline)) {
        const float l = lane_from_left(c[i][NC - 1]), r = lane_from_right(c[i][0]);
#pragma unroll
        for (int k = 0; k < NC; k++)
            s[k] = __fadd_rn(__fadd_rn(k > 0 ? c[i][k > 0 ? k - 1 : 0] : l, c[i][k]),
                             k + 1 < NC ? c[i][k + 1 < NC ? k + 1 : k] : r);
    };
    auto generations = [&](auto kInside, auto kFast) __attribute__((always_inline)) {
        for (int s = 0; s < steps; s++) {
            float rs[RPW + 2][NC];  // row sums of rows gy0-1 .. gy0+RPW
            // the wave's edge rows first: their sums go to the neighbouring
            // waves; the inner rows' sums follow the exchange, in the block of
            // the column sums, where each lane shift folds into its add
            rowsum(0, rs[1]);
            rowsum(RPW - 1, rs[RPW]);
            float(&e)[NW][2][W] = edge[s & 1];
#pragma unroll
            for (int k = 0; k < NC; k++) {
                e[wave][0][NC * lane + k] = rs[1][k];
                e[wave][1][NC * lane + k] = rs[RPW][k];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NC; k++) {
                rs[0][k] = e[wave > 0 ? wave - 1 : 0][1][NC * lane + k];
                rs[RPW + 1][k] = e[wave < NW - 1 ? wave + 1 : wave][0][NC * lane + k];
            }
            if (!decltype(kInside)::value && !live) continue;
#pragma unroll
            for (int i = 1; i < RPW - 1; i++) rowsum(i, rs[i + 1]);
#pragma unroll
            for (int i = 0; i < RPW; i++)
#pragma unroll
                for (int k = 0; k < NC; k++) {
                    // the column sum without its leading +0
                    const float t = __fadd_rn(__fadd_rn(rs[i][k], rs[i + 1][k]), rs[i + 2][k]);
                    const float q = decltype(kFast)::value ? div_pair(t, pair) : div_plus0(t, denom, rcp);
                    c[i][k] = decltype(kInside)::value ? q : __uint_as_float((__float_as_uint(q) & colmask[k]) | nvcol[k]);
                }
            if (!decltype(kInside)::value && !rows_in) {
#pragma unroll
                for (int i = 0; i < RPW; i++)
                    if ((unsigned)(gy0 + i) >= (unsigned)rows)
#pragma unroll
                        for (int k = 0; k < NC; k++) c[i][k] = nv;
            }
        }
    };
    const bool fast = __syncthreads_and(domain.ok());
    if (inside && fast)
        generations(std::true_type{}, std::true_type{});
    else if (inside)
        generations(std::true_type{}, std::false_type{});
    else if (fast)
        generations(std::false_type{}, std::true_type{});
    else
        generations(std::false_type{}, std::false_type{});

    if (NC * lane >= K && NC * lane < W - K) {
#pragma unroll
        for (int i = 0; i < RPW; i++) {
            const int r = wave * RPW + i, gy = gy0 + i;
            if (r < K || r >= H - K || gy >= rows) continue;
            float *o = out + (size_t)gy * cols + gx;
            if (gx + NC <= cols) {
                __builtin_memcpy(o, c[i], sizeof(c[i]));
            } else {
#pragma unroll
                for (int k = 0; k < NC; k++)
                    if (gx + k < cols) o[k] = c[i][k];
            }
        }
    }
}

constexpr int kMean3K = 6;     // generations per launch
template <int NC, int RPW, int NW>
static int launch_mean3(float *out, const float *in, int rows, int cols, float nv, int steps) {
    constexpr int TW = 64 * NC - 2 * kMean3K, TH = NW * RPW - 2 * kMean3K;
    const int tiles_x = (cols + TW - 1) / TW;
    const long blocks = (long)tiles_x * (((long)rows + TH - 1) / TH);
    const MeanPolicy<1> pol = MeanPolicy<1>::make();
    return launch_split(blocks, 64 * NW, "msl_stencil2d_mean_iterate_f32", [&](int first, int count) {
        mean3_multi_kernel<kMean3K, RPW, NW, NC><<<count, 64 * NW, 0, ctx().stream>>>(
            out, in, rows, cols, nv, steps, tiles_x, first, pol.denom, pol.rcp, rcp_pair(9.0));
    });
}

// 128-column windows once they give two blocks per CU, unless 64-column ones
// cover the rows with fewer lanes.  20 iterations, 64 / 128 columns: 300^2 28.2 /
// 39.4 us, 1024^2 35.5 / 44.9, 2048^2 67.4 / 67.9, 3000^2 117 / 109, 4096^2 177 /
// 162.  64-column ones have eight waves of 8 rows while every block finds a CU of
// its own, else four of 16, which exchange half the edge rows (300^2 24.1 /
// 25.9 us, 1000^2 29.2 / 29.2, 125000 x 40 80 / 70, 156250 x 128 212 / 171).
int mean3_multi_step(float *out, const float *in, int rows, int cols, float nv, int steps) {
    MSL_REQUIRE(steps >= 1 && steps <= kMean3K, "msl_stencil2d_mean_iterate_f32: generations per launch out of range");
    const long tiles2 = (cols + 115) / 116, tiles1 = (cols + 51) / 52;
    const long trows = ((long)rows + 51) / 52;
    if (tiles2 * trows >= 2L * ctx().num_cus && 2 * tiles2 <= tiles1)
        return launch_mean3<2, 8, 8>(out, in, rows, cols, nv, steps);
    return tiles1 * trows <= ctx().num_cus ? launch_mean3<1, 8, 8>(out, in, rows, cols, nv, steps)
                                           : launch_mean3<1, 16, 4>(out, in, rows, cols, nv, steps);
}

}  // namespace mslhip
