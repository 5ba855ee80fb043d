// Game of Life iterations on bit-packed cells.
//
// Reference: examples/gameoflife.cpp:18-43 through DM::mapStencilMM
// (src/dm.cpp:615-1208), one launch and one int per cell per generation.
//
// From the second generation on every cell is 0 or 1, so the grid fits one
// bit per cell.  gol_first_kernel applies generation 1 to the int cells
// (any values) and packs its result, 32 columns per word; gol_bits_kernel
// applies up to 16 generations to packed windows held in registers; the last
// of its launches unpacks to ints.  The packed grids (1/32 of the cells each)
// live in the caller's two buffers, in the one that does not hold the data
// being read or the result.  100 generations of 1024^2 and a fold, which 13
// launches of an int-per-cell register window took 210 us for, take 58 us
// (windows of 64 x 64 ints: 14 us per 8 generations; here 5.4 us per 14,
// mostly launch and load latency; 4096 x 4000: 1.9 us per generation, 10.7
// before).
#include <functional>
#include <string>
#include <vector>

#include "common.hpp"

namespace mslhip {

int gol_step(int32_t *out, const int32_t *in, int rows, int cols);
std::vector<int> generation_plan(int iters, int k);  // stencil2d.hip

// Whole-wave lane shifts with the vacated lane reading 0 (bound_ctrl).
__device__ __forceinline__ uint32_t lane_below(uint32_t v) {  // lane l gets lane l-1 (lane 0: 0)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t lane_above(uint32_t v) {  // lane l gets lane l+1 (lane 63: 0)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xF, 0xF, true);
}

// Up to K generations of int cells per launch: a block owns a 64-column x
// (4 * RPW)-row window, lane l holds column l, wave w rows [w*RPW, (w+1)*RPW) in
// registers.  Each generation exchanges the waves' first and last rows through
// LDS, forms vertical 3-sums in registers and the horizontal ones by DPP; after
// s generations only cells at least s from every window edge are exact, and the
// block stores the window without K cells on each side.  For the counts below,
// where one launch from d_a to d_b leaves the input as it was, and for single
// columns, whose packed grids would not fit the buffers.  3 generations of
// 4096^2 take 35 us, bit-packed 43; 5 of 1024^2 14.5, 20.
template <int K, int RPW>
__global__ __launch_bounds__(256) void gol_window_kernel(int32_t *__restrict__ out, const int32_t *__restrict__ in,
                                                         int rows, int cols, int steps, int tiles_x, int tile0) {
    constexpr int H = 4 * RPW, TW = 64 - 2 * K, TH = H - 2 * K;
    __shared__ uint32_t edge[4][2][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int tile = tile0 + (int)xcd_tile(blockIdx.x, gridDim.x);
    const int gx = tile % tiles_x * TW - K + lane;
    const int gy0 = tile / tiles_x * TH - K + wave * RPW;
    const bool colok = (unsigned)gx < (unsigned)cols;
    uint32_t c[RPW + 2];  // rows gy0-1 .. gy0+RPW
#pragma unroll
    for (int i = 0; i < RPW; i++) {
        const int gy = gy0 + i;
        c[i + 1] = colok && (unsigned)gy < (unsigned)rows ? (uint32_t)in[(size_t)gy * cols + gx] : 0u;
    }
    for (int s = 0; s < steps; s++) {
        edge[wave][0][lane] = c[1];
        edge[wave][1][lane] = c[RPW];
        __syncthreads();
        c[0] = wave > 0 ? edge[wave - 1][1][lane] : 0u;
        c[RPW + 1] = wave < 3 ? edge[wave + 1][0][lane] : 0u;
        __syncthreads();
        uint32_t nw[RPW];
#pragma unroll
        for (int i = 0; i < RPW; i++) {
            const uint32_t vs = c[i] + c[i + 1] + c[i + 2], live = c[i + 1];
            const uint32_t sum = lane_below(vs) + vs + lane_above(vs) - live;
            const bool next = (live == 1u && (sum == 2u || sum == 3u)) || (live == 0u && sum == 3u);
            nw[i] = next && colok && (unsigned)(gy0 + i) < (unsigned)rows ? 1u : 0u;
        }
#pragma unroll
        for (int i = 0; i < RPW; i++) c[i + 1] = nw[i];
    }
    if (lane >= K && lane < 64 - K && colok) {
#pragma unroll
        for (int i = 0; i < RPW; i++) {
            const int wy = wave * RPW + i, gy = gy0 + i;
            if (wy >= K && wy < H - K && gy < rows) out[(size_t)gy * cols + gx] = (int32_t)c[i + 1];
        }
    }
}

template <int K, int RPW>
static int gol_window_step(int32_t *out, const int32_t *in, int rows, int cols, int steps) {
    constexpr int TW = 64 - 2 * K, TH = 4 * RPW - 2 * K;
    const int tiles_x = (cols + TW - 1) / TW;
    const long blocks = (long)tiles_x * (((long)rows + TH - 1) / TH);
    MSL_REQUIRE(steps >= 1 && steps <= K, "msl_gol_iterate_i32: generations per launch out of range");
    return launch_split(blocks, 256, "msl_gol_iterate_i32", [&](int first, int count) {
        gol_window_kernel<K, RPW><<<count, 256, 0, ctx().stream>>>(out, in, rows, cols, steps, tiles_x, first);
    });
}

// Up to 2^20 cells, where launches bound the run, 8 generations of 64 x 64
// windows, above 4 of 64 x 32.
constexpr long kGolSmallCells = 1L << 20;
static int gol_window_gens(int rows, int cols) { return (long)rows * cols <= kGolSmallCells ? 8 : 4; }
static int gol_windows(int32_t *out, const int32_t *in, int rows, int cols, int steps) {
    return gol_window_gens(rows, cols) == 8 ? gol_window_step<8, 16>(out, in, rows, cols, steps)
                                            : gol_window_step<4, 8>(out, in, rows, cols, steps);
}

// Generation 1 of 64 columns x kFirstRows rows per wave, lane = column: the
// rule of the one-step kernel on the int cells, then one ballot per row.
// Bound by the 4 bytes per cell it reads (the two neighbour loads of a row
// hit the L1); 8 rows keep 30 loads in flight per lane.
constexpr int kFirstRows = 8;

__global__ __launch_bounds__(64) void gol_first_kernel(uint32_t *__restrict__ out, const int32_t *__restrict__ in,
                                                       int rows, int cols, int words, int tiles_x, int tile0) {
    const int lane = threadIdx.x;
    const int tile = tile0 + (int)xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const int x = tx * 64 + lane, y0 = ty * kFirstRows;
    const int xl = max(min(x - 1, cols - 1), 0), xc = min(x, cols - 1), xr = min(x + 1, cols - 1);
    uint32_t l[kFirstRows + 2], c[kFirstRows + 2], r[kFirstRows + 2];
#pragma unroll
    for (int i = 0; i < kFirstRows + 2; i++) {
        const int32_t *row = in + (size_t)min(max(y0 - 1 + i, 0), rows - 1) * cols;
        l[i] = (uint32_t)row[xl];
        c[i] = (uint32_t)row[xc];
        r[i] = (uint32_t)row[xr];
    }
    uint32_t h[kFirstRows + 2];
#pragma unroll
    for (int i = 0; i < kFirstRows + 2; i++) {
        const bool rowok = (unsigned)(y0 - 1 + i) < (unsigned)rows;
        c[i] = rowok && x < cols ? c[i] : 0u;
        h[i] = (rowok && x >= 1 && x - 1 < cols ? l[i] : 0u) + c[i] + (rowok && x + 1 < cols ? r[i] : 0u);
    }
    uint64_t mine = 0;  // lane i < kFirstRows keeps the word pair of row y0 + i
#pragma unroll
    for (int i = 0; i < kFirstRows; i++) {
        const uint32_t live = c[i + 1];
        const uint32_t sum = h[i] + h[i + 1] + h[i + 2] - live;
        const bool next = x < cols && ((live == 1u && (sum == 2u || sum == 3u)) || (live == 0u && sum == 3u));
        const uint64_t m = __ballot(next);
        if (lane == i) mine = m;
    }
    if (lane < kFirstRows && y0 + lane < rows) {
        uint32_t *o = out + (size_t)(y0 + lane) * words + 2 * tx;
        o[0] = (uint32_t)mine;
        if (2 * tx + 1 < words) o[1] = (uint32_t)(mine >> 32);
    }
}

// Up to kBitSteps generations of packed cells per launch.  One wave holds a
// window of 64 rows (lane = row) x kBitWords words of 32 columns: vertical
// neighbours come from the adjacent lanes by DPP, horizontal ones by funnel
// shifts, and the eight neighbour bits are added with carry-save logic (three-
// input boolean operations, about 17 per word and generation, for 2048
// cells).  The window edges lack neighbours, so after s generations only
// cells at least s from them are exact: the wave stores the rows of lanes
// kBitSteps .. 63 - kBitSteps and the inner words.  No LDS, no barrier; one
// wave per workgroup spreads small grids over all CUs.
// Cells outside the grid stay 0.
constexpr int kBitSteps = 16;
constexpr int kBitWords = 4;
constexpr int kBitRows = 64 - 2 * kBitSteps;        // rows stored per window
constexpr int kBitInner = kBitWords - 2;            // words stored per window
static_assert(kBitSteps <= 32, "one halo word per side covers 32 generations");
static_assert(kBitInner == 2, "the unpacking store writes 64 columns per row");

template <bool kUnpack>
__global__ __launch_bounds__(64) void gol_bits_kernel(void *__restrict__ out, const uint32_t *__restrict__ in,
                                                      int rows, int cols, int words, int steps, int tiles_x,
                                                      int tile0) {
    const int lane = threadIdx.x;
    const int tile = tile0 + (int)xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const int w0 = tx * kBitInner - 1;
    const int y = ty * kBitRows - kBitSteps + lane;
    const bool rowok = (unsigned)y < (unsigned)rows;
    uint32_t c[kBitWords], valid[kBitWords];
#pragma unroll
    for (int q = 0; q < kBitWords; q++) {
        const int w = w0 + q;
        const bool ok = rowok && (unsigned)w < (unsigned)words;
        c[q] = ok ? in[(size_t)y * words + w] : 0u;
        // columns of the last word beyond the grid stay 0
        valid[q] = ok ? (w == words - 1 && (cols & 31) ? (1u << (cols & 31)) - 1u : ~0u) : 0u;
    }
    for (int s = 0; s < steps; s++) {
        uint32_t nw[kBitWords];
#pragma unroll
        for (int q = 0; q < kBitWords; q++) {
            const uint32_t cc = c[q];
            // bit k of a word is column 32w + k
            const uint32_t lf = (cc << 1) | (q > 0 ? c[q - 1] >> 31 : 0u);
            const uint32_t rt = (cc >> 1) | (q + 1 < kBitWords ? c[q + 1] << 31 : 0u);
            const uint32_t s0 = lf ^ cc ^ rt, s1 = (lf & cc) | (lf & rt) | (cc & rt);  // left + self + right
            const uint32_t m0 = lf ^ rt, m1 = lf & rt;                                 // left + right
            const uint32_t u0 = lane_below(s0), u1 = lane_below(s1);                   // the row above
            const uint32_t d0 = lane_above(s0), d1 = lane_above(s1);                   // the row below
            const uint32_t bit0 = u0 ^ d0 ^ m0;
            const uint32_t c1 = (u0 & d0) | (u0 & m0) | (d0 & m0);
            // neighbours = bit0 + 2 (c1 + u1 + d1 + m1): 2 or 3 when exactly
            // one of the four twos is set
            const uint32_t none = ~(u1 | d1 | m1);
            const uint32_t one = (u1 ^ d1 ^ m1) & ~((u1 & d1) | (u1 & m1) | (d1 & m1));
            const uint32_t two = (c1 & none) | (~c1 & one);
            nw[q] = two & (bit0 | cc) & valid[q];  // 3 neighbours, or 2 and alive
        }
#pragma unroll
        for (int q = 0; q < kBitWords; q++) c[q] = nw[q];
    }
    if constexpr (kUnpack) {
        // one row at a time: its 64 inner columns as one bit mask, expanded
        // to one int per lane (lane = column), 256 bytes per store
        int32_t *o = static_cast<int32_t *>(out);
        const int x = (w0 + 1) * 32 + lane;
#pragma unroll
        for (int i = 0; i < kBitRows; i++) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)c[1], kBitSteps + i);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)c[2], kBitSteps + i);
            const int yo = ty * kBitRows + i;
            const uint64_t m = ((uint64_t)hi << 32) | lo;
            const int32_t v = __builtin_amdgcn_inverse_ballot_w64(m) ? 1 : 0;
            if (yo < rows && x < cols) o[(size_t)yo * cols + x] = v;
        }
    } else {
        uint32_t *o = static_cast<uint32_t *>(out);
        if (lane >= kBitSteps && lane < 64 - kBitSteps && y < rows) {
#pragma unroll
            for (int q = 1; q <= kBitInner; q++)
                if (w0 + q < words) o[(size_t)y * words + w0 + q] = c[q];
        }
    }
}

static int gol_bits_step(void *out, const uint32_t *in, int rows, int cols, int words, int steps, bool unpack) {
    const int tiles_x = (words + kBitInner - 1) / kBitInner;
    const long blocks = (long)tiles_x * (((long)rows + kBitRows - 1) / kBitRows);
    MSL_REQUIRE(steps >= 1 && steps <= kBitSteps, "msl_gol_iterate_i32: generations per launch out of range");
    return launch_split(blocks, 64, "msl_gol_iterate_i32", [&](int first, int count) {
        if (unpack)
            gol_bits_kernel<true><<<count, 64, 0, ctx().stream>>>(out, in, rows, cols, words, steps, tiles_x, first);
        else
            gol_bits_kernel<false><<<count, 64, 0, ctx().stream>>>(out, in, rows, cols, words, steps, tiles_x, first);
    });
}

// iters generations from d_a, the result in d_b when iters is odd, else in
// d_a.  Single columns, and odd counts that one launch of windows holds, run
// those.  Else the first launch reads d_a and packs into d_b; the launches after it
// alternate between two packed grids in the buffer that the result does not
// go to (for odd counts the first of them moves the packed grid from d_b to
// d_a, so at least two follow).  Two packed grids of rows * ceil(cols / 32)
// words fit one buffer from two columns on.
static int gol_run(int32_t *d_a, int32_t *d_b, int rows, int cols, int iters) {
    if (iters == 1) return gol_step(d_b, d_a, rows, cols);
    if (cols < 2 || ((iters & 1) && iters <= gol_window_gens(rows, cols))) {
        const std::vector<int> plan = generation_plan(iters, gol_window_gens(rows, cols));
        for (size_t k = 0; k < plan.size(); k++) {
            const int rc = gol_windows((k & 1) ? d_a : d_b, (k & 1) ? d_b : d_a, rows, cols, plan[k]);
            if (rc) return rc;
        }
        return MSL_OK;
    }
    const bool odd = iters & 1;
    const int words = (cols + 31) / 32;
    const size_t packed = (size_t)rows * words;
    const int tiles_x = (cols + 63) / 64;
    const long blocks = (long)tiles_x * (((long)rows + kFirstRows - 1) / kFirstRows);
    uint32_t *src = reinterpret_cast<uint32_t *>(d_b);
    int rc = launch_split(blocks, 64, "msl_gol_iterate_i32", [&](int first, int count) {
        gol_first_kernel<<<count, 64, 0, ctx().stream>>>(src, d_a, rows, cols, words, tiles_x, first);
    });
    if (rc) return rc;
    uint32_t *home = reinterpret_cast<uint32_t *>(odd ? d_a : d_b);  // the packed grids' buffer
    int left = iters - 1;
    int launches = (left + kBitSteps - 1) / kBitSteps;
    if (odd && launches < 2) launches = 2;
    for (int k = 0; k < launches; k++) {
        const int steps = (left + (launches - k) - 1) / (launches - k);
        left -= steps;
        const bool last = k + 1 == launches;
        void *dst;
        if (last)
            dst = odd ? d_b : d_a;
        else
            dst = src == home ? home + packed : home;
        rc = gol_bits_step(dst, src, rows, cols, words, steps, last);
        if (rc) return rc;
        src = static_cast<uint32_t *>(dst);
    }
    return MSL_OK;
}

}  // namespace mslhip

using namespace mslhip;

extern "C" {

int msl_gol_iterate_i32(int32_t *d_a, int32_t *d_b, int rows, int cols, int iters, int *h_result_in_b) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(iters >= 0, "msl_gol_iterate_i32: negative iteration count");
    MSL_REQUIRE(rows >= 0 && cols >= 0, "msl_gol_iterate_i32: negative shape");
    if (h_result_in_b) *h_result_in_b = iters & 1;
    if (iters == 0 || rows == 0 || cols == 0) return MSL_OK;
    MSL_REQUIRE((int64_t)rows * cols <= INT32_MAX, "msl_gol_iterate_i32: grid too large");
    MSL_REQUIRE(d_a && d_b && d_a != d_b, "msl_gol_iterate_i32: null or aliased buffers");
    const std::string key = graph_key("gol", d_a, d_b, rows, cols, iters, 0, 0);
    return run_cached_graph(key, [&]() { return gol_run(d_a, d_b, rows, cols, iters); });
}

}  // extern "C"
