// 2-D stencils on a rows x cols grid: mean blur of radius R and Game of Life.
//
// Reference: DM::mapStencil<f> launches one thread per output that makes
// (2r+1)^2 bounds-checked global reads through NPLMatrix::operator()
// (include/detail/map_kernels.cuh:159-168, include/nplmatrix.h:123-139).
//
// Here one wavefront owns a strip of 256 columns (64 lanes x 4 columns) and
// a segment of rows and marches down it with a register ring of row sums
// (strip_march): each input element is read once from HBM, each output is
// written once, and every output keeps the exact operation order of the
// scalar definition (bit-exact), with 2(2R+1) adds per output instead of
// (2R+1)^2.  The division by (2R+1)^2 is div_odd_square (multiply plus one
// FMA correction, checked bit-identical to IEEE division on all inputs).
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "blur_tile.hpp"
#include "strip.hpp"

namespace mslhip {

constexpr int kStripW = StripConsts<1, 4>::SW;  // columns per wave strip

// One wave per (strip, segment) item, four independent waves per 256-thread
// workgroup; each wave stages rows in its own LDS region, so only
// wave-level ordering is needed (no workgroup barrier).  C columns per lane:
// 4 (256-column strips) in general, 1 (64-column strips) for small grids,
// where four times as many strips keep more waves busy.
// Radii 9 and 10 with 256-column strips: at most two waves per SIMD (the
// register budget of the wave-uniform row addressing would allow three, but
// three waves per SIMD measured slower: spills, and a partial last round of
// the waves strip_shape launches).
template <int R, int C>
constexpr int strip_max_waves_per_eu() { return (C == 4 && R >= 9 && R <= 10) ? 2 : 8; }

// How the single-grid march ends its last ring period (strip_march_dir's
// kTail): r = 10 runs 128-row segments on streamed grids (see strip_shape),
// 148 input rows, one more than 7 ring periods of 21, so it ends with one
// checked period (8192^2: 4.39 -> 4.69 TB/s against whole periods of 64-row
// segments); every other radius keeps whole periods (r = 9 at 128 rows
// marches 146 of 147 rows anyway and lost 2 % to the checked copy).
constexpr bool strip_checked_tail(int r, int c) { return c == 4 && r == 10; }
template <int R, int C>
constexpr int strip_tail_mode() { return strip_checked_tail(R, C) ? 2 : 0; }

template <typename Pol, int MODE, bool NT = true, int C = 4>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, strip_max_waves_per_eu<Pol::R, C>())))
void strip_stencil_kernel(typename Pol::T *__restrict__ out,
                                                            const typename Pol::T *__restrict__ in, int rows, int cols,
                                                            typename Pol::T nv, int seg, int strips_x, int nitems,
                                                            Pol pol) {
    typedef typename Pol::T T;
    constexpr int R = Pol::R;
    __shared__ __attribute__((aligned(16))) T lds[4][2][StripConsts<R, C>::LDSW];

    const int wave = threadIdx.x >> 6;
    // the item is wave-uniform: with readfirstlane the row indices, clamps
    // and row bases of the march are scalar (r = 10: 205 -> 190 VALU
    // instructions per marched row, 170 -> 154 VGPRs)
    const int item = __builtin_amdgcn_readfirstlane((int)xcd_tile(blockIdx.x, gridDim.x) * 4 + wave);
    if (item >= nitems) return;
    const int sx = item % strips_x;
    const int sy = item / strips_x;
    const int y0 = sy * seg;
    // Grids that stay in the Infinity Cache run fewer waves per CU (see
    // strip_shape), so radii up to 10 that otherwise prefetch one row ahead
    // prefetch three there (measured: r = 5, 6 and 8 gain 4-25 % on 4096^2).
    constexpr int DQ = (NT || StripConsts<R, C>::D > 1 || R > 10) ? 0 : 3;
    strip_march<Pol, C, MODE, false, DQ, NT, strip_tail_mode<R, C>()>(out, in, rows, cols, nv, sx * StripConsts<R, C>::SW, y0,
                                             min(y0 + seg, rows), pol, lds[wave], nullptr, sy & 1);
}

// Two generations of the radius-R mean blur per wave item (strip2_march_dir):
// output strips of 256 - 2RP columns, segments marched in alternating
// directions as in strip_stencil_kernel.  Aligned or unaligned rows.
template <int R, int MODE, bool NT>
__global__ __launch_bounds__(256) void strip2_mean_kernel(float *__restrict__ out, const float *__restrict__ in,
                                                          int rows, int cols, float nv, int seg, int strips_x,
                                                          int nitems, MeanPolicy<R> pol) {
    typedef StripConsts<R, 4> K;
    __shared__ __attribute__((aligned(16))) float lds[4][4][K::LDSW];
    const int wave = threadIdx.x >> 6;
    // wave-uniform item: row indices and row bases of the march are scalar
    const int item = __builtin_amdgcn_readfirstlane((int)xcd_tile(blockIdx.x, gridDim.x) * 4 + wave);
    if (item >= nitems) return;
    const int sx = item % strips_x;
    const int sy = item / strips_x;
    const int y0 = sy * seg;
    const int xs = sx * (K::SW - 2 * K::RP);
    if (sy & 1)
        strip2_march_dir<R, MODE, true, NT>(out, in, rows, cols, nv, xs, y0, min(y0 + seg, rows), pol, lds[wave]);
    else
        strip2_march_dir<R, MODE, false, NT>(out, in, rows, cols, nv, xs, y0, min(y0 + seg, rows), pol, lds[wave]);
}

// Row access mode of a 4-column-per-lane march over these buffers.
template <typename T>
inline int row_mode(const T *in, const T *out, int cols) {
    const uintptr_t a = (uintptr_t)in | (uintptr_t)out;
    if ((cols & 3) == 0 && (a & 15u) == 0) return kAligned;
    if (cols >= 4 && (a & 3u) == 0) return kUnaligned;
    return kScalar;
}

// Grids whose single steps run the tile kernel (blur_tile.hip), and their
// tiles: 16-wave tiles (one row per thread) of the fewest rows that give at most
// one per CU, else 8-wave tiles of 64 rows once those give two per CU and of 32
// below; 128-column tiles, which read the fewest LDS cells per output, above
// kTile1WideCells and at radii above 10 (whose 64-column tiles hold few
// outputs) from four tiles per CU.  us per step, march / tile, on the same
// buffers: 300 x 1000 r = 2 4.1 / 3.6, 4 5.1 / 3.7; 1201 x 1999 r = 2 8.1 / 5.8, 4 9.2
// / 6.4; 2048^2 r = 2 7.5 / 7.8, 4 9.1 / 8.8, 5 11.6 / 9.3, 10 17.4 / 11.3, 16 34.1 / 15.3;
// 3000^2 r = 5 16.5 / 14.2, 9 19.6 / 17.8, 10 20.1 / 18.8, 11 24.4 / 20.0; 4000^2 r = 5
// 24.6 / 21.8, 8 26.5 / 24.2, 9 30.1 / 27.5, 11 37.6 / 31.0; 4096^2 r = 2 23.4 / 23.5;
// 5000^2 r = 5 33.5 / 31.8, 8 36.7 / 34.9, 9 41.4 / 40.4, 11 52.7 / 47.1; 5001^2 r = 5
// 39.2 / 31.8, 10 44.2 / 42.7; 5792^2 r = 5 47.0 / 42.4, 8 49.4 / 49.9, 16 77.5 / 87.8.
// On buffers that come from memory both take 4-8 us more.  Rows of 1024 to 6144
// columns in steps of 1024 do not differ from others (25 million cells r = 5 33.8
// / 31.7, at 4096 columns 34.1 / 34.4).  The radius whose march ends with a checked
// period (strip_checked_tail: a quarter faster than its neighbour's at most
// heights) marches on aligned rows from 13.6 million cells: r = 10 3400 x 3600 22.5 /
// 23.1, 4000^2 26.9 / 29.1, 5000^2 37.4 / 42.5, from memory 29.0 / 27.4, 33.4 / 34.0,
// 47.7 / 50.1 (r = 9 33.9 / 26.6, 37.1 / 32.9, 52.2 / 48.8).
constexpr long kTile1WideCells = 9L << 19;

// Whether the environment sets the shape of the march (strip_shape): the mean
// blur then marches at every size.
static bool march_forced() {
    static const bool forced = [] {
        const int c = tune_int("MSL_STRIP_C", 0);
        return tune_int("MSL_STRIP_SEG", 0) > 0 || c == 1 || c == 4;
    }();
    return forced;
}

// Grids of few rows: a tile costs about the same however few of its rows lie
// in the grid, a strip only the rows that do, so once there are several tiles
// per CU the march wins.  us per step, march / tile: 1 x 300000 r = 2 3.5 / 9.1,
// 10 8.7 / 17.4; 3 x 100000 4.0 / 4.7, 9.6 / 7.6; 4 x 750000 6.8 / 20.3, 19.5 /
// 40.4; 16 x 187500 6.8 / 8.1, 17.0 / 15.4; 24 x 125000 6.0 / 6.9, 17.1 / 12.3;
// r = 13 8 x 375000 24.7 / 24.4, 10 x 2000000 94 / 122, 12 x 1666666 102 / 104.
static bool thin_step(int rows, int cols, int r) {
    const int tiles = cols / (r > 10 ? 128 - 2 * r : 64 - 2 * r), cus = ctx().num_cus;
    return tiles >= 8 * cus && rows <= (r <= 10 ? 16 : (tiles >= 48 * cus ? 12 : 8));
}

// The same for iterations, whose tiles take several generations at once.  us
// per generation, march / tile: 1 x 300000 r = 2 3.8 / 5.8, 10 9.1 / 17.9; 2 x
// 150000 4.4 / 3.6, 9.5 / 10.6; 6 x 500000 6.3 / 10.4, 12.7 / 29.5; 10 x 300000
// 7.6 / 6.7, 14.7 / 21.4; 12 x 250000 8.0 / 6.3, 15.5 / 18.7; 16 x 187500 8.5 /
// 5.1, 17.4 / 15.8; two-generation march: 8 x 2500000 r = 2 18 / 44, 16 x 1250000 15
// / 25, 24 x 833333 20 / 20.
static bool thin_iterate(int rows, int cols, int r) {
    const int tiles = cols / (64 - 2 * r), cus = ctx().num_cus;
    return tiles >= 16 * cus && rows <= (tiles >= 64 * cus ? 16 : (r >= 8 ? 12 : 8));
}

static bool tile1_default(const float *in, const float *out, int r, int rows, int cols) {
    if (r < 2 || march_forced() || thin_step(rows, cols, r)) return false;
    const bool tail = strip_checked_tail(r, 4) && row_mode(in, out, cols) == kAligned;
    return (long)rows * cols <= (r <= 4 ? 3L << 20 : tail ? 13L << 20 : 25L << 20);
}

static TileShape tile1_shape(int rows, int cols, int r) {
    const int cus = ctx().num_cus, tile_w = (64 - 2 * r) / 4 * 4;
    auto tiles = [&](int h) { return (long)((cols + tile_w - 1) / tile_w) * ((rows + h - 1) / h); };
    for (int h = 8; h <= 32; h *= 2)
        if (tiles(h) <= cus) return TileShape{64, 1, h, 0.0};
    if ((long)rows * cols > kTile1WideCells || (r > 10 && tiles(64) > 4L * cus)) return TileShape{128, 4, 64, 0.0};
    return TileShape{64, 2, tiles(64) < 2L * cus ? 32 : 64, 0.0};
}

struct StripShape {
    int seg, strips_x, segs, nitems, c;
};

// Columns per lane and segment length (measured on 512^2 .. 8192^2 grids,
// r = 1, 5, 10).  A grid whose 256-column strips cannot give 8 waves per CU
// at 8-row segments marches 64-column strips (one column per lane) instead.
// Segments aim at 8 waves per CU with 256-column strips on grids that stay
// in the Infinity Cache, 16 on grids streamed from HBM (longer load latency
// to cover), and 32 with 64-column strips, which carry a quarter of the
// loads per row each.  They stay at least 4, 8 or 16 rows long for R <= 2,
// <= 6 and larger, so that the 2R halo rows read by each segment stay a
// modest fraction of its rows.
inline StripShape strip_shape(int rows, int cols, int r, int seg, bool streamed) {
    StripShape s;
    const long cus = ctx().num_cus;
    const long strips4 = (cols + kStripW - 1) / kStripW;
    s.c = tune_int("MSL_STRIP_C", 0);
    if (s.c != 1 && s.c != 4) s.c = r == 1 && strips4 * ((rows + 7) / 8) < 8 * cus ? 1 : 4;
    const int sw = 64 * s.c;
    s.strips_x = (cols + sw - 1) / sw;
    if (seg <= 0) seg = tune_int("MSL_STRIP_SEG", 0);
    if (seg <= 0) {
        // radii 9 and 10 run at most two waves per SIMD with 256-column
        // strips: one round of them (8 per CU) halves the 2R halo rows of
        // each output row against two rounds (8192^2: r = 9 4.45 -> 4.68
        // TB/s, r = 10 with the checked last period 4.39 -> 4.69)
        const bool two_waves = s.c == 4 && r >= 9 && r <= 10;  // strip_max_waves_per_eu
        const long target = cus * (s.c == 1 ? 32 : (streamed && !two_waves ? 16 : 8));
        // at most target waves (whole rounds, no trailing partial one)
        const long segs = std::max(1L, target / s.strips_x);
        seg = (int)((rows + segs - 1) / segs);
        const int seg_min = r <= 2 ? 4 : (r <= 6 ? 8 : 16);
        if (seg < seg_min) seg = seg_min;
    }
    s.seg = seg;
    s.segs = (rows + seg - 1) / seg;
    s.nitems = s.strips_x * s.segs;
    return s;
}

template <typename Pol>
int launch_strip(typename Pol::T *out, const typename Pol::T *in, int rows, int cols, typename Pol::T nv, Pol pol,
                 int seg, const char *name) {
    const bool nt = stream_stores((size_t)rows * cols * sizeof(*out));
    StripShape s = strip_shape(rows, cols, Pol::R, seg, nt);
    const int blocks = (s.nitems + 3) / 4;
    const int mode = row_mode(in, out, cols);
    if (s.c == 1)  // (above R = 1 only where MSL_STRIP_C asks for it)
        strip_stencil_kernel<Pol, kAligned, false, 1><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, s.seg,
                                                                                          s.strips_x, s.nitems, pol);
    else if (mode == kAligned && nt)
        strip_stencil_kernel<Pol, kAligned, true><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, s.seg,
                                                                                      s.strips_x, s.nitems, pol);
    else if (mode == kAligned)
        strip_stencil_kernel<Pol, kAligned, false><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, s.seg,
                                                                                       s.strips_x, s.nitems, pol);
    else if (mode == kUnaligned)
        strip_stencil_kernel<Pol, kUnaligned><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, s.seg,
                                                                                  s.strips_x, s.nitems, pol);
    else
        strip_stencil_kernel<Pol, kScalar><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, s.seg,
                                                                               s.strips_x, s.nitems, pol);
    return check_launch(name);
}

template <int R>
int launch_mean_r(float *out, const float *in, int rows, int cols, float nv, int seg) {
    return launch_strip(out, in, rows, cols, nv, MeanPolicy<R>::make(), seg, "msl_stencil2d_mean_f32");
}

typedef int (*MeanLauncher)(float *, const float *, int, int, float, int);
static const MeanLauncher kMeanLaunchers[] = {
    nullptr,           launch_mean_r<1>,  launch_mean_r<2>,  launch_mean_r<3>,  launch_mean_r<4>,
    launch_mean_r<5>,  launch_mean_r<6>,  launch_mean_r<7>,  launch_mean_r<8>,  launch_mean_r<9>,
    launch_mean_r<10>, launch_mean_r<11>, launch_mean_r<12>, launch_mean_r<13>, launch_mean_r<14>,
    launch_mean_r<15>, launch_mean_r<16>};
constexpr int kMaxMeanR = 16;

// Two generations per launch (strip2_mean_kernel) for radii 2 .. kMaxMean2R.
template <int R>
int launch_mean2_r(float *out, const float *in, int rows, int cols, float nv, int seg) {
    typedef StripConsts<R, 4> K;
    constexpr int sw = K::SW - 2 * K::RP;  // output columns per strip
    const bool nt = stream_stores((size_t)rows * cols * sizeof(float));
    const long cus = ctx().num_cus;
    const int strips_x = (cols + sw - 1) / sw;
    if (seg <= 0) seg = tune_int("MSL_STRIP2_SEG", 0);
    if (seg <= 0) {
        // waves per CU on streamed grids: 24 for r = 2, 8 above: one round
        // of long segments halves the 4R warm-up rows of each segment
        // (8192^2, 20 iterations, TB/s with 8 / 16 / 24 waves per CU:
        // r = 2 8.70 / 8.68 / 8.79, r = 3 8.05 / 7.44 / 7.83, r = 5
        // 7.05 / 6.06 / 5.86, r = 7 6.01 / 5.59 / 5.12);
        // MSL_STRIP2_WAVES overrides (tune_int caches one value per name, so
        // the radius-dependent default is applied here, not passed to it)
        int waves = tune_int("MSL_STRIP2_WAVES", 0);
        if (waves <= 0) waves = nt && R <= 2 ? 24 : 8;
        // whole rounds: at most target waves, so no partial round trails
        const long target = cus * waves;
        const long segs = std::max(1L, target / strips_x);
        seg = (int)((rows + segs - 1) / segs);
        if (seg < 8 * R) seg = 8 * R;
    }
    const long nitems = (long)strips_x * ((rows + seg - 1) / seg);
    MSL_REQUIRE(nitems <= INT32_MAX - 3, "msl_stencil2d_mean_iterate_f32: grid too large");
    const int blocks = (int)((nitems + 3) / 4);
    const MeanPolicy<R> pol = MeanPolicy<R>::make();
    const int mode = row_mode(in, out, cols);
    MSL_REQUIRE(mode != kScalar, "msl_stencil2d_mean_iterate_f32: two generations need rows of 4 or more cells");
    if (mode == kAligned && nt)
        strip2_mean_kernel<R, kAligned, true><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, seg,
                                                                               strips_x, (int)nitems, pol);
    else if (mode == kAligned)
        strip2_mean_kernel<R, kAligned, false><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, seg,
                                                                                strips_x, (int)nitems, pol);
    else
        strip2_mean_kernel<R, kUnaligned, false><<<blocks, 256, 0, ctx().stream>>>(out, in, rows, cols, nv, seg,
                                                                                  strips_x, (int)nitems, pol);
    return check_launch("msl_stencil2d_mean_iterate_f32");
}

static const MeanLauncher kMean2Launchers[] = {nullptr, nullptr, launch_mean2_r<2>, launch_mean2_r<3>,
                                               launch_mean2_r<4>, launch_mean2_r<5>, launch_mean2_r<6>,
                                               launch_mean2_r<7>};
constexpr int kMaxMean2R = 7;

// Radius 1, up to kMean3Steps generations per launch (mean3.hip).
int mean3_multi_step(float *out, const float *in, int rows, int cols, float nv, int steps);

int mean_step(float *out, const float *in, int rows, int cols, int r, float nv, int seg) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(rows >= 0 && cols >= 0, "msl_stencil2d_mean_f32: negative shape");
    MSL_REQUIRE(r >= 1 && r <= kMaxMeanR, "msl_stencil2d_mean_f32: radius must be in [1, 16]");
    MSL_REQUIRE((int64_t)rows * cols <= INT32_MAX && cols < (1 << 30), "msl_stencil2d_mean_f32: grid too large");
    if (rows == 0 || cols == 0) return MSL_OK;
    MSL_REQUIRE(out && in && out != in, "msl_stencil2d_mean_f32: null or aliased buffers");
    if (seg <= 0 && tile1_default(in, out, r, rows, cols))
        return blur_tile_step(out, in, rows, cols, r, nv, 1, tile1_shape(rows, cols, r));
    return kMeanLaunchers[r](out, in, rows, cols, nv, seg);
}

int gol_step(int32_t *out, const int32_t *in, int rows, int cols) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(rows >= 0 && cols >= 0, "msl_gol_i32: negative shape");
    MSL_REQUIRE((int64_t)rows * cols <= INT32_MAX && cols < (1 << 30), "msl_gol_i32: grid too large");
    if (rows == 0 || cols == 0) return MSL_OK;
    MSL_REQUIRE(out && in && out != in, "msl_gol_i32: null or aliased buffers");
    LifePolicy pol;
    pol.denom = 1.0f;
    return launch_strip(out, in, rows, cols, (int32_t)0, pol, 0, "msl_gol_i32");
}

constexpr int kMean3Steps = 6;  // most generations per launch of the radius-1 kernel and of the tiles

// Launch plan for `iters` generations of at most k per launch, alternating
// buffers: the result must end in b exactly when iters is odd (as with one
// launch per generation), so the number of launches must have the parity of
// iters; when it does not, one launch of several generations is split in
// two (there is one, since launches of one generation each number iters).
std::vector<int> generation_plan(int iters, int k) {
    std::vector<int> plan;
    for (int done = 0; done < iters; done += plan.back()) plan.push_back(std::min(k, iters - done));
    if ((int)(plan.size() & 1) != (iters & 1)) {
        for (size_t j = plan.size(); j-- > 0;)
            if (plan[j] >= 2) {
                plan[j] -= 1;
                plan.insert(plan.begin() + j + 1, 1);
                break;
            }
    }
    return plan;
}

// The same parity with the generations dealt evenly to as few launches as at
// most k each allow (LDS tiles: a launch's cost grows with its generations).
static std::vector<int> even_plan(int iters, int k) {
    std::vector<int> plan;
    int launches = iters > 0 ? (iters - 1) / k + 1 : 0;
    if ((launches ^ iters) & 1) launches++;
    for (; launches > 0; launches--) {
        plan.push_back((iters - 1) / launches + 1);
        iters -= plan.back();
    }
    return plan;
}

// Whether iterations of radius r run two generations per launch by default.
// Measured (GB/s, one vs two generations per launch): radii 2-4 gain from
// 4096^2 on (2 and 3 are asked for thin grids only, see tile_default), radii 5-7
// only on grids streamed from HBM (8192^2: r = 5 4.7 -> 7.2, r = 7 4.5 -> 6.1);
// on grids that stay in the Infinity Cache their longer halo recomputation
// costs more than the saved traffic (5792^2: r = 5 5.2 -> 4.6).
static bool mean2_default(int r, int rows, int cols) {
    const size_t bytes = (size_t)rows * cols * sizeof(float);
    if (r < 2 || r > kMaxMean2R) return false;
    return r <= 4 ? bytes >= ((size_t)32 << 20) : stream_stores(bytes);
}

// Grids whose iterations run in tiles (several generations per launch in
// LDS): radii 2 and 3 at every size, 4 to 8 up to 2^24 cells, above up to 2^22.2,
// thin grids apart.
// us per generation of the best tile and of the march: 8192^2 r = 2 42.7 / 59.0,
// 3 57.8 / 60.3, 4 63.9 / 60.9, 5 79.9 / 63.2; 4096^2 r = 4 17.0 / 19.3, 5 20.4
// / 26.4, 6 21.6 / 26.0, 8 28.0 / 28.3; 3000^2 r = 8 16.9 / 20.3, 9 20.6 / 22.5,
// 10 23.8 / 22.2; 2048^2 r = 10 13.0 / 17.7; 500 x 517 r = 3 2.1 / 4.9.
// At radii 2 and 3 from 32 MiB on, rows that one strip of the two-generation
// march (248 columns) holds stay with it, tiles / march: 125000 x 160 r = 2 20.0 /
// 18.8, 3 25.4 / 23.2; 250000 x 240 2 47 / 50, 3 69 / 54; 80000 x 250 3 23 / 38.
static bool one_strip(int r, int rows, int cols) {
    return r <= 3 && cols >= 150 && cols <= (r == 2 ? 190 : 248) && (long)rows * cols >= 8L << 20;
}

static bool tile_default(int r, int rows, int cols) {
    const long cells = (long)rows * cols;
    if (one_strip(r, rows, cols)) return false;
    return r >= 2 && !march_forced() && !thin_iterate(rows, cols, r) && (r <= 3 || cells <= (r <= 8 ? 1L << 24 : 9L << 19));
}

// Launches of an iteration; kLaunchStep is one generation by mean_step.
enum LaunchKind { kLaunchStep, kLaunchMulti3, kLaunchPair, kLaunchTile };

struct MeanLaunch {
    int gens;
    LaunchKind kind;
    TileShape tile;
};

// The launches of msl_stencil2d_mean_iterate_f32, in order: the
// six-generation register-window kernel at r = 1, tiles with the number of
// generations that the model prices lowest (tile_default), the two-generation
// march up to kMaxMean2R on larger grids with rows of 4 or more cells, else the
// one-step kernel.  MSL_MEAN_GENS = 1 or 2 forces one or two
// generations per launch for r >= 2 (read on every call, so a process can
// compare both).
static int mean_gens_env() {  // 0: not forced (unset, or any other value)
    const char *ge = getenv("MSL_MEAN_GENS");
    const int gens = ge ? atoi(ge) : 0;
    return gens == 1 || gens == 2 ? gens : 0;
}

static std::vector<MeanLaunch> mean_iterate_plan(const float *d_a, const float *d_b, int rows, int cols, int r,
                                                 int iters) {
    auto launches = [](const std::vector<int> &gens, LaunchKind kind) {
        std::vector<MeanLaunch> plan;
        for (int g : gens) plan.push_back(MeanLaunch{g, g == 1 ? kLaunchStep : kind, TileShape{}});
        return plan;
    };
    if (r == 1) return launches(generation_plan(iters, kMean3Steps), kLaunchMulti3);
    const int gens_env = mean_gens_env();
    const bool tiles = gens_env == 0 && iters > 1 && tile_default(r, rows, cols);
    const bool pairs = !tiles && r <= kMaxMean2R && row_mode(d_a, d_b, cols) != kScalar &&
                       (gens_env == 2 || (gens_env != 1 && mean2_default(r, rows, cols)));
    if (pairs) return launches(generation_plan(iters, 2), kLaunchPair);
    if (tiles) {
        TileShape shape[kMean3Steps + 1];
        std::vector<int> best;
        double best_us = 1e30;
        for (int k = 1; k <= kMean3Steps; k++) {
            shape[k] = tile_shape(rows, cols, r, k);
            if (shape[k].w == 0) break;
            const std::vector<int> gens = even_plan(iters, k);
            double us = 0.0;
            for (int g : gens) us += shape[g].us;
            if (us < best_us) {
                best_us = us;
                best = gens;
            }
        }
        // one generation by itself: as a single step runs it, but narrow rows in the
        // tile that was priced, where the step would march mostly empty strips (us
        // per generation, march / tile: 500000 x 120 r = 3 115 / 70, 1071428 x 56 182 /
        // 76)
        const bool step = cols >= 192 || tile1_default(d_a, d_b, r, rows, cols);
        std::vector<MeanLaunch> plan = launches(best, kLaunchTile);
        for (MeanLaunch &l : plan) {
            if (l.gens == 1 && !step) l.kind = kLaunchTile;
            if (l.kind == kLaunchTile) l.tile = shape[l.gens];
        }
        return plan;
    }
    return launches(std::vector<int>(iters, 1), kLaunchStep);
}

// ---- exhaustive check of div_odd_square against IEEE division -------------
__global__ void zero_u64_kernel(unsigned long long *p) { *p = 0ull; }

// Every 32-bit pattern x: compare div_odd_square(x) (or div6, the heat
// division, or div_plus0 against (0 + x) / d) with x / d bit for bit (NaN against NaN counts as equal);
// one atomic per block.
// kKind 0: div_odd_square, 1: div6, 2: div_plus0, 3: div6_plus0, 4: div6_fast
// where div6_suspect passes it and 5: div_pair on its domain, the last four
// against (0 + x) / d
template <int kKind>
__global__ __launch_bounds__(256) void div_check_kernel(float d, float rcp, unsigned long long *count,
                                                         RcpPair pair = RcpPair{}) {
    __shared__ unsigned int part[256];
    unsigned int bad = 0;
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < (1ull << 32); i += stride) {
        const float x = __uint_as_float((unsigned int)i);
        const float ref = __fdiv_rn(kKind >= 2 ? __fadd_rn(0.0f, x) : x, d);
        float got;
        if constexpr (kKind == 1) {
            got = div6(x);
        } else if constexpr (kKind == 2) {
            got = div_plus0(x, d, rcp);
        } else if constexpr (kKind == 3) {
            got = div6_plus0(x);
        } else if constexpr (kKind == 4) {
            got = div6_fast(x);
            if (div6_suspect(got)) got = ref;
        } else if constexpr (kKind == 5) {
            got = x == 0.0f || (x >= 0x1p-93f && x <= 0x1p112f) ? div_pair(__fadd_rn(0.0f, x), pair) : ref;
        } else {
            got = div_odd_square(x, d, rcp);
        }
        const bool same = (__float_as_uint(ref) == __float_as_uint(got)) || (ref != ref && got != got);
        bad += same ? 0u : 1u;
    }
    part[threadIdx.x] = bad;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0 && part[0]) atomicAdd(count, (unsigned long long)part[0]);
}

}  // namespace mslhip

using namespace mslhip;

extern "C" {

int msl_stencil2d_mean_f32(float *d_out, const float *d_in, int rows, int cols, int r, float nv) {
    return mean_step(d_out, d_in, rows, cols, r, nv, 0);
}

int msl_stencil2d_mean_iterate_f32(float *d_a, float *d_b, int rows, int cols, int r, float nv, int iters,
                                   int *h_result_in_b) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(iters >= 0, "msl_stencil2d_mean_iterate_f32: negative iteration count");
    MSL_REQUIRE(r >= 1 && r <= kMaxMeanR, "msl_stencil2d_mean_iterate_f32: radius must be in [1, 16]");
    MSL_REQUIRE(rows >= 0 && cols >= 0, "msl_stencil2d_mean_iterate_f32: negative shape");
    if (h_result_in_b) *h_result_in_b = iters & 1;
    if (iters == 0 || rows == 0 || cols == 0) return MSL_OK;
    union {
        float f;
        int32_t i;
    } nvb;
    nvb.f = nv;
    MSL_REQUIRE((int64_t)rows * cols <= INT32_MAX && cols < (1 << 30), "msl_stencil2d_mean_iterate_f32: grid too large");
    MSL_REQUIRE(d_a && d_b && d_a != d_b, "msl_stencil2d_mean_iterate_f32: null or aliased buffers");
    std::string key = graph_key("mean2d", d_a, d_b, rows, cols, r, nvb.i, iters);
    key += "|" + std::to_string(mean_gens_env());
    return run_cached_graph(key, [&]() {
        const std::vector<MeanLaunch> plan = mean_iterate_plan(d_a, d_b, rows, cols, r, iters);
        for (size_t k = 0; k < plan.size(); k++) {
            const MeanLaunch &l = plan[k];
            float *src = (k & 1) ? d_b : d_a;
            float *dst = (k & 1) ? d_a : d_b;
            int brc = MSL_OK;
            switch (l.kind) {
                case kLaunchStep: brc = mean_step(dst, src, rows, cols, r, nv, 0); break;
                case kLaunchMulti3: brc = mean3_multi_step(dst, src, rows, cols, nv, l.gens); break;
                case kLaunchPair: brc = kMean2Launchers[r](dst, src, rows, cols, nv, 0); break;
                case kLaunchTile: brc = blur_tile_step(dst, src, rows, cols, r, nv, l.gens, l.tile); break;
            }
            if (brc) return brc;
        }
        return MSL_OK;
    });
}

int msl_stencil2d_mean_iterate_plan(const float *d_a, const float *d_b, int rows, int cols, int r, int iters,
                                    int *h_gens, int capacity, int *h_launches) {
    MSL_REQUIRE(iters >= 0 && rows >= 0 && cols >= 0, "msl_stencil2d_mean_iterate_plan: negative argument");
    MSL_REQUIRE(r >= 1 && r <= kMaxMeanR, "msl_stencil2d_mean_iterate_plan: radius must be in [1, 16]");
    MSL_REQUIRE(h_launches != nullptr && capacity >= 0, "msl_stencil2d_mean_iterate_plan: bad output arguments");
    std::vector<MeanLaunch> plan;
    if (iters > 0 && rows > 0 && cols > 0) plan = mean_iterate_plan(d_a, d_b, rows, cols, r, iters);
    *h_launches = (int)plan.size();
    MSL_REQUIRE(h_gens != nullptr || plan.empty() || capacity == 0, "msl_stencil2d_mean_iterate_plan: null output");
    for (size_t k = 0; k < plan.size() && (int)k < capacity; k++) h_gens[k] = plan[k].gens;
    return MSL_OK;
}

int msl_stencil2d_mean_iterate_kernels(const float *d_a, const float *d_b, int rows, int cols, int r, int iters,
                                       int *h_kernels, int capacity, int *h_launches) {
    MSL_REQUIRE(iters >= 0 && rows >= 0 && cols >= 0, "msl_stencil2d_mean_iterate_kernels: negative argument");
    MSL_REQUIRE(r >= 1 && r <= kMaxMeanR, "msl_stencil2d_mean_iterate_kernels: radius must be in [1, 16]");
    MSL_REQUIRE(h_launches != nullptr && capacity >= 0, "msl_stencil2d_mean_iterate_kernels: bad output arguments");
    std::vector<MeanLaunch> plan;
    if (iters > 0 && rows > 0 && cols > 0) plan = mean_iterate_plan(d_a, d_b, rows, cols, r, iters);
    *h_launches = (int)plan.size();
    MSL_REQUIRE(h_kernels != nullptr || plan.empty() || capacity == 0, "msl_stencil2d_mean_iterate_kernels: null output");
    for (size_t k = 0; k < plan.size() && (int)k < capacity; k++) {
        switch (plan[k].kind) {
            case kLaunchStep:
                h_kernels[k] = tile1_default(d_a, d_b, r, rows, cols) ? MSL_MEAN_TILE : MSL_MEAN_MARCH;
                break;
            case kLaunchMulti3: h_kernels[k] = MSL_MEAN_WINDOW; break;
            case kLaunchPair: h_kernels[k] = MSL_MEAN_PAIR; break;
            case kLaunchTile: h_kernels[k] = MSL_MEAN_TILE; break;
        }
    }
    return MSL_OK;
}

int msl_selftest_div_odd_square(int r, uint64_t *h_mismatches) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(r >= 1 && r <= kMaxMeanR, "msl_selftest_div_odd_square: r must be in [1, 16]");
    MSL_REQUIRE(h_mismatches != nullptr, "msl_selftest_div_odd_square: null out-pointer");
    unsigned long long *d_count = nullptr;
    MSL_HIP_TRY(hipMalloc(&d_count, sizeof(unsigned long long)));
    zero_u64_kernel<<<1, 1, 0, ctx().stream>>>(d_count);
    const float d = (float)((2 * r + 1) * (2 * r + 1));
    div_check_kernel<0><<<ctx().num_cus * 8, 256, 0, ctx().stream>>>(d, 1.0f / d, d_count);
    div_check_kernel<2><<<ctx().num_cus * 8, 256, 0, ctx().stream>>>(d, 1.0f / d, d_count);
    div_check_kernel<5><<<ctx().num_cus * 8, 256, 0, ctx().stream>>>(d, 1.0f / d, d_count, rcp_pair(d));
    rc = check_launch("msl_selftest_div_odd_square");
    unsigned long long h = 0;
    hipError_t e = hipMemcpyAsync(&h, d_count, sizeof h, hipMemcpyDeviceToHost, ctx().stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx().stream);
    (void)hipFree(d_count);
    if (rc) return rc;
    if (e != hipSuccess) return hip_fail(e, "msl_selftest_div_odd_square");
    *h_mismatches = h;
    return MSL_OK;
}

int msl_selftest_div_six(uint64_t *h_mismatches) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(h_mismatches != nullptr, "msl_selftest_div_six: null out-pointer");
    unsigned long long *d_count = nullptr;
    MSL_HIP_TRY(hipMalloc(&d_count, sizeof(unsigned long long)));
    zero_u64_kernel<<<1, 1, 0, ctx().stream>>>(d_count);
    div_check_kernel<1><<<ctx().num_cus * 8, 256, 0, ctx().stream>>>(6.0f, 1.0f / 6.0f, d_count);
    div_check_kernel<3><<<ctx().num_cus * 8, 256, 0, ctx().stream>>>(6.0f, 1.0f / 6.0f, d_count);
    div_check_kernel<4><<<ctx().num_cus * 8, 256, 0, ctx().stream>>>(6.0f, 1.0f / 6.0f, d_count);
    rc = check_launch("msl_selftest_div_six");
    unsigned long long h = 0;
    hipError_t e = hipMemcpyAsync(&h, d_count, sizeof h, hipMemcpyDeviceToHost, ctx().stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx().stream);
    (void)hipFree(d_count);
    if (rc) return rc;
    if (e != hipSuccess) return hip_fail(e, "msl_selftest_div_six");
    *h_mismatches = h;
    return MSL_OK;
}

int msl_gol_i32(int32_t *d_out, const int32_t *d_in, int rows, int cols) { return gol_step(d_out, d_in, rows, cols); }

}  // extern "C"
