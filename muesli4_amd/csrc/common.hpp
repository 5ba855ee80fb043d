// Internal helpers shared by the translation units of libmsl_hip.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <functional>
#include <string>

#include "msl_hip.h"

namespace mslhip {

// ---- error state ---------------------------------------------------------
void set_error(const std::string &msg);
int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *what);

#define MSL_HIP_TRY(expr)                                   \
    do {                                                    \
        hipError_t _e = (expr);                             \
        if (_e != hipSuccess) return ::mslhip::hip_fail(_e, #expr); \
    } while (0)

#define MSL_REQUIRE(cond, msg)                                          \
    do {                                                                \
        if (!(cond)) return ::mslhip::fail(MSL_E_INVALID, (msg));       \
    } while (0)

// ---- context --------------------------------------------------------------
struct Context {
    bool ready = false;
    int device = 0;
    int num_cus = 256;
    hipStream_t stream = nullptr;
    hipEvent_t t0 = nullptr, t1 = nullptr;
    bool capturing = false;
};

Context &ctx();
// Returns MSL_OK when the context is initialised (initialising device 0 on
// first use), else an error code.
int ensure_ready();
// Launch-error check after a kernel launch.
int check_launch(const char *what);

// Scratch workspace owned by the context (grown outside graph capture only).
int workspace(size_t bytes, void **ptr);
// Results that a kernel posts to the host itself.  host_post_slot gives a
// 16-byte entry of pinned memory and a sequence number for one launch, whose
// last thread calls post_result; host_post_wait returns the posted 64 bits.
int host_post_slot(void **slot, uint32_t *seq);
int host_post_wait(const void *slot, uint32_t seq, uint64_t *bits, const char *name);

// Looks up, with `device` current, the device address of the fixed scratch
// array of the allocation-free fold (fold.hip); called once per device by
// msl_init.
int noalloc_setup(int device);

// Integer tuning knob from the environment, else dflt.  The result of the
// first call is cached per name, dflt included: callers whose default
// varies pass a fixed sentinel (0) and apply their default themselves.
int tune_int(const char *name, int dflt);

// Iteration loops captured once into a HIP graph and replayed: runs the
// graph cached under `key`, capturing body()'s launches first when there is
// none (runtime.hip).
std::string graph_key(const char *kind, const void *a, const void *b, long p0, long p1, long p2, long p3, long p4);
int run_cached_graph(const std::string &key, const std::function<int()> &body);

// Most workgroups of one launch: HIP takes fewer than 2^32 threads per launch
// (MSL_LAUNCH_THREADS in the environment lowers that bound).
long launch_limit(int threads);
// Launches workgroups [0, blocks) of a kernel whose grid grows with the data,
// in as many launches of (first workgroup, count) as that bound asks for.
template <typename Part>
int launch_split_plan(long blocks, int threads, const char *name, Part part) {
    MSL_REQUIRE(blocks <= INT32_MAX, std::string(name) + ": grid too large");
    const long most = launch_limit(threads);
    for (long first = 0; first < blocks; first += most) {
        const int rc = part((int)first, (int)(blocks - first < most ? blocks - first : most));
        if (rc) return rc;
    }
    return MSL_OK;
}
template <typename Launch>
int launch_split(long blocks, int threads, const char *name, Launch launch) {
    return launch_split_plan(blocks, threads, name, [&](int first, int count) {
        launch(first, count);
        return check_launch(name);
    });
}

// Number of workgroups that fills the device for a streaming kernel.
inline int streaming_blocks(size_t work_items, int threads, int per_cu) {
    size_t want = (work_items + threads - 1) / threads;
    size_t cap = (size_t)ctx().num_cus * per_cu;
    if (want > cap) want = cap;
    if (want < 1) want = 1;
    return (int)want;
}

// Store policy of the stencil marches.  A grid of up to 128 MiB ping-pongs
// with its partner (256 MiB together) inside the 256 MiB Infinity Cache
// well enough that ordinary stores win: the next step finds its input there.
// Larger grids use non-temporal stores, which do not allocate in the
// Infinity Cache and so leave it to the input being read (measured on
// 8192^2 and 512^3 ping-pongs: ordinary stores lose 2-7 %).
constexpr size_t kCachedStoreMaxBytes = (size_t)128 << 20;
inline bool stream_stores(size_t grid_bytes) { return grid_bytes > kCachedStoreMaxBytes; }

// ---- device-side helpers --------------------------------------------------
__host__ __device__ inline uint64_t hash64(uint64_t seed, uint64_t idx) {
    uint64_t z = seed + (idx + 1) * 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

// One 16-byte store of the value, its sequence number and a check word over
// both: the host takes the entry only when the three agree, so the order in
// which its bytes arrive does not matter.
__host__ __device__ inline uint32_t post_check(uint64_t bits, uint32_t seq) {
    return ((uint32_t)bits * 0x9E3779B1u) ^ ((uint32_t)(bits >> 32) * 0x85EBCA77u) ^ (seq * 0xC2B2AE3Du) ^ 0x27D4EB2Fu;
}
__device__ __forceinline__ void post_result(void *slot, uint32_t seq, uint64_t bits) {
    typedef uint32_t post_t __attribute__((ext_vector_type(4)));
    const post_t v = {(uint32_t)bits, (uint32_t)(bits >> 32), seq, post_check(bits, seq)};
    __builtin_nontemporal_store(v, static_cast<post_t *>(slot));
}

// IEEE single operations that the compiler may not contract into an FMA.
__device__ __forceinline__ float add_rn(float a, float b) { return __fadd_rn(a, b); }
__device__ __forceinline__ float mul_rn(float a, float b) { return __fmul_rn(a, b); }

// Knuth's TwoSum: s = RN(a + b) and the exact rounding error e, so that
// a + b == s + e in real arithmetic.
__device__ __forceinline__ void two_sum(float a, float b, float &s, float &e) {
    s = __fadd_rn(a, b);
    float bp = __fsub_rn(s, a);
    float ap = __fsub_rn(s, bp);
    e = __fadd_rn(__fsub_rn(a, ap), __fsub_rn(b, bp));
}

// Workgroup barrier that orders LDS accesses only.  __syncthreads() also
// waits for every outstanding global load of the wave, which would drain the
// software prefetch queues of the stencil marches at each step; the
// "local"-only fences make the barrier wait for LDS operations alone.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Orders one wave's own LDS accesses (RAW/WAR between its lanes).  A wave's
// LDS instructions execute in issue order, so this is a compiler-level
// barrier only: no wait on outstanding global loads, no workgroup barrier.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Correctly rounded x / d for the divisors d = (2r+1)^2, r = 1..16, without
// the IEEE division sequence: q0 = x*rcp (rcp = RN(1/d)), the remainder
// x - q0*d is exact with one FMA, and one FMA correction gives RN(x/d).
// When the remainder is 0 (q0 exact; covers -0) or NaN (x infinite or NaN)
// q0 itself is the answer.  Checked bit-for-bit against IEEE division for
// all 2^32 inputs of every such d by msl_selftest_div_odd_square.
__device__ __forceinline__ float div_odd_square(float x, float d, float rcp) {
    float q0 = __fmul_rn(x, rcp);
    float r = __fmaf_rn(-q0, d, x);
    float q1 = __fmaf_rn(r, rcp, q0);
    return (r != 0.0f && r == r) ? q1 : q0;
}

// Correctly rounded (0 + x) / d for the same divisors: the finish of a sum
// that the caller formed without its leading "0 +" (which only turns a -0
// sum into +0).  The sequence of div_odd_square, with the remainder clamped
// to a finite value instead of selecting q0: for infinite x the correction
// then adds a finite term to q0 = +-inf, for NaN x it stays NaN, for x = -0
// the remainder +0 gives +0 + -0 = +0, and for an exact quotient q0 + 0 =
// q0.  Checked bit-for-bit against IEEE division of 0 + x on all 2^32
// inputs by msl_selftest_div_odd_square.
__device__ __forceinline__ float div_plus0(float x, float d, float rcp) {
    const float q0 = __fmul_rn(x, rcp);
    const float r = __fmaf_rn(-q0, d, x);
    const float rc = __builtin_amdgcn_fmed3f(r, -3.0e38f, 3.0e38f);  // NaN -> -3e38
    return __fmaf_rn(rc, rcp, q0);
}

// Correctly rounded x / d by two operations: 1/d = hi + lo with hi rounded
// down (so lo >= 0), and RN(x * hi + RN(x * lo)) is the quotient as long as the
// second product keeps its precision (Brisebarre and Muller, "Correctly
// rounded multiplication by arbitrary precision constants"; for these d the
// quotient stays at least ulp / 2d away from a rounding boundary).  For x = +0
// and 2^-93 <= x <= 2^112 only: checked bit-for-bit against IEEE division on
// all of them by msl_selftest_div_odd_square.
struct RcpPair {
    float hi, lo;
};
inline RcpPair rcp_pair(double d) {
    const double q = 1.0 / d;
    float hi = (float)q;
    if ((double)hi > q) hi = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, hi) - 1u);
    return RcpPair{hi, (float)(q - (double)hi)};
}
__device__ __forceinline__ float div_pair(float x, RcpPair p) { return __fmaf_rn(x, p.hi, __fmul_rn(x, p.lo)); }

// Collects whether cells are all +0 or in [2^-40, 2^100], so that several
// generations of means of them stay in the domain of div_pair: a mean of
// (2r+1)^2 such cells is 0 or at least a (2r+1)^2-th of the smallest.
struct PairDomain {
    uint32_t most = 0u, least = ~0u;
    __device__ __forceinline__ void push(float x) {
        const uint32_t u = __float_as_uint(x);  // negative cells, -0 and NaN are above every bound
        most = u > most ? u : most;
        least = u - 1u < least ? u - 1u : least;  // +0 becomes the largest
    }
    __device__ __forceinline__ bool ok() const {
        return most <= 0x71800000u && least >= 0x2B800000u - 1u;  // 2^100, 2^-40
    }
};

// Correctly rounded x / 6 (the heat functor's division) by the sequence of
// div_odd_square with rcp = RN(1/6), plus one case that sequence misses: a
// quotient exactly halfway between two subnormals (x = (6k+3) * 2^-149, where
// the remainder r = x - 6*q0 is +-3 * 2^-149 and the inexact reciprocal
// always rounds away from q0), which must round to the even one of q0 and
// q1 = q0 +- 2^-149.  Branch-free; checked bit-for-bit against IEEE
// division on all 2^32 inputs by msl_selftest_div_six.
__device__ __forceinline__ float div6(float x) {
    constexpr float kRcp6 = 1.0f / 6.0f;
    const float q0 = __fmul_rn(x, kRcp6);
    const float r = __fmaf_rn(-q0, 6.0f, x);
    const float q1 = __fmaf_rn(r, kRcp6, q0);
    const bool keep_even_q0 = fabsf(r) == 0x1.8p-148f && (__float_as_uint(q0) & 1u) == 0u;
    return (r != 0.0f && r == r && !keep_even_q0) ? q1 : q0;
}

// Correctly rounded (0 + x) / 6 for a sum formed without its leading "0 +":
// div6 with the remainder clamped to a finite value as in div_plus0.
// Checked on all 2^32 inputs by msl_selftest_div_six.
__device__ __forceinline__ float div6_plus0(float x) {
    constexpr float kRcp6 = 1.0f / 6.0f;
    const float q0 = __fmul_rn(x, kRcp6);
    const float r = __fmaf_rn(-q0, 6.0f, x);
    const bool keep_even_q0 = fabsf(r) == 0x1.8p-148f && (__float_as_uint(q0) & 1u) == 0u;
    const float q = __fmaf_rn(__builtin_amdgcn_fmed3f(r, -3.0e38f, 3.0e38f), kRcp6, q0);
    return keep_even_q0 ? q0 : q;
}

// div6_plus0 by the plain multiply-and-correct sequence (3 operations instead
// of 9): right whenever its result is zero or normal.  Infinite and NaN sums
// give NaN, and a halfway quotient that the sequence rounds the wrong way is
// subnormal, so callers check their results with div6_suspect (one compare)
// and redo the ones that it flags with div6_plus0.  Checked on all 2^32
// inputs by msl_selftest_div_six.
__device__ __forceinline__ float div6_fast(float x) {
    constexpr float kRcp6 = 1.0f / 6.0f;
    const float q0 = __fmul_rn(x, kRcp6);
    return __fmaf_rn(__fmaf_rn(-q0, 6.0f, x), kRcp6, q0);
}
__device__ __forceinline__ bool div6_suspect(float q) {
    return __builtin_amdgcn_classf(q, 0x297);  // NaN, +-infinity, +-subnormal
}

// Remap blockIdx so that each XCD (blocks are dealt round-robin to the 8
// XCDs) receives a contiguous range of logical tiles; neighbouring tiles
// then share one L2.  The first nblocks % 8 XCDs get one tile more.  (With the
// identity for grids that do not split evenly, a radius-7 step of a 1024^2 grid by
// 484 tiles took 7.1 us, and now 5.3; 1201 x 1999, r = 7: 8.9 -> 7.0 us.)
__device__ __forceinline__ unsigned xcd_tile(unsigned bid, unsigned nblocks) {
    constexpr unsigned kXcd = 8;
    const unsigned xcd = bid % kXcd, rest = nblocks % kXcd;
    return xcd * (nblocks / kXcd) + (xcd < rest ? xcd : rest) + bid / kXcd;
}

// The same for launches whose tiles differ in cost (the hardware hands out
// workgroups in order as others end, so costs balance by themselves): within
// each 64 workgroups, every XCD takes 8 neighbours.
__device__ __forceinline__ unsigned xcd_mixed_tile(unsigned bid, unsigned nblocks) {
    constexpr unsigned kXcd = 8, kNear = 8, kGroup = kXcd * kNear;
    const unsigned base = bid / kGroup * kGroup, k = bid - base;
    return base + kGroup > nblocks ? bid : base + k % kXcd * kNear + k / kXcd;
}

}  // namespace mslhip
