// Runtime: context, stream, error state, residency, timing and graph capture.
//
// Replaces the device side of msl::initSkeletons / terminateSkeletons /
// syncStreams (reference src/muesli.cpp:63-158, 213-223): one process, one
// device, one stream; skeletons are stream-ordered instead of synchronising
// after every call.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <vector>

#include "common.hpp"

namespace mslhip {

static thread_local std::string g_last_error;
static Context g_ctx;
static std::mutex g_init_mutex;
static void *g_ws = nullptr;
// Pinned, device-accessible host buffer for small device-to-host copies: a
// kernel writes the bytes there, which avoids the copy engine's latency
// (a scalar fold result otherwise costs about as much as the fold).
constexpr size_t kSmallCopyBytes = 64 << 10;
static char *g_small = nullptr;
// Entries of host_post_slot, taken in turn: far more than calls can be waiting.
constexpr uint32_t kPostSlots = 1024;
static char *g_posts = nullptr;
static std::atomic<uint32_t> g_post_seq{0};
static size_t g_ws_bytes = 0;
static std::vector<void *> g_ws_retired;

void set_error(const std::string &msg) { g_last_error = msg; }

int fail(int code, const std::string &msg) {
    set_error(msg);
    return code;
}

int hip_fail(hipError_t e, const char *what) {
    std::string m = std::string(what) + ": " + hipGetErrorString(e);
    set_error(m);
    return e == hipErrorOutOfMemory ? MSL_E_NOMEM : MSL_E_HIP;
}

Context &ctx() { return g_ctx; }

int ensure_ready() {
    if (g_ctx.ready) return MSL_OK;
    return msl_init(0);
}

int tune_int(const char *name, int dflt) {
    static std::mutex mu;
    static std::map<std::string, int> cache;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(name);
    if (it != cache.end()) return it->second;
    int v = dflt;
    if (const char *e = std::getenv(name)) {
        char *end = nullptr;
        long x = std::strtol(e, &end, 10);
        if (end != e && x > 0 && x < (1 << 20)) v = (int)x;
    }
    cache[name] = v;
    return v;
}

long launch_limit(int threads) {
    static const long most_threads = [] {
        const int forced = tune_int("MSL_LAUNCH_THREADS", 0);
        return forced > 0 ? (long)forced : (1L << 32) - 1;
    }();
    return most_threads / threads > 0 ? most_threads / threads : 1;
}

__global__ void small_copy_kernel(char *__restrict__ dst, const char *__restrict__ src, size_t bytes) {
    for (size_t i = threadIdx.x; i < bytes; i += blockDim.x) dst[i] = src[i];
}

int check_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, what);
    return MSL_OK;
}

int host_post_slot(void **slot, uint32_t *seq) {
    int rc = ensure_ready();
    if (rc) return rc;
    do {
        *seq = g_post_seq.fetch_add(1) + 1;
    } while (*seq == 0);  // 0: nothing posted
    *slot = g_posts + 16 * (size_t)(*seq % kPostSlots);
    return MSL_OK;
}

// Polls for some 200 us (a posted result arrives 5 us before
// hipStreamSynchronize returns: a fold of 10007 floats 13.9 -> 8.7 us), then
// leaves the wait, and any error, to the stream.
int host_post_wait(const void *slot, uint32_t seq, uint64_t *bits, const char *name) {
    const volatile uint32_t *w = static_cast<const volatile uint32_t *>(slot);
    auto taken = [&]() {
        const uint32_t lo = w[0], hi = w[1], s = w[2], check = w[3];
        *bits = ((uint64_t)hi << 32) | lo;
        return s == seq && check == post_check(*bits, seq);
    };
    if (!g_ctx.capturing) {
        for (int k = 0; k < 4000; k++) {
            if (taken()) return MSL_OK;
            for (int p = 0; p < 2; p++) __builtin_ia32_pause();
        }
    }
    MSL_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
    if (!taken()) return fail(MSL_E_HIP, std::string(name) + ": the result did not arrive");
    return MSL_OK;
}

int workspace(size_t bytes, void **ptr) {
    if (bytes <= g_ws_bytes && g_ws) {
        *ptr = g_ws;
        return MSL_OK;
    }
    if (g_ctx.capturing) return fail(MSL_E_STATE, "workspace must grow outside graph capture; call once before capturing");
    // A smaller workspace is retired, not freed: graphs captured earlier may
    // still reference it.  Retired blocks are released by msl_finalize.
    if (g_ws) {
        g_ws_retired.push_back(g_ws);
        g_ws = nullptr;
        g_ws_bytes = 0;
    }
    size_t want = bytes < (1u << 20) ? (1u << 20) : bytes;
    MSL_HIP_TRY(hipMalloc(&g_ws, want));
    g_ws_bytes = want;
    *ptr = g_ws;
    return MSL_OK;
}

// ---- graph cache for iteration loops ---------------------------------------
struct GraphCache {
    std::mutex mu;
    std::map<std::string, hipGraphExec_t> graphs;
};
static GraphCache g_cache;

int run_cached_graph(const std::string &key, const std::function<int()> &body) {
    hipGraphExec_t exec = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_cache.mu);
        auto it = g_cache.graphs.find(key);
        if (it != g_cache.graphs.end()) exec = it->second;
    }
    if (!exec) {
        int rc = msl_graph_begin();
        if (rc) return rc;
        int brc = body();
        void *g = nullptr;
        int erc = msl_graph_end(&g);
        if (brc) {
            if (g) msl_graph_destroy(g);
            return brc;
        }
        if (erc) return erc;
        exec = (hipGraphExec_t)g;
        std::lock_guard<std::mutex> lock(g_cache.mu);
        if (g_cache.graphs.size() > 64) {
            // a cached graph may still be running: drain the stream first
            MSL_HIP_TRY(hipStreamSynchronize(ctx().stream));
            for (auto &kv : g_cache.graphs) (void)hipGraphExecDestroy(kv.second);
            g_cache.graphs.clear();
        }
        g_cache.graphs[key] = exec;
    }
    MSL_HIP_TRY(hipGraphLaunch(exec, ctx().stream));
    return MSL_OK;
}

std::string graph_key(const char *kind, const void *a, const void *b, long p0, long p1, long p2, long p3, long p4) {
    char buf[256];
    snprintf(buf, sizeof buf, "%s|%p|%p|%ld|%ld|%ld|%ld|%ld", kind, a, b, p0, p1, p2, p3, p4);
    return std::string(buf);
}

}  // namespace mslhip

using namespace mslhip;

extern "C" {

int msl_init(int device) {
    std::lock_guard<std::mutex> lock(g_init_mutex);
    if (g_ctx.ready) {
        if (g_ctx.device != device) return fail(MSL_E_STATE, "msl_init: already initialised on another device");
        return MSL_OK;
    }
    int count = 0;
    MSL_HIP_TRY(hipGetDeviceCount(&count));
    if (device < 0 || device >= count) return fail(MSL_E_INVALID, "msl_init: no such device");
    MSL_HIP_TRY(hipSetDevice(device));
    hipDeviceProp_t prop;
    MSL_HIP_TRY(hipGetDeviceProperties(&prop, device));
    // the allocation-free fold's scratch address on this device
    int rc = noalloc_setup(device);
    if (rc) return rc;
    g_ctx.device = device;
    g_ctx.num_cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    // Default-priority, non-blocking stream (one per device as in the reference).
    MSL_HIP_TRY(hipStreamCreateWithFlags(&g_ctx.stream, hipStreamNonBlocking));
    MSL_HIP_TRY(hipEventCreate(&g_ctx.t0));
    MSL_HIP_TRY(hipEventCreate(&g_ctx.t1));
    MSL_HIP_TRY(hipHostMalloc((void **)&g_small, kSmallCopyBytes, hipHostMallocDefault));
    MSL_HIP_TRY(hipHostMalloc((void **)&g_posts, 16 * kPostSlots, hipHostMallocDefault));
    std::memset(g_posts, 0, 16 * kPostSlots);
    g_ctx.ready = true;
    return MSL_OK;
}

int msl_finalize(void) {
    std::lock_guard<std::mutex> lock(g_init_mutex);
    if (!g_ctx.ready) return MSL_OK;
    MSL_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
    if (g_ws) {
        MSL_HIP_TRY(hipFree(g_ws));
        g_ws = nullptr;
        g_ws_bytes = 0;
    }
    for (void *p : g_ws_retired) hipFree(p);
    g_ws_retired.clear();
    if (g_small) {
        (void)hipHostFree(g_small);
        g_small = nullptr;
    }
    if (g_posts) {
        (void)hipHostFree(g_posts);
        g_posts = nullptr;
    }
    hipEventDestroy(g_ctx.t0);
    hipEventDestroy(g_ctx.t1);
    hipStreamDestroy(g_ctx.stream);
    g_ctx = Context();
    return MSL_OK;
}

const char *msl_last_error(void) { return g_last_error.c_str(); }

void *msl_stream(void) {
    if (ensure_ready() != MSL_OK) return nullptr;
    return (void *)g_ctx.stream;
}

int msl_synchronize(void) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
    return MSL_OK;
}

int msl_device_info(int *num_cus, int *warp_size, size_t *total_mem, char *name, int name_len) {
    int rc = ensure_ready();
    if (rc) return rc;
    hipDeviceProp_t prop;
    MSL_HIP_TRY(hipGetDeviceProperties(&prop, g_ctx.device));
    if (num_cus) *num_cus = prop.multiProcessorCount;
    if (warp_size) *warp_size = prop.warpSize;
    if (total_mem) *total_mem = prop.totalGlobalMem;
    if (name && name_len > 0) {
        std::snprintf(name, (size_t)name_len, "%s", prop.gcnArchName);
    }
    return MSL_OK;
}

int msl_malloc(void **d_ptr, size_t bytes) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(d_ptr != nullptr, "msl_malloc: null out-pointer");
    if (g_ctx.capturing) return fail(MSL_E_STATE, "msl_malloc: not allowed during graph capture");
    *d_ptr = nullptr;
    if (bytes == 0) return MSL_OK;
    MSL_HIP_TRY(hipMalloc(d_ptr, bytes));
    return MSL_OK;
}

int msl_free(void *d_ptr) {
    int rc = ensure_ready();
    if (rc) return rc;
    if (!d_ptr) return MSL_OK;
    if (g_ctx.capturing) return fail(MSL_E_STATE, "msl_free: not allowed during graph capture");
    MSL_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
    MSL_HIP_TRY(hipFree(d_ptr));
    return MSL_OK;
}

int msl_memcpy_h2d(void *d_dst, const void *h_src, size_t bytes) {
    int rc = ensure_ready();
    if (rc) return rc;
    if (bytes == 0) return MSL_OK;
    MSL_REQUIRE(d_dst && h_src, "msl_memcpy_h2d: null pointer");
    MSL_HIP_TRY(hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, g_ctx.stream));
    MSL_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
    return MSL_OK;
}

int msl_memcpy_d2h(void *h_dst, const void *d_src, size_t bytes) {
    int rc = ensure_ready();
    if (rc) return rc;
    if (bytes == 0) return MSL_OK;
    MSL_REQUIRE(h_dst && d_src, "msl_memcpy_d2h: null pointer");
    if (bytes <= kSmallCopyBytes && g_small && !g_ctx.capturing) {
        small_copy_kernel<<<1, 256, 0, g_ctx.stream>>>(g_small, (const char *)d_src, bytes);
        rc = check_launch("msl_memcpy_d2h");
        if (rc) return rc;
        MSL_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
        std::memcpy(h_dst, g_small, bytes);
        return MSL_OK;
    }
    MSL_HIP_TRY(hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, g_ctx.stream));
    MSL_HIP_TRY(hipStreamSynchronize(g_ctx.stream));
    return MSL_OK;
}

int msl_result_slot(void **h_slot, size_t *h_bytes) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(h_slot != nullptr, "msl_result_slot: null out-pointer");
    MSL_REQUIRE(g_small != nullptr, "msl_result_slot: no pinned slot");
    *h_slot = g_small;
    if (h_bytes) *h_bytes = kSmallCopyBytes;
    return MSL_OK;
}

int msl_memcpy_d2d(void *d_dst, const void *d_src, size_t bytes) {
    int rc = ensure_ready();
    if (rc) return rc;
    if (bytes == 0) return MSL_OK;
    MSL_REQUIRE(d_dst && d_src, "msl_memcpy_d2d: null pointer");
    MSL_HIP_TRY(hipMemcpyAsync(d_dst, d_src, bytes, hipMemcpyDeviceToDevice, g_ctx.stream));
    return MSL_OK;
}

int msl_timer_start(void) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_HIP_TRY(hipEventRecord(g_ctx.t0, g_ctx.stream));
    return MSL_OK;
}

int msl_timer_stop(float *h_ms) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(h_ms != nullptr, "msl_timer_stop: null out-pointer");
    MSL_HIP_TRY(hipEventRecord(g_ctx.t1, g_ctx.stream));
    MSL_HIP_TRY(hipEventSynchronize(g_ctx.t1));
    MSL_HIP_TRY(hipEventElapsedTime(h_ms, g_ctx.t0, g_ctx.t1));
    return MSL_OK;
}

int msl_selftest_launch_split(int64_t blocks, int threads, int *h_launches, int64_t *h_most_threads) {
    MSL_REQUIRE(blocks >= 0 && threads >= 1 && threads <= 1024, "msl_selftest_launch_split: bad launch");
    MSL_REQUIRE(h_launches != nullptr && h_most_threads != nullptr, "msl_selftest_launch_split: null out-pointer");
    *h_launches = 0;
    *h_most_threads = 0;
    int64_t next = 0;
    bool gapless = true;
    const int rc = launch_split_plan((long)blocks, threads, "msl_selftest_launch_split", [&](int first, int count) {
        gapless = gapless && first == next;
        next = (int64_t)first + count;
        ++*h_launches;
        if ((int64_t)count * threads > *h_most_threads) *h_most_threads = (int64_t)count * threads;
        return MSL_OK;
    });
    if (rc) return rc;
    return gapless && next == blocks ? MSL_OK : fail(MSL_E_STATE, "msl_selftest_launch_split: workgroups left out");
}

int msl_graph_begin(void) {
    int rc = ensure_ready();
    if (rc) return rc;
    if (g_ctx.capturing) return fail(MSL_E_STATE, "msl_graph_begin: capture already active");
    MSL_HIP_TRY(hipStreamBeginCapture(g_ctx.stream, hipStreamCaptureModeThreadLocal));
    g_ctx.capturing = true;
    return MSL_OK;
}

int msl_graph_end(void **graph) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(graph != nullptr, "msl_graph_end: null out-pointer");
    if (!g_ctx.capturing) return fail(MSL_E_STATE, "msl_graph_end: no capture active");
    hipGraph_t g = nullptr;
    g_ctx.capturing = false;
    MSL_HIP_TRY(hipStreamEndCapture(g_ctx.stream, &g));
    hipGraphExec_t exec = nullptr;
    hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (e != hipSuccess) return hip_fail(e, "hipGraphInstantiate");
    *graph = (void *)exec;
    return MSL_OK;
}

int msl_graph_launch(void *graph) {
    int rc = ensure_ready();
    if (rc) return rc;
    MSL_REQUIRE(graph != nullptr, "msl_graph_launch: null graph");
    MSL_HIP_TRY(hipGraphLaunch((hipGraphExec_t)graph, g_ctx.stream));
    return MSL_OK;
}

int msl_graph_destroy(void *graph) {
    if (!graph) return MSL_OK;
    MSL_HIP_TRY(hipGraphExecDestroy((hipGraphExec_t)graph));
    return MSL_OK;
}

}  // extern "C"
