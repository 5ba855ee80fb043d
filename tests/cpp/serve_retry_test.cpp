// A serving round that fails for want of memory, then runs again: the jobs'
// final states and sums are those of an undisturbed server.  The failure is
// forced on the host: this program's hipMalloc, which the library's calls bind
// to, refuses while g_refuse is set.
#include <dlfcn.h>

#include <cstdio>
#include <cstring>
#include <vector>

#include "msl_hip.h"

static bool g_refuse = false;

extern "C" int hipMalloc(void **p, size_t bytes) {
    typedef int (*Fn)(void **, size_t);
    static const Fn next = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "hipMalloc"));
    if (g_refuse || !next) return 2;  // hipErrorOutOfMemory
    return next(p, bytes);
}

#define CHECK(cond)                                                              \
    do {                                                                         \
        if (!(cond)) {                                                           \
            std::printf("line %d: %s (%s)\n", __LINE__, #cond, msl_last_error()); \
            return 1;                                                            \
        }                                                                        \
    } while (0)

static msl_job job(int kind, int steps, int r, int d0, int d1, int d2, unsigned seed) {
    msl_job j;
    std::memset(&j, 0, sizeof j);
    j.kind = kind;
    j.steps = steps;
    j.r = r;
    j.d0 = d0;
    j.d1 = d1;
    j.d2 = d2;
    j.nv = 0.5f;
    j.seed = seed;
    j.keep_final = 1;
    return j;
}

// The jobs' states and sums; `fail`: the first round is refused its memory.
static int serve(const std::vector<msl_job> &jobs, bool fail, std::vector<std::vector<float>> &states,
                 std::vector<double> &sums) {
    void *server = nullptr;
    CHECK(msl_server_create((size_t)64 << 20, 16, &server) == MSL_OK);
    std::vector<int64_t> ids(jobs.size());
    for (size_t k = 0; k < jobs.size(); k++) CHECK(msl_server_submit(server, &jobs[k], -1.0, &ids[k]) == MSL_OK);
    if (fail) {
        g_refuse = true;
        const int rc = msl_server_step(server, nullptr, nullptr);
        g_refuse = false;
        CHECK(rc == MSL_E_NOMEM);
    }
    CHECK(msl_server_drain(server) == MSL_OK);
    for (size_t k = 0; k < jobs.size(); k++) {
        const msl_job &j = jobs[k];
        std::vector<float> state((size_t)j.d0 * j.d1 * (j.kind == MSL_JOB_HEAT3D ? j.d2 : 1));
        msl_job_result res;
        CHECK(msl_server_poll(server, ids[k], &res, state.data(), state.size() * sizeof(float)) == MSL_OK);
        states.push_back(state);
        sums.push_back(res.sum);
    }
    CHECK(msl_server_destroy(server) == MSL_OK);
    return 0;
}

int main() {
    CHECK(msl_init(0) == MSL_OK);
    const std::vector<msl_job> jobs = {job(MSL_JOB_BLUR2D, 5, 3, 60, 70, 0, 1), job(MSL_JOB_BLUR2D, 70, 2, 90, 33, 0, 2),
                                       job(MSL_JOB_HEAT3D, 3, 0, 20, 18, 16, 3), job(MSL_JOB_HEAT3D, 1, 0, 9, 8, 7, 4)};
    std::vector<std::vector<float>> want, got;
    std::vector<double> want_sums, got_sums;
    if (serve(jobs, false, want, want_sums) || serve(jobs, true, got, got_sums)) return 1;
    for (size_t k = 0; k < jobs.size(); k++) {
        CHECK(std::memcmp(want[k].data(), got[k].data(), want[k].size() * sizeof(float)) == 0);
        CHECK(want_sums[k] == got_sums[k]);
    }
    std::printf("ok\n");
    return 0;
}
