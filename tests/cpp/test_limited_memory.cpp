// A tree whose device memory runs out: this program's hipMalloc and hipFree stand before the HIP
// library's and refuse what would pass a limit, and the calls have to do with what there is or
// leave the tree as it was.
//
//   test_limited_memory points    tables of a growing tree
//   test_limited_memory copies    a stage that fails leaves no copy of the caller's points under way
//   test_limited_memory equal     equal points over such an end: the first of them are kept
//   test_limited_memory compact   a run that ends for lack of records, taken up again with compaction
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <random>
#include <vector>

#include "voronoids.h"

static std::map<void*, size_t> g_sizes;
static size_t g_used = 0, g_limit = SIZE_MAX;

extern "C" hipError_t hipMalloc(void** p, size_t bytes) {
    using Fn = hipError_t (*)(void**, size_t);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "hipMalloc");
    if (bytes > g_limit || g_used > g_limit - bytes) return hipErrorOutOfMemory;
    const hipError_t e = real(p, bytes);
    if (e == hipSuccess) {
        g_sizes[*p] = bytes;
        g_used += bytes;
    }
    return e;
}
extern "C" hipError_t hipFree(void* p) {
    using Fn = hipError_t (*)(void*);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "hipFree");
    const auto it = g_sizes.find(p);
    if (it != g_sizes.end()) {
        g_used -= it->second;
        g_sizes.erase(it);
    }
    return real(p);
}

// copies from the caller's points not yet waited for
static const char *g_lo = nullptr, *g_hi = nullptr;
static int g_copies = 0, g_waited = 0;
extern "C" hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
    using Fn = hipError_t (*)(void*, const void*, size_t, hipMemcpyKind, hipStream_t);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "hipMemcpyAsync");
    if ((const char*)src >= g_lo && (const char*)src < g_hi) ++g_copies;
    return real(dst, src, bytes, kind, s);
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t s) {
    using Fn = hipError_t (*)(hipStream_t);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "hipStreamSynchronize");
    const hipError_t e = real(s);
    g_waited = g_copies;
    return e;
}

#define CHECK(x)                                                                                     \
    do {                                                                                             \
        if (!(x)) {                                                                                  \
            std::printf("line %d: %s (%s)\n", __LINE__, #x, vo_last_error() ? vo_last_error() : ""); \
            return 1;                                                                                \
        }                                                                                            \
    } while (0)

static std::vector<double> points(int dim, int64_t n, unsigned seed) {
    std::mt19937_64 g(seed);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    std::vector<double> p((size_t)n * dim);
    for (double& x : p) x = u(g);
    return p;
}

static int run_points() {
    const int64_t n = 200000;
    const std::vector<double> p = points(2, n, 1), more = points(2, 20, 2);
    vo_tri* t = nullptr;
    CHECK(vo_tri_create(0, 2, p.data(), n, &t) == VO_OK);
    CHECK(vo_tri_insert(t, p.data(), n, 0) == VO_OK);
    // records enough for a few points more: what is left to ask for are the point tables, 32 bytes a
    // point: 6.4 MB as needed, 9.6 MB with half as many points again
    CHECK(vo_tri_config(t, "reuse", 1) == VO_OK);
    const size_t used = g_used;
    g_limit = used + 5000000;                // neither
    for (int k = 0; k < 3; ++k) {
        CHECK(vo_tri_stage(t, more.data(), 10, 0) == VO_ERR_OOM);
        CHECK(g_used == used);
    }
    g_limit = used + 8500000;                // the tables needed
    CHECK(vo_tri_insert(t, more.data(), 10, 0) == VO_OK);
    g_limit = SIZE_MAX;
    CHECK(vo_tri_insert(t, more.data() + 20, 10, 0) == VO_OK);
    int64_t bad = -1, nv = 0;
    CHECK(vo_tri_check(t, &bad) == VO_OK && bad == 0);
    CHECK(vo_tri_counts(t, &nv, nullptr, nullptr) == VO_OK && nv == n + 20 + 3);
    vo_tri_destroy(t);
    CHECK(g_used == 0);
    return 0;
}

static int run_copies() {
    const int64_t n = 100000;
    const std::vector<double> p = points(3, n, 4);
    vo_tri* t = nullptr;
    CHECK(vo_tri_create(0, 3, p.data(), 100, &t) == VO_OK);
    g_lo = (const char*)p.data();
    g_hi = g_lo + sizeof(double) * p.size();
    // the tables fit (56 bytes a point), then less and less of what follows: scratch, the hint grid, records
    int refused = 0;
    for (size_t more = 5 << 20; more < ((size_t)64 << 20); more += 128 << 10) {
        g_limit = g_used + more;
        const int rc = vo_tri_stage(t, p.data(), n, 0);
        CHECK(rc == VO_OK || rc == VO_ERR_OOM);
        CHECK(g_waited == g_copies);
        if (rc == VO_OK) break;
        ++refused;
    }
    g_limit = SIZE_MAX;
    CHECK(refused > 0);
    g_lo = g_hi = nullptr;
    vo_tri_destroy(t);
    CHECK(g_used == 0);
    return 0;
}

static int run_equal() {
    const int64_t n = 30000;
    for (const int dim : {3, 2}) {
        std::vector<double> p = points(dim, n, 5);
        for (int64_t i = 0; i < n / 3; ++i)              // a third of the points twice
            for (int k = 0; k < dim; ++k) p[(size_t)(n - 1 - i) * dim + k] = p[(size_t)i * dim + k];
        int32_t *T[2] = {}, *E[2] = {};
        int64_t nT[2] = {}, nE[2] = {};
        for (int ended = 0; ended < 2; ++ended) {
            vo_tri* t = nullptr;
            CHECK(vo_tri_create(0, dim, p.data(), n, &t) == VO_OK);
            // (windows as large as the tree, and records for less than that, as below)
            CHECK(vo_tri_config(t, "alloc_stripes", 0) == VO_OK && vo_tri_config(t, "window_gamma_milli", 1000) == VO_OK);
            CHECK(vo_tri_config(t, "small_frac_lo_milli", 1) == VO_OK && vo_tri_config(t, "small_frac_hi_milli", 999) == VO_OK);
            CHECK(vo_tri_config(t, "walk_budget", 1) == VO_OK);
            CHECK(vo_tri_stage(t, p.data(), n, 0) == VO_OK);
            int rc = 0;
            if (ended) {
                g_limit = g_used + 1000000;
                CHECK(vo_tri_run(t) == VO_ERR_OOM);
                g_limit = SIZE_MAX;
            }
            rc = vo_tri_run(t);
            CHECK(rc == VO_ERR_DUPLICATE || (ended && rc == VO_OK));
            CHECK(vo_tri_canonical(t, &T[ended], &nT[ended], &E[ended], &nE[ended]) == VO_OK);
            vo_tri_destroy(t);
        }
        CHECK(nT[0] == nT[1] && nE[0] == nE[1]);
        CHECK(!std::memcmp(T[0], T[1], sizeof(int32_t) * nT[0] * (dim + 1)) && !std::memcmp(E[0], E[1], sizeof(int32_t) * nE[0] * 2));
        for (int k = 0; k < 2; ++k) {
            vo_free(T[k]);
            vo_free(E[k]);
        }
    }
    return 0;
}

static int run_compact() {
    const int64_t n = 30000;
    for (const int dim : {3, 2}) {
        const std::vector<double> p = points(dim, n, 3);
        vo_tri* t = nullptr;
        CHECK(vo_tri_create(0, dim, p.data(), n, &t) == VO_OK);
        // reserved at the stage: 30 (2D: 8) records a point, while windows as large as the tree reserve
        // 64 (16) for each of their points: that fails with about a third of the points inserted,
        // when points beyond the window have walked ahead
        CHECK(vo_tri_config(t, "alloc_stripes", 0) == VO_OK);
        CHECK(vo_tri_config(t, "window_gamma_milli", 1000) == VO_OK);
        CHECK(vo_tri_config(t, "small_frac_lo_milli", 1) == VO_OK);
        CHECK(vo_tri_config(t, "small_frac_hi_milli", 999) == VO_OK);
        CHECK(vo_tri_stage(t, p.data(), n, 0) == VO_OK);
        g_limit = g_used + 1000000;
        CHECK(vo_tri_run(t) == VO_ERR_OOM);
        g_limit = SIZE_MAX;
        int64_t nv = 0, bad = -1;
        CHECK(vo_tri_counts(t, &nv, nullptr, nullptr) == VO_OK);
        std::printf("%dD: %lld of %lld points in when the records ran out\n", dim, (long long)nv, (long long)n);
        std::fflush(stdout);
        CHECK(nv > n / 10 && nv < n / 2);
        CHECK(vo_tri_config(t, "compact_min", 16) == VO_OK);
        CHECK(vo_tri_config(t, "compact_ratio_milli", 1500) == VO_OK);
        CHECK(vo_tri_run(t) == VO_OK);
        CHECK(vo_tri_check(t, &bad) == VO_OK && bad == 0);
        CHECK(vo_tri_counts(t, &nv, nullptr, nullptr) == VO_OK && nv == n + dim + 1);
        vo_tri_destroy(t);
    }
    CHECK(g_used == 0);
    return 0;
}

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    int failed = 1;
    if (!std::strcmp(what, "points")) failed = run_points();
    if (!std::strcmp(what, "copies")) failed = run_copies();
    if (!std::strcmp(what, "equal")) failed = run_equal();
    if (!std::strcmp(what, "compact")) failed = run_compact();
    if (!failed) std::printf("%s: ok\n", what);
    return failed;
}
