// match_ridge (voronoids_amd/csrc/ridges.hpp) on the CPU, one lane after another: closed
// boundaries, where every ridge has its partner, and broken ones, where the search has to end.
#include <cstdio>
#include <vector>

struct int4 {
    int x, y, z, w;
};
#define __device__
#define __forceinline__ inline
static int atomicCAS(int* p, int expect, int value) {
    const int old = *p;
    if (old == expect) *p = value;
    return old;
}
#include "../../voronoids_amd/csrc/ridges.hpp"

static int failed = 0;
#define CHECK(x)                                                  \
    do {                                                          \
        if (!(x)) {                                               \
            std::printf("line %d: %s\n", __LINE__, #x);           \
            failed = 1;                                           \
        }                                                         \
    } while (0)

constexpr int MC = 64, SIZE = 128;

struct Result {
    std::vector<int> o;
    int pairs = 0, first = 0, none = 0;
};
static Result match(const std::vector<int4>& fv) {
    std::vector<int> tab(SIZE, -1);
    Result r;
    for (int q = 0; q < 3 * (int)fv.size(); ++q) {
        int h = -1;
        r.o.push_back(vo::match_ridge<SIZE>(fv.data(), tab.data(), q, h));
        if (r.o.back() >= 0) CHECK(vo::take_ridge(tab.data(), h, r.o.back()) == r.o.back());
        (r.o.back() >= 0 ? r.pairs : r.o.back() == vo::kRidgeFirst ? r.first : r.none)++;
    }
    return r;
}
static std::vector<int> ridge(const int4& f, int k) {
    const int a[3] = {f.y, f.z, f.w};
    std::vector<int> r;
    for (int i = 0; i < 3; ++i)
        if (i != k) r.push_back(a[i]);
    if (r[0] > r[1]) std::swap(r[0], r[1]);
    return r;
}

int main() {
    // a double pyramid over a ring of n vertices, 2 n facets: closed
    for (int n : {3, 4, 15, MC / 2})
        for (int stride : {1, 7, 65536}) {
            std::vector<int4> fv;
            for (int i = 0; i < n; ++i)
                for (int top = 0; top < 2; ++top) fv.push_back({9, (2 + i) * stride, (2 + (i + 1) % n) * stride, top * stride});
            const Result r = match(fv);
            CHECK(2 * r.pairs == 3 * (int)fv.size() && r.first == r.pairs && r.none == 0);
            for (int q = 0; q < (int)r.o.size(); ++q)
                if (r.o[q] >= 0) CHECK(ridge(fv[q / 3], q % 3) == ridge(fv[r.o[q] / 3], r.o[q] % 3));
        }
    // facets that share nothing: more ridges than entries
    {
        std::vector<int4> fv;
        for (int i = 0; i < MC; ++i) fv.push_back({9, 3 * i, 3 * i + 1, 3 * i + 2});
        const Result r = match(fv);
        CHECK(r.pairs == 0 && r.first == SIZE && r.none == 3 * MC - SIZE);
    }
    // two lanes that matched one entry in one step: one of them gets it
    {
        std::vector<int> tab(SIZE, -1);
        const std::vector<int4> fv = {{9, 0, 1, 2}, {9, 0, 1, 3}, {9, 0, 1, 4}};
        int h0 = -1, h1 = -1, h2 = -1;
        CHECK(vo::match_ridge<SIZE>(fv.data(), tab.data(), 2, h0) == vo::kRidgeFirst);
        CHECK(vo::match_ridge<SIZE>(fv.data(), tab.data(), 5, h1) == 2 && vo::match_ridge<SIZE>(fv.data(), tab.data(), 8, h2) == 2);
        CHECK(h1 == h0 && h2 == h0 && vo::take_ridge(tab.data(), h1, 2) == 2 && vo::take_ridge(tab.data(), h2, 2) != 2);
    }
    // three facets on one ridge, and ridges alone: the third is nobody's partner
    {
        const Result r = match({{9, 0, 1, 2}, {9, 0, 1, 3}, {9, 0, 1, 4}, {9, 5, 6, 7}});
        CHECK(r.pairs == 1 && r.first == 11 && r.none == 0);
    }
    if (!failed) std::printf("ridges: ok\n");
    return failed;
}
