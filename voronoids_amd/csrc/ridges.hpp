// ridges.hpp -- partners of the ridges of a 3D cavity boundary.
//
// fv: the new simplices' vertex tuples in LDS, p first, then the facet's three vertices; ridge k of
// facet j is the facet's vertices other than fv[j][k].  The boundary of a cavity is a closed
// manifold, so exactly one other facet holds all of the ridge; its new simplex shares the face
// across the ridge.
#pragma once

namespace vo {

constexpr int kRidgeFirst = -1;    // the first of its two to come; also a free entry of the table
constexpr int kRidgeNoRoom = -2;   // no entry left
constexpr int kRidgePaired = -3;   // entry of a ridge whose partner has come

// A hash table of ridges in LDS (open addressing; an entry is j * 3 + k - 1 of the ridge that came
// first).  Returns the entry of the ridge with the same two vertices and its place h, kRidgeFirst for
// the first of the two to come, kRidgeNoRoom where every entry is taken by others.  A scan of the facets reads
// up to nf tuples per ridge, 3 nf ridges, 30 facets on average and up to 100: run at n = 4M
// 74.6 -> 66.8 ms, 10^5 16.6 -> 13.6 ms.
//
// On a closed boundary every ridge finds its one partner, and 1.5 entries a facet fill at most
// three quarters of the table.  A tree whose vertices were moved or swapped by hand need not have
// one: then ridges without a partner can be more than the table holds, so a search ends after
// SIZE entries, and three facets may hold one ridge, so the caller has to take an entry (take_ridge)
// and counts the ones it got.
template <int SIZE> __device__ __forceinline__ int match_ridge(const int4* fv, int* tab, int q, int& h) {
    static_assert((SIZE & (SIZE - 1)) == 0, "a power of two");
    const int4 a = fv[q / 3];
    const int k = q % 3;
    const int u = k == 0 ? a.z : a.y, w = k == 2 ? a.z : a.w;
    const int lo = u < w ? u : w, hi = u < w ? w : u;
    h = (int)((((unsigned)lo * 0x9E3779B1u) ^ ((unsigned)hi * 0x85EBCA77u)) >> 16) & (SIZE - 1);
    for (int n = 0; n < SIZE; ++n) {
        const int o = atomicCAS(&tab[h], kRidgeFirst, q);
        if (o == kRidgeFirst) return kRidgeFirst;
        if (o >= 0) {
            const int4 b = fv[o / 3];
            const int m = o % 3;
            const int bu = m == 0 ? b.z : b.y, bw = m == 2 ? b.z : b.w;
            if ((bu == u && bw == w) || (bu == w && bw == u)) return o;
        }
        h = (h + 1) & (SIZE - 1);
    }
    return kRidgeNoRoom;
}

// Entry o at h to its second ridge: o for the one that gets it (lanes that matched in one step may
// be two).  Apart from the search, so that its trip to LDS runs under the links' stores (with it
// inside, a round at 3D n = 10^4 took 0.3 us longer).
__device__ __forceinline__ int take_ridge(int* tab, int h, int o) {
    return o >= 0 ? atomicCAS(&tab[h], o, kRidgePaired) : kRidgePaired;
}

}  // namespace vo
