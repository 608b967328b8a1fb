// canon.hpp -- canonical form of a triangulation on the device: the simplices with only real
// vertices as sorted vertex tuples in lexicographic order, and the unique edges between real
// vertices, sorted (the form the parity tests compare; the reference's check_delaunay walks the
// DashMaps instead, src/delaunay_tree.rs:512-541, :642-671).
//
// Two ways to it:
//  * buckets (k_canon_rows .. k_canon_edges): simplices and edges go to the bucket of their least
//    vertex, whose few entries are then sorted in LDS.  A vertex has about 7 simplices and 13 edge
//    entries, so one scatter and one short sort take the place of a radix sort's 14 to 18 passes
//    over all of them;
//  * where a vertex's bucket outgrows LDS (kCanonBig), the same rows and edge entries by a stable
//    least-significant-digit radix sort of 64-bit keys (8-bit digits, optional 32-bit payload).  Each
//    sort pass is per-tile digit histograms (tile = 4,096 elements, one block), a scan of the
//    histograms in digit-major order (tile offsets of every digit), and a stable scatter in which
//    each wavefront ranks its 64 elements per digit with ballots.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"

namespace vo {

// ---------------------------------------------------------------- buckets
constexpr int kCanonSmall = 64;           // bucket entries sorted by a group of 16 lanes
constexpr int kCanonBig = 4096;           // bucket entries sorted by one block in LDS
constexpr int kCanonNone = 0x3fffffff;    // "no point" (a super vertex); point indices are below 2^30
constexpr int kScanTile = 4096;

struct CanonTot {
    unsigned rows;         // simplices with at least two points
    unsigned n_big;        // vertices with a bucket above kCanonSmall
    unsigned max_bucket;
    unsigned pad;
    unsigned long long te; // simplex total | edge entry total << 32
    unsigned long long ne; // unique edges
};

// One simplex: r = its point indices in any order (kCanonNone for a super vertex), bit k of
// `least` set when the simplex index is below that of its neighbor across face k.  Counts the
// simplex (low word) and the edges it answers for (high word) at their least vertices and
// returns the sorted row, with the edge mask in the two top bits of its first three entries, and
// the places taken in the buckets.
//
// An edge lies in every simplex of the ring around it.  A simplex answers for it when its index
// is below both ring neighbors' (the neighbors across the faces that hold the edge): the ring's
// least simplex always does, and of the 5.1 simplices around an edge on average 1.7 do, so the
// buckets hold a third of the entries that all simplices would give (2D: exactly one).
template <int M>
__device__ __forceinline__ void canon_row(int4 r, unsigned least, unsigned long long* cnt, int4& row, int4& rank) {
    unsigned k0 = ((unsigned)r.x << 1) | (least & 1u), k1 = ((unsigned)r.y << 1) | ((least >> 1) & 1u);
    unsigned k2 = ((unsigned)r.z << 1) | ((least >> 2) & 1u);
    unsigned k3 = M == 4 ? ((unsigned)r.w << 1) | ((least >> 3) & 1u) : 0u;
    auto cs = [](unsigned& a, unsigned& b) {
        const unsigned lo = a < b ? a : b, hi = a < b ? b : a;
        a = lo;
        b = hi;
    };
    if constexpr (M == 4) { cs(k0, k1); cs(k2, k3); cs(k0, k2); cs(k1, k3); cs(k1, k2); }
    else { cs(k0, k1); cs(k1, k2); cs(k0, k1); }
    const int r0 = (int)(k0 >> 1), r1 = (int)(k1 >> 1), r2 = (int)(k2 >> 1), r3 = (int)(k3 >> 1);
    const bool l0 = k0 & 1u, l1 = k1 & 1u, l2 = k2 & 1u, l3 = M == 4 ? (k3 & 1u) : true;
    // (points come first: an edge is one of two points when its second entry is a point)
    const bool p1 = r1 != kCanonNone, p2 = r2 != kCanonNone, p3 = M == 4 && r3 != kCanonNone;
    const bool e01 = p1 && l2 && l3, e02 = p2 && l1 && l3, e12 = p2 && l0 && l3;
    const bool e03 = p3 && l1 && l2, e13 = p3 && l0 && l2, e23 = p3 && l0 && l1;
    const bool real = M == 4 ? p3 : p2;
    rank = make_int4(0, 0, 0, 0);
    const unsigned n0 = (unsigned)e01 + e02 + e03, n1 = (unsigned)e12 + e13;
    const unsigned long long add = (unsigned long long)real | ((unsigned long long)n0 << 32);
    if (add) {
        const unsigned long long o = atomicAdd(&cnt[r0], add);
        rank.x = (int)(unsigned)o;
        rank.y = (int)(unsigned)(o >> 32);
    }
    if (n1) rank.z = (int)(unsigned)(atomicAdd(&cnt[r1], (unsigned long long)n1 << 32) >> 32);
    if (e23) rank.w = (int)(unsigned)(atomicAdd(&cnt[r2], 1ull << 32) >> 32);
    row.x = r0 | (int)((unsigned)e01 << 30) | (int)((unsigned)e02 << 31);
    row.y = r1 | (int)((unsigned)e03 << 30) | (int)((unsigned)e12 << 31);
    row.z = r2 | (int)((unsigned)e13 << 30) | (int)((unsigned)e23 << 31);
    row.w = M == 4 ? r3 : (real ? 0 : kCanonNone);
}

// Rows of the live simplices of a tree.  Bound by the stream over the records: a dead record
// costs its line too (3D n = 4M: 144 M records, 18.4 GB).  A block reads 1,024 records, four per
// thread with their adjacency (the same line), keeps the live ones in LDS and then works on them
// densely: about one record in five is live, and a lane per record would leave most lanes idle
// behind the gathers (vmap) and the returning atomics of canon_row.  One atomic per 1,024 records
// places the rows; their order is free.  all: every simplex answers for every edge (a tree whose
// adjacency was edited by hand).
template <int D>
__global__ void __launch_bounds__(256) k_canon_rows_tree(Ctx c, const int* vmap, int n, int all, int4* rows, int4* ranks,
                                                         unsigned cap, unsigned long long* cnt, CanonTot* tot) {
    constexpr int M = D + 1;
    __shared__ int4 s_v[1024], s_a[1024];
    __shared__ int s_t[1024];
    __shared__ int s_w[4], s_base, s_n;
    const int wv = threadIdx.x >> 6;
    for (int b0 = blockIdx.x * 1024; b0 < n; b0 += gridDim.x * 1024) {
        int4 v[4], a[4];
        int k = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = b0 + j * 256 + (int)threadIdx.x;
            v[j] = make_int4(-1, -1, -1, -1);
            if (t < n) {
                if constexpr (D == 3) {
                    v[j] = ld_v<3>(c, t);
                    a[j] = ld_a<3>(c, t);
                } else {
                    const int4* q = reinterpret_cast<const int4*>(rp<2>(c, t));
                    const int4 w0 = q[0], w1 = q[1];
                    v[j] = make_int4(w0.x, w0.y, w0.z, -1);
                    a[j] = make_int4(w0.w, w1.x, w1.y, -1);
                }
            }
        }
        bool keep[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int pts = (v[j].x >= M) + (v[j].y >= M) + (v[j].z >= M) + (D == 3 && v[j].w >= M);
            keep[j] = v[j].x >= 0 && pts >= 2;
            k += keep[j];
        }
        int wtot = 0;
        int at = wave_excl_scan(k, wtot);
        if ((threadIdx.x & 63) == 0) s_w[wv] = wtot;
        __syncthreads();
        if (threadIdx.x == 0) {
            s_n = s_w[0] + s_w[1] + s_w[2] + s_w[3];
            s_base = s_n ? (int)atomicAdd(&tot->rows, (unsigned)s_n) : 0;
        }
        for (int w = 0; w < wv; ++w) at += s_w[w];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (keep[j]) {
                s_v[at] = v[j];
                s_a[at] = a[j];
                s_t[at] = b0 + j * 256 + (int)threadIdx.x;
                ++at;
            }
        __syncthreads();
        for (int i = threadIdx.x; i < s_n; i += 256) {
            const int4 vv = s_v[i], aa = s_a[i];
            const int t = s_t[i];
            auto point = [&](int x) { return x >= M ? vmap[x] - 2 * M : kCanonNone; };
            const int4 r = make_int4(point(vv.x), point(vv.y), point(vv.z), D == 3 ? point(vv.w) : 0);
            unsigned least = 15u;
            if (!all) {
                auto below = [&](int nb) { return nb < 0 || t < (nb >> 2); };
                least = (unsigned)below(aa.x) | (unsigned)below(aa.y) << 1 | (unsigned)below(aa.z) << 2 |
                        (unsigned)(D == 3 ? below(aa.w) : true) << 3;
            }
            int4 row, rank;
            canon_row<M>(r, least, cnt, row, rank);
            if ((unsigned)(s_base + i) < cap) {
                rows[s_base + i] = row;
                ranks[s_base + i] = rank;
            }
        }
        __syncthreads();                   // the lists are rewritten by the next step
    }
}

// The same for a list of simplices in reference ids (first = the first point's) without adjacency:
// every simplex answers for all its edges.  A point index of n or more is noted as a bucket too
// large to sort here.
template <int M>
__global__ void __launch_bounds__(256) k_canon_rows_list(const int32_t* simp, int n_simp, int first, int n, int4* rows,
                                                         int4* ranks, unsigned long long* cnt, CanonTot* tot) {
    if (blockIdx.x == 0 && threadIdx.x == 0) tot->rows = (unsigned)n_simp;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n_simp; i += gridDim.x * 256) {
        int r[4] = {0, 0, 0, 0};
        bool ok = true;
        for (int k = 0; k < M; ++k) {
            const int v = simp[(int64_t)i * M + k];
            r[k] = v >= first ? v - first : kCanonNone;
            ok &= r[k] < n || r[k] == kCanonNone;
        }
        int4 row = make_int4(kCanonNone, kCanonNone, kCanonNone, kCanonNone), rank = make_int4(0, 0, 0, 0);
        if (ok) canon_row<M>(make_int4(r[0], r[1], r[2], r[3]), 15u, cnt, row, rank);
        else atomicMax(&tot->max_bucket, 0xffffffffu);
        rows[i] = row;
        ranks[i] = rank;
    }
}

// Exclusive scan of n 64-bit values, 4,096 per block: block sums, then each block adds the sums
// before its own (n / 4096 of them) and scans its tile.  out[n] = the total.  With `big` (the
// bucket counts): vertices with a bucket above kCanonSmall are listed and the largest noted.
__global__ void __launch_bounds__(256) k_scan64_sums(const unsigned long long* in, unsigned long long* bsum, int64_t n) {
    __shared__ unsigned long long s_w[4];
    unsigned long long x = 0;
    const int64_t b0 = (int64_t)blockIdx.x * kScanTile;
    for (int j = threadIdx.x; j < kScanTile; j += 256)
        if (b0 + j < n) x += in[b0 + j];
    x = wave_sum(x);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

__global__ void __launch_bounds__(256) k_scan64_apply(const unsigned long long* in, const unsigned long long* bsum,
                                                      unsigned long long* out, int64_t n, unsigned long long* total,
                                                      int* big, CanonTot* tot) {
    __shared__ unsigned long long s_w[4];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    unsigned long long base = 0;
    for (int64_t j = threadIdx.x; j < blockIdx.x; j += 256) base += bsum[j];
    base = wave_sum(base);
    if (lane == 0) s_w[wv] = base;
    __syncthreads();
    base = s_w[0] + s_w[1] + s_w[2] + s_w[3];
    __syncthreads();
    const int64_t b0 = (int64_t)blockIdx.x * kScanTile;
    unsigned mx = 0;
    for (int j0 = 0; j0 < kScanTile; j0 += 256) {
        const int64_t i = b0 + j0 + threadIdx.x;
        const unsigned long long v = i < n ? in[i] : 0ull;
        if (big) {
            const unsigned t = (unsigned)v, e = (unsigned)(v >> 32), m = t > e ? t : e;
            mx = m > mx ? m : mx;
            if (m > (unsigned)kCanonSmall) big[atomicAdd(&tot->n_big, 1u)] = (int)i;
        }
        unsigned long long x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) s_w[wv] = x;
        __syncthreads();
        unsigned long long before = base;
        for (int w = 0; w < wv; ++w) before += s_w[w];
        if (i < n) out[i] = before + x - v;
        if (i == n - 1) {
            out[n] = before + x;
            *total = before + x;
        }
        base += s_w[0] + s_w[1] + s_w[2] + s_w[3];
        __syncthreads();
    }
    if (big && mx > (unsigned)kCanonSmall) atomicMax(&tot->max_bucket, mx);
}

// The buckets can be worked on: the rows fit their arrays and the largest bucket fits LDS.  (Else
// the host reports the first, and takes the radix sort for the second.)
__device__ __forceinline__ bool canon_ok(const CanonTot* tot, unsigned cap) {
    return tot->rows <= cap && tot->max_bucket <= (unsigned)kCanonBig;
}

// every row and edge entry with its place in the buckets: row(place, r0, r1, r2, r3), edge(place,
// least, other)
template <class Row, class Edge>
__device__ __forceinline__ void canon_places(const int4* rows, const int4* ranks, unsigned n, const unsigned long long* ofs,
                                             Row row, Edge edge) {
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const int4 q = rows[i], k = ranks[i];
        constexpr int low = 0x3fffffff;
        const int r0 = q.x & low, r1 = q.y & low, r2 = q.z & low, r3 = q.w;
        const bool e01 = (q.x >> 30) & 1, e02 = q.x < 0, e03 = (q.y >> 30) & 1, e12 = q.y < 0;
        const bool e13 = (q.z >> 30) & 1, e23 = q.z < 0;
        const bool real = r3 != kCanonNone;
        if (real || e01 || e02 || e03) {
            const unsigned long long o = ofs[r0];
            if (real) row((size_t)(unsigned)o + (unsigned)k.x, r0, r1, r2, r3);
            size_t e = (size_t)(unsigned)(o >> 32) + (unsigned)k.y;
            if (e01) edge(e++, r0, r1);
            if (e02) edge(e++, r0, r2);
            if (e03) edge(e, r0, r3);
        }
        if (e12 || e13) {
            size_t e = (size_t)(unsigned)(ofs[r1] >> 32) + (unsigned)k.z;
            if (e12) edge(e++, r1, r2);
            if (e13) edge(e, r1, r3);
        }
        if (e23) edge((size_t)(unsigned)(ofs[r2] >> 32) + (unsigned)k.w, r2, r3);
    }
}

// rows to their buckets: a simplex's other vertices (16 B) and the edges' other ends (4 B)
__global__ void __launch_bounds__(256) k_canon_scatter(const int4* rows, const int4* ranks, unsigned cap, const CanonTot* tot,
                                                       const unsigned long long* ofs, int4* tb, int* eb) {
    if (!canon_ok(tot, cap)) return;
    canon_places(rows, ranks, tot->rows, ofs, [&](size_t o, int, int r1, int r2, int r3) { tb[o] = make_int4(r1, r2, r3, 0); },
                 [&](size_t e, int, int y) { eb[e] = y; });
}

template <int M> __device__ __forceinline__ bool canon_less(int4 a, int4 b) {
    if (a.x != b.x) return a.x < b.x;
    if (M == 3 || a.y != b.y) return a.y < b.y;
    return a.z < b.z;
}
template <int M> __device__ __forceinline__ void canon_put(int32_t* T, size_t at, int v, int4 o) {
    if constexpr (M == 4) reinterpret_cast<int4*>(T)[at] = make_int4(v, o.x, o.y, o.z);
    else {
        T[3 * at] = v;
        T[3 * at + 1] = o.x;
        T[3 * at + 2] = o.y;
    }
}

// Buckets of at most kCanonSmall entries: 16 lanes per vertex, the entries in LDS, each entry's
// place the number of lesser ones (a bucket of 7 simplices or 13 edge entries is 7 or 13 LDS
// reads per lane; a sorting network over 16 or 64 would move them more often).  Simplex rows go
// to their final place; an edge's further entries are dropped, the rest go back in order and
// their number to ucnt.
template <int M>
__global__ void __launch_bounds__(256) k_canon_sort(const unsigned long long* ofs, int64_t n, const int4* tb, int* eb,
                                                    int32_t* T, unsigned long long* ucnt, const CanonTot* tot,
                                                    unsigned cap) {
    if (!canon_ok(tot, cap)) return;
    constexpr int L = 16, V = 256 / L;
    // a row as its entries in order and its place: equal rows (a list given by the caller may hold
    // some) differ by the last, and two comparisons of 64 bits order any two
    __shared__ ulonglong2 s_t[V][kCanonSmall];
    __shared__ int s_e[V][kCanonSmall];
    __shared__ int s_u[V];
    const int g = threadIdx.x / L, l = threadIdx.x % L;
    for (int64_t v0 = (int64_t)blockIdx.x * V; v0 < n; v0 += (int64_t)gridDim.x * V) {
        const int64_t v = v0 + g;
        unsigned long long a = 0, b = 0;
        if (v < n) {
            a = ofs[v];
            b = ofs[v + 1];
        }
        const size_t t0 = (size_t)(unsigned)a, e0 = (size_t)(unsigned)(a >> 32);
        int nt = (int)((unsigned)b - (unsigned)a), ne = (int)((unsigned)(b >> 32) - (unsigned)(a >> 32));
        const bool small = nt <= kCanonSmall && ne <= kCanonSmall;
        if (!small) nt = ne = 0;
        for (int i = l; i < nt; i += L) {
            const int4 q = tb[t0 + i];
            s_t[g][i] = make_ulonglong2((unsigned long long)(unsigned)q.x << 32 | (unsigned)q.y,
                                        (unsigned long long)(unsigned)(M == 4 ? q.z : 0) << 32 | (unsigned)i);
        }
        for (int i = l; i < ne; i += L) s_e[g][i] = eb[e0 + i];
        if (l == 0) s_u[g] = 0;
        __syncthreads();
        for (int i = l; i < nt; i += L) {
            const ulonglong2 x = s_t[g][i];
            int rank = 0;
            for (int j = 0; j < nt; ++j) {
                const ulonglong2 y = s_t[g][j];
                rank += (y.x < x.x) | ((y.x == x.x) & (y.y < x.y));
            }
            canon_put<M>(T, t0 + rank, (int)v, make_int4((int)(x.x >> 32), (int)x.x, (int)(x.y >> 32), 0));
        }
        // entries repeated by a later one are dropped: the last of equal entries stays
        bool keep[kCanonSmall / L];
#pragma unroll
        for (int q = 0; q < kCanonSmall / L; ++q) {
            const int i = l + q * L;
            keep[q] = i < ne;
            if (!keep[q]) continue;
            const int x = s_e[g][i];
            for (int j = i + 1; j < ne; ++j) keep[q] &= s_e[g][j] != x;
        }
        __syncthreads();
        int x[kCanonSmall / L];
#pragma unroll
        for (int q = 0; q < kCanonSmall / L; ++q) {
            const int i = l + q * L;
            if (i >= ne) continue;
            x[q] = s_e[g][i];
            if (keep[q]) atomicAdd(&s_u[g], 1);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kCanonSmall / L; ++q) {
            const int i = l + q * L;
            if (i < ne && !keep[q]) s_e[g][i] = 0x7fffffff;      // behind every point index
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kCanonSmall / L; ++q) {
            const int i = l + q * L;
            if (i >= ne || !keep[q]) continue;
            int rank = 0;
            for (int j = 0; j < ne; ++j) rank += s_e[g][j] < x[q];
            eb[e0 + rank] = x[q];
        }
        if (l == 0 && v < n && small) ucnt[v] = (unsigned long long)s_u[g];
        __syncthreads();
    }
}

// Buckets of kCanonSmall + 1 .. kCanonBig entries (the vertices listed in big): a block per
// vertex, bitonic sort in LDS, edges after simplices in the same LDS.
template <int M>
__global__ void __launch_bounds__(256) k_canon_sort_big(const unsigned long long* ofs, const int* big, const CanonTot* tot,
                                                        unsigned cap, const int4* tb, int* eb, int32_t* T, unsigned long long* ucnt) {
    __shared__ int s_x[kCanonBig], s_y[kCanonBig], s_z[kCanonBig];
    __shared__ int s_w[4], s_acc;
    if (!canon_ok(tot, cap)) return;
    const int n_big = (int)tot->n_big;
    auto pow2 = [](int n) {
        int p = 1;
        while (p < n) p <<= 1;
        return p;
    };
    for (int w = blockIdx.x; w < n_big; w += gridDim.x) {
        const int v = big[w];
        const unsigned long long a = ofs[v], b = ofs[v + 1];
        const size_t t0 = (size_t)(unsigned)a, e0 = (size_t)(unsigned)(a >> 32);
        const int nt = (int)((unsigned)b - (unsigned)a), ne = (int)((unsigned)(b >> 32) - (unsigned)(a >> 32));
        const int pt = pow2(nt), pe = pow2(ne);
        for (int i = threadIdx.x; i < pt; i += 256) {
            const int4 q = i < nt ? tb[t0 + i] : make_int4(0x7fffffff, 0x7fffffff, 0x7fffffff, 0);
            s_x[i] = q.x;
            s_y[i] = q.y;
            s_z[i] = q.z;
        }
        __syncthreads();
        for (int k = 2; k <= pt; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int i = threadIdx.x; i < pt; i += 256) {
                    const int o = i ^ j;
                    if (o > i) {
                        const int4 p = make_int4(s_x[i], s_y[i], s_z[i], 0), q = make_int4(s_x[o], s_y[o], s_z[o], 0);
                        if (canon_less<M>(q, p) == ((i & k) == 0)) {
                            s_x[i] = q.x; s_y[i] = q.y; s_z[i] = q.z;
                            s_x[o] = p.x; s_y[o] = p.y; s_z[o] = p.z;
                        }
                    }
                }
                __syncthreads();
            }
        for (int i = threadIdx.x; i < nt; i += 256) canon_put<M>(T, t0 + i, v, make_int4(s_x[i], s_y[i], s_z[i], 0));
        __syncthreads();
        for (int i = threadIdx.x; i < pe; i += 256) s_x[i] = i < ne ? eb[e0 + i] : 0x7fffffff;
        __syncthreads();
        for (int k = 2; k <= pe; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int i = threadIdx.x; i < pe; i += 256) {
                    const int o = i ^ j;
                    if (o > i) {
                        const int p = s_x[i], q = s_x[o];
                        if ((q < p) == ((i & k) == 0)) {
                            s_x[i] = q;
                            s_x[o] = p;
                        }
                    }
                }
                __syncthreads();
            }
        if (threadIdx.x == 0) s_acc = 0;
        __syncthreads();
        for (int i0 = 0; i0 < ne; i0 += 256) {
            const int i = i0 + (int)threadIdx.x;
            const bool first = i < ne && (i == 0 || s_x[i] != s_x[i - 1]);
            int wt = 0;
            int at = wave_excl_scan(first, wt);
            if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = wt;
            __syncthreads();
            at += s_acc;
            for (int q = 0; q < (int)(threadIdx.x >> 6); ++q) at += s_w[q];
            if (first) eb[e0 + at] = s_x[i];
            __syncthreads();
            if (threadIdx.x == 0) s_acc += s_w[0] + s_w[1] + s_w[2] + s_w[3];
            __syncthreads();
        }
        if (threadIdx.x == 0) ucnt[v] = (unsigned long long)s_acc;
        __syncthreads();
    }
}

// the unique edges of every vertex to their final place
__global__ void __launch_bounds__(256) k_canon_edges(const unsigned long long* ofs, const unsigned long long* uofs,
                                                     int64_t n, const int* eb, int2* E, const CanonTot* tot, unsigned cap) {
    if (!canon_ok(tot, cap)) return;
    constexpr int L = 16, V = 256 / L;
    const int g = threadIdx.x / L, l = threadIdx.x % L;
    for (int64_t v = (int64_t)blockIdx.x * V + g; v < n; v += (int64_t)gridDim.x * V) {
        const size_t e0 = (size_t)(ofs[v] >> 32), u0 = (size_t)uofs[v];
        const int m = (int)(uofs[v + 1] - uofs[v]);
        for (int i = l; i < m; i += L) E[u0 + i] = make_int2((int)v, eb[e0 + i]);
    }
}

// ---------------------------------------------------------------- radix sort

constexpr int kRadixThreads = 256;
constexpr int kRadixTile = 4096;                         // 16 elements per thread
constexpr int kRadixWaves = kRadixThreads / 64;
constexpr int kRadixPerWave = kRadixTile / kRadixWaves;  // contiguous elements per wavefront

// per-tile histogram of the digit at `shift`: hist[d * ntiles + tile]
__global__ void __launch_bounds__(kRadixThreads) k_radix_hist(const unsigned long long* keys, int64_t n, int shift,
                                                             unsigned long long* hist, int ntiles) {
    __shared__ int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kRadixTile;
    for (int i = threadIdx.x; i < kRadixTile; i += kRadixThreads) {
        const int64_t j = base + i;
        if (j < n) atomicAdd(&h[(int)((keys[j] >> shift) & 255ull)], 1);
    }
    __syncthreads();
    hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = (unsigned long long)h[threadIdx.x];
}

// Stable scatter of one tile: wavefront w owns elements [w * kRadixPerWave, (w + 1) * ...) of
// the tile; it counts its digits, the block turns the counts into per-wavefront offsets on top
// of the tile's offsets (off[d * ntiles + tile]), and each wavefront then places its elements
// in order, ranking equal digits among its 64 lanes with ballots.
__global__ void __launch_bounds__(kRadixThreads) k_radix_scatter(const unsigned long long* keys, const uint32_t* vals,
                                                                unsigned long long* okeys, uint32_t* ovals, int64_t n,
                                                                int shift, const unsigned long long* off, int ntiles) {
    __shared__ unsigned cnt[kRadixWaves][256];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int d = lane; d < 256; d += 64) cnt[w][d] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kRadixTile + (int64_t)w * kRadixPerWave;
    for (int i = lane; i < kRadixPerWave; i += 64) {
        const int64_t j = base + i;
        if (j < n) atomicAdd(&cnt[w][(int)((keys[j] >> shift) & 255ull)], 1u);
    }
    __syncthreads();
    // per-wavefront starting positions: tile offset of the digit + counts of earlier wavefronts
    for (int d = threadIdx.x; d < 256; d += kRadixThreads) {
        unsigned acc = (unsigned)off[(int64_t)d * ntiles + blockIdx.x];
        for (int v = 0; v < kRadixWaves; ++v) {
            const unsigned c = cnt[v][d];
            cnt[v][d] = acc;
            acc += c;
        }
    }
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int i0 = 0; i0 < kRadixPerWave; i0 += 64) {
        const int64_t j = base + i0 + lane;
        const bool valid = j < n;
        unsigned long long k = 0;
        uint32_t v = 0;
        int d = 256;                                   // invalid lanes form a group of their own
        if (valid) {
            k = keys[j];
            if (vals) v = vals[j];
            d = (int)((k >> shift) & 255ull);
        }
        unsigned long long same = __ballot(true);
        for (int b = 0; b < 9; ++b) {
            const unsigned long long bb = __ballot((d >> b) & 1);
            same &= ((d >> b) & 1) ? bb : ~bb;
        }
        const int rank = __popcll(same & below);
        const unsigned start = valid ? cnt[w][d] : 0u;
        if (valid) {
            const unsigned pos = start + rank;
            okeys[pos] = k;
            if (vals) ovals[pos] = v;
        }
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) cnt[w][d] = start + __popcll(same);
        __builtin_amdgcn_wave_barrier();
    }
}

__global__ void k_iota_u32(uint32_t* v, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        v[i] = (uint32_t)i;
}

// The rows and their two 64-bit sort keys, lo = columns (2, 3) (2D: column 2) and hi = columns (0, 1),
// and the edge entries' keys (least, other), each column `nb` bits wide, at their places in the buckets.
template <int M>
__global__ void __launch_bounds__(256) k_canon_keys(const int4* rows, const int4* ranks, unsigned n, const unsigned long long* ofs,
                                                    int nb, int4* crow, unsigned long long* klo, unsigned long long* khi,
                                                    unsigned long long* ekeys) {
    auto two = [&](int a, int b) { return ((unsigned long long)a << nb) | (unsigned long long)b; };
    canon_places(rows, ranks, n, ofs,
                 [&](size_t o, int r0, int r1, int r2, int r3) {
                     crow[o] = make_int4(r0, r1, r2, r3);
                     klo[o] = M == 4 ? two(r2, r3) : (unsigned long long)r2;
                     khi[o] = two(r0, r1);
                 },
                 [&](size_t e, int x, int y) { ekeys[e] = two(x, y); });
}

// key of every row in the permutation's order: dst[i] = khi[perm[i]]
__global__ void k_gather_u64(const unsigned long long* src, const uint32_t* perm, unsigned long long* dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[perm[i]];
}

// rows in the sorted order, M columns
template <int M>
__global__ void k_canon_out_rows(const int4* crow, const uint32_t* perm, int64_t n, int32_t* out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int4 r = crow[perm[i]];
        out[i * M + 0] = r.x;
        out[i * M + 1] = r.y;
        out[i * M + 2] = r.z;
        if (M == 4) out[i * M + 3] = r.w;
    }
}

// first occurrence of each edge key in the sorted list
__global__ void k_canon_edge_flags(const unsigned long long* keys, int64_t n, unsigned long long* flag) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        flag[i] = i == 0 || keys[i] != keys[i - 1];
}

__global__ void k_canon_edge_out(const unsigned long long* keys, const unsigned long long* pos, int64_t n, int nb,
                                 int32_t* out) {
    const unsigned long long mask = (1ull << nb) - 1ull;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t o = (int64_t)pos[i];
        if ((int64_t)pos[i + 1] == o) continue;
        out[2 * o] = (int32_t)(keys[i] >> nb);
        out[2 * o + 1] = (int32_t)(keys[i] & mask);
    }
}

}  // namespace vo
