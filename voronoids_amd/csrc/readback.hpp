// readback.hpp -- large results from the device to the caller's memory.
//
// A copy to pageable memory is staged by one runtime thread at about 16 GB/s, and when the
// destination is fresh memory, as a result's is, that thread also takes the page faults: 683 MB
// (the canonical form of 4 M points) took 220 ms, where the link needs 12.  Here the device copies
// into a ring of pinned slots at the link's rate and several threads move the slots on, so that
// faults and copies run beside each other and beside the link.  With huge pages for the results
// and no further copy of them in Python: the canonical form at 3D n = 4M 225 -> 25 ms (7 of it on
// the device), 2D n = 10M 157 -> 17.5 ms, the export at 3D n = 4M (868 MB into the caller's arrays,
// on small pages) 92 -> 33 ms, 29 where the pages were there before.  Eight or fifteen threads
// instead of four measured the same.
//
// For up to two seconds after a gigabyte or more of device memory was freed, by any process, the
// system clears it with the copy engine, and copies to the host run at a quarter of the rate (pieces
// of a slot 12 GB/s instead of 45): then the canonical form takes 65 ms and the export 81.
#pragma once
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <thread>
#include <vector>

#include "host_common.hpp"

namespace vo_host {

struct Segment {
    void* dst;
    const void* src;
    size_t bytes;
};

// Pinned slots and their events; kept by the handle from its first large result on (24 MB), freed
// with it.  One user at a time, as the handle.
struct PinnedRing {
    static constexpr int kSlots = 12;
    static constexpr size_t kSlot = (size_t)2 << 20;
    char* p = nullptr;
    hipEvent_t ev[kSlots] = {};
    PinnedRing() = default;
    PinnedRing(const PinnedRing&) = delete;
    ~PinnedRing() {
        for (auto& e : ev)
            if (e) hipEventDestroy(e);
        if (p) hipHostFree(p);
    }
    bool ready() {
        if (!p && hipHostMalloc((void**)&p, kSlots * kSlot) != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();       // (not for the next launch to report)
            return false;
        }
        for (auto& e : ev)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
        return true;
    }
};

// From this size on the ring and its threads are used: starting them takes about 0.2 ms, the
// runtime's copy of 8 MB into fresh pages about 2.
constexpr size_t kRingBytes = (size_t)8 << 20;

inline int read_back_plain(hipStream_t s, const std::vector<Segment>& segs) {
    for (const Segment& g : segs)
        if (g.bytes) VO_HIP(hipMemcpyAsync(g.dst, g.src, g.bytes, hipMemcpyDeviceToHost, s));
    VO_HIP(hipStreamSynchronize(s));
    return 0;
}

// every segment copied when this returns
inline int read_back(hipStream_t s, int dev, PinnedRing& ring, const std::vector<Segment>& segs) {
    size_t total = 0;
    for (const Segment& g : segs) total += g.bytes;
    if (total < kRingBytes || !ring.ready()) return read_back_plain(s, segs);
    constexpr size_t kSlot = PinnedRing::kSlot;
    constexpr int S = PinnedRing::kSlots;
    std::vector<Segment> part;
    for (const Segment& g : segs)
        for (size_t o = 0; o < g.bytes; o += kSlot)
            part.push_back({(char*)g.dst + o, (const char*)g.src + o, std::min(kSlot, g.bytes - o)});
    const int n = (int)part.size();
    // part i goes through slot i mod S: issued once part i - S is done with it
    std::unique_ptr<std::atomic<bool>[]> done(new std::atomic<bool>[n]);
    for (int i = 0; i < n; ++i) done[i].store(false, std::memory_order_relaxed);
    std::atomic<int> issued{0}, next{0};
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&] {
        if (hipSetDevice(dev) != hipSuccess) {
            err.store((int)hipErrorInvalidDevice);
            return;
        }
        for (;;) {
            const int i = next.fetch_add(1);
            if (i >= n) return;
            while (issued.load(std::memory_order_acquire) <= i) {
                if (err.load() != (int)hipSuccess) return;
                std::this_thread::yield();
            }
            const hipError_t e = hipEventSynchronize(ring.ev[i % S]);
            if (e != hipSuccess) {
                err.store((int)e);
                return;
            }
            std::memcpy(part[i].dst, ring.p + (size_t)(i % S) * kSlot, part[i].bytes);
            done[i].store(true, std::memory_order_release);
        }
    };
    const int want = std::max(1, std::min({4, (int)std::thread::hardware_concurrency() / 2, n}));
    std::vector<std::thread> pool;
    try {
        pool.reserve((size_t)want);
        for (int k = 0; k < want; ++k) pool.emplace_back(work);
    } catch (...) {                        // no more threads to be had: the ones that started do it
    }
    if (pool.empty()) return read_back_plain(s, segs);
    for (int i = 0; i < n && err.load() == (int)hipSuccess; ++i) {
        while (i >= S && !done[i - S].load(std::memory_order_acquire) && err.load() == (int)hipSuccess)
            std::this_thread::yield();
        if (err.load() != (int)hipSuccess) break;
        hipError_t e = hipMemcpyAsync(ring.p + (size_t)(i % S) * kSlot, part[i].src, part[i].bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ring.ev[i % S], s);
        if (e != hipSuccess) {
            err.store((int)e);
            break;
        }
        issued.store(i + 1, std::memory_order_release);
    }
    for (auto& t : pool) t.join();
    const hipError_t last = hipStreamSynchronize(s);
    if (err.load() != (int)hipSuccess || last != hipSuccess)
        return fail(VO_ERR_HIP, std::string("result copy: ") +
                                    hipGetErrorString(err.load() != (int)hipSuccess ? (hipError_t)err.load() : last));
    return 0;
}

// Memory for a result, released with free() (vo_free).  Large ones on huge pages where the system
// grants them: a fault per 2 MB instead of one per 4 KB.
inline void* result_alloc(size_t bytes) {
    constexpr size_t kHuge = (size_t)2 << 20;
    if (bytes < 2 * kHuge) return std::malloc(std::max<size_t>(bytes, 1));
    void* p = nullptr;
    if (posix_memalign(&p, kHuge, bytes)) return nullptr;
    madvise(p, bytes, MADV_HUGEPAGE);
    return p;
}

}  // namespace vo_host
