// Read-back through pinned staging by several host threads.
//
// A hipMemcpy to memory the caller has just allocated is one host thread that takes the page
// faults of the destination and copies out of the runtime's own staging buffer: 7 GB/s where the
// link carries 55.  Here up to 8 threads each bring a chunk into a pinned slot of their own and
// copy it to its place, so faults, copies and transfers of different chunks overlap: a batch of 33
// views, 463 MB, is read in 25 ms (67 before; 8.4 at the link's rate), a 4K mapping image of 133
// MB in 4.4 (12.8), a 1080p one of 33 MB in 1.15 (1.97).
#include "readback.hpp"

#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace linon {

bool ReadStaging::reserve() {
    if (slots_) return true;
    void* p = nullptr;
    if (hipHostMalloc(&p, THREADS * SLOT, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    for (auto& e : done_) {
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipHostFree(p);
            return false;
        }
    }
    slots_ = p;
    return true;
}

void ReadStaging::release() {
    for (auto& e : done_) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (slots_) (void)hipHostFree(slots_);
    slots_ = nullptr;
}

namespace {

// Pinned, managed and device destinations keep the runtime's own copy.
bool pageable(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t ReadStaging::copy(const HostCopy* copies, int n, hipStream_t stream, int device) {
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += copies[i].bytes;
    const size_t chunks_all = (total + SLOT - 1) / SLOT;
    std::unique_lock<std::mutex> mine(busy_, std::defer_lock);
    // Below 4 MiB the threads' start costs what they save (3.15 MB 190 us staged, 181 by hipMemcpy;
    // 3.84 MB 210 and 214; 4.32 MB 222 and 247; 6.3 MB 303 and 354), and the question what memory the
    // destination is up to 4% of a small read.  A second thread that reads the same context meanwhile
    // has the runtime's copy too.
    bool staged = total >= 4 * SLOT;
    for (int i = 0; staged && i < n; ++i) staged = copies[i].bytes == 0 || pageable(copies[i].dst);
    if (!staged || !mine.try_lock() || !reserve()) {
        for (int i = 0; i < n; ++i) {
            if (!copies[i].bytes) continue;
            const hipError_t e = hipMemcpy(copies[i].dst, copies[i].src, copies[i].bytes, hipMemcpyDeviceToHost);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    std::atomic<size_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int t) noexcept {
        hipError_t e = t ? hipSetDevice(device) : hipSuccess;
        char* slot = static_cast<char*>(slots_) + (size_t)t * SLOT;
        while (e == hipSuccess && failed.load(std::memory_order_relaxed) == (int)hipSuccess) {
            // chunk c of the copies laid end to end, cut at their ends
            size_t c = next.fetch_add(1, std::memory_order_relaxed);
            int i = 0;
            for (; i < n; ++i) {
                const size_t k = (copies[i].bytes + SLOT - 1) / SLOT;
                if (c < k) break;
                c -= k;
            }
            if (i == n) return;
            const size_t off = c * SLOT, left = copies[i].bytes - off, len = left < SLOT ? left : SLOT;
            e = hipMemcpyAsync(slot, static_cast<const char*>(copies[i].src) + off, len, hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(done_[t], stream);
            if (e == hipSuccess) e = hipEventSynchronize(done_[t]);
            if (e == hipSuccess) std::memcpy(static_cast<char*>(copies[i].dst) + off, slot, len);
        }
        if (e != hipSuccess) failed.store((int)e, std::memory_order_relaxed);
    };
    std::thread pool[THREADS - 1];
    int started = 0;
    try {
        for (; started < THREADS - 1 && (size_t)started + 1 < chunks_all; ++started)
            pool[started] = std::thread(work, started + 1);
    } catch (...) {
        // no more threads to be had (std::system_error), or no memory for one (std::bad_alloc): those
        // started, and this one, do the work
    }
    work(0);
    for (int t = 0; t < started; ++t) pool[t].join();
    const hipError_t e = (hipError_t)failed.load();
    if (e != hipSuccess) (void)hipStreamSynchronize(stream);  // no transfer into a slot outlives the call
    return e;
}

}  // namespace linon
