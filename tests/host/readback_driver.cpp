// CPU driver of the staged read-back (linon_amd/csrc/readback.cpp) over HIP calls that copy host
// memory, for tests/test_readback_host.py: `readback_driver CASE` prints what the copies made of
// their sources and exits with 0.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "readback.hpp"

static std::atomic<bool> no_memory{false};      // operator new refuses
static std::atomic<int> staged{0}, plain{0};    // hipMemcpyAsync and hipMemcpy calls
static std::atomic<int> fail_at{-1};            // the hipMemcpyAsync call that fails
static std::atomic<bool> no_pinned{false};
static std::atomic<int> second{0};              // a second reader: 1 expected, 2 done

void* operator new(size_t n) {
    if (no_memory.load()) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (no_pinned.load()) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    ++plain;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (staged++ == fail_at.load()) return hipErrorUnknown;
    while (second.load() == 1) std::this_thread::yield();
    std::memcpy(d, s, n);
    return hipSuccess;
}
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    const size_t bytes = argc > 2 ? std::strtoull(argv[2], nullptr, 10) : (size_t)19 << 19;
    std::vector<unsigned char> src(bytes), dst(bytes, 0);
    for (size_t i = 0; i < bytes; ++i) src[i] = (unsigned char)(i * 2654435761u >> 24);
    linon::ReadStaging staging;
    const size_t cut = bytes / 3;  // two copies, neither a whole number of chunks
    const linon::HostCopy copies[2] = {{dst.data(), src.data(), cut}, {dst.data() + cut, src.data() + cut, bytes - cut}};
    no_pinned = what == "no_pinned";
    fail_at = what == "fail" ? 3 : -1;
    second = what == "second" ? 1 : 0;
    std::thread reader;
    std::vector<unsigned char> other(bytes, 0);
    if (second == 1)
        reader = std::thread([&] {  // while the first holds the slots
            while (!staged.load()) std::this_thread::yield();
            const linon::HostCopy copy{other.data(), src.data(), bytes};
            if (staging.copy(&copy, 1, nullptr, 0) != hipSuccess || other != src) std::exit(4);
            second = 2;
        });
    no_memory = what == "no_memory";
    const hipError_t e = staging.copy(copies, 2, nullptr, 0);
    if (reader.joinable()) reader.join();
    no_memory = false;
    staging.release();
    std::printf("error %d equal %d staged %d plain %d\n", (int)e, (int)(src == dst), staged.load(), plain.load());
    return 0;
}
