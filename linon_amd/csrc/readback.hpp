// Copies of device buffers to ordinary (pageable) host memory through pinned staging.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace linon {

struct HostCopy {
    void* dst;
    const void* src;  // device
    size_t bytes;
};

// Pinned slots and their events, one pair per copying thread; kept by a context from its first
// large read-back until it is destroyed.
class ReadStaging {
  public:
    // Copies whose source is complete (the caller has synchronised); every destination is written
    // when it returns.  Streams' work after the call is the caller's; `stream` orders the copies.
    hipError_t copy(const HostCopy* copies, int n, hipStream_t stream, int device);
    void release();

  private:
    static constexpr int THREADS = 8;
    static constexpr size_t SLOT = size_t{1} << 20;
    bool reserve();
    std::mutex busy_;
    void* slots_ = nullptr;  // THREADS of SLOT bytes
    hipEvent_t done_[THREADS] = {};
};

}  // namespace linon
