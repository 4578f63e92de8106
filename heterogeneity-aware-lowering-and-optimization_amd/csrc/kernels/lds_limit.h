// What a launch may ask for in dynamic LDS beyond 64 KiB.
#ifndef OHIP_LDS_LIMIT_H
#define OHIP_LDS_LIMIT_H

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdint>

namespace ohip {

// One per kernel (a static of its launch): the kernel's limit is raised on every device that it is
// launched on, before its first launch there returns to any thread.
class LdsLimit {
 public:
  hipError_t raise(const void* kernel, const int bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = dev >= 0 && dev < 64 ? 1ull << dev : 0;   // (any further device: every time)
    if (done_.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);   // (repeating it is harmless)
    if (e == hipSuccess) done_.fetch_or(bit, std::memory_order_release);
    return e;
  }

 private:
  std::atomic<uint64_t> done_{0};
};

}  // namespace ohip
#endif
