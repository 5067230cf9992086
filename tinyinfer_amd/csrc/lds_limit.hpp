// Dynamic LDS above the 64 KiB default.  The limit is an attribute of a kernel on
// one device, so it is raised on every device the kernel is launched on, not once
// per process: a launch on the second device would otherwise be refused.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include <atomic>

namespace tia {

// One per kernel, as a static of its launcher.  Safe with several threads (two
// that meet both set the same value); a failure is returned and tried again by
// the next call.
class LdsLimit {
 public:
  hipError_t raise(const void* kernel, int bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = dev >= 0 && dev < 64 ? uint64_t(1) << dev : 0;
    if (raised_.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) raised_.fetch_or(bit, std::memory_order_release);
    return e;
  }

 private:
  std::atomic<uint64_t> raised_{0};  // bit per device
};

}  // namespace tia
