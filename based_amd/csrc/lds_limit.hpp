// Kernels with more than 64 KB of dynamic LDS have to be allowed that, on every device by itself.
#pragma once

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstddef>

namespace based {

constexpr int kMaxDevices = 64;

typedef std::atomic<bool> LdsAllowed[kMaxDevices];  // of one kernel

// Lets a kernel have `bytes` of LDS on the current device, once for each device; what is refused is asked for again.
static inline hipError_t allow_lds(const void* kernel, size_t bytes, LdsAllowed& allowed) {
  if (bytes <= 64 * 1024) return hipSuccess;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess && (dev < 0 || dev >= kMaxDevices)) e = hipErrorInvalidDevice;
  if (e != hipSuccess || allowed[dev].load(std::memory_order_acquire)) return e;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) allowed[dev].store(true, std::memory_order_release);
  return e;
}

}  // namespace based
