#pragma once

// A kernel's limit of dynamic LDS.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstddef>

namespace tk {

struct LdsLimits {      // of one kernel, zeros before the first launch
  std::atomic<bool> raised[64];
};

// Raises the limit on the current device, once a device: the attribute belongs to a function on a device.
inline bool raise_lds_limit(const void* kernel, size_t bytes, LdsLimits& limits) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  if (limits.raised[dev].load(std::memory_order_relaxed)) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  limits.raised[dev].store(true, std::memory_order_relaxed);
  return true;
}

}  // namespace tk
