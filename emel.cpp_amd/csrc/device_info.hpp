// Host-side facts about the current device.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <stdint.h>

namespace emelk {

// Compute units of the current device, cached per device id.  Racing first
// calls store the same value, so relaxed atomics are enough.
inline int32_t device_cu_count() {
  static std::atomic<int32_t> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int32_t cus = cached[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    int c = 0;
    if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        c <= 0) {
      c = 256;
    }
    cus = c;
    cached[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

}  // namespace emelk
