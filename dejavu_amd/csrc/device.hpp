// What the launch plans ask of the current device.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

namespace dv {

constexpr int kMaxDevices = 64;

inline int current_device() {
  int dev = 0;
  return (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices) ? dev : -1;
}

// Compute units of the current device (remembered per device).
inline int compute_units() {
  static std::atomic<int> cus[kMaxDevices];
  const int dev = current_device();
  if (dev < 0) return 256;
  int v = cus[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cus[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

}  // namespace dv
