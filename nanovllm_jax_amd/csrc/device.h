// What the host side of a launch asks of the current device.
#ifndef NVJ_DEVICE_H_
#define NVJ_DEVICE_H_

#include <hip/hip_runtime.h>

#include <atomic>

namespace nvj {

// Compute units of the current device (256 on an MI355X), looked up once per
// device; 256 when no device can be asked (argument checks without a GPU).
inline int compute_units() {
  constexpr int kMaxDevicesSeen = 64;
  static std::atomic<int> cached[kMaxDevicesSeen];
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevicesSeen) {
    (void)hipGetLastError();   // not an error of any launch
    return 256;
  }
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      n <= 0) {
    (void)hipGetLastError();
    return 256;
  }
  cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

}  // namespace nvj

#endif  // NVJ_DEVICE_H_
