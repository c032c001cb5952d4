// Division by a number that only the host knows.
#ifndef NVJ_DIVISOR_H_
#define NVJ_DIVISOR_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvj {

// x / d for 0 <= x < 2^31 as a multiplication (a division by a number only known at run time is 20
// instructions and more, and a
// launch's workgroups are in front of their first load meanwhile).  With
// bits = ceil(log2 d) the multiplier m = ceil(2^(31 + bits) / d) has 32 bits, and x * m / 2^(31 +
// bits) exceeds x / d by less than x / 2^31 / d: the whole part is the same.
struct Divisor {
  uint32_t multiplier, bits;
  int32_t d;
  Divisor() = default;
  explicit Divisor(int64_t divisor) : bits(0), d((int32_t)divisor) {
    while (((int64_t)1 << bits) < divisor) ++bits;
    multiplier = (uint32_t)((((uint64_t)1 << (31 + bits)) + divisor - 1) / divisor);
  }
  __device__ __forceinline__ int divide(int x) const {
    return (int)(__umulhi(2u * (uint32_t)x, multiplier) >> bits);
  }
};

}  // namespace nvj

#endif
