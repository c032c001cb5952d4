// Division by a number that only the host knows.
#ifndef NVJ_DIVISOR_H_
#define NVJ_DIVISOR_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvj {

// x / d for 0 <= x < 2^31 as a multiplication (a division by a number only known at run time is 20
// instructions and more, and a launch's workgroups are in front of their first load meanwhile).  With
// bits = ceil(log2 d) the multiplier m = ceil(2^(31 + bits) / d) has 32 bits, and x * m / 2^(31 + bits)
// exceeds x / d by less than x / 2^31 / d: the whole part is the same.
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

// x / d for unsigned x of 32 bits by a reciprocal of d: (x + 0.5) / d is at least 0.5 / d away from a
// whole number, and the reciprocal, one Newton step behind an estimate of 20 bits and more, is off
// by less than 2^-39 of itself.  A wave divides by the same two numbers a dozen times in a launch,
// at some 25 instructions each by way of the compiler and at four here.
__device__ __forceinline__ double reciprocal(int d) {   // d: wave-uniform
  const double x = d, r = __builtin_amdgcn_rcp(x);
  const uint2 bits = __builtin_bit_cast(uint2, __builtin_fma(__builtin_fma(-x, r, 1.0), r, r));
  return __builtin_bit_cast(double, make_uint2(__builtin_amdgcn_readfirstlane(bits.x),
                                               __builtin_amdgcn_readfirstlane(bits.y)));
}
__device__ __forceinline__ uint32_t quotient(uint32_t x, double per) {
  return (uint32_t)(((double)x + 0.5) * per);
}

}  // namespace nvj

#endif
