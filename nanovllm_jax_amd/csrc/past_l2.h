// Stores that do not stay in the writing XCD's L2 (non-temporal): for rows that other XCDs
// read next, which have to leave it anyway, and for rows nobody reads soon, which would
// displace what is read.
#ifndef NVJ_PAST_L2_H_
#define NVJ_PAST_L2_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvj {

__device__ __forceinline__ void store_past_l2(uint4* to, const uint4& v) {
  typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
  const u32x4 t = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(t, reinterpret_cast<u32x4*>(to));
}
__device__ __forceinline__ void store_past_l2(uint2* to, const uint2& v) {
  typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
  const u32x2 t = {v.x, v.y};
  __builtin_nontemporal_store(t, reinterpret_cast<u32x2*>(to));
}

}  // namespace nvj

#endif  // NVJ_PAST_L2_H_
