// 16-bit elements and matrix operands.
#ifndef NVJ_BF16_H_
#define NVJ_BF16_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvj {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;     // operand of a 16x16x32 product
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;       // its accumulator

__device__ __forceinline__ float bf16_to_f32(uint16_t b) {
  return __uint_as_float((uint32_t)b << 16);
}

// round to nearest even, NaN kept quiet (the hardware conversion)
__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}

// two values, rounded to nearest even, as one word
__device__ __forceinline__ uint32_t pack2_bf16(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  const bf16x2 p = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, p);
}
__device__ __forceinline__ uint32_t pack2_f16(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
  const f16x2 p = {(_Float16)lo, (_Float16)hi};
  return __builtin_bit_cast(uint32_t, p);
}

}  // namespace nvj

#endif  // NVJ_BF16_H_
