// New K/V rows on their way into the cache: a piece of 8 elements, rounded where the
// source is float32.
#ifndef NVJ_CACHE_ROWS_H_
#define NVJ_CACHE_ROWS_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvj {

// fp32 -> bf16 bits, round to nearest even, NaN kept quiet.  Integer
// arithmetic so the result is bit-identical on every path.
__device__ __forceinline__ uint32_t f32_to_bf16_rne(uint32_t u) {
  uint32_t r = (u + (((u >> 16) & 1u) + 0x7FFFu)) >> 16;
  const bool is_nan = (u & 0x7FFFFFFFu) > 0x7F800000u;
  return is_nan ? ((u >> 16) | 0x0040u) : r;
}

// fp32 -> IEEE half bits, round to nearest even (the hardware conversion).
__device__ __forceinline__ uint32_t f32_to_f16_rne(uint32_t u) {
  const _Float16 h = (_Float16)__uint_as_float(u);
  return (uint32_t)__builtin_bit_cast(uint16_t, h);
}

// One piece of a source row as 8 cache elements.  F32: the source is float32
// and is rounded to the cache's type (CF16: IEEE half, else bf16); otherwise
// the source already has the cache's type and is copied.
template <bool F32, bool CF16>
__device__ __forceinline__ uint4 load_piece_as_cache_type(const void* src, int64_t piece) {
  if constexpr (!F32) {
    return reinterpret_cast<const uint4*>(src)[piece];
  } else {
    const uint4* p = reinterpret_cast<const uint4*>(src) + 2 * piece;
    const uint4 a = p[0], b = p[1];
    auto cvt = [](uint32_t u) { return CF16 ? f32_to_f16_rne(u) : f32_to_bf16_rne(u); };
    uint4 o;
    o.x = cvt(a.x) | (cvt(a.y) << 16);
    o.y = cvt(a.z) | (cvt(a.w) << 16);
    o.z = cvt(b.x) | (cvt(b.y) << 16);
    o.w = cvt(b.z) | (cvt(b.w) << 16);
    return o;
  }
}

}  // namespace nvj

#endif  // NVJ_CACHE_ROWS_H_
