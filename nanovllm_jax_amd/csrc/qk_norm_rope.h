// QK-RMSNorm and rotary embedding of one 128-wide head row held by 16 lanes: lane i
// holds elements 4i .. 4i+3 and 64+4i .. 64+4i+3, whole rotary pairs, as two packed
// groups of four bf16.  The arithmetic is the fixed sequence of IEEE fp32 operations
// documented in qk_norm_rope_store.hip.
#ifndef NVJ_QK_NORM_ROPE_H_
#define NVJ_QK_NORM_ROPE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bf16.h"
#include "wave_ops.h"

namespace nvj {

__device__ __forceinline__ void unpack4(uint2 p, float (&f)[4]) {
  f[0] = __uint_as_float(p.x << 16); f[1] = __uint_as_float(p.x & 0xFFFF0000u);
  f[2] = __uint_as_float(p.y << 16); f[3] = __uint_as_float(p.y & 0xFFFF0000u);
}
__device__ __forceinline__ uint2 pack4(const float (&f)[4]) {
  return make_uint2(pack2_bf16(f[0], f[1]), pack2_bf16(f[2], f[3]));
}

// WIDE: the pointers are 16-byte aligned.
template <bool WIDE>
__device__ __forceinline__ float4 load4(const float* p) {
  if (WIDE) return *reinterpret_cast<const float4*>(p);
  return make_float4(p[0], p[1], p[2], p[3]);
}

// `norm`: with the RMSNorm, of weights wl and wh (the lane's elements 4i .. and 64 + 4i ..);
// c4, s4: the lane's four cosines and sines of this position (all 16 lanes are active).
__device__ __forceinline__ void qk_norm_rope(uint2& lo, uint2& hi, bool norm, const float4& wl,
                                             const float4& wh, float eps, const float4& c4,
                                             const float4& s4) {
#pragma clang fp contract(off)
  float x1[4], x2[4];
  unpack4(lo, x1);
  unpack4(hi, x2);
  if (norm) {
    const float w1[4] = {wl.x, wl.y, wl.z, wl.w}, w2[4] = {wh.x, wh.y, wh.z, wh.w};
    float s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = __builtin_fmaf(x2[e], x2[e], x1[e] * x1[e]);
    // butterfly over l = 4 * lane + e: masks 32 .. 4 are lanes 8 .. 1 apart (inside a
    // row of 16: DPP moves), masks 2 and 1 elements of a lane
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += row_move<0x128>(s[e]);                    // row_ror:8
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += row_move<0x124>(s[e]);   // row_ror:4, i ^ 4 or i ^ 4 ^ 8
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += row_move<0x4E>(s[e]);                     // i ^ 2
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += row_move<0xB1>(s[e]);                     // i ^ 1
    const float sum = (s[0] + s[2]) + (s[1] + s[3]);
    const float r = 1.0f / __builtin_sqrtf(sum * (1.0f / 128) + eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x1[e] = x1[e] * r * w1[e];
      x2[e] = x2[e] * r * w2[e];
    }
    unpack4(pack4(x1), x1);
    unpack4(pack4(x2), x2);
  }
  const float c[4] = {c4.x, c4.y, c4.z, c4.w}, sn[4] = {s4.x, s4.y, s4.z, s4.w};
  float y1[4], y2[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    y1[e] = x1[e] * c[e] - x2[e] * sn[e];
    y2[e] = x2[e] * c[e] + x1[e] * sn[e];
  }
  lo = pack4(y1);
  hi = pack4(y2);
}
// `weight`: [128] or null (no norm); i: the lane in its group of 16.
template <bool WIDE>
__device__ __forceinline__ void qk_norm_rope(uint2& lo, uint2& hi, const float* weight, float eps,
                                             const float4& c4, const float4& s4, int i) {
  float4 wl = {}, wh = {};
  if (weight != nullptr) {
    wl = load4<WIDE>(weight + 4 * i);
    wh = load4<WIDE>(weight + 64 + 4 * i);
  }
  qk_norm_rope(lo, hi, weight != nullptr, wl, wh, eps, c4, s4);
}

}  // namespace nvj

#endif  // NVJ_QK_NORM_ROPE_H_
