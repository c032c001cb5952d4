// Fused per-head QK-RMSNorm + rotary embedding + KV-cache store for gfx950.
//
// One launch replaces the chain the reference runs between the QKV projection
// and the attention call of a decode (or prefill) step:
//   q, k = q_norm(q), k_norm(k)        models/qwen3.py:157-160, layers/layernorm.py:31-48
//   q, k = rotary_emb(positions, q, k) models/qwen3.py:163, layers/rotary_embedding.py:13-37,96-106
//   q -> cache dtype                   layers/attention.py:386-387
//   store_kv_to_cache(k, v, ...)       layers/attention.py:42-77 (cast at :70-71)
// It reads the packed QKV projection output once and writes q (bf16) plus the
// K and V cache rows; nothing else touches HBM.
//
// Bytes in and out are what bounds it with many rows, the chain of dependent loads
// (slot, position, its table row) with few.  16 lanes per (token, head), four heads
// per wave: lane i holds elements 4i .. 4i+3 and 64+4i .. 64+4i+3, whole rotary
// pairs in 8-byte loads, so the rotation needs no cross-lane traffic.  (One wave per
// head, 2-byte loads, took 42.6 us for 4400 rows of 32 heads.)  With l the element
// of the lower half, the mean of squares is the same xor butterfly over l whatever
// lanes hold it.  The arithmetic is a fixed sequence of IEEE fp32 operations (no
// contraction, no approximate rsqrt) so that a CPU restatement reproduces it bit for
// bit:
//   s_l   = fma(x2, x2, x1 * x1)            (fp32 values of the bf16 inputs)
//   s_l  += s_(l ^ m)  for m = 32, 16, 8, 4, 2, 1
//   r     = 1 / sqrt(s / 128 + eps)
//   n_i   = bf16(x_i * r * w_i)             (cast back to the input dtype)
//   y1    = n1 * cos - n2 * sin,  y2 = n2 * cos + n1 * sin   (fp32)
//   out   = bf16(y)                         (round to nearest even)
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.h"
#include "nvj_paged_attn.h"
#include "qk_norm_rope.h"

namespace {

constexpr int kHeadDim = 128;

struct QkArgs {
  const uint16_t* qkv;        // [T, >= (Hq+2Hkv)*128] bf16
  int64_t qkv_row_stride;
  const int32_t* positions;   // [T]
  const float* cos_sin;       // [max_position, 128]: cos | sin
  const float* q_weight;      // [128] or null
  const float* k_weight;
  const int32_t* slot_mapping;   // [T]
  uint16_t* k_cache;          // [num_slots, Hkv, 128]
  uint16_t* v_cache;
  uint16_t* q_out;            // [T, >= Hq*128]; may be qkv itself
  int64_t q_row_stride;
  uint16_t* k_out;            // [T, >= Hkv*128] the new rows besides the cache, or null; may lie in qkv
  uint16_t* v_out;
  int64_t kv_row_stride;
  float eps;
  int max_position, num_tokens, num_heads, num_kv_heads;
  int64_t num_slots;
};

// WIDE: everything is aligned for 8- and 16-byte accesses; otherwise element by
// element (rows at odd offsets inside a larger buffer).
template <bool WIDE>
__device__ __forceinline__ uint2 load4(const uint16_t* p) {
  if (WIDE) return *reinterpret_cast<const uint2*>(p);
  return make_uint2(p[0] | ((uint32_t)p[1] << 16), p[2] | ((uint32_t)p[3] << 16));
}
template <bool WIDE>
__device__ __forceinline__ void store4(uint16_t* p, uint2 v) {
  if (WIDE) {
    *reinterpret_cast<uint2*>(p) = v;
  } else {
    p[0] = (uint16_t)v.x; p[1] = (uint16_t)(v.x >> 16);
    p[2] = (uint16_t)v.y; p[3] = (uint16_t)(v.y >> 16);
  }
}

// grid.x = ceil(num_tokens * heads_total / 16), block = 256: 16 groups of 16 lanes.
// Every load that depends on nothing but the (token, head) is issued together.
template <bool WIDE>
__global__ __launch_bounds__(256) void qk_norm_rope_store_kernel(QkArgs a) {
  const int heads_total = a.num_heads + 2 * a.num_kv_heads;
  const int64_t unit = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (unit >= (int64_t)a.num_tokens * heads_total) return;
  const int token = (int)(unit / heads_total);
  const int head = (int)(unit - (int64_t)token * heads_total);
  const int i = threadIdx.x & 15;
  const uint16_t* src = a.qkv + (int64_t)token * a.qkv_row_stride + (int64_t)head * kHeadDim + 4 * i;
  uint2 lo = load4<WIDE>(src), hi = load4<WIDE>(src + 64);
  const int pos = min(max(a.positions[token], 0), a.max_position - 1);
  const int64_t slot = a.slot_mapping[token];
  const bool is_q = head < a.num_heads;
  const bool is_k = !is_q && head < a.num_heads + a.num_kv_heads;
  if (is_q || is_k) {
    const float* cs = a.cos_sin + (int64_t)pos * kHeadDim + 4 * i;
    nvj::qk_norm_rope<WIDE>(lo, hi, is_q ? a.q_weight : a.k_weight, a.eps, nvj::load4<WIDE>(cs),
                            nvj::load4<WIDE>(cs + 64), i);
  }
  auto put = [&](uint16_t* row) {
    store4<WIDE>(row + 4 * i, lo);
    store4<WIDE>(row + 64 + 4 * i, hi);
  };
  if (is_q) {
    put(a.q_out + (int64_t)token * a.q_row_stride + (int64_t)head * kHeadDim);
    return;
  }
  const int kvh = head - a.num_heads - (is_k ? 0 : a.num_kv_heads);
  uint16_t* rows = is_k ? a.k_out : a.v_out;
  if (rows != nullptr) put(rows + (int64_t)token * a.kv_row_stride + (int64_t)kvh * kHeadDim);
  if (slot >= 0 && slot < a.num_slots)   // else: skipped / dropped token
    put((is_k ? a.k_cache : a.v_cache) + (slot * a.num_kv_heads + kvh) * kHeadDim);
}

}  // namespace

extern "C" int nvj_qk_norm_rope_rows_launch(
    void* stream, const void* qkv, int64_t qkv_row_stride, const int32_t* positions,
    const float* cos_sin_cache, int32_t max_position, const float* q_norm_weight,
    const float* k_norm_weight, float eps, const int32_t* slot_mapping, void* k_cache,
    void* v_cache, void* q_out, int64_t q_row_stride, void* k_out, void* v_out,
    int64_t kv_row_stride, int32_t num_tokens, int32_t num_heads, int32_t num_kv_heads,
    int32_t head_dim, int64_t num_slots) {
  if (num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 || max_position <= 0 || num_slots < 0)
    return NVJ_ERR_BAD_SHAPE;
  if (head_dim != kHeadDim) return NVJ_ERR_UNSUPPORTED;
  const int64_t heads_total = (int64_t)num_heads + 2 * (int64_t)num_kv_heads;
  if (qkv_row_stride < heads_total * kHeadDim || (qkv_row_stride & 1) ||
      q_row_stride < (int64_t)num_heads * kHeadDim ||
      ((k_out || v_out) && kv_row_stride < (int64_t)num_kv_heads * kHeadDim))
    return NVJ_ERR_BAD_SHAPE;
  if (num_tokens == 0) return NVJ_OK;
  if (!qkv || !positions || !cos_sin_cache || !slot_mapping || !k_cache || !v_cache || !q_out)
    return NVJ_ERR_NULL_POINTER;
  if ((q_norm_weight == nullptr) != (k_norm_weight == nullptr)) return NVJ_ERR_NULL_POINTER;
  const uintptr_t rows = reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(k_cache) |
                         reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(q_out) |
                         reinterpret_cast<uintptr_t>(k_out) | reinterpret_cast<uintptr_t>(v_out);
  const int64_t strides = qkv_row_stride | q_row_stride | ((k_out || v_out) ? kv_row_stride : 0);
  if ((rows & 3u) || (strides & 1)) return NVJ_ERR_ALIGNMENT;
  const uintptr_t tables = reinterpret_cast<uintptr_t>(cos_sin_cache) |
                           reinterpret_cast<uintptr_t>(q_norm_weight) |
                           reinterpret_cast<uintptr_t>(k_norm_weight);
  const bool wide = (rows & 7u) == 0 && (strides & 3) == 0 && (tables & 15u) == 0;
  const int64_t units = (int64_t)num_tokens * heads_total;
  const int64_t blocks = (units + 15) / 16;
  if (blocks > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  QkArgs a;
  a.qkv = static_cast<const uint16_t*>(qkv);
  a.qkv_row_stride = qkv_row_stride;
  a.positions = positions;
  a.cos_sin = cos_sin_cache;
  a.q_weight = q_norm_weight;
  a.k_weight = k_norm_weight;
  a.slot_mapping = slot_mapping;
  a.k_cache = static_cast<uint16_t*>(k_cache);
  a.v_cache = static_cast<uint16_t*>(v_cache);
  a.q_out = static_cast<uint16_t*>(q_out);
  a.q_row_stride = q_row_stride;
  a.k_out = static_cast<uint16_t*>(k_out);
  a.v_out = static_cast<uint16_t*>(v_out);
  a.kv_row_stride = kv_row_stride;
  a.eps = eps;
  a.max_position = max_position;
  a.num_tokens = num_tokens;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.num_slots = num_slots;
  const auto kernel = wide ? qk_norm_rope_store_kernel<true> : qk_norm_rope_store_kernel<false>;
  const hipError_t rc = nvj::launch(kernel, dim3((unsigned)blocks), dim3(256),
                                    static_cast<hipStream_t>(stream), a);
  return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
}

extern "C" int nvj_qk_norm_rope_store_launch(void* stream, const void* qkv, int64_t qkv_row_stride,
                                             const int32_t* positions, const float* cos_sin_cache,
                                             int32_t max_position, const float* q_norm_weight,
                                             const float* k_norm_weight, float eps,
                                             const int32_t* slot_mapping, void* k_cache,
                                             void* v_cache, void* q_out, int32_t num_tokens,
                                             int32_t num_heads, int32_t num_kv_heads,
                                             int32_t head_dim, int64_t num_slots) {
  return nvj_qk_norm_rope_rows_launch(stream, qkv, qkv_row_stride, positions, cos_sin_cache,
                                      max_position, q_norm_weight, k_norm_weight, eps, slot_mapping,
                                      k_cache, v_cache, q_out, (int64_t)num_heads * kHeadDim,
                                      nullptr, nullptr, 0, num_tokens, num_heads, num_kv_heads,
                                      head_dim, num_slots);
}
