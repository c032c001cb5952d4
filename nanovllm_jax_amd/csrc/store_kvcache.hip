// KV-cache store for gfx950: scatter the new K/V rows of a step through
// slot_mapping into the block-paged cache, in place.
//
// Stands in for store_kv_to_cache (layers/attention.py:42-77 of the
// reference): cast to the cache dtype (:70-71), then cache[slot] = row for
// every in-range slot (:74-75).  Out-of-range slots are dropped, negative
// slots are skipped.  HBM-bound byte shuffling: every lane moves one 16-byte
// piece of a row (8 cache elements, bf16 or IEEE half), reading either 16
// bytes (source already in the cache's type) or 32 bytes (f32 source, rounded
// to nearest even here).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cache_rows.h"
#include "launch.h"
#include "nvj_paged_attn.h"

namespace {

using nvj::load_piece_as_cache_type;

// One lane per 16-byte piece of one token row, for K and V both.
// pieces_per_row = num_kv_heads * head_dim / 8.
template <bool KF32, bool VF32, bool CF16>
__global__ __launch_bounds__(256) void store_kvcache_kernel(
    const void* __restrict__ key, const void* __restrict__ value,
    uint4* __restrict__ k_cache, uint4* __restrict__ v_cache,
    const int32_t* __restrict__ slot_mapping, int num_tokens,
    int pieces_per_row, int64_t num_slots) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)num_tokens * pieces_per_row;
  if (gid >= total) return;
  const int token = (int)(gid / pieces_per_row);
  const int piece = (int)(gid - (int64_t)token * pieces_per_row);
  const int64_t slot = slot_mapping[token];
  if (slot < 0 || slot >= num_slots) return;
  const uint4 kb = load_piece_as_cache_type<KF32, CF16>(key, gid);
  const uint4 vb = load_piece_as_cache_type<VF32, CF16>(value, gid);
  const int64_t dst = slot * pieces_per_row + piece;
  k_cache[dst] = kb;
  v_cache[dst] = vb;
}

// The same with what a caller would otherwise launch (and on a small call wait for) next to
// it: packed copies of the rows in the cache's type for all tokens (k_rows / v_rows, or
// null), and `clear_words` words at `clear` zeroed by the blocks behind the rows'.  A
// kernel of its own: the longer argument list and the branches cost the plain store 0.5
// of its 2.8 us on a small call.
template <bool KF32, bool VF32, bool CF16>
__global__ __launch_bounds__(256) void store_kvcache_rows_kernel(
    const void* __restrict__ key, const void* __restrict__ value,
    uint4* __restrict__ k_cache, uint4* __restrict__ v_cache,
    const int32_t* __restrict__ slot_mapping, int num_tokens,
    int pieces_per_row, int64_t num_slots, uint4* __restrict__ k_rows, uint4* __restrict__ v_rows,
    int32_t* __restrict__ clear, int clear_words, int row_blocks) {
  if ((int)blockIdx.x >= row_blocks) {
    const int w = ((int)blockIdx.x - row_blocks) * 256 + (int)threadIdx.x;
    if (w < clear_words) clear[w] = 0;
    return;
  }
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)num_tokens * pieces_per_row;
  if (gid >= total) return;
  const int token = (int)(gid / pieces_per_row);
  const int piece = (int)(gid - (int64_t)token * pieces_per_row);
  const int64_t slot = slot_mapping[token];
  const uint4 kb = load_piece_as_cache_type<KF32, CF16>(key, gid);
  const uint4 vb = load_piece_as_cache_type<VF32, CF16>(value, gid);
  if (k_rows != nullptr) k_rows[gid] = kb;
  if (v_rows != nullptr) v_rows[gid] = vb;
  if (slot < 0 || slot >= num_slots) return;
  const int64_t dst = slot * pieces_per_row + piece;
  k_cache[dst] = kb;
  v_cache[dst] = vb;
}

}  // namespace

extern "C" int nvj_store_kvcache_rows_launch(void* stream, const void* key, const void* value,
                                             void* k_cache, void* v_cache,
                                             const int32_t* slot_mapping, int32_t num_tokens,
                                             int32_t num_kv_heads, int32_t head_dim,
                                             int64_t num_slots, int32_t k_dtype,
                                             int32_t v_dtype, int32_t cache_dtype, void* k_rows,
                                             void* v_rows, void* clear, size_t clear_bytes) {
  if (num_tokens < 0 || num_kv_heads <= 0 || head_dim <= 0 || num_slots < 0)
    return NVJ_ERR_BAD_SHAPE;
  if (cache_dtype != NVJ_DTYPE_BF16 && cache_dtype != NVJ_DTYPE_F16) return NVJ_ERR_BAD_DTYPE;
  // a source is float32 (rounded here) or already has the cache's type
  if ((k_dtype != cache_dtype && k_dtype != NVJ_DTYPE_F32) ||
      (v_dtype != cache_dtype && v_dtype != NVJ_DTYPE_F32))
    return NVJ_ERR_BAD_DTYPE;
  const int64_t row = (int64_t)num_kv_heads * head_dim;
  if (row % 8 != 0 || row / 8 > INT32_MAX) return NVJ_ERR_UNSUPPORTED;
  if (num_tokens == 0) return NVJ_OK;
  if (!key || !value || !k_cache || !v_cache || !slot_mapping) return NVJ_ERR_NULL_POINTER;
  if ((reinterpret_cast<uintptr_t>(key) | reinterpret_cast<uintptr_t>(value) |
       reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache) |
       reinterpret_cast<uintptr_t>(k_rows) | reinterpret_cast<uintptr_t>(v_rows)) & 15u)
    return NVJ_ERR_ALIGNMENT;
  if (clear ? ((reinterpret_cast<uintptr_t>(clear) | clear_bytes) & 3u) != 0 : clear_bytes != 0)
    return NVJ_ERR_ALIGNMENT;
  const int pieces = (int)(row / 8);
  const int64_t total = (int64_t)num_tokens * pieces;
  const int64_t blocks = (total + 255) / 256;
  const int64_t clear_words = (int64_t)(clear_bytes / 4);
  const int64_t clear_blocks = (clear_words + 255) / 256;
  if (blocks + clear_blocks > INT32_MAX || clear_words > INT32_MAX - 256) return NVJ_ERR_BAD_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid((unsigned)(blocks + clear_blocks)), block(256);
  uint4* kc = static_cast<uint4*>(k_cache);
  uint4* vc = static_cast<uint4*>(v_cache);
  const bool kf = k_dtype == NVJ_DTYPE_F32, vf = v_dtype == NVJ_DTYPE_F32;
  const bool cf16 = cache_dtype == NVJ_DTYPE_F16;
  hipError_t rc;
  const bool plain = !k_rows && !v_rows && clear_words == 0;
#define NVJ_LAUNCH_STORE(KF, VF, CF)                                                          \
  rc = plain ? nvj::launch(store_kvcache_kernel<KF, VF, CF>, grid, block, s, key, value, kc,  \
                           vc, slot_mapping, num_tokens, pieces, num_slots)                   \
             : nvj::launch(store_kvcache_rows_kernel<KF, VF, CF>, grid, block, s, key, value, \
                           kc, vc, slot_mapping, num_tokens, pieces, num_slots,               \
                           static_cast<uint4*>(k_rows), static_cast<uint4*>(v_rows),          \
                           static_cast<int32_t*>(clear), (int)clear_words, (int)blocks)
  switch ((kf ? 4 : 0) | (vf ? 2 : 0) | (cf16 ? 1 : 0)) {
    case 0: NVJ_LAUNCH_STORE(false, false, false); break;   // copies: the type does not matter
    case 1: NVJ_LAUNCH_STORE(false, false, false); break;
    case 2: NVJ_LAUNCH_STORE(false, true, false); break;
    case 3: NVJ_LAUNCH_STORE(false, true, true); break;
    case 4: NVJ_LAUNCH_STORE(true, false, false); break;
    case 5: NVJ_LAUNCH_STORE(true, false, true); break;
    case 6: NVJ_LAUNCH_STORE(true, true, false); break;
    default: NVJ_LAUNCH_STORE(true, true, true); break;
  }
#undef NVJ_LAUNCH_STORE
  return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
}

extern "C" int nvj_store_kvcache_launch(void* stream, const void* key, const void* value,
                                        void* k_cache, void* v_cache,
                                        const int32_t* slot_mapping, int32_t num_tokens,
                                        int32_t num_kv_heads, int32_t head_dim,
                                        int64_t num_slots, int32_t k_dtype,
                                        int32_t v_dtype, int32_t cache_dtype) {
  return nvj_store_kvcache_rows_launch(stream, key, value, k_cache, v_cache, slot_mapping,
                                       num_tokens, num_kv_heads, head_dim, num_slots, k_dtype,
                                       v_dtype, cache_dtype, nullptr, nullptr, nullptr, 0);
}
