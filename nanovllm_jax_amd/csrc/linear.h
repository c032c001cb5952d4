// Products of activation rows with weights, with the stage that follows them (linear.hip).
#ifndef NVJ_LINEAR_H_
#define NVJ_LINEAR_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "read_ahead.h"

namespace nvj {

struct LinearArgs {
  const char* x;      // [M, K] bf16
  const char* w;      // [N, K] bf16
  uint16_t* out;      // [M, N] bf16; linear_silu_mul: [M, N / 2]
  int M, N, K;
  // linear_qk_rope: N = (num_heads + 2 * num_kv_heads) * 128
  uint16_t* q_out;               // [M, num_heads * 128]
  bool keep_kv;                  // K and V also to their columns of out (q is never written there)
  const int32_t* positions;      // [M]
  const float* cos_sin;          // [max_position, 128]: cos | sin
  const float* q_norm;           // [128], or null with k_norm
  const float* k_norm;
  const int32_t* slot_mapping;   // [M]
  uint16_t* k_cache;             // [num_slots, num_kv_heads, 128]
  uint16_t* v_cache;
  float eps;
  int max_position, num_heads, num_kv_heads;
  int64_t num_slots;
  ReadAhead ahead;                 // by workgroups behind the product's own (not linear_chained)
  int m_tiles, n_tiles;            // filled in by the launch
  int tile;                        // 1 + index of the tile shape, 0: by the sizes
};

// Whether the kernels can be given these sizes at all.
bool linear_takes(int64_t m, int64_t n, int64_t k);

// bf16 rows; `for_later`: no launch of this step reads them.  (An argument of the host alone: one
// more field in LinearArgs and the QKV kernel loads its arguments in four pieces, 7.6 -> 8.3 us.)
hipError_t linear(hipStream_t s, LinearArgs a, bool for_later = false);
hipError_t linear_silu_mul(hipStream_t s, LinearArgs a);   // SiLU(gate) * up; N / 2 a multiple of 16
hipError_t linear_qk_rope(hipStream_t s, LinearArgs a);    // QK-norm, RoPE, KV store
// The reduction cut into `chains` interleaved runs of `run` steps of 32, summed in order:
// (4, 1), (4, 2) or (2, 4); K a multiple of 32 * chains * run.
hipError_t linear_chained(hipStream_t s, const LinearArgs& a, int chains, int run);

}  // namespace nvj

#endif  // NVJ_LINEAR_H_
