// One step of the whole decoder stack (a decode batch, or the prefill of new prompts)
// as a chain of launches enqueued in one call for gfx950.
//
// Covers the layer body of models/qwen3.py:130-172 and :285-318 of the reference
// (fused QKV, per-head QK-RMSNorm, RoPE, store, attention, output projection,
// pre-norm with fused residual, SiLU MLP), the embedding and the tied LM head
// (:366-393, :472-491):
// With up to 16 token rows, six launches per layer:
//   1. norm_gemm QKV       RMSNorm in the prologue
//   2. qk_norm_rope_store
//   3. attention           the paged decode or the prefill kernel
//   4. residual_gemm O     adds into the residual stream
//   5. norm_gemm GATE_UP   RMSNorm in the prologue, SiLU(gate) * up in the epilogue
//   6. residual_gemm DOWN
// With more, the products of linear.hip between the norms of layer_glue.hip: QKV with
// norm, RoPE and store in its epilogue, attention, O, add + norm, GATE_UP with SiLU * up
// in its epilogue, DOWN, add + norm.
// The residual stream h holds the unrounded fp32 sums that the next norm is taken
// over; the sum that follows adds to their bf16 rounding, so every value is
// rounded where the separate kernels (layer_glue.hip) round it.
//
// What bounds the first form: with few rows every product streams its weights once and the rest
// is latency, so a launch is worth its fixed 2-3 us only if the weights it
// needs are all requested before anything else is waited for, by all CUs (one CU
// alone draws some 50 GB/s).  Each wave therefore issues the loads of its whole
// share of the weights at once, straight into the registers the matrix core reads
// them from (a wave's share is used by that wave only, LDS would add nothing), and
// does the norm prologue under them.  The token rows are the N side of
// v_mfma_f32_16x16x32_bf16 (weights A, rows B), 16 per column tile.
//
// Order of the sums.  A network of random bf16 weights doubles any difference of one
// ulp from stage to stage until all roundings differ (two GEMM kernels that sum in
// different orders end 2-3 % apart in the logits after 28 layers).  The reduction of these
// products is therefore cut into `chains` interleaved runs of `run` steps of 32, each chain
// accumulated in order and the chains added in order, as the library GEMMs that the step ran
// through before did at hidden 1024 / intermediate 3072 (found by comparing the bits of each
// form with theirs over 1 .. 4400 rows):
//   rows          QKV, gate/up   O       down
//   1 .. 16       4 x 1          4 x 1   2 x 4
//   17 .. 128     one chain      4 x 1   2 x 4 up to 64 but 32, else 4 x 2
//   more          one chain      one chain
// That keeps a program's logits where they were at that width, and is all it does: at other
// widths the library sums in other orders, any of these is as exact (fp32 sums), and a
// library of another version may differ everywhere.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bf16.h"
#include "launch.h"
#include "linear.h"
#include "nvj_paged_attn.h"
#include "read_ahead.h"
#include "wave_ops.h"

namespace {

using nvj::bf16_to_f32;
using nvj::bf16x8;
using nvj::f32_to_bf16_rne;
using nvj::f32x4;
using nvj::pack2_bf16;

constexpr int kMaxRows = 16;   // token rows of one step: one column tile

__device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
enum Epilogue { kPlain, kSiluMul };

struct NormGemmArgs {
  const float4* h;            // [rows, hidden] residual stream
  const int32_t* row_index;   // rows to take from h (row_of_index), or null: row m is row m
  const float* norm_weight;   // [hidden]
  const char* weight;         // [outputs, hidden] bf16
  uint16_t* out;              // kPlain [rows, outputs], kSiluMul [rows, outputs / 2]
  float eps;
  int num_tokens, outputs;
  int num_rows;               // of h, with row_index
};

// The row of `rows` that an index names: a negative one counts from the end, as tensor
// indexing on the host does (a sequence without new tokens in front of all others has
// index -1).  One that names no row gives `real` = false and row 0, which is in range:
// its output is NaN.
struct IndexedRow {
  int row;
  bool real;
};
__device__ __forceinline__ IndexedRow row_of_index(int index, int rows) {
  if (index < 0) index += rows;
  const bool real = (uint32_t)index < (uint32_t)rows;
  return {real ? index : 0, real};
}

// RMSNorm of up to 16 rows of h into LDS as bf16, `WAVES` waves, a row each at a time;
// the arithmetic and its order are those of add_rms_norm_kernel (layer_glue.hip).
// 16-byte pieces are XOR-permuted by the row so that the B-operand reads are free of
// bank conflicts.  hidden = 256 * RV.  Two halves, so that the caller can issue other
// loads in between.
template <int RV, int ROWS>
struct NormPrologue {
  static constexpr int kHidden = 256 * RV;
  static constexpr int kPieces = kHidden / 8;               // of a row
  static constexpr int kPerLane = (kPieces + 63) / 64;
  float4 x[ROWS][kPerLane][2], g[kPerLane][2];

  __device__ __forceinline__ void load(const NormGemmArgs& a, int wave, int waves, int lane) {
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      const int token = min(wave + waves * j, a.num_tokens - 1);
      IndexedRow at = {token, true};
      if (a.row_index) at = row_of_index(a.row_index[token], a.num_rows);
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) {
        const int p = min(lane + 64 * i, kPieces - 1);
        const float4* src = a.h + (int64_t)at.row * (kHidden / 4) + 2 * p;
        x[j][i][0] = src[0];
        x[j][i][1] = src[1];
      }
      if (!at.real) x[j][0][0].x = __builtin_nanf("");   // reaches the whole row by its norm
    }
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int p = min(lane + 64 * i, kPieces - 1);
      g[i][0] = reinterpret_cast<const float4*>(a.norm_weight)[2 * p];
      g[i][1] = reinterpret_cast<const float4*>(a.norm_weight)[2 * p + 1];
    }
  }

  __device__ __forceinline__ void store(uint4* lds, float eps, int wave, int waves, int lane) const {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      const int m = wave + waves * j;   // (a row beyond the last token repeats it)
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) {
        if (kPieces % 64 == 0 || lane + 64 * i < kPieces) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const float4 v = x[j][i][u];
            sum = sum + v.x * v.x;
            sum = sum + v.y * v.y;
            sum = sum + v.z * v.z;
            sum = sum + v.w * v.w;
          }
        }
      }
      sum = nvj::wave_sum(sum);
      const float rs = 1.0f / __builtin_sqrtf(sum * (1.0f / (float)kHidden) + eps);
#pragma unroll
      for (int i = 0; i < kPerLane; ++i) {
        const int p = lane + 64 * i;
        const float4 u = x[j][i][0], v = x[j][i][1], gu = g[i][0], gv = g[i][1];
        if (kPieces % 64 == 0 || p < kPieces)
          lds[m * kPieces + (p ^ m)] =
              make_uint4(pack2_bf16(u.x * rs * gu.x, u.y * rs * gu.y),
                         pack2_bf16(u.z * rs * gu.z, u.w * rs * gu.w),
                         pack2_bf16(v.x * rs * gv.x, v.y * rs * gv.y),
                         pack2_bf16(v.z * rs * gv.z, v.w * rs * gv.w));
      }
    }
  }
};

// out[m][n] = bf16(norm(h[m]) . weight[n]) for up to 16 rows, four chains of single
// steps: one 16-output tile per workgroup, a chain per wave.  kSiluMul: the tile is 8
// gate and the matching 8 up columns.
template <int RV, int ROWS, Epilogue EPI>
__global__ __launch_bounds__(256) void norm_gemm_kernel(NormGemmArgs a) {
  constexpr int kWaves = 4;                  // = chains
  constexpr int kPieces = 32 * RV;
  constexpr int kSteps = 8 * RV / kWaves;    // reduction steps of one chain
  constexpr int kStride = 20;                // floats per row of partial sums
  __shared__ uint4 rows[16 * kPieces];
  __shared__ float red[kWaves][16 * kStride];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int half = a.outputs / 2;
  const int n = EPI == kSiluMul ? (int)blockIdx.x * 8 + (r & 7) + (r < 8 ? 0 : half)
                                : (int)blockIdx.x * 16 + r;
  const char* wrow = a.weight + (int64_t)n * (kPieces * 16) + 64 * wave + 16 * kg;
  NormPrologue<RV, ROWS> norm;
  norm.load(a, wave, kWaves, lane);
  // loads return in order: the weights are asked for right behind the rows, so that
  // the norm waits for the rows alone
  uint4 w[kSteps];
#pragma unroll
  for (int i = 0; i < kSteps; ++i)
    w[i] = *reinterpret_cast<const uint4*>(wrow + 64 * kWaves * i);
  __builtin_amdgcn_sched_barrier(0);
  norm.store(rows, a.eps, wave, kWaves, lane);
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};   // D[output][row]
  // (with fewer than 16 rows in LDS the other columns read what is there: not stored)
  const int m = ROWS * kWaves >= 16 ? r : r % (ROWS * kWaves);
#pragma unroll
  for (int i = 0; i < kSteps; ++i)
    acc = mfma(w[i], rows[m * kPieces + ((4 * (kWaves * i + wave) + kg) ^ m)], acc);
  *reinterpret_cast<f32x4*>(&red[wave][r * kStride + 4 * kg]) = acc;
  __syncthreads();
  auto total = [&](int row, int col) {
    float v = red[0][row * kStride + col];
#pragma unroll
    for (int p = 1; p < kWaves; ++p) v += red[p][row * kStride + col];
    return f32_to_bf16_rne(v);
  };
  if constexpr (EPI == kSiluMul) {
    const int row = threadIdx.x >> 3, col = threadIdx.x & 7;
    if (row < a.num_tokens) {
      const float g = bf16_to_f32(total(row, col)), u = bf16_to_f32(total(row, 8 + col));
      a.out[(int64_t)row * half + blockIdx.x * 8 + col] =
          f32_to_bf16_rne(g / (1.0f + expf(-g)) * u);
    }
  } else {
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    if (row < a.num_tokens)
      a.out[(int64_t)row * a.outputs + blockIdx.x * 16 + col] = total(row, col);
  }
}

// The same with one chain, for many outputs (the LM head): every wave owns a whole
// 16-output tile, its weights in flight together.  NORM: the rows are normalised here;
// otherwise a.h holds bf16 rows that have been.
template <int RV, int ROWS, bool NORM>
__global__ __launch_bounds__(256) void norm_gemm_wide_kernel(NormGemmArgs a) {
  constexpr int kWaves = 4;
  constexpr int kPieces = 32 * RV;
  constexpr int kSteps = 8 * RV;
  constexpr int kDepth = kSteps < 32 ? kSteps : 32;
  __shared__ uint4 rows[16 * kPieces];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int n0 = (blockIdx.x * kWaves + wave) * 16;
  const char* wrow =
      a.weight + (int64_t)min(n0 + r, a.outputs - 1) * (kPieces * 16) + 16 * kg;
  NormPrologue<RV, ROWS> norm;
  if constexpr (NORM) {
    norm.load(a, wave, kWaves, lane);
  } else {
    const uint4* x = reinterpret_cast<const uint4*>(a.h);
#pragma unroll
    for (int j = 0; j < ROWS; ++j) {
      const int m = wave + kWaves * j;
      for (int p = lane; p < kPieces; p += 64)
        rows[m * kPieces + (p ^ m)] = x[(int64_t)min(m, a.num_tokens - 1) * kPieces + p];
    }
  }
  uint4 w[kDepth];
#pragma unroll
  for (int i = 0; i < kDepth; ++i) w[i] = *reinterpret_cast<const uint4*>(wrow + 64 * i);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NORM) norm.store(rows, a.eps, wave, kWaves, lane);
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int m = ROWS * kWaves >= 16 ? r : r % (ROWS * kWaves);
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    acc = mfma(w[i % kDepth], rows[m * kPieces + ((4 * i + kg) ^ m)], acc);
    if (i + kDepth < kSteps)
      w[i % kDepth] = *reinterpret_cast<const uint4*>(wrow + 64 * (i + kDepth));
  }
  if (r < a.num_tokens) {
    uint16_t* dst = a.out + (int64_t)r * a.outputs + n0 + 4 * kg;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n0 + 4 * kg + e < a.outputs) dst[e] = f32_to_bf16_rne(acc[e]);
  }
}

// h[m][n] = bf16(x[m][:] . weight[n][:]) + bf16(h[m][n]) for up to 16 rows.  A
// workgroup owns NR outputs (the A rows repeat NR of them: narrower tiles put more CUs
// on a matrix of few outputs) and has a wave for each of CHAINS x PARTS shares of the
// reduction: T steps, whose operands all waves fetch at once.  The parts of a chain
// hand its sum on through LDS, in order; the chains are added at the end.
template <int NR, int CHAINS, int RUN, int PARTS, int T>
__global__ __launch_bounds__(CHAINS * PARTS * 64) void residual_gemm_kernel(
    const char* __restrict__ x, const char* __restrict__ weight, float* __restrict__ h,
    int num_tokens, int outputs) {
  constexpr int64_t kRowBytes = (int64_t)CHAINS * PARTS * T * 64;
  __shared__ f32x4 sums[CHAINS][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chain = wave % CHAINS, part = wave / CHAINS;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * NR;
  const char* wrow = weight + (int64_t)(n0 + r % NR) * kRowBytes + 16 * kg;
  const char* xrow = x + min(r, num_tokens - 1) * kRowBytes + 16 * kg;
  uint4 w[T], b[T];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int j = part * T + i;   // step of the chain
    const int at = 64 * (j / RUN * (CHAINS * RUN) + chain * RUN + j % RUN);
    w[i] = *reinterpret_cast<const uint4*>(wrow + at);
    b[i] = *reinterpret_cast<const uint4*>(xrow + at);
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < PARTS; ++p) {
    if (part == p) {
      if (p > 0) acc = sums[chain][lane];
#pragma unroll
      for (int i = 0; i < T; ++i) acc = mfma(w[i], b[i], acc);
      sums[chain][lane] = acc;
    }
    __syncthreads();
  }
  if (wave == 0 && r < num_tokens && 4 * kg < NR) {
    f32x4 v = sums[0][lane];
#pragma unroll
    for (int c = 1; c < CHAINS; ++c) v += sums[c][lane];
    float4* at = reinterpret_cast<float4*>(h + (int64_t)r * outputs + n0 + 4 * kg);
    const float4 old = *at;
    auto round = [](float f) { return bf16_to_f32(f32_to_bf16_rne(f)); };
    *at = make_float4(round(v[0]) + round(old.x), round(v[1]) + round(old.y),
                      round(v[2]) + round(old.z), round(v[3]) + round(old.w));
  }
}

// Waves per chain: the shares are at most 12 steps (96 registers of operands).
template <int CHAINS, int RUN, int PARTS>
hipError_t launch_residual_gemm(hipStream_t s, const void* x, const void* weight, float* h,
                                int num_tokens, int outputs, int reduction) {
  constexpr int NR = 8;
  const dim3 grid((unsigned)(outputs / NR)), block(CHAINS * PARTS * 64);
#define NVJ_CASE(TV)                                                                              \
  case TV:                                                                                        \
    return nvj::launch(residual_gemm_kernel<NR, CHAINS, RUN, PARTS, TV>, grid, block, s,          \
                       static_cast<const char*>(x), static_cast<const char*>(weight), h,          \
                       num_tokens, outputs)
  switch (reduction / (CHAINS * PARTS * 32)) {
    NVJ_CASE(1); NVJ_CASE(2); NVJ_CASE(3); NVJ_CASE(4); NVJ_CASE(5); NVJ_CASE(6);
    NVJ_CASE(7); NVJ_CASE(8); NVJ_CASE(9); NVJ_CASE(10); NVJ_CASE(11); NVJ_CASE(12);
    default: return hipErrorInvalidValue;
  }
#undef NVJ_CASE
}
bool residual_gemm_takes(int64_t reduction) {
  return reduction % 256 == 0 && reduction <= 12 * 256;   // both of the forms below: 8 waves
}

__device__ constexpr uint4 kNanPiece = {0x7FC07FC0u, 0x7FC07FC0u, 0x7FC07FC0u, 0x7FC07FC0u};

// h[m] = float(embed[ids[m]]), one wave per row; NaN for an id outside the table, which then
// shows in the logits of its sequence and in no other.
__global__ __launch_bounds__(256) void embed_rows_kernel(const uint4* __restrict__ embed,
                                                         const int32_t* __restrict__ ids,
                                                         float4* __restrict__ h, int num_tokens,
                                                         int pieces, int vocab) {
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= num_tokens) return;
  const int lane = threadIdx.x & 63;
  const int id = ids[m];
  const bool real = (uint32_t)id < (uint32_t)vocab;
  for (int p = lane; p < pieces; p += 64) {
    const uint4 v = real ? embed[(int64_t)id * pieces + p] : kNanPiece;
    float4* dst = h + ((int64_t)m * pieces + p) * 2;
    dst[0] = make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xFFFF0000u),
                         __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xFFFF0000u));
    dst[1] = make_float4(__uint_as_float(v.z << 16), __uint_as_float(v.z & 0xFFFF0000u),
                         __uint_as_float(v.w << 16), __uint_as_float(v.w & 0xFFFF0000u));
  }
}

// dst[m] = src[index[m]], bf16 rows of `pieces` 16-byte pieces, one wave per row; NaN where
// the index names none.  FROM_END: a negative one counts from the end (row_of_index).
template <bool FROM_END>
__global__ __launch_bounds__(256) void copy_rows_kernel(const uint4* __restrict__ src,
                                                        const int32_t* __restrict__ index,
                                                        uint4* __restrict__ dst, int num_rows,
                                                        int pieces, int src_rows) {
  const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= num_rows) return;
  const int i = index[m];
  const IndexedRow at = row_of_index(!FROM_END && i < 0 ? src_rows : i, src_rows);
  for (int p = threadIdx.x & 63; p < pieces; p += 64)
    dst[(int64_t)m * pieces + p] = at.real ? src[(int64_t)at.row * pieces + p] : kNanPiece;
}

// hidden 256, 512, 1024 or 2048; one row per wave for up to 4 rows, else four
#define NVJ_BY_ROW(LAUNCH)                                     \
  switch (hidden) {                                            \
    case 256: return few ? LAUNCH(1, 1) : LAUNCH(1, 4);        \
    case 512: return few ? LAUNCH(2, 1) : LAUNCH(2, 4);        \
    case 1024: return few ? LAUNCH(4, 1) : LAUNCH(4, 4);       \
    default: return few ? LAUNCH(8, 1) : LAUNCH(8, 4);         \
  }
template <Epilogue EPI>
hipError_t launch_norm_gemm(hipStream_t s, const NormGemmArgs& a, int hidden) {
  const bool few = a.num_tokens <= 4;
  const dim3 grid((unsigned)(a.outputs / 16)), block(256);
#define NVJ_LAUNCH(RV, ROWS) nvj::launch(norm_gemm_kernel<RV, ROWS, EPI>, grid, block, s, a)
  NVJ_BY_ROW(NVJ_LAUNCH)
#undef NVJ_LAUNCH
}
template <bool NORM>
hipError_t launch_norm_gemm_wide(hipStream_t s, const NormGemmArgs& a, int hidden) {
  const bool few = a.num_tokens <= 4;
  const dim3 grid((unsigned)((a.outputs + 63) / 64)), block(256);
#define NVJ_LAUNCH(RV, ROWS) nvj::launch(norm_gemm_wide_kernel<RV, ROWS, NORM>, grid, block, s, a)
  NVJ_BY_ROW(NVJ_LAUNCH)
#undef NVJ_LAUNCH
}
#undef NVJ_BY_ROW

constexpr size_t round256(size_t n) { return (n + 255) / 256 * 256; }

// Up to kMaxRows rows go through the first form where it is built for the sizes.
bool few_rows_takes(const nvj_decoder_model& m, int64_t tokens, int64_t sequences) {
  return tokens <= kMaxRows && sequences <= kMaxRows &&
         (m.hidden == 256 || m.hidden == 512 || m.hidden == 1024 || m.hidden == 2048) &&
         residual_gemm_takes((int64_t)m.num_heads * m.head_dim) &&
         residual_gemm_takes(m.intermediate);
}

struct StepBuffers {
  size_t h, y, t, qkv, q, o, k_rows, act, last, bytes;
};
StepBuffers step_buffers(const nvj_decoder_model& m, int64_t tokens, int64_t sequences) {
  StepBuffers b;
  size_t at = 0;
  auto take = [&](size_t bytes_per_token) {
    const size_t here = at;
    at += round256((size_t)tokens * bytes_per_token);
    return here;
  };
  const size_t row = (size_t)m.hidden * 2;
  const size_t q_row = (size_t)m.num_heads * m.head_dim * 2;
  const size_t kv_row = (size_t)m.num_kv_heads * m.head_dim * 2;
  b.h = take(2 * row);           // few rows: float32; else the bf16 residual
  b.y = take(row);               // normalised rows
  b.t = take(row);               // output of a projection
  b.qkv = take(q_row + 2 * kv_row);
  b.q = take(q_row);
  b.o = take(q_row);
  b.k_rows = take(kv_row);       // packed K (few rows)
  take(kv_row);                  // and V
  b.act = take((size_t)m.intermediate * 2);
  b.last = at;                   // the rows that get logits, when not all do
  at += round256((size_t)sequences * row);
  b.bytes = at;
  return b;
}

int check_model(const nvj_decoder_model* m) {
  if (!m) return NVJ_ERR_NULL_POINTER;
  if (m->num_layers <= 0 || m->hidden <= 0 || m->num_heads <= 0 || m->num_kv_heads <= 0 ||
      m->intermediate <= 0 || m->vocab <= 0 || m->max_position <= 0 || m->block_size <= 0 ||
      m->num_blocks <= 0 || m->num_heads % m->num_kv_heads != 0)
    return NVJ_ERR_BAD_SHAPE;
  const int64_t q_width = (int64_t)m->num_heads * m->head_dim;
  const int64_t qkv = q_width + 2 * (int64_t)m->num_kv_heads * m->head_dim;
  if (m->head_dim != 128 || m->hidden > 8192 || m->intermediate % 16 != 0 ||
      !nvj::linear_takes(1, qkv, m->hidden) || !nvj::linear_takes(1, m->hidden, q_width) ||
      !nvj::linear_takes(1, 2 * (int64_t)m->intermediate, m->hidden) ||
      !nvj::linear_takes(1, m->hidden, m->intermediate) ||
      !nvj::linear_takes(1, m->vocab, m->hidden))
    return NVJ_ERR_UNSUPPORTED;
  return NVJ_OK;
}

// Whether the products can be given that many rows (32-bit offsets into the operands).
bool takes_rows(const nvj_decoder_model& m, int64_t tokens, int64_t sequences) {
  const int64_t q_width = (int64_t)m.num_heads * m.head_dim;
  return nvj::linear_takes(tokens, m.hidden, m.hidden) &&
         nvj::linear_takes(tokens, m.hidden, q_width) &&
         nvj::linear_takes(tokens, m.hidden, m.intermediate) &&
         nvj::linear_takes(sequences, m.vocab, m.hidden);
}

int attention(void* stream, const nvj_decoder_model& m, const nvj_decoder_layer& l,
              const nvj_decoder_batch& b, bool first_layer, const void* q,
              const void* k, const void* v, int64_t kv_stride, void* out,
              const nvj::ReadAhead* ahead = nullptr) {
  if (b.is_prefill && !b.block_tables)
    return nvj_prefill_attention_rows_launch(stream, q, (int64_t)m.num_heads * m.head_dim, k, v, kv_stride, b.cu_seqlens_q,
                                             b.cu_seqlens_k, out, b.num_tokens, b.num_sequences,
                                             m.num_heads, m.num_kv_heads, m.head_dim, m.scale,
                                             NVJ_DTYPE_BF16);
  if (b.is_prefill)
    return nvj_paged_prefill_attention_launch(
        stream, q, l.k_cache, l.v_cache, b.block_tables, b.cu_seqlens_q, b.cu_seqlens_k,
        out, b.num_tokens, b.num_sequences, m.num_heads, m.num_kv_heads, m.head_dim, m.block_size,
        b.max_blocks, m.num_blocks, m.scale, NVJ_DTYPE_BF16);
  const uint32_t phases = NVJ_PHASE_SPLITK | NVJ_PHASE_COMBINE;
  if (b.chunk == 0)
    return nvj::paged_decode_launch_ahead(
        stream, q, l.k_cache, l.v_cache, b.block_tables, b.context_lens, out, b.partials,
        b.partial_bytes, b.counters, b.counter_bytes, b.num_sequences, m.num_heads, m.num_kv_heads,
        m.head_dim, m.block_size, b.max_blocks, m.num_blocks, m.scale, NVJ_DTYPE_BF16,
        phases | (b.clear_counters && first_layer ? NVJ_PHASE_CLEAR_COUNTERS : 0), ahead);
  return nvj_paged_decode_launch_phases(
      stream, q, l.k_cache, l.v_cache, b.block_tables, b.context_lens, out, b.partials,
      b.partial_bytes, b.num_sequences, m.num_heads, m.num_kv_heads, m.head_dim, m.block_size,
      b.max_blocks, m.num_blocks, m.scale, b.chunk, NVJ_DTYPE_BF16, phases);
}

// Whether the weights of a layer have left the Infinity Cache (256 MB) by the time the next step
// comes to it; else there is nothing to read ahead.  us without / with: 12 layers of 1024 (3072),
// 378 MB, 64 rows 763 / 698, a prompt of 400 tokens 887 / 827; 28 of 512 (1536), 245 MB, 1319 /
// 1289; 6 of 1024, 189 MB, 337 / 342 and 392 / 392; 3 of 1024 178 / 182.  Close to the line the LM
// head decides what stays: 7 of 1024, 220 MB, 20 rows 413 / 386 with a head of 311 MB, 303 / 313 with
// one of 16.
bool weights_leave_the_cache(const nvj_decoder_model& m) {
  const int64_t q = (int64_t)m.num_heads * m.head_dim, kv = (int64_t)m.num_kv_heads * m.head_dim;
  const int64_t rows = 2 * (q + kv) + 3 * (int64_t)m.intermediate;   // of `hidden` elements
  return rows * m.hidden * 2 * m.num_layers > (200 << 20);
}

int step_of_few_rows(void* stream, const nvj_decoder_model& m, const nvj_decoder_layer* layers,
                     const nvj_decoder_batch& b, char* ws, const StepBuffers& at) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* h = reinterpret_cast<float*>(ws + at.h);
  const int tokens = b.num_tokens;
  const int q_width = m.num_heads * m.head_dim, kv_width = m.num_kv_heads * m.head_dim;
  if (nvj::launch(embed_rows_kernel, dim3((unsigned)((tokens + 3) / 4)), dim3(256), s,
                  static_cast<const uint4*>(m.embed), b.input_ids, reinterpret_cast<float4*>(h),
                  tokens, m.hidden / 8, m.vocab) != hipSuccess)
    return NVJ_ERR_LAUNCH;
  NormGemmArgs a = {};
  a.h = reinterpret_cast<const float4*>(h);
  a.eps = m.eps;
  a.num_tokens = tokens;
  const bool packed = b.is_prefill && !b.block_tables;
  char* k_rows = packed ? ws + at.k_rows : nullptr;
  char* v_rows = packed ? k_rows + round256((size_t)tokens * kv_width * 2) : nullptr;
  // The attention reads weights ahead (read_ahead.h), in the order in which they are needed, as
  // many as HBM moves beside the K and V that the table holds in the 10 us that the launch
  // takes of its own.  A chunk is what one workgroup of the product takes, so that it goes to
  // the L2 of the XCD that asks for it (16 rows of the gate/up matrix instead of 8 and 8: 1058
  // us instead of 1036).  us a step without / with: 4 rows of 100 .. 900 positions 1080 / 1036,
  // 1 of 500 1023 / 982, 16 of 100 .. 400 (output and gate/up) 1250 / 1221; with all four
  // behind 8 rows of 1000 .. 2500 it would be 1349 / 1440.
  const int64_t ahead_bytes =
      b.is_prefill || !weights_leave_the_cache(m) ? 0
                   : (50 << 20) - (int64_t)tokens * b.max_blocks * m.block_size * kv_width * 4;
  for (int i = 0; i < m.num_layers; ++i) {
    const nvj_decoder_layer& l = layers[i];
    a.weight = static_cast<const char*>(l.qkv);
    a.norm_weight = l.ln1;
    a.outputs = q_width + 2 * kv_width;
    a.out = reinterpret_cast<uint16_t*>(ws + at.qkv);
    if (launch_norm_gemm<kPlain>(s, a, m.hidden) != hipSuccess) return NVJ_ERR_LAUNCH;
    int code = nvj_qk_norm_rope_rows_launch(
        stream, ws + at.qkv, a.outputs, b.positions, m.cos_sin, m.max_position, l.q_norm, l.k_norm,
        m.eps, b.slot_mapping, l.k_cache, l.v_cache, ws + at.q, q_width, k_rows, v_rows, kv_width,
        tokens, m.num_heads, m.num_kv_heads, m.head_dim, (int64_t)m.num_blocks * m.block_size);
    if (code != NVJ_OK) return code;
    nvj::ReadAhead ahead = {};
    int64_t left = ahead_bytes;
    const auto fits = [&](int64_t rows, int64_t columns) {
      return (left -= rows * columns * 2) >= 0;
    };
    const char* gate_up = static_cast<const char*>(l.gate_up);
    if (fits(m.hidden, q_width)) ahead.add_matrix(l.o, m.hidden, q_width, 8);
    if (fits(2 * (int64_t)m.intermediate, m.hidden)) {
      ahead.add_matrix(gate_up, m.intermediate, m.hidden, 8);
      ahead.add_matrix(gate_up + (int64_t)m.intermediate * m.hidden * 2, m.intermediate, m.hidden,
                       8);
    }
    if (fits(m.hidden, m.intermediate)) ahead.add_matrix(l.down, m.hidden, m.intermediate, 8);
    if (i + 1 < m.num_layers && fits(q_width + 2 * kv_width, m.hidden))
      ahead.add_matrix(layers[i + 1].qkv, q_width + 2 * kv_width, m.hidden, 16);
    code = attention(stream, m, l, b, i == 0, ws + at.q, k_rows, v_rows, kv_width,
                     ws + at.o, &ahead);
    if (code != NVJ_OK) return code;
    if (launch_residual_gemm<4, 1, 2>(s, ws + at.o, l.o, h, tokens, m.hidden, q_width) !=
        hipSuccess)
      return NVJ_ERR_LAUNCH;
    a.weight = static_cast<const char*>(l.gate_up);
    a.norm_weight = l.ln2;
    a.outputs = 2 * m.intermediate;
    a.out = reinterpret_cast<uint16_t*>(ws + at.act);
    if (launch_norm_gemm<kSiluMul>(s, a, m.hidden) != hipSuccess) return NVJ_ERR_LAUNCH;
    if (launch_residual_gemm<2, 4, 4>(s, ws + at.act, l.down, h, tokens, m.hidden,
                                      m.intermediate) != hipSuccess)
      return NVJ_ERR_LAUNCH;
  }
  if (!b.logits || b.num_sequences == 0) return NVJ_OK;
  a.weight = static_cast<const char*>(m.embed);
  a.norm_weight = m.final_norm;
  a.outputs = m.vocab;
  a.out = static_cast<uint16_t*>(b.logits);
  a.row_index = b.is_prefill ? b.last_token_indices : nullptr;
  a.num_rows = tokens;
  a.num_tokens = b.num_sequences;
  return launch_norm_gemm_wide<true>(s, a, m.hidden) == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
}

// The orders of the sums of the output and down projections (see the top).
hipError_t output_projection(hipStream_t s, const nvj::LinearArgs& a) {
  if (a.M <= 128 && a.K % 128 == 0) return nvj::linear_chained(s, a, 4, 1);
  return nvj::linear(s, a);
}
hipError_t down_projection(hipStream_t s, const nvj::LinearArgs& a) {
  if (a.M <= 128 && a.K % 256 == 0)
    return a.M > 64 || a.M == 32 ? nvj::linear_chained(s, a, 4, 2) : nvj::linear_chained(s, a, 2, 4);
  return nvj::linear(s, a);
}

// Weights are read ahead (read_ahead.h) by the norms, whose few workgroups leave HBM idle, and by
// the gate/up product, which is long and has the next layer's first products behind it.  The
// norm in front of the MLP takes the down projection, so that the gate/up product carries less;
// up to kReadRows rows it takes the gate/up matrix instead, which that product is still waiting
// for then, and the norm behind the MLP the next layer's first two.  us a step without / by the
// gate/up product alone / like this, up to kReadRows first: 17 rows of 50 .. 200 positions 1433 /
// 1354 / 1335, 24 of 100 .. 1000 1680 / 1570 / 1552, 64 of 500 1880 / 1774 / 1739; like this,
// and as with fewer rows: 80 of 200 .. 400 1893 / 1850 / 1830, 1847, 100 of 200 .. 400 1911 / 1895 /
// 1880, 1890, 128 of 1024 3475 / 3400 / 3378, 3375; a prompt of 200 tokens 1830 / 1648 / 1636, 1666
// (the middle one with the output projection's help), of 4268 6110 / 5837 / 5815, 5865.
constexpr int kReadRows = 64;

// A norm is over in 5 us, and waits for what it reads ahead.
constexpr int64_t kNormReads = 20 << 20;

// A gate/up product is given what makes up 128 MB with its own weights.  Beyond that it waits
// for HBM itself, whatever the order of the reads; us of 6 layers without / with: 2048 (6144)
// with 50 + 50 MB, 64 rows 542 / 520; 2560 (9728), 4 rows, with 100 + 31 MB 581 / 566 and with
// 100 + 81 581 / 618; 4096 (12288), 4 rows, with 201 + 50 MB 823 / 855.
constexpr int64_t kProductReads = 128 << 20;

bool read_ahead(nvj::ReadAhead& ahead, int64_t limit, const void* w, int64_t rows, int64_t columns,
                int chunk = 8) {
  if (ahead.total() + rows * columns * 2 > limit) return false;
  ahead.add_matrix(w, rows, columns, chunk);
  return true;
}

int step_of_many_rows(void* stream, const nvj_decoder_model& m, const nvj_decoder_layer* layers,
                      const nvj_decoder_batch& b, char* ws, const StepBuffers& at) {
  const bool ahead = weights_leave_the_cache(m);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int tokens = b.num_tokens, pieces = m.hidden / 8;
  const int q_width = m.num_heads * m.head_dim, kv_width = m.num_kv_heads * m.head_dim;
  const int qkv_width = q_width + 2 * kv_width;
  char *h = ws + at.h, *y = ws + at.y, *t = ws + at.t, *qkv = ws + at.qkv, *o = ws + at.o;
  char* act = ws + at.act;
  // the embedding rows are the residual
  if (nvj::launch(copy_rows_kernel<false>, dim3((unsigned)((tokens + 3) / 4)), dim3(256), s,
                  static_cast<const uint4*>(m.embed), b.input_ids, reinterpret_cast<uint4*>(h),
                  tokens, pieces, m.vocab) != hipSuccess)
    return NVJ_ERR_LAUNCH;
  int code = nvj_add_rms_norm_launch(stream, h, nullptr, layers[0].ln1, m.eps, y, nullptr, tokens,
                                     m.hidden);
  if (code != NVJ_OK) return code;
  nvj::LinearArgs a = {};
  a.M = tokens;
  a.positions = b.positions;
  a.cos_sin = m.cos_sin;
  a.slot_mapping = b.slot_mapping;
  a.eps = m.eps;
  a.max_position = m.max_position;
  a.num_heads = m.num_heads;
  a.num_kv_heads = m.num_kv_heads;
  a.num_slots = (int64_t)m.num_blocks * m.block_size;
  a.q_out = reinterpret_cast<uint16_t*>(ws + at.q);
  a.keep_kv = b.is_prefill && !b.block_tables;   // packed prefill reads K and V from the projection
  auto product = [&](const void* x, const void* w, void* out, int n, int k) {
    a.x = static_cast<const char*>(x);
    a.w = static_cast<const char*>(w);
    a.out = static_cast<uint16_t*>(out);
    a.N = n;
    a.K = k;
  };
  for (int i = 0; i < m.num_layers; ++i) {
    const nvj_decoder_layer& l = layers[i];
    product(y, l.qkv, qkv, qkv_width, m.hidden);
    a.q_norm = l.q_norm;
    a.k_norm = l.k_norm;
    a.k_cache = static_cast<uint16_t*>(l.k_cache);
    a.v_cache = static_cast<uint16_t*>(l.v_cache);
    if (nvj::linear_qk_rope(s, a) != hipSuccess) return NVJ_ERR_LAUNCH;
    code = attention(stream, m, l, b, i == 0, ws + at.q, qkv + 2 * (int64_t)q_width,
                     qkv + 2 * (int64_t)(q_width + kv_width), qkv_width, o);
    if (code != NVJ_OK) return code;
    product(o, l.o, t, m.hidden, q_width);
    if (output_projection(s, a) != hipSuccess) return NVJ_ERR_LAUNCH;
    const int64_t gate_up = 2 * (int64_t)m.intermediate;
    const int64_t norm_reads = ahead ? kNormReads : 0;
    const int64_t left = ahead ? kProductReads - gate_up * m.hidden * 2 : 0;
    const bool few = tokens <= kReadRows;
    nvj::ReadAhead by_norm2 = {}, by_norm1 = {}, by_product = {};
    if (few) read_ahead(by_norm2, norm_reads, l.gate_up, gate_up, m.hidden, 16);
    if (i + 1 < m.num_layers) {
      const nvj_decoder_layer& next = layers[i + 1];
      if (!few || !read_ahead(by_norm1, norm_reads, next.qkv, qkv_width, m.hidden))
        read_ahead(by_product, left, next.qkv, qkv_width, m.hidden);
      if (!few || !read_ahead(by_norm1, norm_reads, next.o, m.hidden, q_width))
        read_ahead(by_product, left, next.o, m.hidden, q_width);
    }
    if (few || !read_ahead(by_norm2, norm_reads, l.down, m.hidden, m.intermediate))
      read_ahead(by_product, left, l.down, m.hidden, m.intermediate);
    code = nvj::add_rms_norm(stream, t, h, l.ln2, m.eps, y, h, tokens, m.hidden, by_norm2);
    if (code != NVJ_OK) return code;
    product(y, l.gate_up, act, 2 * m.intermediate, m.hidden);
    a.ahead = by_product;
    if (nvj::linear_silu_mul(s, a) != hipSuccess) return NVJ_ERR_LAUNCH;
    a.ahead = {};
    product(act, l.down, t, m.hidden, m.intermediate);
    if (down_projection(s, a) != hipSuccess) return NVJ_ERR_LAUNCH;
    const float* next = i + 1 < m.num_layers ? layers[i + 1].ln1 : m.final_norm;
    code = nvj::add_rms_norm(stream, t, h, next, m.eps, y, h, tokens, m.hidden, by_norm1);
    if (code != NVJ_OK) return code;
  }
  if (!b.logits || b.num_sequences == 0) return NVJ_OK;
  const char* rows = y;
  if (b.is_prefill) {
    if (nvj::launch(copy_rows_kernel<true>, dim3((unsigned)((b.num_sequences + 3) / 4)), dim3(256), s,
                    reinterpret_cast<const uint4*>(y), b.last_token_indices,
                    reinterpret_cast<uint4*>(ws + at.last), b.num_sequences, pieces,
                    tokens) != hipSuccess)
      return NVJ_ERR_LAUNCH;
    rows = ws + at.last;
  }
  if (few_rows_takes(m, 1, b.num_sequences)) {
    NormGemmArgs n = {};
    n.h = reinterpret_cast<const float4*>(rows);
    n.weight = static_cast<const char*>(m.embed);
    n.out = static_cast<uint16_t*>(b.logits);
    n.num_tokens = b.num_sequences;
    n.outputs = m.vocab;
    return launch_norm_gemm_wide<false>(s, n, m.hidden) == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
  }
  a.M = b.num_sequences;
  product(rows, m.embed, b.logits, m.vocab, m.hidden);
  return nvj::linear(s, a, true) == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
}

}  // namespace

extern "C" size_t nvj_decoder_step_workspace_bytes(const nvj_decoder_model* model,
                                                   int32_t num_tokens,
                                                   int32_t num_sequences) {
  if (check_model(model) != NVJ_OK || num_tokens <= 0 || num_sequences < 0 ||
      !takes_rows(*model, num_tokens, num_sequences > 0 ? num_sequences : 1))
    return 0;
  return step_buffers(*model, num_tokens, num_sequences).bytes;
}

extern "C" int nvj_decoder_step_launch(void* stream, const nvj_decoder_model* model,
                                       const nvj_decoder_layer* layers,
                                       const nvj_decoder_batch* batch, void* workspace,
                                       size_t workspace_bytes) {
  const int bad = check_model(model);
  if (bad != NVJ_OK) return bad;
  if (!batch) return NVJ_ERR_NULL_POINTER;
  const nvj_decoder_model& m = *model;
  const nvj_decoder_batch& b = *batch;
  if (b.num_tokens < 0 || b.num_sequences < 0 || (!b.is_prefill && b.num_tokens != b.num_sequences))
    return NVJ_ERR_BAD_SHAPE;
  if (!takes_rows(m, b.num_tokens > 0 ? b.num_tokens : 1, b.num_sequences > 0 ? b.num_sequences : 1))
    return NVJ_ERR_UNSUPPORTED;
  if (b.num_tokens == 0) return NVJ_OK;
  if (!layers || !m.embed || !m.final_norm || !m.cos_sin || !b.input_ids || !b.positions ||
      !b.slot_mapping || !workspace)
    return NVJ_ERR_NULL_POINTER;
  if (b.is_prefill ? (!b.cu_seqlens_q || !b.cu_seqlens_k || (b.logits && !b.last_token_indices))
                   : !b.context_lens)
    return NVJ_ERR_NULL_POINTER;
  const StepBuffers at = step_buffers(m, b.num_tokens, b.num_sequences);
  if (workspace_bytes < at.bytes) return NVJ_ERR_WORKSPACE;
  uintptr_t bits = reinterpret_cast<uintptr_t>(workspace) | reinterpret_cast<uintptr_t>(m.embed) |
                   reinterpret_cast<uintptr_t>(m.final_norm) |
                   reinterpret_cast<uintptr_t>(m.cos_sin) | reinterpret_cast<uintptr_t>(b.logits);
  for (int i = 0; i < m.num_layers; ++i) {
    const nvj_decoder_layer& l = layers[i];
    if (!l.qkv || !l.o || !l.gate_up || !l.down || !l.ln1 || !l.ln2 || !l.k_cache || !l.v_cache)
      return NVJ_ERR_NULL_POINTER;
    if ((l.q_norm == nullptr) != (l.k_norm == nullptr)) return NVJ_ERR_NULL_POINTER;
    for (const void* p : {l.qkv, l.o, l.gate_up, l.down, (const void*)l.ln1, (const void*)l.ln2,
                          (const void*)l.q_norm, (const void*)l.k_norm, (const void*)l.k_cache,
                          (const void*)l.v_cache})
      bits |= reinterpret_cast<uintptr_t>(p);
  }
  if (bits & 15u) return NVJ_ERR_ALIGNMENT;

  char* ws = static_cast<char*>(workspace);
  return few_rows_takes(m, b.num_tokens, b.num_sequences)
             ? step_of_few_rows(stream, m, layers, b, ws, at)
             : step_of_many_rows(stream, m, layers, b, ws, at);
}
