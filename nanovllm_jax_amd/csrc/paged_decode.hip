// Split-K paged decode attention for gfx950 (CDNA4, wave64) and its combine pass.
//
// Stands in for paged_attention -> paged_decode_attention_vectorized
// (layers/pallas_attention.py:465-507, :146-238 of the reference) and for the
// gather + dot_product_attention fallback (layers/attention.py:399-434).
//
// Work split.  A workgroup handles a run of positions for NW KV heads at once,
// one wave per KV head, so the workgroup as a whole streams whole 2 KiB cache
// rows (all heads of a position are contiguous in the [page, position, head,
// dim] layout).  A wave owns the G query heads of its KV head, so every K/V
// byte is fetched once per group.  The runs are either equal cuts of all the
// steps of the batch, derived on the device from context_lens (balanced split,
// the default), or fixed chunks of each sequence.  A third mode finishes every
// sequence inside one workgroup (its waves are a few KV heads x equal parts of
// the sequence, merged through LDS): one launch, no workspace, for batches of
// similar lengths.
//
// Inner step = 32 positions of one page:
//   * K: 8 x 16-byte loads per lane, quarter-wave = one 256-byte (position,
//     head) row; staged through a wave-private, padded LDS tile and read back
//     in the MFMA A-operand layout (lane = position, 8 consecutive dims).
//   * S^T[pos, qhead] = K . Q^T with v_mfma_f32_16x16x32_bf16 (query heads
//     padded to 16 columns, held in registers for the whole chunk).
//   * fp32 online softmax on the accumulator layout (lane = query head,
//     4 positions per tile), running max shared across the 4 lane groups.
//   * V: 8 x 16-byte loads per lane straight from HBM, one per position the
//     lane's P^T operand holds, transposed inside the lane with v_perm_b32
//     into 8 A operands (lane = 8 dims x 8 positions), so no LDS for V.
//   * O^T[dim, qhead] += V^T . P^T with 16 MFMAs: P enters twice, as its values
//     rounded to the cache's 16-bit type and as the rest of that rounding.
// Loads for step i+1 are issued before the arithmetic of step i.
//
// In the first two modes the partial (unnormalised O, running max, running
// sum) of every segment goes to the workspace and the combine kernel merges the
// segments of a sequence; a sequence that is one segment is written directly.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <mutex>

#include "bf16.h"
#include "cache_rows.h"
#include "device.h"
#include "divisor.h"
#include "launch.h"
#include "nvj_paged_attn.h"
#include "read_ahead.h"
#include "wave_ops.h"

namespace {

typedef __attribute__((address_space(3))) char* lds_ptr;
using nvj::bf16x8;
using nvj::compute_units;
using nvj::f16x8;
using nvj::f32x4;
using nvj::quotient;
using nvj::reciprocal;
using nvj::wave_inclusive_scan;
using nvj::wave_max;
using nvj::wave_xor_add;
using nvj::wave_xor_max;

constexpr int kMaxHeadDim = 128;     // head_dim is a template parameter: 128 or 64
constexpr int kStep = 32;            // positions per inner step
// A (position, head) row of D bf16 is D/8 16-byte pieces; the LDS tile pads a
// row by one piece so that the 16 rows an MFMA operand read touches fall on
// different banks.
template <int D> struct HeadDim {
  static_assert(D == 128 || D == 64, "head_dim 128 or 64");
  static constexpr int kPieces = D / 8;             // 16 or 8
  static constexpr int kLdsRowPieces = kPieces + 1;
  static constexpr int kPosPerLoad = 64 / kPieces;  // positions one 64-lane load covers: 4 or 8
  static constexpr int kKLoads = kStep / kPosPerLoad;  // K loads per lane per step: 8 or 4
  static constexpr int kQkSteps = D / 32;           // MFMA reduction steps of Q.K: 4 or 2
};
constexpr float kNegBig = -1.0e30f;  // stands for -inf without inf-inf hazards
constexpr float kLog2e = 1.4426950408889634f;

// The cache element type: bf16 (F16 = false) or IEEE half (F16 = true).  The
// kernels move 16-bit patterns; only the matrix instruction, the rounding of
// the probabilities and of the output depend on the type.
template <bool F16> struct Elem;
template <> struct Elem<false> {
  static __device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    return nvj::pack2_bf16(lo, hi);
  }
  // the two values a packed pair stands for
  static __device__ __forceinline__ float low_of(uint32_t pair) {
    return __builtin_bit_cast(float, pair << 16);
  }
  static __device__ __forceinline__ float high_of(uint32_t pair) {
    return __builtin_bit_cast(float, pair & 0xFFFF0000u);
  }
};
template <> struct Elem<true> {
  static __device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    return nvj::pack2_f16(lo, hi);
  }
  static __device__ __forceinline__ float low_of(uint32_t pair) {
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    return (float)__builtin_bit_cast(f16x2, pair)[0];
  }
  static __device__ __forceinline__ float high_of(uint32_t pair) {
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    return (float)__builtin_bit_cast(f16x2, pair)[1];
  }
};

// A pair of fp32 values as two packed pairs of the cache's 16-bit type: the
// rounded values and what the rounding left over, rounded again.  Their sum
// carries 16 (bf16) or 22 (float16) mantissa bits of the fp32 values.
template <bool F16>
__device__ __forceinline__ void pack2_with_rest(float a, float b, uint32_t& main, uint32_t& rest) {
  main = Elem<F16>::pack2(a, b);
  rest = Elem<F16>::pack2(a - Elem<F16>::low_of(main), b - Elem<F16>::high_of(main));
}


// K/V are read exactly once per call: non-temporal loads stream them past the
// caches instead of allocating lines that will never be hit again.  `base` is
// wave-uniform (scalar registers), `off` the lane's 32-bit byte offset: a step
// never leaves its page, so offsets stay below block_size * row_bytes.
__device__ __forceinline__ uint4 load_piece(const char* base, uint32_t off) {
  typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
  const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(base + off));
  return make_uint4(t[0], t[1], t[2], t[3]);
}

// K of one step: 64 lanes cover kPosPerLoad whole (position, head) rows per
// load (lane -> position lane / kPieces, piece lane % kPieces), so every group
// of kPieces lanes reads one contiguous row (a quarter-wave at head_dim 128).
// In a full step the position splits into a uniform part (folded into the
// scalar base) and one per-lane offset shared by all loads; a TAIL step clamps
// every slot to the last live position so that nothing at or beyond the
// context length is ever read.
template <bool TAIL, int D>
__device__ __forceinline__ void issue_k_loads(uint4 (&kreg)[HeadDim<D>::kKLoads],
                                              const char* base, int lane, int last,
                                              uint32_t row_bytes) {
  using H = HeadDim<D>;
  const int pos_lane = lane / H::kPieces;
  const uint32_t piece_bytes = (uint32_t)(lane % H::kPieces) * 16u;
#pragma unroll
  for (int i = 0; i < H::kKLoads; ++i) {
    if constexpr (TAIL) {
      kreg[i] = load_piece(
          base, (uint32_t)min(H::kPosPerLoad * i + pos_lane, last) * row_bytes + piece_bytes);
    } else {
      kreg[i] = load_piece(base + (size_t)(H::kPosPerLoad * i) * row_bytes,
                           (uint32_t)pos_lane * row_bytes + piece_bytes);
    }
  }
}

// V of one step: load slot j of lane (kg, r) is the position that reduction
// slot j of k-group kg stands for in the P^T operand: 4*kg + j from the first
// S^T tile, 16 + 4*kg + (j - 4) from the second.
template <bool TAIL, int D>
__device__ __forceinline__ void issue_v_loads(uint4 (&vreg)[8], const char* base, int kg, int r,
                                              int last, uint32_t row_bytes) {
  // lane (kg, r) fetches piece r (dims 8r .. 8r+7) of its 8 positions; at
  // head_dim 64 there are only 8 pieces and lanes r >= 8 hold zeros
  const bool live = r < HeadDim<D>::kPieces;
  const uint32_t lane_bytes = (uint32_t)r * 16u;
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int uni = (j < 4) ? j : (16 + j - 4);   // uniform part of the position
    if (!live) {
      vreg[j] = zero;
    } else if constexpr (TAIL) {
      vreg[j] = load_piece(base, (uint32_t)min(4 * kg + uni, last) * row_bytes + lane_bytes);
    } else {
      vreg[j] = load_piece(base + (size_t)uni * row_bytes,
                           (uint32_t)(4 * kg) * row_bytes + lane_bytes);
    }
  }
}

// Read-only int32 metadata (block tables, context lengths) is never written
// while a launch runs.  Reading it through the constant address space tells
// the compiler so: a wave-uniform index then becomes a scalar load (s_load)
// even after the kernel has issued stores of its own, instead of a vector load
// whose result has to be moved back to the scalar unit.
typedef const __attribute__((address_space(4))) int32_t* const_i32_ptr;
__device__ __forceinline__ const_i32_ptr as_constant(const int32_t* p) {
  return (const_i32_ptr)(uintptr_t)p;
}

// Everything shared by the launch: pointers and problem shape.
struct DecodeArgs {
  const uint4* q;              // [B, Hq, 16] pieces
  const char* k_cache;         // [NB, bs, Hkv, 128] bf16
  const char* v_cache;
  const int32_t* block_tables; // [B, MB]
  const int32_t* context_lens; // [B]
  uint4* out;                  // [B, Hq, 16] pieces (bf16)
  float* part_o;               // [slots, Hq, 128]
  float* part_ml;              // [slots, Hq, 2]
  // num_kv_heads and group describe the heads as the kernels walk them: with
  // more than 16 query heads per cache head, a cache head is walked as kv_rep
  // "virtual" KV heads of group = G / kv_rep query heads each (kv_rep = 1
  // otherwise); cache_kv_heads is the number of heads a cache row really holds.
  int num_heads, num_kv_heads, group, kv_rep, cache_kv_heads, block_size, max_blocks, num_blocks;
  nvj::Divisor page;   // block_size
  float scale_log2e;
  __device__ __forceinline__ int cache_head(int kvh) const {
    return kv_rep == 1 ? kvh : kvh / kv_rep;
  }
};

// The new K/V rows of the step, stored by the same launch (NEW kernels: head_dim 128, up to
// 64 rows).  A store kernel in front of the attention is 2.8 us that a small call waits
// for.  Here nobody waits for the rows to arrive in the cache: a wave that walks 32 slots
// of the cache with a new row among them takes that row from `key` and `value` instead
// (compute_segment).  One compare per step against the slots of all the rows, one per lane,
// finds it, so that any slot mapping means what it means with the store in front, rows of
// one sequence in several batch entries included.
struct NewRows {
  const void* key;       // [B, Hkv, 128], the cache's type or float32
  const void* value;
  const int32_t* slots;  // [B]; < 0 or >= num_slots: not stored
  int num_slots;
  bool key_f32, value_f32;
  int main_wgs;          // workgroups behind these store a row each; 0: workgroup b stores row b
  int32_t* clear;        // balanced kernel: kNullStreamWords words for workgroup 0 to zero, or null
};
constexpr int kMaxNewRows = 64;
constexpr int kNullStreamWords = 512;   // see null_stream_counters: one per thread of a workgroup

template <bool F16>
__device__ __forceinline__ uint4 new_piece(const void* rows, bool f32, int64_t piece) {
  return f32 ? nvj::load_piece_as_cache_type<true, F16>(rows, piece)
             : nvj::load_piece_as_cache_type<false, F16>(rows, piece);
}

// This lane's new slot (of row `lane`), -1 where there is none.
__device__ __forceinline__ int new_slot_of_lane(const NewRows& n, int batch, int lane) {
  const int slot = lane < batch ? n.slots[lane] : -1;
  return slot < n.num_slots ? max(slot, -1) : -1;
}

// Row `row` into the cache, by one workgroup of `threads` threads.
template <bool F16>
__device__ __forceinline__ void store_new_row(const DecodeArgs& a, const NewRows& n, int row,
                                              int threads) {
  const int64_t slot = n.slots[row];
  if (slot < 0 || slot >= n.num_slots) return;
  const int pieces = a.cache_kv_heads * (kMaxHeadDim / 8);
  for (int p = threadIdx.x; p < 2 * pieces; p += threads) {
    const bool is_k = p < pieces;
    const int at = is_k ? p : p - pieces;
    char* cache = const_cast<char*>(is_k ? a.k_cache : a.v_cache);
    reinterpret_cast<uint4*>(cache)[slot * pieces + at] =
        is_k ? new_piece<F16>(n.key, n.key_f32, (int64_t)row * pieces + at)
             : new_piece<F16>(n.value, n.value_f32, (int64_t)row * pieces + at);
  }
}

// One wave's share of one segment: positions [t0, t1) of sequence b for KV head
// kvh; t0 is a multiple of 32, t0 < t1.  Leaves the unnormalised result in
// registers: acc[jd][e] is O[head kvh*group + r][dim 32*kg + 8*e + jd] for the
// lane (r = lane & 15, kg = lane >> 4), m_run the maximum raw score and l_run
// the sum of exp((score - m_run) * scale) of that head (the same in the four
// lanes that share r).  Lanes with r >= group hold padding.
// NEW: `new_slot` is new_slot_of_lane.  first_block: the first step's entry of the block table, if
// the caller has it (>= 0).
template <int D, bool F16, bool NEW = false>
__device__ __forceinline__ void compute_segment(const DecodeArgs& a, uint4* lds, int b, int kvh,
                                                int t0, int t1, int lane, f32x4 (&acc)[8],
                                                float& m_run, float& l_run,
                                                const NewRows* fresh = nullptr,
                                                int new_slot = -1, int first_block = -1) {
  using H = HeadDim<D>;
  const int r = lane & 15;   // MFMA row/column index inside a 16-wide tile
  const int kg = lane >> 4;  // MFMA k-group (which 8 of the 32 reduction slots)
  const uint4* __restrict__ q = a.q;
  const char* __restrict__ k_cache = a.k_cache;
  const char* __restrict__ v_cache = a.v_cache;
  const int num_heads = a.num_heads, group = a.group, block_size = a.block_size;
  const int num_blocks = a.num_blocks;
  const float scale_log2e = a.scale_log2e;
  const int nsteps = (t1 - t0 + kStep - 1) / kStep;

  // Q^T as MFMA B operand for the D/32 reduction steps over head_dim:
  // lane (column r = query head of the group, k-group kg) holds dims
  // 32*s + 8*kg .. +8.  Columns >= group are zero.
  uint4 qreg[H::kQkSteps];
  {
    // lanes of padding columns read the group's last head (always in range)
    // and then drop it, so the loads stay unconditional 16-byte loads
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    const uint4* qrow =
        q + ((int64_t)b * num_heads + (int64_t)kvh * group + min(r, group - 1)) * H::kPieces;
#pragma unroll
    for (int s = 0; s < H::kQkSteps; ++s) {
      const uint4 v = qrow[4 * s + kg];
      qreg[s] = r < group ? v : zero;
    }
  }

  const uint32_t row_bytes = (uint32_t)a.cache_kv_heads * (D * 2);  // one position, all heads
  const int64_t head_bytes = (int64_t)a.cache_head(kvh) * (D * 2);
  const const_i32_ptr table = as_constant(a.block_tables + (int64_t)b * a.max_blocks);

  // wave-uniform place of the first position of a step in the cache: its slot if NEW, else
  // its byte offset at once
  auto step_place = [&](int step, int known) -> int64_t {
    const int ts = t0 + step * kStep;
    const int page = a.page.divide(ts);
    const int phys = min(max(known >= 0 ? known : table[page], 0), num_blocks - 1);
    const int64_t slot = (int64_t)phys * block_size + (ts - page * block_size);
    return NEW ? slot : slot * row_bytes + head_bytes;
  };
  auto offset_of = [&](int64_t place) { return NEW ? place * row_bytes + head_bytes : place; };
  // NEW: this KV head's piece of a new row
  auto fresh_piece = [&](int row, int piece) {
    return ((int64_t)row * a.cache_kv_heads + a.cache_head(kvh)) * H::kPieces + piece;
  };

  uint4 kreg[H::kKLoads], vreg[8];
  int64_t place;   // of the step at hand
  {
    place = step_place(0, first_block);
    const int64_t off = offset_of(place);
    const int last = min(kStep, t1 - t0) - 1;
    issue_k_loads<true, D>(kreg, k_cache + off, lane, last, row_bytes);
    issue_v_loads<true, D>(vreg, v_cache + off, kg, r, last, row_bytes);
  }

#pragma unroll
  for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
  m_run = kNegBig;  // running max of raw scores (q.k, unscaled) of column r
  l_run = 0.f;      // this lane's share of the running sum

  // the page lookup of a step is started two steps ahead, so that its latency
  // is not in front of the loads that need the address
  int64_t place_ahead = nsteps > 1 ? step_place(1, -1) : 0;
  for (int step = 0; step < nsteps; ++step) {
    const int nvalid = min(kStep, t1 - (t0 + step * kStep));
    const bool more = step + 1 < nsteps;
    const int64_t next_place = place_ahead, next_off = offset_of(next_place);
    int next_last = kStep - 1;
    if (more) next_last = min(kStep, t1 - (t0 + (step + 1) * kStep)) - 1;
    if (step + 2 < nsteps) place_ahead = step_place(step + 2, -1);

    // the new rows among this step's positions; the pieces of the first are asked for here
    // already, while the step's own loads are still on their way
    unsigned long long hits = 0;
    uint4 fresh_k, fresh_v;
    if constexpr (NEW) {
      hits = __ballot((uint32_t)(new_slot - (int)place) < (uint32_t)nvalid);
      if (hits != 0) {
        const int64_t piece = fresh_piece(__builtin_ctzll(hits), r);
        fresh_k = new_piece<F16>(fresh->key, fresh->key_f32, piece);
        fresh_v = new_piece<F16>(fresh->value, fresh->value_f32, piece);
      }
    }

    // ---- K: registers -> LDS (row = position, padded), then next K loads ----
#pragma unroll
    for (int i = 0; i < H::kKLoads; ++i)
      lds[(H::kPosPerLoad * i + lane / H::kPieces) * H::kLdsRowPieces + lane % H::kPieces] =
          kreg[i];
    if constexpr (NEW) {
      for (unsigned long long h = hits; h != 0; h &= h - 1) {
        const int row = __builtin_ctzll(h);
        const int pos = __builtin_amdgcn_readlane(new_slot, row) - (int)place;
        const uint4 piece = h == hits ? fresh_k : new_piece<F16>(fresh->key, fresh->key_f32,
                                                                 fresh_piece(row, r));
        if (kg == 0) lds[pos * H::kLdsRowPieces + r] = piece;
      }
    }
    // Other lanes read these rows below.  The wave's own LDS accesses complete
    // in order; the fences keep the compiler from moving the reads ahead of the
    // writes (and, at the end of the step, the next writes ahead of the reads).
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (more) {
      if (next_last == kStep - 1)
        issue_k_loads<false, D>(kreg, k_cache + next_off, lane, next_last, row_bytes);
      else
        issue_k_loads<true, D>(kreg, k_cache + next_off, lane, next_last, row_bytes);
    }

    // ---- S^T = K . Q^T for two 16-position tiles ----
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < H::kQkSteps; ++s) {
      const uint4 a0 = lds[r * H::kLdsRowPieces + 4 * s + kg];
      const uint4 a1 = lds[(16 + r) * H::kLdsRowPieces + 4 * s + kg];
      s0 = Elem<F16>::mfma(a0, qreg[s], s0);
      s1 = Elem<F16>::mfma(a1, qreg[s], s1);
    }

    // ---- online softmax; lane holds positions 4*kg+e (s0) and 16+4*kg+e (s1) ----
    if (nvalid < kStep) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (4 * kg + e >= nvalid) s0[e] = kNegBig;
        if (16 + 4 * kg + e >= nvalid) s1[e] = kNegBig;
      }
    }
    float mx = fmaxf(fmaxf(fmaxf(s0[0], s0[1]), fmaxf(s0[2], s0[3])),
                     fmaxf(fmaxf(s1[0], s1[1]), fmaxf(s1[2], s1[3])));
    mx = wave_xor_max<16>(mx);
    mx = wave_xor_max<32>(mx);
    const float m_new = fmaxf(m_run, mx);
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2e);
    const float mneg = -m_new * scale_log2e;
    m_run = m_new;
    float p0[4], p1[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p0[e] = __builtin_amdgcn_exp2f(fmaf(s0[e], scale_log2e, mneg));
      p1[e] = __builtin_amdgcn_exp2f(fmaf(s1[e], scale_log2e, mneg));
    }
    if (nvalid < kStep) {
      // positions past the end weigh exactly 0 whatever the scale (at scale 0
      // the exponential of a masked score is 1, not 0)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (4 * kg + e >= nvalid) p0[e] = 0.f;
        if (16 + 4 * kg + e >= nvalid) p1[e] = 0.f;
      }
    }
    float psum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) psum += p0[e] + p1[e];
    l_run = fmaf(l_run, alpha, psum);
    // The probabilities go to the matrix core as two operands of the cache's
    // 16-bit type, the rounded values and the rest of the rounding, so that
    // P.V sees them to 16 bits or more, as good as the fp32 probabilities of the
    // reference's vectorised path (layers/pallas_attention.py:227-236); the
    // second product is free under the K/V stream.
    uint4 pbits, prest;
    pack2_with_rest<F16>(p0[0], p0[1], pbits.x, prest.x);
    pack2_with_rest<F16>(p0[2], p0[3], pbits.y, prest.y);
    pack2_with_rest<F16>(p1[0], p1[1], pbits.z, prest.z);
    pack2_with_rest<F16>(p1[2], p1[3], pbits.w, prest.w);

    if constexpr (NEW) {
      // Load slot j of k-group kg is position 4 * kg + (j & 3) + 16 * (j >> 2).  Positions
      // behind the last hold copies of the last: they weigh 0, but what the cache held
      // there before the step need not be finite.
      for (unsigned long long h = hits; h != 0; h &= h - 1) {
        const int row = __builtin_ctzll(h);
        const int pos = __builtin_amdgcn_readlane(new_slot, row) - (int)place;
        const uint4 piece = h == hits ? fresh_v : new_piece<F16>(fresh->value, fresh->value_f32,
                                                                 fresh_piece(row, r));
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (min(4 * kg + (j & 3) + 16 * (j >> 2), nvalid - 1) == pos) vreg[j] = piece;
      }
    }

    // ---- V: in-lane 8x8 transpose (positions x dims), then next V loads ----
    uint4 vt[8];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint32_t vw[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        vw[j] = w == 0 ? vreg[j].x : w == 1 ? vreg[j].y : w == 2 ? vreg[j].z : vreg[j].w;
      // even dim of the pair: low halves; odd dim: high halves
      vt[2 * w].x = __builtin_amdgcn_perm(vw[1], vw[0], 0x05040100u);
      vt[2 * w].y = __builtin_amdgcn_perm(vw[3], vw[2], 0x05040100u);
      vt[2 * w].z = __builtin_amdgcn_perm(vw[5], vw[4], 0x05040100u);
      vt[2 * w].w = __builtin_amdgcn_perm(vw[7], vw[6], 0x05040100u);
      vt[2 * w + 1].x = __builtin_amdgcn_perm(vw[1], vw[0], 0x07060302u);
      vt[2 * w + 1].y = __builtin_amdgcn_perm(vw[3], vw[2], 0x07060302u);
      vt[2 * w + 1].z = __builtin_amdgcn_perm(vw[5], vw[4], 0x07060302u);
      vt[2 * w + 1].w = __builtin_amdgcn_perm(vw[7], vw[6], 0x07060302u);
    }
    if (more) {
      if (next_last == kStep - 1)
        issue_v_loads<false, D>(vreg, v_cache + next_off, kg, r, next_last, row_bytes);
      else
        issue_v_loads<true, D>(vreg, v_cache + next_off, kg, r, next_last, row_bytes);
    }

    // ---- O^T = alpha * O^T + V^T . P^T ----
#pragma unroll
    for (int jd = 0; jd < 8; ++jd) {
      acc[jd] *= alpha;
      acc[jd] = Elem<F16>::mfma(vt[jd], pbits, acc[jd]);
      acc[jd] = Elem<F16>::mfma(vt[jd], prest, acc[jd]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    place = next_place;
  }

  // total of the running sum over the 4 k-groups that share column r
  l_run = wave_xor_add<16>(l_run);
  l_run = wave_xor_add<32>(l_run);
}

// ---------------------------------------------------------------------------
// Measurement variant: the same segment with both products on the vector ALU
// (v_dot2c_f32_bf16) instead of the matrix cores, so that the choice between
// the two can be timed rather than argued.  head_dim 128, bf16, exactly G = 2,
// 4 or 8 query heads per KV head.  Same loads, same page walk, same results
// layout as compute_segment; only the arithmetic between them differs:
//   * Q.K: lane (pl = lane / 16, pc = lane % 16) holds dims 8*pc .. +8 of
//     position 4*i + pl for its 8 K loads i and the same dims of all G query
//     rows, so 4 dot2 give a 1/16 partial of score (i, h).  The 8*G partials
//     per lane are summed over the 16 lanes of a row by a halving exchange
//     (DPP mirror, half mirror, two quad permutes): each step a lane keeps
//     one half of its values and adds the partner's copy of that half, which
//     leaves lane pc with the 8*G/16 complete scores of one head.
//   * softmax on those few scores per lane; the probabilities (bf16) and the
//     rescale factors travel to the P.V layout through the wave's LDS tile.
//   * P.V: lane (kg, r) holds 8 positions x 8 dims of V, transposed in-lane
//     into (position pair) x dim words as in the MFMA path, then 4 dot2 per
//     (head, dim) against the matching probability pairs; the four position
//     groups kg are summed once at the end.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a),
                                         __builtin_bit_cast(bf16x2, b), c, false);
}

// value of the lane that DPP control CTRL pairs this lane with (same row of 16)
template <int CTRL> __device__ __forceinline__ float dpp_partner(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}

// One halving step over v[0 .. 2*HALF): the lane whose `upper` is false keeps
// the even entries, its partner (upper true) the odd ones; each adds the
// partner's copy of what it keeps.  Result in v[0 .. HALF).
template <int CTRL, int HALF, int N>
__device__ __forceinline__ void halve_across(float (&v)[N], bool upper) {
#pragma unroll
  for (int j = 0; j < HALF; ++j) {
    const float keep = upper ? v[2 * j + 1] : v[2 * j];
    const float send = upper ? v[2 * j] : v[2 * j + 1];
    v[j] = keep + dpp_partner<CTRL>(send);
  }
}

constexpr int kDppQuadXor1 = 0xB1;      // quad_perm [1,0,3,2]
constexpr int kDppQuadXor2 = 0x4E;      // quad_perm [2,3,0,1]
constexpr int kDppRowMirror = 0x140;    // lane i <-> 15 - i
constexpr int kDppHalfMirror = 0x141;   // lane i <-> i ^ 7

template <int G>
__device__ __forceinline__ void compute_segment_valu(const DecodeArgs& a, uint4* lds, int b,
                                                     int kvh, int t0, int t1, int lane,
                                                     f32x4 (&acc_out)[8], float& m_out,
                                                     float& l_out) {
  static_assert(G == 2 || G == 4 || G == 8, "vector-ALU variant: 2, 4 or 8 query heads");
  constexpr int D = 128;
  using H = HeadDim<D>;
  // the 8 K loads of a step are scored in batches of LB loads = NB partial
  // scores per lane, which the exchange turns into NB / 16 complete ones
  constexpr int LB = G <= 4 ? 8 : 32 / G;   // K loads per batch
  constexpr int NB = LB * G;                // partial scores per lane and batch (16 or 32)
  constexpr int CB = NB / 16;               // complete scores per lane and batch
  constexpr int NS = 8 / LB * CB;           // complete scores per lane and step
  const int r = lane & 15, kg = lane >> 4;   // (piece, position group) in either layout
  const char* __restrict__ k_cache = a.k_cache;
  const char* __restrict__ v_cache = a.v_cache;
  const int block_size = a.block_size, num_blocks = a.num_blocks;
  const float scale_log2e = a.scale_log2e;
  const int nsteps = (t1 - t0 + kStep - 1) / kStep;

  // wave-private LDS: probabilities [G][32] bf16, rescale factors [G] f32,
  // and at the end of the segment the results [G][128] f32 + (max, sum) [G][2]
  uint16_t* lds_p = reinterpret_cast<uint16_t*>(lds);
  float* lds_alpha = reinterpret_cast<float*>(lds) + 256;   // byte 1024
  float* lds_o = reinterpret_cast<float*>(lds) + 512;       // byte 2048
  float* lds_ml = lds_o + G * D;
  static_assert((512 + 8 * 128 + 16) * 4 <= kStep * H::kLdsRowPieces * 16, "fits the K tile");

  // dims 8*r .. +8 of every query row of the group: in registers up to 4 rows,
  // in the wave's LDS tile beyond (read back per batch, the same address in
  // the four lanes that share r), which keeps the 8-row form free of spills
  constexpr bool kQInLds = G > 4;
  uint4* lds_q = lds + 400;   // byte 6400, behind the hand-over area; G * 16 pieces
  static_assert(400 + 8 * 16 <= kStep * H::kLdsRowPieces, "q pieces fit the K tile");
  uint4 qv[kQInLds ? 1 : G];
  if constexpr (kQInLds) {
#pragma unroll
    for (int h = kg; h < G; h += 4)
      lds_q[h * H::kPieces + r] =
          a.q[((int64_t)b * a.num_heads + (int64_t)kvh * G + h) * H::kPieces + r];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
#pragma unroll
    for (int h = 0; h < G; ++h)
      qv[h] = a.q[((int64_t)b * a.num_heads + (int64_t)kvh * G + h) * H::kPieces + r];
  }

  // the scores this lane owns after the exchange: entry c of a batch is partial
  // index n = low + 16 * c, low = the bits of r in reverse order; n = h + G * i
  // with i the load inside the batch
  const int low = ((r >> 3) & 1) | ((r >> 1) & 2) | ((r << 1) & 4) | ((r << 3) & 8);
  const int my_h = low % G;
  int my_pos[NS];   // position inside the step, entry = batch * CB + c
#pragma unroll
  for (int bt = 0; bt < 8 / LB; ++bt)
#pragma unroll
    for (int c = 0; c < CB; ++c) my_pos[bt * CB + c] = 4 * (bt * LB + (low + 16 * c) / G) + kg;
  // one lane per head publishes that head's values: the first of those that share it
  const bool publisher = kg == 0 && (r & (16 / G - 1)) == 0;

  const uint32_t row_bytes = (uint32_t)a.cache_kv_heads * (D * 2);
  const int64_t head_bytes = (int64_t)a.cache_head(kvh) * (D * 2);
  const const_i32_ptr table = as_constant(a.block_tables + (int64_t)b * a.max_blocks);
  auto step_base = [&](int step) -> int64_t {
    const int ts = t0 + step * kStep;
    const int page = a.page.divide(ts);
    const int phys = min(max(table[page], 0), num_blocks - 1);
    return ((int64_t)phys * block_size + (ts - page * block_size)) * row_bytes + head_bytes;
  };

  uint4 kreg[H::kKLoads], vreg[8];
  {
    const int64_t off = step_base(0);
    const int last = min(kStep, t1 - t0) - 1;
    issue_k_loads<true, D>(kreg, k_cache + off, lane, last, row_bytes);
    issue_v_loads<true, D>(vreg, v_cache + off, kg, r, last, row_bytes);
  }

  float acc[G][8];   // O[head h][dim 8*r + jd], this lane's position group only
#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int jd = 0; jd < 8; ++jd) acc[h][jd] = 0.f;
  float m_run = kNegBig, l_run = 0.f;   // of head my_h; l_run is this lane's share

  // the page lookup of a step is started two steps ahead, so that its latency
  // is not in front of the loads that need the address
  int64_t off_ahead = nsteps > 1 ? step_base(1) : 0;
  for (int step = 0; step < nsteps; ++step) {
    const int nvalid = min(kStep, t1 - (t0 + step * kStep));
    const bool more = step + 1 < nsteps;
    const int64_t next_off = off_ahead;
    int next_last = kStep - 1;
    if (more) next_last = min(kStep, t1 - (t0 + (step + 1) * kStep)) - 1;
    if (step + 2 < nsteps) off_ahead = step_base(step + 2);

    // ---- scores, batch by batch, then next K loads ----
    float v[NS];
#pragma unroll
    for (int bt = 0; bt < 8 / LB; ++bt) {
      float part[NB];
#pragma unroll
      for (int i = 0; i < LB; ++i)
#pragma unroll
        for (int h = 0; h < G; ++h) {
          const uint4 kk = kreg[bt * LB + i];
          const uint4 qq = kQInLds ? lds_q[h * H::kPieces + r] : qv[kQInLds ? 0 : h];
          float s = dot2_bf16(kk.x, qq.x, 0.f);
          s = dot2_bf16(kk.y, qq.y, s);
          s = dot2_bf16(kk.z, qq.z, s);
          part[h + G * i] = dot2_bf16(kk.w, qq.w, s);
        }
      halve_across<kDppRowMirror, NB / 2>(part, (r & 8) != 0);
      halve_across<kDppHalfMirror, NB / 4>(part, (r & 4) != 0);
      halve_across<kDppQuadXor2, NB / 8>(part, (r & 2) != 0);
      halve_across<kDppQuadXor1, NB / 16>(part, (r & 1) != 0);
#pragma unroll
      for (int c = 0; c < CB; ++c) v[bt * CB + c] = part[c];
    }
    if (more) {
      if (next_last == kStep - 1)
        issue_k_loads<false, D>(kreg, k_cache + next_off, lane, next_last, row_bytes);
      else
        issue_k_loads<true, D>(kreg, k_cache + next_off, lane, next_last, row_bytes);
    }

    // ---- online softmax of head my_h over the lanes that share it ----
    float mx = kNegBig;
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      if (my_pos[c] >= nvalid) v[c] = kNegBig;
      mx = fmaxf(mx, v[c]);
    }
    mx = fmaxf(mx, dpp_partner<kDppQuadXor1>(mx));
    if (G <= 4) mx = fmaxf(mx, dpp_partner<kDppQuadXor2>(mx));
    if (G <= 2) mx = fmaxf(mx, dpp_partner<kDppHalfMirror>(mx));
    mx = wave_xor_max<16>(mx);
    mx = wave_xor_max<32>(mx);
    const float m_new = fmaxf(m_run, mx);
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2e);
    const float mneg = -m_new * scale_log2e;
    m_run = m_new;
    float psum = 0.f;
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      float p = __builtin_amdgcn_exp2f(fmaf(v[c], scale_log2e, mneg));
      if (my_pos[c] >= nvalid) p = 0.f;   // exactly 0 whatever the scale
      psum += p;
      lds_p[my_h * kStep + my_pos[c]] = (uint16_t)(Elem<false>::pack2(p, 0.f) & 0xFFFFu);
    }
    l_run = fmaf(l_run, alpha, psum);
    const bool rescale = __builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0ull;
    if (rescale && publisher) lds_alpha[my_h] = alpha;
    // the wave's own LDS accesses complete in order; the fence keeps the
    // compiler from moving the reads below ahead of the writes above
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- V: in-lane 8x8 transpose (positions x dims), then next V loads ----
    uint4 vt[8];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint32_t vw[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        vw[j] = w == 0 ? vreg[j].x : w == 1 ? vreg[j].y : w == 2 ? vreg[j].z : vreg[j].w;
      vt[2 * w].x = __builtin_amdgcn_perm(vw[1], vw[0], 0x05040100u);
      vt[2 * w].y = __builtin_amdgcn_perm(vw[3], vw[2], 0x05040100u);
      vt[2 * w].z = __builtin_amdgcn_perm(vw[5], vw[4], 0x05040100u);
      vt[2 * w].w = __builtin_amdgcn_perm(vw[7], vw[6], 0x05040100u);
      vt[2 * w + 1].x = __builtin_amdgcn_perm(vw[1], vw[0], 0x07060302u);
      vt[2 * w + 1].y = __builtin_amdgcn_perm(vw[3], vw[2], 0x07060302u);
      vt[2 * w + 1].z = __builtin_amdgcn_perm(vw[5], vw[4], 0x07060302u);
      vt[2 * w + 1].w = __builtin_amdgcn_perm(vw[7], vw[6], 0x07060302u);
    }
    if (more) {
      if (next_last == kStep - 1)
        issue_v_loads<false, D>(vreg, v_cache + next_off, kg, r, next_last, row_bytes);
      else
        issue_v_loads<true, D>(vreg, v_cache + next_off, kg, r, next_last, row_bytes);
    }

    // ---- O = alpha * O + P . V for every head of the group ----
#pragma unroll
    for (int h = 0; h < G; ++h) {
      // probabilities of positions 4*kg .. +4 and 16 + 4*kg .. +4, as pairs
      const uint2 plo = *reinterpret_cast<const uint2*>(lds_p + h * kStep + 4 * kg);
      const uint2 phi = *reinterpret_cast<const uint2*>(lds_p + h * kStep + 16 + 4 * kg);
      if (rescale) {
        const float al = lds_alpha[h];
#pragma unroll
        for (int jd = 0; jd < 8; ++jd) acc[h][jd] *= al;
      }
#pragma unroll
      for (int jd = 0; jd < 8; ++jd) {
        float o = dot2_bf16(vt[jd].x, plo.x, acc[h][jd]);
        o = dot2_bf16(vt[jd].y, plo.y, o);
        o = dot2_bf16(vt[jd].z, phi.x, o);
        acc[h][jd] = dot2_bf16(vt[jd].w, phi.y, o);
      }
    }
    // the next step's writes must not overtake these reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // ---- totals: the sum of head my_h over the lanes that share it; O over the
  // four position groups ----
  l_run += dpp_partner<kDppQuadXor1>(l_run);
  if (G <= 4) l_run += dpp_partner<kDppQuadXor2>(l_run);
  if (G <= 2) l_run += dpp_partner<kDppHalfMirror>(l_run);
  l_run = wave_xor_add<16>(l_run);
  l_run = wave_xor_add<32>(l_run);
#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int jd = 0; jd < 8; ++jd) {
      float o = acc[h][jd];
      o = wave_xor_add<16>(o);
      o = wave_xor_add<32>(o);
      acc[h][jd] = o;
    }

  // ---- hand over in the layout the MFMA path leaves: lane (r = head, kg)
  // holds O[head r][dim 32*kg + 8*e + jd] in acc_out[jd][e] ----
  if (kg == 0) {
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float4* dst = reinterpret_cast<float4*>(lds_o + h * D + 8 * r);
      dst[0] = make_float4(acc[h][0], acc[h][1], acc[h][2], acc[h][3]);
      dst[1] = make_float4(acc[h][4], acc[h][5], acc[h][6], acc[h][7]);
    }
  }
  if (publisher) {
    lds_ml[2 * my_h] = m_run;
    lds_ml[2 * my_h + 1] = l_run;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int hr = min(r, G - 1);   // padding lanes read a real head and are ignored later
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float4* src = reinterpret_cast<const float4*>(lds_o + hr * D + 32 * kg + 8 * e);
    const float4 x = src[0], y = src[1];
    acc_out[0][e] = x.x; acc_out[1][e] = x.y; acc_out[2][e] = x.z; acc_out[3][e] = x.w;
    acc_out[4][e] = y.x; acc_out[5][e] = y.y; acc_out[6][e] = y.z; acc_out[7][e] = y.w;
  }
  m_out = lds_ml[2 * hr];
  l_out = lds_ml[2 * hr + 1];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------
// Measurement variant: the load stream of a segment and nothing else.  Same
// page walk, same K and V loads (addresses, order, one step fetched ahead) as
// compute_segment, but what arrives is only folded into one word per lane: no
// LDS, no matrix or softmax work.  Timing it against the real kernel shows how
// much of the kernel's time the arithmetic adds on top of the memory stream.
// The "result" is meaningless (and finite).  head_dim 128 only.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void compute_segment_loads_only(const DecodeArgs& a, int b, int kvh,
                                                           int t0, int t1, int lane,
                                                           f32x4 (&acc)[8], float& m_run,
                                                           float& l_run) {
  constexpr int D = 128;
  using H = HeadDim<D>;
  const int r = lane & 15, kg = lane >> 4;
  const int block_size = a.block_size, num_blocks = a.num_blocks;
  const int nsteps = (t1 - t0 + kStep - 1) / kStep;
  const uint32_t row_bytes = (uint32_t)a.cache_kv_heads * (D * 2);
  const int64_t head_bytes = (int64_t)a.cache_head(kvh) * (D * 2);
  const const_i32_ptr table = as_constant(a.block_tables + (int64_t)b * a.max_blocks);
  auto step_base = [&](int step) -> int64_t {
    const int ts = t0 + step * kStep;
    const int page = a.page.divide(ts);
    const int phys = min(max(table[page], 0), num_blocks - 1);
    return ((int64_t)phys * block_size + (ts - page * block_size)) * row_bytes + head_bytes;
  };
  uint4 kreg[H::kKLoads], vreg[8];
  {
    const int64_t off = step_base(0);
    const int last = min(kStep, t1 - t0) - 1;
    issue_k_loads<true, D>(kreg, a.k_cache + off, lane, last, row_bytes);
    issue_v_loads<true, D>(vreg, a.v_cache + off, kg, r, last, row_bytes);
  }
#pragma unroll
  for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
  m_run = 0.f;
  l_run = 0.f;
  uint32_t folded = 0;
  int64_t off_ahead = nsteps > 1 ? step_base(1) : 0;
  for (int step = 0; step < nsteps; ++step) {
    const bool more = step + 1 < nsteps;
    const int64_t next_off = off_ahead;
    int next_last = kStep - 1;
    if (more) next_last = min(kStep, t1 - (t0 + (step + 1) * kStep)) - 1;
    if (step + 2 < nsteps) off_ahead = step_base(step + 2);
#pragma unroll
    for (int i = 0; i < H::kKLoads; ++i) folded ^= kreg[i].x ^ kreg[i].y ^ kreg[i].z ^ kreg[i].w;
#pragma unroll
    for (int j = 0; j < 8; ++j) folded ^= vreg[j].x ^ vreg[j].y ^ vreg[j].z ^ vreg[j].w;
    if (more) {
      if (next_last == kStep - 1) {
        issue_k_loads<false, D>(kreg, a.k_cache + next_off, lane, next_last, row_bytes);
        issue_v_loads<false, D>(vreg, a.v_cache + next_off, kg, r, next_last, row_bytes);
      } else {
        issue_k_loads<true, D>(kreg, a.k_cache + next_off, lane, next_last, row_bytes);
        issue_v_loads<true, D>(vreg, a.v_cache + next_off, kg, r, next_last, row_bytes);
      }
    }
    l_run += 1.0f;
  }
  acc[0][0] = (float)(folded & 0xFFu);
}

// Folds the partial another wave of the workgroup left in its LDS tile into this
// wave's (acc, m_run, l_run): value v of a lane at float v * STRIDE of `theirs`
// (already offset by the lane), v = 4 * jd + e for acc[jd][e], 32 the running
// max, 33 the running sum.  All 34 values are fetched before the first is used:
// read one by one, as the compiler orders them when left alone, the 17 LDS
// round trips of every part follow each other (1.3 us for 3 parts).
template <int STRIDE>
__device__ __forceinline__ void add_partial_from_lds(const float* theirs, float scale_log2e,
                                                     f32x4 (&acc)[8], float& m_run, float& l_run) {
  float t[34];
#pragma unroll
  for (int v = 0; v < 34; ++v) t[v] = theirs[v * STRIDE];
  __builtin_amdgcn_sched_barrier(0);
  const float m_new = fmaxf(m_run, t[32]);
  const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2e);
  const float w = __builtin_amdgcn_exp2f((t[32] - m_new) * scale_log2e);
  m_run = m_new;
  l_run = fmaf(l_run, keep, w * t[33]);
#pragma unroll
  for (int jd = 0; jd < 8; ++jd)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[jd][e] = fmaf(acc[jd][e], keep, w * t[4 * jd + e]);
}

// Normalised bf16 result of a whole sequence straight to `out`.
template <int D, bool F16>
__device__ __forceinline__ void write_output(const DecodeArgs& a, int b, int kvh, int lane,
                                             const f32x4 (&acc)[8], float l_run) {
  using H = HeadDim<D>;
  const int r = lane & 15, kg = lane >> 4;
  // at head_dim 64 only k-groups 0 and 1 hold real dims
  if (r >= a.group || 32 * kg >= D) return;
  const int head = kvh * a.group + r;
  const float inv = 1.0f / (l_run + 1e-9f);
  uint4* orow = a.out + ((int64_t)b * a.num_heads + head) * H::kPieces + 4 * kg;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint4 o;
    o.x = Elem<F16>::pack2(acc[0][e] * inv, acc[1][e] * inv);
    o.y = Elem<F16>::pack2(acc[2][e] * inv, acc[3][e] * inv);
    o.z = Elem<F16>::pack2(acc[4][e] * inv, acc[5][e] * inv);
    o.w = Elem<F16>::pack2(acc[6][e] * inv, acc[7][e] * inv);
    orow[e] = o;
  }
}

// A row (or a piece of one) that the 8 waves of a workgroup have walked in up to 8 parts: every part
// lies in the K tile of its wave as add_partial_from_lds expects it (park_part), and wave w
// merges its eighth of the head dimensions (4 in every 32: dims 32 * kg + 8 * e + jd .. + 3 of
// query head r in lane (r, kg), e = w / 2, jd = 4 * (w % 2)), each value by the recurrence of
// add_partial_from_lds over the parts in order: the same bits as one wave merging all of
// it, without its 7 x 34 LDS reads in a row (6.7 -> 5.7 us for rows of 256 positions).
template <int D>
__device__ __forceinline__ void park_part(uint4* tile, int lane, const f32x4 (&acc)[8], float m_run,
                                          float l_run) {
  constexpr int STRIDE = D / 32 * 16;
  if (lane >= STRIDE) return;   // (lanes whose k-group holds no dims)
  float* mine = reinterpret_cast<float*>(tile) + lane;
#pragma unroll
  for (int jd = 0; jd < 8; ++jd)
#pragma unroll
    for (int e = 0; e < 4; ++e) mine[(4 * jd + e) * STRIDE] = acc[jd][e];
  mine[32 * STRIDE] = m_run;
  mine[33 * STRIDE] = l_run;
}
template <int D, int TILE>
__device__ __forceinline__ void merge_parts(const DecodeArgs& a, const uint4 (&k_tile)[8][TILE],
                                            int wave, int lane, float (&acc)[4], float& m_run,
                                            float& l_run, int parts) {
  constexpr int STRIDE = D / 32 * 16;
  const int e = wave >> 1, jd = 4 * (wave & 1);
  float v[8][4], ml[8][2];
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const float* t = reinterpret_cast<const float*>(k_tile[p]) + lane;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[p][i] = t[(4 * (jd + i) + e) * STRIDE];
    ml[p][0] = t[32 * STRIDE];
    ml[p][1] = t[33 * STRIDE];
  }
  m_run = ml[0][0];
  l_run = ml[0][1];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = v[0][i];
#pragma unroll
  for (int p = 1; p < 8; ++p) {
    if (p >= parts) break;
    const float m_new = fmaxf(m_run, ml[p][0]);
    const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2e);
    const float w = __builtin_amdgcn_exp2f((ml[p][0] - m_new) * a.scale_log2e);
    m_run = m_new;
    l_run = fmaf(l_run, keep, w * ml[p][1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(acc[i], keep, w * v[p][i]);
  }
}
// The wave's eighth of a finished row, by lanes with r < group and real dims.
template <int D, bool F16>
__device__ __forceinline__ void write_eighth(const DecodeArgs& a, int b, int kvh, int wave, int r,
                                             int kg, const float (&acc)[4], float l_run) {
  const float inv = 1.0f / (l_run + 1e-9f);
  uint2 o;
  o.x = Elem<F16>::pack2(acc[0] * inv, acc[1] * inv);
  o.y = Elem<F16>::pack2(acc[2] * inv, acc[3] * inv);
  const int head = kvh * a.group + r;
  reinterpret_cast<uint2*>(a.out + ((int64_t)b * a.num_heads + head) * HeadDim<D>::kPieces)
      [8 * kg + wave] = o;   // piece 4 * kg + e, half wave % 2
}

// Unnormalised partial (D f32 per head) + (max, sum) to the workspace.  A
// partial record is D + 2 floats of one query head; `rec_base` is the record of
// the first query head of this wave's KV head.
template <int D>
__device__ __forceinline__ void write_partial(const DecodeArgs& a, int64_t rec_base, int lane,
                                              const f32x4 (&acc)[8], float m_run, float l_run) {
  const int r = lane & 15, kg = lane >> 4;
  if (r >= a.group || 32 * kg >= D) return;
  const int64_t row = rec_base + r;
  float4* prow = reinterpret_cast<float4*>(a.part_o + row * D + 32 * kg);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    prow[2 * e] = make_float4(acc[0][e], acc[1][e], acc[2][e], acc[3][e]);
    prow[2 * e + 1] = make_float4(acc[4][e], acc[5][e], acc[6][e], acc[7][e]);
  }
  if (kg == 0) reinterpret_cast<float2*>(a.part_ml)[row] = make_float2(m_run, l_run);
}

// Fixed-chunk split: grid.x = batch * max_chunks, grid.y = num_kv_heads / NW,
// block = NW * 64.  Workgroup (b, c) owns positions [c*chunk, (c+1)*chunk) of
// sequence b; partial slot = b * max_chunks + c holds all query heads.
template <int NW, int D, bool F16>
__global__ __launch_bounds__(NW * 64) void paged_decode_splitk_kernel(DecodeArgs a, int chunk,
                                                                      int max_chunks) {
  __shared__ uint4 k_tile[NW][kStep * HeadDim<D>::kLdsRowPieces];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int b = blockIdx.x / max_chunks;
  const int c = blockIdx.x - b * max_chunks;
  // A length beyond what the block table can describe is clamped to it.
  const int ctx = min(a.context_lens[b], a.max_blocks * a.block_size);
  const int t0 = c * chunk;
  if (t0 >= ctx) return;  // also every chunk of an empty sequence
  const int t1 = min(ctx, t0 + chunk);
  const int kvh = blockIdx.y * NW + wave;
  f32x4 acc[8];
  float m_run, l_run;
  compute_segment<D, F16>(a, k_tile[wave], b, kvh, t0, t1, lane, acc, m_run, l_run);
  if (ctx <= chunk) write_output<D, F16>(a, b, kvh, lane, acc, l_run);
  else write_partial<D>(a, ((int64_t)b * max_chunks + c) * a.num_heads + kvh * a.group, lane, acc,
                        m_run, l_run);
}

// The steps [first, end) of part `part` of NPARTS: one each while there are no more steps than
// parts (the first parts have one then, which leaves fewer to merge), else equal shares.
struct PartOfSteps {
  int first, end;
};
template <int NPARTS>
__device__ __forceinline__ PartOfSteps part_of_steps(int part, int steps) {
  if (steps <= NPARTS) return {min(part, steps), min(part + 1, steps)};
  return {part * steps / NPARTS, (part + 1) * steps / NPARTS};
}

// Whole-sequence split: every sequence is finished inside one workgroup, so
// there is no workspace and no second pass.  grid.x = batch * (num_kv_heads /
// hpw), block = NW * 64.  Workgroup (b, head group hg) owns `hpw` KV heads of
// sequence b; its NW waves are hpw heads x NW / hpw parts: wave w takes head
// hg * hpw + w % hpw and the (w / hpw)-th of NW / hpw equal runs of the
// sequence's 32-position steps.  The parts of a head meet through LDS (each
// wave's K tile is free by then and exactly holds its 34 floats per lane) and
// the wave of part 0 merges them and writes the output.  Meant for batches of
// similar lengths: a workgroup's time follows its sequence's length.
// With a handful of steps the instructions in front of the first load count: divisions by hpw, by
// its number of parts and by the block size, five in a row, were 0.8 us and more of a launch (one
// sequence of 100 positions 6.9 -> 5.3 us, of 300 8.7 -> 8.0).
// VG < 0 selects the loads-only measurement variant; VG > 0 selects the
// vector-ALU measurement variant for exactly VG query heads
// per KV head (head_dim 128, bf16 only).
template <int NW, int D, bool F16, int VG = 0, bool NEW = false>
__global__ __launch_bounds__(NW * 64) void paged_decode_whole_kernel(DecodeArgs a, int hpw,
                                                                     nvj::Divisor groups,
                                                                     NewRows fresh, int batch) {
  using H = HeadDim<D>;
  __shared__ uint4 k_tile[NW][kStep * H::kLdsRowPieces];
  constexpr int kLanesWithDims = D / 32 * 16;   // lanes whose k-group holds real dims
  static_assert(sizeof(uint4) * kStep * H::kLdsRowPieces >= 34 * kLanesWithDims * sizeof(float),
                "a wave's K tile must hold its partial");
  int new_slot = -1;
  if constexpr (NEW) {
    if (fresh.main_wgs > 0 && (int)blockIdx.x >= fresh.main_wgs) {
      store_new_row<F16>(a, fresh, blockIdx.x - fresh.main_wgs, NW * 64);
      return;
    }
    if (fresh.main_wgs == 0 && (int)blockIdx.x < batch)
      store_new_row<F16>(a, fresh, blockIdx.x, NW * 64);
    new_slot = new_slot_of_lane(fresh, batch, threadIdx.x & 63);
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int log_hpw = __builtin_ctz(hpw), parts = NW >> log_hpw;
  const int b = groups.divide(blockIdx.x);
  const int hg = blockIdx.x - b * groups.d;
  const int part = wave >> log_hpw;
  const int kvh = hg * hpw + (wave - part * hpw);
  const int ctx = min(max(as_constant(a.context_lens)[b], 0), a.max_blocks * a.block_size);
  const int steps = (ctx + kStep - 1) / kStep;
  const bool all_merge = NW == 8 && hpw == 1;
  const PartOfSteps mine =
      all_merge ? part_of_steps<NW>(part, steps)
                : PartOfSteps{part * steps * hpw / NW, (part + 1) * steps * hpw / NW};
  const int s0 = mine.first, s1 = mine.end;

  f32x4 acc[8];
#pragma unroll
  for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegBig, l_run = 0.f;
  if (s1 > s0) {
    if constexpr (VG > 0)
      compute_segment_valu<VG>(a, k_tile[wave], b, kvh, s0 * kStep, min(ctx, s1 * kStep), lane,
                               acc, m_run, l_run);
    else if constexpr (VG < 0)
      compute_segment_loads_only(a, b, kvh, s0 * kStep, min(ctx, s1 * kStep), lane, acc, m_run,
                                 l_run);
    else
      compute_segment<D, F16, NEW>(a, k_tile[wave], b, kvh, s0 * kStep, min(ctx, s1 * kStep),
                                   lane, acc, m_run, l_run, &fresh, new_slot);
  }
  if (parts > 1) {
    // value v of lane l at float v * kLanesWithDims + l of the wave's tile
    const int parked = all_merge ? max(min(steps, NW), 1) : parts;   // (an empty row: zeros)
    if ((part > 0 || all_merge) && part < parked) park_part<D>(k_tile[wave], lane, acc, m_run, l_run);
    __syncthreads();
    if constexpr (NW == 8) {
      if (all_merge) {
        const int r = lane & 15, kg = lane >> 4;
        if (r >= a.group || 32 * kg >= D) return;
        float merged[4];
        merge_parts<D>(a, k_tile, wave, lane, merged, m_run, l_run, parked);
        write_eighth<D, F16>(a, b, kvh, wave, r, kg, merged, l_run);
        return;
      }
    }
    if (part > 0) return;
    if (lane < kLanesWithDims) {
      for (int p = 1; p < parts; ++p) {
        add_partial_from_lds<kLanesWithDims>(
            reinterpret_cast<const float*>(k_tile[wave + p * hpw]) + lane, a.scale_log2e, acc, m_run,
            l_run);
      }
    }
  }
  write_output<D, F16>(a, b, kvh, lane, acc, l_run);
}

// ---------------------------------------------------------------------------
// Balanced split: one launch for any mix of lengths.
//
// A workgroup is 8 waves = `hpw` KV heads x R = 8 / hpw parts (hpw is 4, 2 or
// 1 by the size of the launch, see balanced_heads_per_workgroup on the host side).
// The unit of work is a "row step": one 32-position step of one row, a row
// being (sequence b, head group hg of hpw KV heads).  All row steps, ordered
// by (b, hg, step), form one axis of length T = (num_kv_heads / hpw) * sum of
// steps.  The axis is cut into `nsub` sub-runs of equal length to within one
// step (`Cut` below): nsub = workgroups x R when there is at least one step for
// each, fewer otherwise.  Sub-run j belongs to workgroup j / R, part j % R, and
// is walked by the hpw waves of that part, one KV head each.  Every wave
// derives the cut from context_lens itself (a wave-wide prefix sum over the
// batch), so the host never needs the lengths.
//
// A sub-run that covers a whole row writes the output directly.  Otherwise a
// row is shared by several sub-runs; the piece of row `row` in sub-run j is a
// segment and owns partial slot j + row (unique, because j and row only grow
// along the axis, and consecutive within a row).  When the whole run of a
// workgroup lies inside one row, its parts are first merged through LDS (a
// wave's K tile is free by then) and part 0 writes one partial for all of
// them; the slots of the other parts stay unused, which the merging wave knows
// from the cut.
//
// Merge without a second launch: `counters` holds one int32 per (sequence, KV
// head), zero between launches.  A wave that has written partials for a row
// adds the number of sub-runs they stand for; the wave whose addition
// completes the row's count (the number of sub-runs that touch the row, known
// from the cut) merges the row's partials (in an order fixed by the cut alone,
// so that the result does not depend on who merges), writes the output and puts
// the counter back to zero.  Nothing ever waits for another workgroup.
// ---------------------------------------------------------------------------

// Sequences whose (length, steps before) pairs every wave keeps in registers
// after its one pass over the lengths; further ones are read again when needed.
constexpr int kKeptSequences = 256;

// Whole rows in the order of the batch, several rows per workgroup: only when
// no workgroup gets more than 1 + 8/256 of the mean (beyond that the order by
// length, which the caller's tolerance applies to, usually does better).
constexpr int kWholeRowTightTolerance = 8;
// The whole-row layout is offered for launches of up to this many workgroups
// (every wave checks the deal of all of them, 64 per pass).
constexpr int kMaxWholeRowWorkgroups = 256;

// The cut of the axis: sub-run j covers the axis positions whose unit
// (position >> shift) lies in [floor(j * units / nsub), floor((j+1) * units / nsub)).
// shift is 0 unless the axis is so long that units * nsub would not fit 31 bits
// (the host picks it from the largest axis the shapes allow).  Every sub-run
// holds at least one position.
struct Cut {
  int axis;    // row steps in all
  int units;   // ceil(axis >> shift)
  int nsub;    // sub-runs in use, 1 <= nsub <= units
  int shift;
  double per_unit, per_subrun;   // reciprocals of units and nsub
  __device__ __forceinline__ Cut(int axis, int shift, int most, int min_steps)
      : axis(axis), units((axis + (1 << shift) - 1) >> shift), shift(shift) {
    nsub = max(1, min(most, min_steps == 1 ? units : units / min_steps));
    per_unit = reciprocal(max(units, 1));
    per_subrun = reciprocal(nsub);
  }
  __device__ __forceinline__ int start_of(int j) const {
    const uint32_t u = quotient((uint32_t)j * (uint32_t)units, per_subrun);
    return min(axis, (int)(u << shift));
  }
  __device__ __forceinline__ int subrun_of(int x) const {
    return (int)quotient(((uint32_t)(x >> shift) + 1u) * (uint32_t)nsub - 1u, per_unit);
  }
};

// Record (see write_partial) of query head 0 of KV head `h_in_row` of a slot.
__device__ __forceinline__ int64_t balanced_record(const DecodeArgs& a, int64_t slot, int hpw,
                                                   int h_in_row) {
  return (slot * hpw + h_in_row) * a.group;
}

// Partials of the balanced split travel between workgroups of one launch, and
// workgroups on different XCDs do not share an L2.  They are therefore written
// and read with device-scope accesses (cache policy sc1: written through to,
// and read from, the point where the XCDs meet), ordered against the row's
// counter by waiting for the stores to be acknowledged.  No cache-wide
// write-back or invalidate is ever issued; those stall the K/V stream of every
// other wave on the XCD.  The accesses are 16-byte buffer instructions over a
// window that starts at a wave-uniform address.
//
// Layout of the partial of one (slot, KV head), chosen so that every store
// instruction of a wave writes one contiguous run: 16-byte piece i (0..7) of
// lane (r = query head, kg = dim group) sits at piece index
// i * (D/32 * G) + kg * G + r.  Piece 2e holds acc[0..3][e], piece 2e+1
// acc[4..7][e] of that lane.  The (max, sum) pairs follow the record order.
typedef __attribute__((ext_vector_type(4))) float vfloat4;
typedef __attribute__((ext_vector_type(2))) float vfloat2;
typedef __attribute__((ext_vector_type(4))) unsigned int vuint4;
typedef __attribute__((ext_vector_type(2))) unsigned int vuint2;
constexpr int kDeviceScope = 16;   // buffer cache policy: sc1

__device__ __forceinline__ __amdgpu_buffer_rsrc_t device_window(const void* base, int64_t bytes) {
  const int n = (int)(bytes < 0x7fffffff ? bytes : 0x7fffffff);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, n, 0x00020000);
}

template <int D>
__device__ __forceinline__ void write_partial_coherent(const DecodeArgs& a, int64_t rec_base,
                                                       int lane, const f32x4 (&acc)[8],
                                                       float m_run, float l_run) {
  constexpr int KG = D / 32;
  const int r = lane & 15, kg = lane >> 4;
  if (r >= a.group || kg >= KG) return;
  const __amdgpu_buffer_rsrc_t wo =
      device_window(a.part_o + rec_base * D, (int64_t)a.group * D * sizeof(float));
  const int lane_off = (kg * a.group + r) * 16, piece_stride = KG * a.group * 16;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const vfloat4 lo = {acc[0][e], acc[1][e], acc[2][e], acc[3][e]};
    const vfloat4 hi = {acc[4][e], acc[5][e], acc[6][e], acc[7][e]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(vuint4, lo), wo,
                                           lane_off + 2 * e * piece_stride, 0, kDeviceScope);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(vuint4, hi), wo,
                                           lane_off + (2 * e + 1) * piece_stride, 0, kDeviceScope);
  }
  if (kg == 0) {
    const __amdgpu_buffer_rsrc_t wm =
        device_window(a.part_ml + rec_base * 2, (int64_t)a.group * 2 * sizeof(float));
    const vfloat2 ml = {m_run, l_run};
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(vuint2, ml), wm, r * 8, 0,
                                          kDeviceScope);
  }
}

// All earlier stores of this wave have been acknowledged (and no later memory
// operation is moved ahead of this point by the compiler).
__device__ __forceinline__ void wait_for_stores() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// arrive: the wave has written its partials of row [r0, r1) (row steps on the
// axis) of (sequence b, KV head kvh), standing for `n` sub-runs, and publishes
// them.  merge_row: all partials of the row are there; merge them and write the
// output.  `lds` is the wave's own tile (free at that point).
//
// The merge keeps the chain of dependent memory round trips short: which slots
// hold a partial is computed from the cut, not read; the (max, sum) pairs of up
// to 64 slots are fetched by loads issued together and spread to the lanes
// through LDS; the accumulators of four partials are in flight at once.
// Returns true when this arrival completed the row: the caller then owes the
// row its merge (merge_row), at a time of its choosing.
__device__ __forceinline__ bool arrive(const DecodeArgs& a, int32_t* counters, int b, int kvh,
                                       int r0, int r1, const Cut& cut, int n, int lane) {
  // the partial stores of every lane have reached the device before the count does
  wait_for_stores();
  // word 0 of the counter region is the stale flag, the counters follow
  int32_t* counter = counters + 1 + (int64_t)b * a.num_kv_heads + kvh;
  int old = 0;
  if (lane == 0)
    old = __hip_atomic_fetch_add(counter, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  old = __builtin_amdgcn_readfirstlane(old);
  const int expected = cut.subrun_of(r1 - 1) - cut.subrun_of(r0) + 1;
  if (old < 0 || old + n > expected) {
    // The counter did not start at zero: the region was never cleared, an earlier
    // launch on it was cut short, or two launches overlap on it.  This row's
    // output is lost; say so where the host can see it and put the counter
    // back, so that a launch after this one starts from zero again.
    if (lane == 0) {
      __hip_atomic_store(counters, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return false;
  }
  if (old + n != expected) return false;
  // last to arrive: every other partial of the row was acknowledged before its
  // writer's count, which this wave has just seen
  asm volatile("" ::: "memory");
  if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// x of the lane n places further on in its row of 16 lanes (wrapping around)
template <int N>
__device__ __forceinline__ float row_rotate(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 | N, 0xf, 0xf, false));
}

template <int D, bool F16>
__device__ __forceinline__ void merge_row(const DecodeArgs& a, uint4* lds, int b, int kvh,
                                          int hpw, int r0, int r1, const Cut& cut, int lane) {
  using H = HeadDim<D>;
  // slots whose (max, sum) pairs fit the wave's tile at 16 heads x 8 bytes each
  constexpr int kSlots = (kStep * H::kLdsRowPieces * 16) / 128 >= 64 ? 64 : 32;
  static_assert(kStep * H::kLdsRowPieces * 16 >= kSlots * 128 + kSlots, "room for the slot list");
  constexpr int KG = D / 32;
  const int parts = 8 / hpw;
  const int first = cut.subrun_of(r0);
  const int expected = cut.subrun_of(r1 - 1) - first + 1;
  const int hg = kvh / hpw;
  const int rows_per_seq = a.num_kv_heads / hpw;
  const int64_t slot0 = (int64_t)first + (int64_t)b * rows_per_seq + hg;
  // A row of 16 lanes has room for 16 query heads; with fewer, the row is cut
  // into 16 / gp lane groups of gp >= group lanes (gp a power of two) and every
  // lane group merges partials of its own, so that 4 * 16 / gp partials are in
  // flight at once; the lane groups are added up at the end.  Lanes of padding
  // heads / padding dims read a real record and drop it later.
  const int gp = a.group > 8 ? 16 : a.group > 4 ? 8 : a.group > 2 ? 4 : a.group > 1 ? 2 : 1;
  const int lane_groups = 16 / gp;
  const int lg = (lane & 15) / gp;                        // this lane's group
  const int r = min((lane & 15) - lg * gp, a.group - 1);  // its query head
  const int kg = (32 * (lane >> 4) < D) ? (lane >> 4) : 0;
  const int64_t rec0 = balanced_record(a, slot0, hpw, kvh - hg * hpw);   // slot0, head 0
  const int64_t rec_stride = (int64_t)hpw * a.group;                     // per slot
  const __amdgpu_buffer_rsrc_t wm = device_window(
      a.part_ml + rec0 * 2, ((int64_t)(expected - 1) * rec_stride + a.group) * 2 * sizeof(float));
  const __amdgpu_buffer_rsrc_t wo = device_window(
      a.part_o + rec0 * D, ((int64_t)(expected - 1) * rec_stride + a.group) * D * sizeof(float));
  const int slot_bytes = (int)rec_stride * D * (int)sizeof(float);
  const int lane_off = (kg * a.group + r) * 16, piece_stride = KG * a.group * 16;
  vfloat2* lds_ml = reinterpret_cast<vfloat2*>(lds);   // [kSlots][16 heads]
  uint8_t* lds_list = reinterpret_cast<uint8_t*>(lds_ml + kSlots * 16);   // [kSlots]
  f32x4 acc[8];
#pragma unroll
  for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegBig, l_run = 0.f;
  for (int base = 0; base < expected; base += kSlots) {
    // Which of the slots base .. base + kSlots - 1 hold a partial follows from the
    // cut: lane L answers for slot base + L.  A workgroup whose whole run lies
    // inside this row merged its parts in LDS and wrote one partial, in the slot
    // of its part 0; any other workgroup wrote one per sub-run.
    const int count = min(kSlots, expected - base);
    const int j = first + base + lane;
    const int g = j / parts;
    const bool inside = cut.start_of(g * parts) >= r0 &&
                        cut.start_of(min(cut.nsub, g * parts + parts)) <= r1;
    const bool mine_real = lane < count && (!inside || j == g * parts);
    const unsigned long long real = __ballot(mine_real);
    const int nreal = __popcll(real);
    // the slots that hold a partial, in order, as a list
    if (mine_real) lds_list[__popcll(real & ((1ull << lane) - 1ull))] = (uint8_t)lane;
    // (max, sum) of all these slots for the 16 head columns, the loads in flight
    // together: lane (column c, kg) fetches slot base + 4 * i + kg (unused slots
    // hold stale values that are never looked at; slots past the end repeat the last).
    // (Fetching them together with the accumulators of the first partials, one
    // round trip fewer on paper, measured 2 us slower at 8 short sequences.)
    const int c = min(lane & 15, a.group - 1);
    vfloat2 got[kSlots / 4];
#pragma unroll
    for (int i = 0; i < kSlots / 4; ++i) {
      const int s = min(base + 4 * i + (lane >> 4), expected - 1);
      got[i] = __builtin_bit_cast(vfloat2, __builtin_amdgcn_raw_buffer_load_b64(
                                               wm, (int)((s * rec_stride + c) * 8), 0, kDeviceScope));
    }
#pragma unroll
    for (int i = 0; i < kSlots / 4; ++i) lds_ml[(4 * i + (lane >> 4)) * 16 + (lane & 15)] = got[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (nreal > 0) {
      // the largest maximum among the real slots, per head: over the slots this
      // lane fetched, over the four lane rows, then from the head's column
      float m_chunk = kNegBig;
#pragma unroll
      for (int i = 0; i < kSlots / 4; ++i) {
        const int sl = min(4 * i + (lane >> 4), count - 1);
        if ((real >> sl) & 1ull) m_chunk = fmaxf(m_chunk, got[i].x);
      }
      m_chunk = wave_xor_max<16>(m_chunk);
      m_chunk = wave_xor_max<32>(m_chunk);
      m_chunk = __shfl(m_chunk, (lane & 48) | r, 64);
      const float m_new = fmaxf(m_run, m_chunk);
      const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2e);
      m_run = m_new;
      l_run *= keep;
#pragma unroll
      for (int jd = 0; jd < 8; ++jd) acc[jd] *= keep;
      for (int done = 0; done < nreal; done += 4 * lane_groups) {
        // four partials per lane group at a time; absent ones repeat the first
        // of the list with weight 0
        float w[4];
        vfloat4 v[4][8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int n = done + k * lane_groups + lg;
          const bool have = n < nreal;
          const int idx = lds_list[have ? n : 0];
          const int off = (base + idx) * slot_bytes + lane_off;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            v[k][i] = __builtin_bit_cast(
                vfloat4,
                __builtin_amdgcn_raw_buffer_load_b128(wo, off + i * piece_stride, 0, kDeviceScope));
          const vfloat2 ml = lds_ml[idx * 16 + r];
          w[k] = have ? __builtin_amdgcn_exp2f((ml.x - m_new) * a.scale_log2e) : 0.f;
          l_run = fmaf(w[k], ml.y, l_run);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            acc[0][e] = fmaf(w[k], v[k][2 * e].x, acc[0][e]);
            acc[1][e] = fmaf(w[k], v[k][2 * e].y, acc[1][e]);
            acc[2][e] = fmaf(w[k], v[k][2 * e].z, acc[2][e]);
            acc[3][e] = fmaf(w[k], v[k][2 * e].w, acc[3][e]);
            acc[4][e] = fmaf(w[k], v[k][2 * e + 1].x, acc[4][e]);
            acc[5][e] = fmaf(w[k], v[k][2 * e + 1].y, acc[5][e]);
            acc[6][e] = fmaf(w[k], v[k][2 * e + 1].z, acc[6][e]);
            acc[7][e] = fmaf(w[k], v[k][2 * e + 1].w, acc[7][e]);
          }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();   // the next pass overwrites lds_ml and the list
  }
  // the sum over the lane groups, into every lane
#define NVJ_ADD_LANE_GROUPS(N)                                         \
  if (gp <= N) {                                                       \
    l_run += row_rotate<N>(l_run);                                     \
    _Pragma("unroll") for (int jd = 0; jd < 8; ++jd)                   \
      _Pragma("unroll") for (int e = 0; e < 4; ++e)                    \
        acc[jd][e] += row_rotate<N>(acc[jd][e]);                       \
  }
  NVJ_ADD_LANE_GROUPS(8)
  NVJ_ADD_LANE_GROUPS(4)
  NVJ_ADD_LANE_GROUPS(2)
  NVJ_ADD_LANE_GROUPS(1)
#undef NVJ_ADD_LANE_GROUPS
  write_output<D, F16>(a, b, kvh, lane, acc, l_run);
}

// One piece of a row: `parts` of its 8 waves have left a part in the K tiles (park_part).  A row of
// one piece is written at once; else the workgroup publishes the merged piece in slot `slot`
// and the one that comes last, of `pieces` whose slots lie `stride` apart from `slot0`,
// merges them and writes the row.  All 8 waves do both, each for its eighth of the dims, and
// every load of the merge is in flight at once up to 4 pieces per lane group, so that a
// shared row costs one acknowledged store, one count and one round trip.
// counter: of the row (see arrive).  stale: the flag in front of all counters.
template <int D, bool F16, int TILE>
__device__ __forceinline__ void finish_piece(const DecodeArgs& a, const uint4 (&k_tile)[8][TILE],
                                             int* lds_flag, int32_t* stale, int32_t* counter, int b,
                                             int kvh, int slot, int slot0, int stride, int pieces,
                                             int wave, int lane, int parts) {
  static_assert(D == 128, "four k-groups");
  float acc[4], m_run, l_run;
  merge_parts<D>(a, k_tile, wave, lane, acc, m_run, l_run, parts);
  const int group = a.group;
  const int dims = 32 * (lane >> 4) + 4 * wave;   // first of the lane's four
  if (pieces == 1) {
    if ((lane & 15) < group)
      write_eighth<D, F16>(a, b, kvh, wave, lane & 15, lane >> 4, acc, l_run);
    return;
  }
  if ((lane & 15) < group) {
    const int64_t rec = (int64_t)slot * group;
    const __amdgpu_buffer_rsrc_t wo =
        device_window(a.part_o + rec * D, (int64_t)group * D * sizeof(float));
    const vfloat4 mine = {acc[0], acc[1], acc[2], acc[3]};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(vuint4, mine), wo,
                                           ((lane & 15) * D + dims) * 4, 0, kDeviceScope);
    if (wave == 0 && lane < 16) {
      const __amdgpu_buffer_rsrc_t wm =
          device_window(a.part_ml + rec * 2, (int64_t)group * 2 * sizeof(float));
      const vfloat2 ml = {m_run, l_run};
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(vuint2, ml), wm, lane * 8, 0,
                                            kDeviceScope);
    }
  }
  wait_for_stores();
  __syncthreads();   // the whole piece has reached the device before it is counted
  if (threadIdx.x == 0) {
    const int old = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool wrong = old < 0 || old >= pieces;   // see arrive
    if (wrong) __hip_atomic_store(stale, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (wrong || old + 1 == pieces)
      __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *lds_flag = !wrong && old + 1 == pieces;
  }
  __syncthreads();
  if (*lds_flag == 0) return;
  // A row of 16 lanes holds 16 / gp lane groups of gp >= group lanes; lane group lg merges pieces
  // lg, lg + 16 / gp, ..., then the lane groups are merged; up to four pieces need one group
  // only, and no merge of groups.  Lanes of padding heads read a real record and are dropped.
  const int gp = group > 8 || pieces <= 4 ? 16 : group > 4 ? 8 : group > 2 ? 4 : group > 1 ? 2 : 1;
  const int lane_groups = 16 / gp;
  const int lg = (lane & 15) / gp;
  const int r = min((lane & 15) - lg * gp, group - 1);
  const int64_t rec0 = (int64_t)slot0 * group;
  const int64_t span = (int64_t)(pieces - 1) * stride * group + group;   // records
  const __amdgpu_buffer_rsrc_t wo = device_window(a.part_o + rec0 * D, span * D * sizeof(float));
  const __amdgpu_buffer_rsrc_t wm = device_window(a.part_ml + rec0 * 2, span * 2 * sizeof(float));
  m_run = kNegBig;
  l_run = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = 0.f;
  for (int p0 = lg; __any(p0 < pieces); p0 += 4 * lane_groups) {
    vfloat4 v[4];
    vfloat2 ml[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // (absent ones repeat the last with weight 0: a branch around a load costs more than
      // the load)
      const int rec = min(p0 + k * lane_groups, pieces - 1) * stride * group + r;
      v[k] = __builtin_bit_cast(vfloat4, __builtin_amdgcn_raw_buffer_load_b128(
                                             wo, (rec * D + dims) * 4, 0, kDeviceScope));
      ml[k] = __builtin_bit_cast(
          vfloat2, __builtin_amdgcn_raw_buffer_load_b64(wm, rec * 8, 0, kDeviceScope));
    }
    const float m_new =
        fmaxf(m_run, fmaxf(fmaxf(ml[0].x, ml[1].x), fmaxf(ml[2].x, ml[3].x)));
    const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2e);
    l_run *= keep;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] *= keep;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float w = p0 + k * lane_groups < pieces
                          ? __builtin_amdgcn_exp2f((ml[k].x - m_new) * a.scale_log2e)
                          : 0.f;
      l_run = fmaf(w, ml[k].y, l_run);
      acc[0] = fmaf(w, v[k].x, acc[0]);
      acc[1] = fmaf(w, v[k].y, acc[1]);
      acc[2] = fmaf(w, v[k].z, acc[2]);
      acc[3] = fmaf(w, v[k].w, acc[3]);
    }
    m_run = m_new;
  }
#define NVJ_MERGE_LANE_GROUPS(N)                                               \
  if (gp <= N) {                                                               \
    const float m_there = row_rotate<N>(m_run), m_new = fmaxf(m_run, m_there); \
    const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2e); \
    const float w = __builtin_amdgcn_exp2f((m_there - m_new) * a.scale_log2e); \
    m_run = m_new;                                                             \
    l_run = l_run * keep + w * row_rotate<N>(l_run);                           \
    _Pragma("unroll") for (int i = 0; i < 4; ++i)                              \
      acc[i] = acc[i] * keep + w * row_rotate<N>(acc[i]);                      \
  }
  NVJ_MERGE_LANE_GROUPS(8)
  NVJ_MERGE_LANE_GROUPS(4)
  NVJ_MERGE_LANE_GROUPS(2)
  NVJ_MERGE_LANE_GROUPS(1)
#undef NVJ_MERGE_LANE_GROUPS
  if ((lane & 15) < group) write_eighth<D, F16>(a, b, kvh, wave, r, lane >> 4, acc, l_run);
}

// The balanced split by the equal cut alone, for launches of up to 64 sequences that are offered
// no other layout: the same cut, the same segments and the same order of every sum as
// paged_decode_balanced_kernel, so the same bits, with less in front of the first load and less
// behind the last.  Where a workgroup's run lies inside one row, the waves of a head
// put its parts together, publish the partial and merge the row between them, each for its
// share of the dims; one wave alone took 3.2 us for the parts of a workgroup and 4.5 us for
// a row's partials.  16 / 8 heads, without a store: 1 sequence of 1000 positions 11.7 -> 9.9
// us, 4 of 100 .. 900 12.0 -> 10.2, 8 of 500 .. 8000 21.0 -> 19.1; a stream of K and V hardly
// notices (16 x 32768, 64 / 8 heads 319.4 -> 317.1).
template <bool F16, int HPW>
struct SharedRows {
  static constexpr int D = 128, NW = 8;
  static constexpr int kParts = NW / HPW;
  static constexpr int kPieces = 8 / kParts;   // 16-byte pieces of a lane's 8 that a wave owns
  static constexpr int kTile = kStep * HeadDim<D>::kLdsRowPieces;

  // The parked parts 0 .. nparts - 1 of head `h`, this wave's pieces: piece u of the lane is
  // acc[4 * (i & 1) ..][i >> 1] with i = kPieces * part + u (see add_partial_from_lds).
  static __device__ __forceinline__ void merge_parts_of_head(const DecodeArgs& a,
                                                             const uint4 (&k_tile)[NW][kTile],
                                                             int h, int part, int nparts, int lane,
                                                             f32x4 (&acc)[kPieces], float& m_run,
                                                             float& l_run) {
    constexpr int STRIDE = D / 32 * 16;
    auto tile = [&](int p) {
      return reinterpret_cast<const float*>(k_tile[p * HPW + h]) + lane;
    };
    auto fetch = [&](int p, float (&t)[4 * kPieces + 2]) {
      const float* at = tile(p);
#pragma unroll
      for (int u = 0; u < kPieces; ++u) {
        const int i = kPieces * part + u, jd = 4 * (i & 1), e = i >> 1;
#pragma unroll
        for (int v = 0; v < 4; ++v) t[4 * u + v] = at[(4 * (jd + v) + e) * STRIDE];
      }
      t[4 * kPieces] = at[32 * STRIDE];
      t[4 * kPieces + 1] = at[33 * STRIDE];
    };
    float t[kParts][4 * kPieces + 2];
#pragma unroll
    for (int p = 0; p < kParts; ++p) fetch(min(p, nparts - 1), t[p]);
    m_run = t[0][4 * kPieces];
    l_run = t[0][4 * kPieces + 1];
#pragma unroll
    for (int u = 0; u < kPieces; ++u)
      acc[u] = f32x4{t[0][4 * u], t[0][4 * u + 1], t[0][4 * u + 2], t[0][4 * u + 3]};
#pragma unroll
    for (int p = 1; p < kParts; ++p) {
      if (p < nparts) {
        const float m_new = fmaxf(m_run, t[p][4 * kPieces]);
        const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2e);
        const float w = __builtin_amdgcn_exp2f((t[p][4 * kPieces] - m_new) * a.scale_log2e);
        m_run = m_new;
        l_run = fmaf(l_run, keep, w * t[p][4 * kPieces + 1]);
#pragma unroll
        for (int u = 0; u < kPieces; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[u][v] = fmaf(acc[u][v], keep, w * t[p][4 * u + v]);
      }
    }
  }
  static __device__ __forceinline__ void write_pieces(const DecodeArgs& a, int b, int kvh, int part,
                                                      int lane, const f32x4 (&acc)[kPieces],
                                                      float l_run) {
    if ((lane & 15) >= a.group) return;
#pragma unroll
    for (int u = 0; u < kPieces; ++u) {
      const float mine[4] = {acc[u][0], acc[u][1], acc[u][2], acc[u][3]};
      write_eighth<D, F16>(a, b, kvh, kPieces * part + u, lane & 15, lane >> 4, mine, l_run);
    }
  }
  // merge_row for this wave's pieces.  The whole of it runs once in a launch, so its instructions
  // count as they stand, cold in the instruction cache.  HEADS, up to four query heads a KV head: the
  // (max, sum) pairs are fetched by heads, a slot per lane, 4 loads, LDS writes and masked maxima
  // where by slots, as merge_row has them, they are 16; and the one round of loads left in front of it
  // is the partials' own.  With the reciprocals of Cut, 16 / 8 heads: 4 sequences of 100 .. 900 positions
  // 10.5 -> 8.9 us, 1 of 700 10.1 -> 8.5, of 8000 18.2 -> 13.6, 4 of 3000 15.4 -> 13.9, 16 of 1000 16.6 ->
  // 15.2; 32 / 8 heads the same.  By heads every lane's pair lies in a line of its own, so with more of
  // them it costs more than it saves, us by slots / by heads: 64 / 8 heads, 4 of 3000 15.9 / 17.3, 1 of
  // 8252 among 32 of 20 40.2 / 47.7; 16 / 1, 1 of 700 9.7 / 11.0, of 8000 16.7 / 30.0; only one short
  // sequence with 7 or 8 is the other way round (8 / 1, 1 of 700 9.3 / 8.8, 28 / 4 9.5 / 9.1).
  template <bool HEADS>
  static __device__ __forceinline__ void merge_pieces(const DecodeArgs& a, uint4* lds, int b,
                                                      int kvh, int part, int r0, int r1,
                                                      const Cut& cut, int lane) {
    constexpr int kSlots = 64, KG = D / 32;
    const int first = cut.subrun_of(r0);
    const int expected = cut.subrun_of(r1 - 1) - first + 1;
    const int hg = kvh / HPW;
    const int64_t slot0 = (int64_t)first + (int64_t)b * (a.num_kv_heads / HPW) + hg;
    const int gp = a.group > 8 ? 16 : a.group > 4 ? 8 : a.group > 2 ? 4 : a.group > 1 ? 2 : 1;
    const int lane_groups = 16 / gp;
    const int lg = (lane & 15) / gp;
    const int r = min((lane & 15) - lg * gp, a.group - 1);
    const int kg = lane >> 4;
    const int64_t rec0 = balanced_record(a, slot0, HPW, kvh - hg * HPW);
    const int rec_stride = HPW * a.group;
    const int64_t span = (int64_t)(expected - 1) * rec_stride + a.group;
    const __amdgpu_buffer_rsrc_t wm = device_window(a.part_ml + rec0 * 2, span * 2 * sizeof(float));
    const __amdgpu_buffer_rsrc_t wo = device_window(a.part_o + rec0 * D, span * D * sizeof(float));
    const int slot_bytes = rec_stride * D * (int)sizeof(float);
    const int piece_stride = KG * a.group * 16;
    const int lane_off = (kg * a.group + r) * 16 + kPieces * part * piece_stride;
    vfloat2* lds_ml = reinterpret_cast<vfloat2*>(lds);   // HEADS: [4][kSlots], else [kSlots][16]
    uint8_t* lds_list = reinterpret_cast<uint8_t*>(lds_ml + kSlots * 16);
    f32x4 acc[kPieces];
#pragma unroll
    for (int u = 0; u < kPieces; ++u) acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = kNegBig, l_run = 0.f;
    const auto fence = [] {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const auto rescale = [&](float m_chunk) __attribute__((always_inline)) {
      const float m_new = fmaxf(m_run, m_chunk);
      const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2e);
      m_run = m_new;
      l_run *= keep;
#pragma unroll
      for (int u = 0; u < kPieces; ++u) acc[u] *= keep;
    };
    for (int base = 0; base < expected; base += kSlots) {
      const int count = min(kSlots, expected - base);
      constexpr int kPairs = HEADS ? 4 : kSlots / 4;
      vfloat2 got[kPairs];   // (past the end the last slot or head over again)
#pragma unroll
      for (int i = 0; i < kPairs; ++i) {
        const int slot = min(base + (HEADS ? lane : 4 * i + kg), expected - 1);
        const int head = min(HEADS ? i : lane & 15, a.group - 1);
        got[i] = __builtin_bit_cast(vfloat2, __builtin_amdgcn_raw_buffer_load_b64(
                                                 wm, (slot * rec_stride + head) * 8, 0, kDeviceScope));
      }
      // which slots hold a partial, while these are on their way (see merge_row)
      const int j = first + base + lane;
      const int g = j / kParts;
      const bool inside = cut.start_of(g * kParts) >= r0 &&
                          cut.start_of(min(cut.nsub, g * kParts + kParts)) <= r1;
      const bool mine_real = lane < count && (!inside || j == g * kParts);
      const unsigned long long real = __ballot(mine_real);
      const int nreal = __popcll(real);
      if (mine_real) lds_list[__popcll(real & ((1ull << lane) - 1ull))] = (uint8_t)lane;
      if constexpr (!HEADS) {
        float m_chunk = kNegBig;
#pragma unroll
        for (int i = 0; i < kPairs; ++i) {
          lds_ml[(4 * i + kg) * 16 + (lane & 15)] = got[i];
          const int sl = min(4 * i + kg, count - 1);
          if ((real >> sl) & 1ull) m_chunk = fmaxf(m_chunk, got[i].x);
        }
        fence();
        if (nreal > 0)
          rescale(__shfl(wave_xor_max<32>(wave_xor_max<16>(m_chunk)), (lane & 48) | r, 64));
      } else {
        fence();
      }
      for (int done = 0; done < nreal; done += 4 * lane_groups) {
        // the partials; by heads the first are asked for while the pairs are on their way
        int idx[4];
        vfloat4 v[4][kPieces];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int n = done + k * lane_groups + lg;
          idx[k] = lds_list[n < nreal ? n : 0];
          const int off = (base + idx[k]) * slot_bytes + lane_off;
#pragma unroll
          for (int u = 0; u < kPieces; ++u)
            v[k][u] = __builtin_bit_cast(
                vfloat4, __builtin_amdgcn_raw_buffer_load_b128(wo, off + u * piece_stride, 0,
                                                               kDeviceScope));
        }
        if constexpr (HEADS) {
          if (done == 0) {
            // their maxima over the slots: two halving steps leave lane L with head L % 4
            float m[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              lds_ml[i * kSlots + lane] = got[i];
              m[i] = mine_real ? fmaxf(got[i].x, kNegBig) : kNegBig;
            }
            const bool odd = lane & 1, upper = lane & 2;
            const float m0 = fmaxf(odd ? m[1] : m[0], dpp_partner<kDppQuadXor1>(odd ? m[0] : m[1]));
            const float m2 = fmaxf(odd ? m[3] : m[2], dpp_partner<kDppQuadXor1>(odd ? m[2] : m[3]));
            float most = fmaxf(upper ? m2 : m0, dpp_partner<kDppQuadXor2>(upper ? m0 : m2));
            most = fmaxf(most, row_rotate<4>(most));
            most = fmaxf(most, row_rotate<8>(most));
            most = wave_xor_max<32>(wave_xor_max<16>(most));
            most = __shfl(most, (lane & 48) | r, 64);
            fence();
            rescale(most);
          }
        }
        float w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const vfloat2 ml = lds_ml[HEADS ? r * kSlots + idx[k] : idx[k] * 16 + r];
          w[k] = done + k * lane_groups + lg < nreal
                     ? __builtin_amdgcn_exp2f((ml.x - m_run) * a.scale_log2e)
                     : 0.f;
          l_run = fmaf(w[k], ml.y, l_run);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
          for (int u = 0; u < kPieces; ++u) {
            acc[u][0] = fmaf(w[k], v[k][u].x, acc[u][0]);
            acc[u][1] = fmaf(w[k], v[k][u].y, acc[u][1]);
            acc[u][2] = fmaf(w[k], v[k][u].z, acc[u][2]);
            acc[u][3] = fmaf(w[k], v[k][u].w, acc[u][3]);
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
#define NVJ_ADD_LANE_GROUPS(N)                                         \
  if (gp <= N) {                                                       \
    l_run += row_rotate<N>(l_run);                                     \
    _Pragma("unroll") for (int u = 0; u < kPieces; ++u)                \
      _Pragma("unroll") for (int v = 0; v < 4; ++v)                    \
        acc[u][v] += row_rotate<N>(acc[u][v]);                         \
  }
    NVJ_ADD_LANE_GROUPS(8)
    NVJ_ADD_LANE_GROUPS(4)
    NVJ_ADD_LANE_GROUPS(2)
    NVJ_ADD_LANE_GROUPS(1)
#undef NVJ_ADD_LANE_GROUPS
    write_pieces(a, b, kvh, part, lane, acc, l_run);
  }
};

template <bool F16, int HPW>
__global__ __launch_bounds__(512) void paged_decode_shared_kernel(DecodeArgs a, int batch,
                                                                  int num_wgs, int min_steps,
                                                                  int shift, int32_t* counters,
                                                                  nvj::ReadAhead ahead) {
  using R = SharedRows<F16, HPW>;
  constexpr int D = R::D, NW = R::NW, kParts = R::kParts;
  using H = HeadDim<D>;
  __shared__ uint4 k_tile[NW][R::kTile];
  if ((int)blockIdx.x >= num_wgs) {
    nvj::read_chunk_by_lds<NW * 64>(ahead, (int)blockIdx.x - num_wgs,
                                    (uint32_t)(uintptr_t)(lds_ptr)&k_tile[0][0]);
    return;
  }
  __shared__ int last[HPW];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x;
  const int cap = a.max_blocks * a.block_size;
  const int rows_per_seq = a.num_kv_heads / HPW;
  const int part = wave / HPW, h_in_row = wave % HPW;

  // the lengths, one sequence per lane (the host sees to it that there are no more)
  const int kept_ctx = lane < batch ? min(max(a.context_lens[lane], 0), cap) : 0;
  const int kept_steps = (kept_ctx + kStep - 1) / kStep;
  const int incl = wave_inclusive_scan(kept_steps);
  const int kept_before = incl - kept_steps;
  const int total = __builtin_amdgcn_readlane(incl, 63);
  for (int b = g; b < batch; b += num_wgs) {   // zeros of empty sequences
    if (__builtin_amdgcn_readlane(kept_ctx, b) > 0) continue;
    uint4* orow = a.out + (int64_t)b * a.num_heads * H::kPieces;
    for (int i = threadIdx.x; i < a.num_heads * H::kPieces; i += NW * 64)
      orow[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  const Cut cut(rows_per_seq * total, shift, num_wgs * kParts, min_steps);
  if (cut.axis == 0 || g * kParts >= cut.nsub) return;

  // the sequence whose rows hold axis position x
  auto locate = [&](int x, int& b, int& before, int& ctx) __attribute__((always_inline)) {
    const int lo = rows_per_seq * kept_before;
    const unsigned long long hit = __ballot(lo <= x && x < lo + rows_per_seq * kept_steps);
    b = hit != 0ull ? __builtin_ctzll(hit) : batch;
    before = __builtin_amdgcn_readlane(kept_before, b & 63);
    ctx = hit != 0ull ? __builtin_amdgcn_readlane(kept_ctx, b & 63) : 0;
  };
  const int nparts = min(kParts, cut.nsub - g * kParts);   // parts that have work
  const int start = cut.start_of(g * kParts), end = cut.start_of(g * kParts + nparts);
  int b, before, ctx;
  locate(start, b, before, ctx);
  if (b >= batch || ctx <= 0) return;   // cannot happen when the prefix sums are right
  const int nb0 = (ctx + kStep - 1) / kStep;
  const int hg0 = (int)quotient(start - rows_per_seq * before, reciprocal(nb0));
  const int row0 = rows_per_seq * before + hg0 * nb0;
  const int xs = part < nparts ? cut.start_of(g * kParts + part) : end;
  const int xe = part < nparts ? cut.start_of(g * kParts + part + 1) : end;
  if (end <= row0 + nb0) {
    // The whole run of the workgroup lies inside one row.
    const int kvh = hg0 * HPW + h_in_row;
    float m_run = kNegBig, l_run = 0.f;
    f32x4 mine[R::kPieces];
    {
      f32x4 acc[8];
#pragma unroll
      for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (xs < xe)
        compute_segment<D, F16>(a, k_tile[wave], b, kvh, (xs - row0) * kStep,
                                min(ctx, (xe - row0) * kStep), lane, acc, m_run, l_run);
      park_part<D>(k_tile[wave], lane, acc, m_run, l_run);
    }
    __syncthreads();
    R::merge_parts_of_head(a, k_tile, h_in_row, part, nparts, lane, mine, m_run, l_run);
    if (start == row0 && end == row0 + nb0) {
      R::write_pieces(a, b, kvh, part, lane, mine, l_run);
      return;
    }
    // the partial, in the slot of part 0 (write_partial_coherent)
    const int64_t slot = (int64_t)g * kParts + (int64_t)b * rows_per_seq + hg0;
    const int64_t rec = balanced_record(a, slot, HPW, h_in_row);
    const int r = lane & 15, kg = lane >> 4;
    if (r < a.group) {
      const __amdgpu_buffer_rsrc_t wo =
          device_window(a.part_o + rec * D, (int64_t)a.group * D * sizeof(float));
      const int piece_stride = D / 32 * a.group * 16;
#pragma unroll
      for (int u = 0; u < R::kPieces; ++u) {
        const vfloat4 v = {mine[u][0], mine[u][1], mine[u][2], mine[u][3]};
        __builtin_amdgcn_raw_buffer_store_b128(
            __builtin_bit_cast(vuint4, v), wo,
            (kg * a.group + r) * 16 + (R::kPieces * part + u) * piece_stride, 0, kDeviceScope);
      }
      if (part == 0 && kg == 0) {
        const __amdgpu_buffer_rsrc_t wm =
            device_window(a.part_ml + rec * 2, (int64_t)a.group * 2 * sizeof(float));
        const vfloat2 ml = {m_run, l_run};
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(vuint2, ml), wm, r * 8, 0,
                                              kDeviceScope);
      }
    }
    wait_for_stores();
    __syncthreads();   // the whole partial has reached the device before it is counted
    if (part == 0) {
      const bool to_merge = arrive(a, counters, b, kvh, row0, row0 + nb0, cut, nparts, lane);
      if (lane == 0) last[h_in_row] = to_merge;
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(last[h_in_row])) {
      if (a.group > 4)
        R::template merge_pieces<false>(a, k_tile[wave], b, kvh, part, row0, row0 + nb0, cut, lane);
      else
        R::template merge_pieces<true>(a, k_tile[wave], b, kvh, part, row0, row0 + nb0, cut, lane);
    }
    return;
  }

  // Every wave walks its own sub-run across the rows.
  if (xs >= xe) return;
  int x = xs;
  if (part > 0) locate(xs, b, before, ctx);
  int owed = 0, owed_b[2] = {0, 0}, owed_kvh[2] = {0, 0}, owed_row[2] = {0, 0}, owed_nb[2] = {1, 1};
  while (x < xe && b < batch) {
    // ---- the next segment: row (sb, hg), steps [st, en) ----
    const int sb = b, nb = (ctx + kStep - 1) / kStep, seq0 = rows_per_seq * before;
    if (x < seq0) break;
    if (nb == 0 || x >= seq0 + rows_per_seq * nb) {   // empty, or this sequence is finished
      before += nb;
      ++b;
      ctx = b < batch ? __builtin_amdgcn_readlane(kept_ctx, b & 63) : 0;
      continue;
    }
    const int hg = (int)quotient(x - seq0, reciprocal(nb)), row = seq0 + hg * nb;
    const int st = x - row, en = min(nb, st + (xe - x));
    const int kvh = hg * HPW + h_in_row;
    f32x4 acc[8];
#pragma unroll
    for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = kNegBig, l_run = 0.f;
    compute_segment<D, F16>(a, k_tile[wave], sb, kvh, st * kStep, min(ctx, en * kStep), lane, acc,
                            m_run, l_run);
    x += en - st;
    if (st == 0 && en == nb) {
      write_output<D, F16>(a, sb, kvh, lane, acc, l_run);
    } else {
      const int64_t slot = (int64_t)g * kParts + part + (int64_t)sb * rows_per_seq + hg;
      write_partial_coherent<D>(a, balanced_record(a, slot, HPW, h_in_row), lane, acc, m_run, l_run);
      if (arrive(a, counters, sb, kvh, row, row + nb, cut, 1, lane)) {
        // at most the first and the last segment of a sub-run are not whole rows
        if (owed == 0) { owed_b[0] = sb; owed_kvh[0] = kvh; owed_row[0] = row; owed_nb[0] = nb; }
        else { owed_b[1] = sb; owed_kvh[1] = kvh; owed_row[1] = row; owed_nb[1] = nb; }
        ++owed;
      }
    }
  }
  for (int i = 0; i < owed; ++i) {
    const int ob = __builtin_amdgcn_readfirstlane(i == 0 ? owed_b[0] : owed_b[1]);
    const int okvh = __builtin_amdgcn_readfirstlane(i == 0 ? owed_kvh[0] : owed_kvh[1]);
    const int orow = __builtin_amdgcn_readfirstlane(i == 0 ? owed_row[0] : owed_row[1]);
    const int onb = __builtin_amdgcn_readfirstlane(i == 0 ? owed_nb[0] : owed_nb[1]);
    merge_row<D, F16>(a, k_tile[wave], ob, okvh, HPW, orow, orow + onb, cut, lane);
  }
}

// x / d for 0 <= x, 0 < d, both below 2^20, as a handful of instructions: (x + 0.5) / d is at least
// 0.5 / d away from a whole number, and its error less than x / d * 2^-21.5.
__device__ __forceinline__ int divide_small(int x, int d) {
  return (int)(((float)x + 0.5f) * __builtin_amdgcn_rcpf((float)d));
}
__device__ __forceinline__ int divide_small_up(int x, int d) { return divide_small(x + d - 1, d); }

// The shortest piece, in steps.  A step less is 0.2 us less of one wave's chain, and pieces of fewer
// than 8 steps leave waves idle but have fewer parts to put together and let more CUs draw a row;
// yet each piece is a partial more for the one that merges them.  So the longest row gets up to
// `per_row` pieces: 12, or what is merged in one round of loads, 8 with more than 4 query heads a KV
// head and 4 with more than 8 (the mean row: a row of 4021 positions among 60 of 1 was 63 pieces of 2
// steps, 18.9 us, in 16 of 8 11.2; one of 1892 among 9 of 20, 64 / 8 heads, 12.3 / 9.7); but no piece
// is longer than 8 steps, one a wave, while there are workgroups.  us,
// one sequence, 8 KV heads, at most 8 / 12 / 16 / 32 pieces a row: 768 positions 7.82 / 7.72 / 7.73 /
// 7.70 (in pieces of 8 steps 8.75, of one 8.81), 1500 8.97 / 8.42 / 8.56 / 9.22, 2048 9.14 / 8.89 /
// 8.91 / 10.21; 64 query heads at most 8 / 12, 1087 positions 8.81 / 9.76, 2 sequences of 1325 9.55 /
// 10.99.  Where a wave has more than a step, the longest of a workgroup has as many as in a piece
// of the next multiple of 8: that is taken if it leaves more than enough pieces (11101 positions in
// 22 of 16 steps 13.55, in 32 of 11 14.03; 3 of 3400, 64 query heads, 7 of 16 14.06, 10 of 11 14.45).
constexpr int kShortestPiece = 2;
constexpr int kHeldEntries = 4;   // registers of a wave for the block table

// Pieces: every row (sequence, KV head) on workgroups of its own, as many as there are, for
// launches of few and short rows, where what counts is the chain of round trips and the
// instructions between them (a wave issues one in 4.5 to 9 cycles here).  A row is cut into
// pieces of equal length to a step, about the shortest that leave no more pieces than `most`
// per KV head; the waves of a workgroup walk a piece in equal shares and put it together in LDS.
// Pieces in multiples of 8 steps, found by bisection, with divisions in front of the first load
// and the block table behind the lengths were 9.1 us for one sequence of 768 positions and 8 KV
// heads, 14.3 for 8 of 100 .. 1500, 10.0 for 8 of 100 .. 900 and 22.7 for 16 of 100 .. 2000; now 8.2,
// 12.9, 8.7 and 21.1.  Of 9000 drawn decode launches (those of the other kernels among them) 0.3 % are
// more than 3 % slower, one of them 18 % (128 / 8 heads, a row of 8145 positions beside one of 1, 20.3 ->
// 24.9).
// grid.x = main_wgs >= most * KV heads workgroups (and those that store new rows), block = 512.
template <bool F16, bool NEW>
__global__ __launch_bounds__(512) void paged_decode_pieces_kernel(DecodeArgs a, int batch,
                                                                  int most, int32_t* counters,
                                                                  NewRows fresh) {
  constexpr int D = 128, NW = 8;
  using H = HeadDim<D>;
  __shared__ uint4 k_tile[NW][kStep * H::kLdsRowPieces];
  __shared__ int last;
  const int g = blockIdx.x;
  int new_slot = -1;
  if constexpr (NEW) {
    if (fresh.main_wgs > 0 && g >= fresh.main_wgs) {
      store_new_row<F16>(a, fresh, g - fresh.main_wgs, NW * 64);
      return;
    }
    if (fresh.main_wgs == 0 && g < batch) store_new_row<F16>(a, fresh, g, NW * 64);
    new_slot = new_slot_of_lane(fresh, batch, threadIdx.x & 63);
    static_assert(NW * 64 == kNullStreamWords, "a word per thread");
    if (g == 0 && fresh.clear != nullptr) fresh.clear[threadIdx.x] = 0;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int cap = a.max_blocks * a.block_size;
  // the lengths, one sequence per lane (the host sees to it that there are no more), and with
  // them a small block table, so that the wave's first load need not wait for another one
  const int len_here = a.context_lens[min(lane, batch - 1)];
  const int64_t entries = (int64_t)batch * a.max_blocks;
  int held[kHeldEntries] = {};
  if (entries <= 64 * kHeldEntries) {
#pragma unroll
    for (int i = 0; i < kHeldEntries; ++i)
      if (i == 0 || entries > 64 * i)
        held[i] = a.block_tables[min(64 * i + lane, (int)entries - 1)];
  }
  // workgroup g: KV head g % heads of piece g / heads of them all
  const int at = __builtin_amdgcn_readfirstlane(divide_small(g, a.num_kv_heads));
  const int kvh = g - at * a.num_kv_heads;
  const int ctx_here = lane < batch ? min(max(len_here, 0), cap) : 0;
  const int steps_here = (ctx_here + kStep - 1) / kStep;
  int total = __builtin_amdgcn_readlane(wave_inclusive_scan(steps_here), 63);
  if (g < batch && __builtin_amdgcn_readlane(ctx_here, g & 63) <= 0) {
    // an empty sequence has no piece: its zeros (0 / (0 + 1e-9)) are written here
    uint4* orow = a.out + (int64_t)g * a.num_heads * H::kPieces;
    for (int i = threadIdx.x; i < a.num_heads * H::kPieces; i += NW * 64)
      orow[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  // Steps per piece.  ceil(total / (most - rows)) always fits, as a row has at most one piece
  // more than its share (with a row for every piece, so does `total`); two shorter lengths are
  // tried with it, in one scan of three counts of 10 bits (none exceeds most + 64): the least
  // there can be, and one between.  (A search by bisection found the shortest, at a scan and a
  // division per try: 1.1 us of 8 ragged sequences' 12.3.)
  const int rows = __popcll(__ballot(steps_here > 0));
  const int per_row = a.group > 8 ? 4 : a.group > 4 ? 8 : 12;   // what is put together at once
  const int enough = max(rows, 1) * per_row;
  // (What follows stays in vector registers: the compiler takes a value that is the same in all lanes
  // to scalar ones and back, and a launch of 7.59 us was 7.87.)
  asm("" : "+v"(total));
  int length0 = max(min(max(divide_small_up(total, enough), kShortestPiece), NW),
                    divide_small_up(total, most));
  if (__any(steps_here > (int)__umul24(per_row, length0)))   // (equal rows pay no maximum: 0.07 us)
    length0 = max(length0, min(divide_small_up(wave_max(steps_here), per_row), NW));
  int length1 = max(length0, divide_small_up(total, most - rows / 2));
  const int length2 = max(length0, divide_small_up(total, max(most - rows, 1)));
  if (length0 > NW && most > enough) length0 = (length0 + NW - 1) / NW * NW;
  // A row of up to a step a wave is one piece whatever the length, as one step would be: it is no
  // longer in one workgroup, and there is nothing to put together across workgroups (one sequence of 83
  // positions, 8 / 1 heads, in tables of 1024, 6.9 us in pieces of 2 steps, 4.9 whole; 44 of 129
  // 7.9 / 6.1).
  const int to_cut = steps_here <= NW ? min(steps_here, 1) : steps_here;
  const uint32_t n2 = divide_small_up(to_cut, length2);
  uint32_t numbers, counts;   // three of 10 bits each
  auto shortest_that_fits = [&]() __attribute__((always_inline)) {   // where its number is
    const uint32_t n0 = divide_small_up(to_cut, length0), n1 = divide_small_up(to_cut, length1);
    numbers = n0 | n1 << 10 | n2 << 20;
    counts = wave_inclusive_scan(numbers);
    const int all = __builtin_amdgcn_readlane(counts, 63);
    return (all & 1023) <= most ? 0 : (all >> 10 & 1023) <= most ? 10 : 20;
  };
  int pick = shortest_that_fits();
  // Lengths that differ much can leave only the one that always fits.  Two multiples of 8 in front of
  // it are tried then: with up to 8 steps more than one of them a wave has one more to walk (10 rows of
  // 1609 positions and 21 of 1, 4 / 4 heads, in pieces of 17 steps 15.0 us, of 16 12.1).
  if (pick == 20 && __builtin_amdgcn_readfirstlane(length2) > NW) {
    length0 = (length1 + NW) / NW * NW;
    length1 = ((length0 + length2) / 2 + NW - 1) / NW * NW;
    pick = shortest_that_fits();
  }
  const int number = numbers >> pick & 1023, incl = counts >> pick & 1023;
  const unsigned long long hit = __ballot(at < incl);
  if (hit == 0ull) return;
  const int b = __builtin_ctzll(hit);
  const int pieces = __builtin_amdgcn_readlane(number, b);
  const int first = __builtin_amdgcn_readlane(incl, b) - pieces;
  const int ctx = __builtin_amdgcn_readlane(ctx_here, b);
  const int nb = __builtin_amdgcn_readlane(steps_here, b);
  const int piece = at - first;
  const int share = __builtin_amdgcn_readfirstlane(divide_small(nb, pieces));
  const int more = nb - share * pieces;   // the first pieces take a step more
  const int s0 = piece * share + min(piece, more), steps = share + (piece < more);
  const int parts = min(steps, NW);
  const PartOfSteps mine = part_of_steps<NW>(wave, steps);
  const int w0 = s0 + mine.first, w1 = s0 + mine.end;
  int first_block = -1;
  if (entries <= 64 * kHeldEntries && w1 > w0) {
    const int at = b * a.max_blocks + a.page.divide(w0 * kStep);
    int entry = held[0];
#pragma unroll
    for (int i = 1; i < kHeldEntries; ++i)
      if (at >> 6 == i) entry = held[i];
    first_block = max(__builtin_amdgcn_readlane(entry, at & 63), 0);
  }
  f32x4 acc[8];
#pragma unroll
  for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegBig, l_run = 0.f;
  if (w1 > w0)
    compute_segment<D, F16, NEW>(a, k_tile[wave], b, kvh, w0 * kStep, min(ctx, w1 * kStep), lane,
                                 acc, m_run, l_run, &fresh, new_slot, first_block);
  if (wave < parts) park_part<D>(k_tile[wave], lane, acc, m_run, l_run);
  __syncthreads();
  finish_piece<D, F16>(a, k_tile, &last, counters, counters + 1 + b * a.num_kv_heads + kvh, b, kvh,
                       g, first * a.num_kv_heads + kvh, a.num_kv_heads, pieces, wave, lane, parts);
}

// grid.x = num_wgs, block = 512.  `min_steps`: fewest steps a sub-run may have
// (in units of 1 << shift steps); `shift`: see Cut.
template <int D, bool F16, int VG = 0, bool NEW = false>
__global__ __launch_bounds__(512) void paged_decode_balanced_kernel(DecodeArgs a, int batch,
                                                                    int num_wgs, int min_steps,
                                                                    int hpw, int wr_hpw, int wr_hpw_alt,
                                                                    int wr_tol, int shift,
                                                                    int short_rows,
                                                                    int32_t* counters,
                                                                    NewRows fresh) {
  using H = HeadDim<D>;
  constexpr int NW = 8;
  int new_slot = -1;
  int main_wgs = gridDim.x;
  if constexpr (NEW) {
    if (fresh.main_wgs > 0) {
      main_wgs = fresh.main_wgs;
      if ((int)blockIdx.x >= main_wgs) {
        store_new_row<F16>(a, fresh, blockIdx.x - main_wgs, NW * 64);
        return;
      }
    } else if ((int)blockIdx.x < batch) {
      store_new_row<F16>(a, fresh, blockIdx.x, NW * 64);
    }
    new_slot = new_slot_of_lane(fresh, batch, threadIdx.x & 63);
  }
  __shared__ uint4 k_tile[NW][kStep * H::kLdsRowPieces];
  constexpr int kLanesWithDims = D / 32 * 16;   // lanes whose k-group holds real dims
  static_assert(sizeof(uint4) * kStep * H::kLdsRowPieces >= 34 * kLanesWithDims * sizeof(float),
                "a wave's K tile must hold its partial");
  // whole-row layout only: the lengths of the batch where any lane can index
  // them, the order the sequences are dealt to the workgroups in, and per wave
  // the partial of a piece that has to wait for the rest of its row
  __shared__ int wr_ctx[kKeptSequences];
  __shared__ int wr_steps[kKeptSequences];    // steps of every sequence
  __shared__ __align__(16) int wr_key[kKeptSequences];   // sorting keys
  __shared__ int wr_order[kKeptSequences];    // sequence of every rank by length
  __shared__ int wr_sorted[kKeptSequences];   // its steps
  __shared__ float wr_parked[NW][34 * kLanesWithDims];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x;
  const int cap = a.max_blocks * a.block_size;

  auto ctx_of = [&](int idx) { return idx < batch ? min(max(a.context_lens[idx], 0), cap) : 0; };
  auto steps_of = [&](int idx) { return (ctx_of(idx) + kStep - 1) / kStep; };

  // One pass over the batch, 64 sequences at a time: total number of steps,
  // and for the first kKeep groups the per-lane (length, steps before) pairs
  // are kept so that locating a position below needs no second read.
  constexpr int kKeep = kKeptSequences / 64;
  int kept_ctx[kKeep], kept_excl[kKeep];
#pragma unroll
  for (int k = 0; k < kKeep; ++k) kept_ctx[k] = kept_excl[k] = 0;
  int total = 0, total_kept = 0;
#pragma unroll
  for (int k = 0; k < kKeep; ++k) {
    if (k * 64 < batch) {
      kept_ctx[k] = ctx_of(k * 64 + lane);
      const int n = (kept_ctx[k] + kStep - 1) / kStep;
      const int incl = wave_inclusive_scan(n);
      kept_excl[k] = total + incl - n;
      total += __builtin_amdgcn_readlane(incl, 63);
    }
  }
  total_kept = total;
  for (int base = kKeep * 64; base < batch; base += 64) {
    const int n = steps_of(base + lane);
    total += __builtin_amdgcn_readlane(wave_inclusive_scan(n), 63);
  }
  if constexpr (NEW) {
    static_assert(NW * 64 == kNullStreamWords, "a word per thread");
    if (g == 0 && fresh.clear != nullptr) fresh.clear[threadIdx.x] = 0;
  }
  // No step belongs to an empty sequence: its output row (zeros, 0 / (0 + 1e-9))
  // is written here, sequence b by workgroup b modulo the grid.  The lengths of
  // the first kKeep * 64 sequences are in registers already.
  for (int b = g; b < batch; b += main_wgs) {
    int c;
    if (b < kKeep * 64) {
      int mine = kept_ctx[0];
#pragma unroll
      for (int k = 1; k < kKeep; ++k) mine = (b >> 6) == k ? kept_ctx[k] : mine;
      c = __builtin_amdgcn_readlane(mine, b & 63);
    } else {
      c = min(as_constant(a.context_lens)[b], cap);
    }
    if (__builtin_amdgcn_readfirstlane(c) <= 0) {
      uint4* orow = a.out + (int64_t)b * a.num_heads * H::kPieces;
      for (int i = threadIdx.x; i < a.num_heads * H::kPieces; i += NW * 64)
        orow[i] = make_uint4(0u, 0u, 0u, 0u);
    }
  }

  // -------------------------------------------------------------------------
  // Short rows: one KV head of one sequence per workgroup, with no more rows than CUs.
  // Publishing partials and merging them costs 5-7 us of a small launch, as much as two
  // rounds of a workgroup's 8 waves over their steps cost it: measured (1 .. 32
  // sequences of 64 .. 8192 positions, 8 KV heads) rows take 5.7 us + 3.2 per round,
  // whatever their number (a CU draws 47 GB/s, with any number of loads in flight), the
  // equal cut 10 us + 2.4 per 1000 wave steps.  4 sequences of 64 / 256 / 512 positions
  // 10.7 / 11.5 / 11.8 us with the equal cut, 5.3 / 8.4 / 10.0 this way; 32 of 2048
  // positions 50.1 / 47.  (Small tables go to paged_decode_whole_kernel or
  // paged_decode_pieces_kernel at once; this is for wide ones with short rows in them.)
  // The row is walked below as a workgroup's run inside one row is: parts meet in LDS.
  // -------------------------------------------------------------------------
  bool short_row = false;
  if (short_rows > 0) {
    int longest = 0;
#pragma unroll
    for (int k = 0; k < kKeep; ++k) longest = max(longest, kept_ctx[k]);
    const int rounds = (wave_max(longest) + NW * kStep - 1) / (NW * kStep);
    short_row = rounds <= 2 || (int64_t)rounds * 1333 < 1792 + (int64_t)a.num_kv_heads * total;
    if (g >= (short_row ? short_rows : num_wgs)) return;
    if (short_row) hpw = 1;
  }

  // -------------------------------------------------------------------------
  // Whole-row layout.  When whole rows can be dealt to the workgroups so that
  // no workgroup gets more than (1 + wr_tol / 256) times its share of the
  // steps, no row is shared between workgroups: a row cut between the parts of
  // one workgroup is put together in LDS, and nothing goes through the
  // workspace or the counters.  The host offers it (wr_hpw > 0: the KV heads
  // per workgroup to use) when all lengths are among the kept ones and there
  // are at least as many rows as workgroups.  Rows are dealt in rounds of
  // num_wgs, forwards and backwards in turn (row of rank p goes to workgroup
  // p % num_wgs in an even round, num_wgs - 1 - p % num_wgs in an odd one),
  // first in the order of the batch - enough for lengths that are equal or
  // nearly so - and, when that is not balanced and there is more than one
  // round, by decreasing length, which pairs long rows with short ones.  Every
  // wave of the launch reads the same lengths and takes the same decision.
  // -------------------------------------------------------------------------
  if (wr_hpw > 0 && total > 0 && !short_row) {
    // every wave writes all the lengths and step counts itself (the same values
    // from each), so no wave has to wait for another before it reads them back
    int key[kKeep];
    int longest = 0, shortest = INT32_MAX;
#pragma unroll
    for (int k = 0; k < kKeep; ++k) {
      const bool real = k * 64 + lane < batch;
      const int n = (kept_ctx[k] + kStep - 1) / kStep;
      wr_ctx[k * 64 + lane] = real ? kept_ctx[k] : 0;
      wr_steps[k * 64 + lane] = real ? n : 0;
      // sorting key: more steps first, among equals the earlier sequence first;
      // unique, and below every real key for the padding behind the batch
      key[k] = real ? (n << 8) | (255 - (k * 64 + lane)) : -1 - (k * 64 + lane);
      longest = max(longest, real ? n : 0);
      shortest = min(shortest, real ? n : INT32_MAX);
    }
    longest = wave_max(longest);
    shortest = -wave_max(-shortest);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // Two candidates: wr_hpw KV heads per workgroup and, when whole rows of
    // that many heads cannot be dealt evenly enough, half as many (twice the
    // rows, another round or more to pair long with short; fewer heads side by
    // side stream a few percent slower, which is why it is second).
    int w_hpw = 0, w_rps = 1, rps_shift = 0, rows = 0, rounds = 0;
    bool whole_rows = false, sorted = false, ranked = false;
    for (int candidate = 0; candidate < 2 && !whole_rows; ++candidate) {
      w_hpw = candidate == 0 ? wr_hpw : wr_hpw_alt;
      if (w_hpw <= 0) break;
      w_rps = a.num_kv_heads / w_hpw;       // a power of two (the host sees to it)
      rps_shift = __builtin_ctz(w_rps);
      rows = batch * w_rps;
      rounds = (rows + num_wgs - 1) / num_wgs;
      // the largest number of steps any workgroup is dealt; steps_of_rank: the
      // steps of the sequence of a given rank (wr_steps in the order of the
      // batch, wr_sorted in the order by length)
      auto largest_deal = [&](const int* steps_of_rank) {
        int worst = 0;
        for (int w0 = 0; w0 < num_wgs; w0 += 64) {
          const int w = w0 + lane;
          int load = 0;
          for (int t = 0; t < rounds; ++t) {
            const int p = t * num_wgs + ((t & 1) ? num_wgs - 1 - w : w);
            if (w < num_wgs && p < rows) load += steps_of_rank[p >> rps_shift];
          }
          worst = max(worst, load);
        }
        return wave_max(worst);
      };
      const int64_t share = (int64_t)w_rps * total;   // num_wgs * a workgroup's share of the steps
      const auto fits = [&](int load, int tol) {
        return (int64_t)load * num_wgs * 256 <= share * (256 + tol);
      };
      // A row longer than the limit rules both orders out.  With one round
      // every workgroup gets one row and the longest row decides.  With more
      // rounds the order of the batch is only taken when it is as good as
      // balanced (and only looked at when the lengths are within an eighth of
      // each other); otherwise the order by length gets its chance.
      if (!fits(longest, wr_tol)) continue;
      sorted = false;
      if (rounds == 1) {
        whole_rows = true;
        break;
      }
      if ((longest - shortest) * 8 <= longest &&
          fits(largest_deal(wr_steps), min(wr_tol, kWholeRowTightTolerance))) {
        whole_rows = true;
        break;
      }
      if (!ranked) {
        // Rank of every sequence by decreasing key: two threads per sequence
        // count, over half of the batch each, the keys above its own.  The keys
        // go through LDS (every wave writes all of them, the same values from
        // each) and are read back four at a time, eight reads in flight.
#pragma unroll
        for (int k = 0; k < kKeep; ++k) wr_key[k * 64 + lane] = key[k];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int i = threadIdx.x >> 1, half = threadIdx.x & 1;
        const int mine = wr_key[i];
        const int quads = (batch + 3) / 4;            // int4 groups that hold real keys
        const int per_half = (quads + 1) / 2;
        int above = 0;
        for (int j0 = half * per_half; j0 < min(quads, (half + 1) * per_half); j0 += 8) {
          int4 k4[8];
#pragma unroll
          for (int u = 0; u < 8; ++u)
            k4[u] = reinterpret_cast<const int4*>(wr_key)[min(j0 + u, kKeptSequences / 4 - 1)];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const bool in = j0 + u < min(quads, (half + 1) * per_half);
            above += (in && k4[u].x > mine ? 1 : 0) + (in && k4[u].y > mine ? 1 : 0) +
                     (in && k4[u].z > mine ? 1 : 0) + (in && k4[u].w > mine ? 1 : 0);
          }
        }
        above += __builtin_amdgcn_update_dpp(0, above, kDppQuadXor1, 0xF, 0xF, false);
        if (half == 0 && i < batch) {
          wr_order[above] = i;
          wr_sorted[above] = mine >> 8;
        }
        __syncthreads();
        ranked = true;
      }
      sorted = true;
      whole_rows = fits(largest_deal(wr_sorted), wr_tol);
    }
    if (whole_rows) {
      const int w_parts = NW / w_hpw;
      const int part = wave / w_hpw;
      const int h_in_row = wave - part * w_hpw;
      // the rows dealt to this workgroup, in the order of the rounds
      auto dealt_row = [&](int t, int& seq, int& hg, int& ctx) {
        const int p = t * num_wgs + ((t & 1) ? num_wgs - 1 - g : g);
        seq = 0; hg = 0; ctx = 0;
        if (p < rows) {
          const int rank = p / w_rps;
          seq = sorted ? wr_order[rank] : rank;
          hg = p - rank * w_rps;
          ctx = wr_ctx[seq];
        }
        seq = __builtin_amdgcn_readfirstlane(seq);
        hg = __builtin_amdgcn_readfirstlane(hg);
        ctx = __builtin_amdgcn_readfirstlane(max(ctx, 0));
      };
      int mine = 0;   // steps dealt to this workgroup
      for (int t = 0; t < rounds; ++t) {
        int seq, hg, ctx;
        dealt_row(t, seq, hg, ctx);
        mine += (ctx + kStep - 1) / kStep;
      }
      // the steps are cut into equal runs for the parts; a part's first piece,
      // when it does not start a row, waits in LDS for the part that does
      const int xs = (int)((int64_t)part * mine / w_parts);
      const int xe = (int)((int64_t)(part + 1) * mine / w_parts);
      f32x4 acc[8];
#pragma unroll
      for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
      float m_run = kNegBig, l_run = 0.f;
      bool owes = false;       // acc holds the first piece of a row that goes on in later parts
      int owed_b = 0, owed_kvh = 0, owed_end = 0;
      const bool holds_dims = lane < kLanesWithDims;
      int row_start = 0;
      for (int t = 0; t < rounds && row_start < xe; ++t) {
        int seq, hg, ctx;
        dealt_row(t, seq, hg, ctx);
        const int nb = (ctx + kStep - 1) / kStep;
        const int lo = max(xs, row_start), hi = min(xe, row_start + nb);
        if (lo < hi) {
          const int st = lo - row_start, en = hi - row_start;
          const int kvh = hg * w_hpw + h_in_row;
          const int t0 = __builtin_amdgcn_readfirstlane(st * kStep);
          const int t1 = __builtin_amdgcn_readfirstlane(min(ctx, en * kStep));
          if constexpr (VG > 0)
            compute_segment_valu<VG>(a, k_tile[wave], seq, kvh, t0, t1, lane, acc, m_run, l_run);
          else if constexpr (VG < 0)
            compute_segment_loads_only(a, seq, kvh, t0, t1, lane, acc, m_run, l_run);
          else
            compute_segment<D, F16, NEW>(a, k_tile[wave], seq, kvh, t0, t1, lane, acc, m_run, l_run,
                                         &fresh, new_slot);
          if (st > 0) {
            // the row started in an earlier part: park the piece for it
            if (holds_dims) {
              float* slot = wr_parked[wave] + lane;
#pragma unroll
              for (int jd = 0; jd < 8; ++jd)
#pragma unroll
                for (int e = 0; e < 4; ++e) slot[(4 * jd + e) * kLanesWithDims] = acc[jd][e];
              slot[32 * kLanesWithDims] = m_run;
              slot[33 * kLanesWithDims] = l_run;
            }
          } else if (en == nb) {
            write_output<D, F16>(a, seq, kvh, lane, acc, l_run);
          } else {
            // the row goes on in the next part(s): this is the run's last segment
            owes = true; owed_b = seq; owed_kvh = kvh; owed_end = row_start + nb;
          }
        }
        row_start += nb;
      }
      __syncthreads();
      if (owes) {
        if (holds_dims) {
          for (int p = part + 1; p < w_parts; ++p) {
            const int ps = (int)((int64_t)p * mine / w_parts);
            const int pe = (int)((int64_t)(p + 1) * mine / w_parts);
            if (ps >= owed_end) break;
            if (pe > ps)
              add_partial_from_lds<kLanesWithDims>(wr_parked[p * w_hpw + h_in_row] + lane,
                                                   a.scale_log2e, acc, m_run, l_run);
          }
        }
        write_output<D, F16>(a, owed_b, owed_kvh, lane, acc, l_run);
      }
      return;
    }
  }
  const int parts = NW / hpw;
  const int rows_per_seq = a.num_kv_heads / hpw;
  const int part = wave / hpw;
  const int h_in_row = wave - part * hpw;
  const Cut cut(rows_per_seq * total, shift, num_wgs * parts, min_steps);
  if (!short_row && (cut.axis == 0 || g * parts >= cut.nsub)) return;

  // the sequence whose rows hold axis position x: its index, the steps before
  // it and its length (all wave-uniform)
  auto locate = [&](int x, int& b, int& before, int& ctx) {
    b = batch; before = total; ctx = 0;
    bool found = false;
#pragma unroll
    for (int k = 0; k < kKeep; ++k) {
      const int n = (kept_ctx[k] + kStep - 1) / kStep;
      const int lo = rows_per_seq * kept_excl[k];
      const unsigned long long hit =
          __ballot(!found && n > 0 && lo <= x && x < lo + rows_per_seq * n);
      if (hit != 0ull) {
        const int src = __builtin_ctzll(hit);
        b = k * 64 + src;
        before = __builtin_amdgcn_readlane(kept_excl[k], src);
        ctx = __builtin_amdgcn_readlane(kept_ctx[k], src);
        found = true;
      }
    }
    if (!found) {
      int running = total_kept;
      for (int base = kKeep * 64; base < batch; base += 64) {
        const int c = ctx_of(base + lane);
        const int n = (c + kStep - 1) / kStep;
        const int incl = wave_inclusive_scan(n);
        const int lo = rows_per_seq * (running + incl - n);
        const unsigned long long hit = __ballot(n > 0 && lo <= x && x < lo + rows_per_seq * n);
        if (hit != 0ull) {
          const int src = __builtin_ctzll(hit);
          b = base + src;
          before = __builtin_amdgcn_readlane(running + incl - n, src);
          ctx = __builtin_amdgcn_readlane(c, src);
          break;
        }
        running += __builtin_amdgcn_readlane(incl, 63);
      }
    }
    b = __builtin_amdgcn_readfirstlane(b);
    before = __builtin_amdgcn_readfirstlane(before);
    ctx = __builtin_amdgcn_readfirstlane(ctx);
  };

  int b0, before0, ctx0, nparts, start, end, hg0, row0, xs, xe;
  if (short_row) {
    b0 = g / a.num_kv_heads;
    hg0 = g - b0 * a.num_kv_heads;
    int mine = kept_ctx[0];
#pragma unroll
    for (int k = 1; k < kKeep; ++k) mine = (b0 >> 6) == k ? kept_ctx[k] : mine;
    ctx0 = __builtin_amdgcn_readlane(mine, b0 & 63);
    if (ctx0 <= 0) return;   // (an empty sequence's zeros are written)
    before0 = start = row0 = 0;
    end = (ctx0 + kStep - 1) / kStep;
    nparts = min(NW, end);
    xs = part < nparts ? part * end / nparts : end;
    xe = part < nparts ? (part + 1) * end / nparts : end;
  } else {
    nparts = min(parts, cut.nsub - g * parts);   // parts of this workgroup that have work
    start = cut.start_of(g * parts);
    end = cut.start_of(g * parts + nparts);
    locate(start, b0, before0, ctx0);
    if (b0 >= batch || ctx0 <= 0) return;   // cannot happen when the prefix sums are right
    const int nb = (ctx0 + kStep - 1) / kStep;
    hg0 = (start - rows_per_seq * before0) / nb;
    row0 = rows_per_seq * before0 + hg0 * nb;   // axis position of the row's step 0
    xs = part < nparts ? cut.start_of(g * parts + part) : end;
    xe = part < nparts ? cut.start_of(g * parts + part + 1) : end;
  }
  const int nb0 = (ctx0 + kStep - 1) / kStep;
  const int64_t subrun = (int64_t)g * parts + part;
  // Does the whole run of the workgroup lie inside one row?  Then every wave has
  // at most one segment, and the parts of a head meet in LDS before anything is
  // written.  Otherwise every wave walks its own sub-run across the rows.
  const bool single = end <= row0 + nb0;
  if (!single && xs >= xe) return;

  int b = b0, before = before0, ctx = ctx0;
  if (!single && part > 0) locate(xs, b, before, ctx);
  // Every quantity of the walk is wave-uniform; readfirstlane says so, so that
  // lengths, page lookups and address arithmetic stay on the scalar unit.  The
  // guards (b inside the batch, x not before the sequence) cannot fire when
  // the prefix sums are right; they keep every index in range regardless.
  int x = xs;
  int owed = 0, owed_b[2] = {0, 0}, owed_kvh[2] = {0, 0}, owed_row[2] = {0, 0}, owed_nb[2] = {1, 1};
  for (;;) {
    // ---- the next segment of this wave's sub-run: row (sb, hg), steps [st, en) ----
    int sb = 0, hg = 0, nb = 1, row = 0, st = 0, en = 0;
    bool have = false;
    while (x < xe && b < batch) {
      sb = __builtin_amdgcn_readfirstlane(b);
      nb = (ctx + kStep - 1) / kStep;
      const int seq0 = rows_per_seq * before;
      if (x < seq0) break;
      if (nb == 0 || x >= seq0 + rows_per_seq * nb) {  // empty sequence, or this one is finished
        before += nb;
        b = sb + 1;
        ctx = b < batch ? __builtin_amdgcn_readfirstlane(
                              min(max(as_constant(a.context_lens)[b], 0), cap))
                        : 0;
        continue;
      }
      hg = (x - seq0) / nb;
      row = seq0 + hg * nb;
      st = x - row;
      en = min(nb, st + (xe - x));
      have = true;
      break;
    }
    if (!have && !single) break;
    const int kvh = (single ? hg0 : hg) * hpw + h_in_row;
    f32x4 acc[8];
#pragma unroll
    for (int jd = 0; jd < 8; ++jd) acc[jd] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = kNegBig, l_run = 0.f;
    if (have) {
      const int t0 = __builtin_amdgcn_readfirstlane(st * kStep);
      const int t1 = __builtin_amdgcn_readfirstlane(min(ctx, en * kStep));
      if constexpr (VG > 0)
        compute_segment_valu<VG>(a, k_tile[wave], sb, kvh, t0, t1, lane, acc, m_run, l_run);
      else if constexpr (VG < 0)
        compute_segment_loads_only(a, sb, kvh, t0, t1, lane, acc, m_run, l_run);
      else
        compute_segment<D, F16, NEW>(a, k_tile[wave], sb, kvh, t0, t1, lane, acc, m_run, l_run,
                                     &fresh, new_slot);
      x += en - st;
    }

    bool direct = st == 0 && en == nb;   // the segment is the whole row
    int covers = 1;                      // sub-runs this wave's partial stands for
    if (single) {
      sb = b0; hg = hg0; nb = nb0; row = row0;
      direct = start == row0 && end == row0 + nb0;
      covers = nparts;
      if (nparts > 1) {
        const bool holds_dims = lane < kLanesWithDims;
        if (part > 0 && have) {
          // value v of lane l at float v * kLanesWithDims + l of the wave's own tile
          if (holds_dims) {
            float* mine = reinterpret_cast<float*>(k_tile[wave]) + lane;
#pragma unroll
            for (int jd = 0; jd < 8; ++jd)
#pragma unroll
              for (int e = 0; e < 4; ++e) mine[(4 * jd + e) * kLanesWithDims] = acc[jd][e];
            mine[32 * kLanesWithDims] = m_run;
            mine[33 * kLanesWithDims] = l_run;
          }
        }
        __syncthreads();
        if (part > 0) return;
        if (holds_dims) {
          for (int p = 1; p < nparts; ++p) {
            add_partial_from_lds<kLanesWithDims>(
                reinterpret_cast<const float*>(k_tile[wave + p * hpw]) + lane, a.scale_log2e, acc,
                m_run, l_run);
          }
        }
      }
      if (part > 0) return;
    }

    if (direct) {
      write_output<D, F16>(a, sb, kvh, lane, acc, l_run);
    } else {
      const int64_t slot = subrun + (int64_t)sb * rows_per_seq + hg;
      write_partial_coherent<D>(a, balanced_record(a, slot, hpw, h_in_row), lane, acc, m_run,
                                l_run);
      if (arrive(a, counters, sb, kvh, row, row + nb, cut, covers, lane)) {
        // at most the first and the last segment of a sub-run are not whole rows
        if (owed == 0) { owed_b[0] = sb; owed_kvh[0] = kvh; owed_row[0] = row; owed_nb[0] = nb; }
        else { owed_b[1] = sb; owed_kvh[1] = kvh; owed_row[1] = row; owed_nb[1] = nb; }
        ++owed;
      }
    }
    if (single) break;
  }
  // the merges this wave owes, after its own work
  for (int i = 0; i < owed; ++i) {
    const int ob = __builtin_amdgcn_readfirstlane(i == 0 ? owed_b[0] : owed_b[1]);
    const int okvh = __builtin_amdgcn_readfirstlane(i == 0 ? owed_kvh[0] : owed_kvh[1]);
    const int orow = __builtin_amdgcn_readfirstlane(i == 0 ? owed_row[0] : owed_row[1]);
    const int onb = __builtin_amdgcn_readfirstlane(i == 0 ? owed_nb[0] : owed_nb[1]);
    merge_row<D, F16>(a, k_tile[wave], ob, okvh, hpw, orow, orow + onb, cut, lane);
  }
}

// Sets n int32 to zero (the counters of the balanced split; a kernel, not a
// memset, so that the launch can be recorded into a graph).
__global__ __launch_bounds__(256) void zero_int32_kernel(int32_t* p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Second pass of the fixed split: merge the partials of one (sequence, query
// head).  grid = (B, Hq), block = head_dim lanes, one per output dim.  The
// partials of sequence b are slots b*max_chunks .. + ceil(ctx/chunk).  A
// sequence with one partial was written by the split kernel itself; an empty
// one gives zeros.
__global__ __launch_bounds__(kMaxHeadDim) void paged_decode_combine_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const int32_t* __restrict__ context_lens, uint16_t* __restrict__ out, int num_heads, int chunk,
    int max_chunks, int max_positions, float scale_log2e, bool f16) {
  const int b = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
  const int head_dim = blockDim.x;
  const int ctx = min(context_lens[b], max_positions);
  const int nparts = ctx <= 0 ? 0 : (ctx + chunk - 1) / chunk;
  const int64_t first = (int64_t)b * max_chunks;
  if (nparts == 1) return;  // written by the split kernel itself
  uint16_t* o = out + ((int64_t)b * num_heads + h) * head_dim + d;
  if (nparts == 0) {  // empty sequence: 0 / (0 + 1e-9)
    *o = 0;
    return;
  }
  const int64_t base = first * num_heads + h;
  const float2* ml = reinterpret_cast<const float2*>(part_ml);
  // One pass, 8 partials at a time with all their loads issued together, merged
  // with the running-max rescale.
  float m = kNegBig, num = 0.f, den = 0.f;
  for (int c0 = 0; c0 < nparts; c0 += 8) {
    float2 mlv[8];
    float po[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t row = base + (int64_t)min(c0 + i, nparts - 1) * num_heads;
      mlv[i] = ml[row];
      po[i] = part_o[row * head_dim + d];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (c0 + i < nparts) {
        const float m_new = fmaxf(m, mlv[i].x);
        const float keep = __builtin_amdgcn_exp2f((m - m_new) * scale_log2e);
        const float w = __builtin_amdgcn_exp2f((mlv[i].x - m_new) * scale_log2e);
        num = fmaf(num, keep, w * po[i]);
        den = fmaf(den, keep, w * mlv[i].y);
        m = m_new;
      }
    }
  }
  const float res = num / (den + 1e-9f);
  *o = (uint16_t)((f16 ? Elem<true>::pack2(res, 0.f) : Elem<false>::pack2(res, 0.f)) & 0xFFFFu);
}

int round_up(int x, int m) { return (x + m - 1) / m * m; }

// A wave covers at most 16 query heads (the MFMA columns).  A cache head with
// more than that is walked as `rep` virtual KV heads, the smallest count that
// divides the group into parts of at most 16; its K/V rows are then read once
// per virtual head.
int virtual_heads_per_cache_head(int group) {
  int rep = 1;
  while (group % rep != 0 || group / rep > 16) ++rep;
  return rep;
}

// KV heads per 8-wave workgroup of the whole-sequence mode: as many as still
// give one (sequence, head group) row per CU, so that a sequence is split over
// the waves of a workgroup no finer than needed; it must divide the number of
// KV heads.
int heads_per_workgroup(int64_t batch, int num_kv_heads) {
  const int cus = compute_units();
  int hpw = 8;
  while (hpw > 1 && (num_kv_heads % hpw != 0 || batch * (num_kv_heads / hpw) < cus)) hpw /= 2;
  return hpw;
}

// KV heads per 8-wave workgroup of the balanced split.  Two forces pull apart.
// The heads of one workgroup read adjacent pieces of every position's row, and
// a stream-bound launch runs faster with more of them side by side: 32
// sequences of 16k..32k positions take 506 / 471 / 457 / 460 us with 1 / 2 / 4
// / 8 heads of 128 per workgroup (head_dim 64 ranks the same way).  Against
// that, the partials one wave has to merge per (sequence, head) grow with the
// heads per workgroup, because the sub-runs are then spread over fewer rows: a
// single sequence of 32k positions takes 38 / 45 / 67 / 109 us.  The rule below
// is the best or within 3 % of it over batch 1..256 x 512..32768 positions x
// 2, 4, 8 KV heads, ragged and uniform lengths: 4 heads from batch 32 up, or
// from batch 16 when the table spans 4096 positions; 1 head for up to 16
// (sequence, head) pairs when the table spans 6144 positions or more; else 2.
int balanced_heads_per_workgroup(int64_t batch, int num_kv_heads, int64_t max_steps) {
  int hpw = 2;
  if (batch * num_kv_heads <= 16 && max_steps >= 192) hpw = 1;
  else if (batch >= 32 || (batch >= 16 && max_steps >= 128)) hpw = 4;
  while (hpw > 1 && num_kv_heads % hpw != 0) hpw /= 2;
  return hpw;
}

// Balanced mode launches at most one workgroup per CU, and never gives a wave
// fewer than this many 32-position steps.
constexpr int kMinBalancedSteps = 1;

// Whole rows are dealt to the workgroups when no workgroup gets more than
// 1 + kWholeRowTolerance / 256 times the mean number of steps.  The launch is
// bound by the memory system as a whole, not by its slowest workgroup: while
// workgroups with less to do finish, the others stream faster, so an uneven
// deal costs far less than its unevenness.  Measured against the equal cut with
// shared rows (256 sequences, 2 rows each, lengths log-uniform or uniform):
// 9 % unevenness 195 against 213 us, 16 % 174 against 187, 34 % 148 against
// 149, 56 % 250 against 231; one row per workgroup (64 sequences around 3500
// positions): 9 % 153 against 165, 15 % 146 against 154, 25 % 137 against 142.
constexpr int kWholeRowTolerance = 64;

// Whether a launch of at most one row per CU goes by pieces (paged_decode_pieces_kernel), from
// what the table can hold; else the balanced kernel looks at the lengths.  Pieces save what
// the balanced kernel's larger head and its merges by single waves cost a small launch, 3 us:
// by pieces / balanced, 1 .. 4 sequences of 1000 positions and 8 KV heads 8.4 .. 9.2 / 13.0 ..
// 14.0 us, 8 of 100 .. 900 8.7 / 13.6, 8 of 128 .. 2048 12.9 / 15.5, 4 of 4096 17.1 / 21.0.
// Against that a row is cut into whole pieces of one length for all rows, which leaves
// workgroups idle when lengths differ and rows are many, and one KV head per workgroup
// streams slower.  At the line, us: 32 rows of 500 .. 32000 positions 56.0 / 62.0, 64 rows of
// 1000 .. 16000 55.6 / 58.9, 128 rows of 300 .. 4096 33.0 / 34.4; equal rows that leave a quarter of the
// workgroups idle are the worst within it: 96 of 4096 39.4 / 40.6, 88 of 5952 52.0 / 50.7; beyond, 64
// rows of 16000 .. 32768 137.7 / 134.2, 128 of 500 .. 8000 60.2 / 57.0.
// Beyond 128 rows the mean row has less than two pieces, and where long rows find none to spare
// one workgroup walks all of a row.  39648 launches drawn from 132 .. 256 rows and 832 .. 1927 positions
// (equal, evenly spread, one, a third, half or most of them long), by pieces / balanced: within the
// line up to 192 rows 0.86 in the mean, 7 % of them above 1.03, to 224 rows 0.88 and 16 %, at worst 1.23
// (176 of 1344 or 20, half of them long, 24.0 / 19.6); beyond it 0.95 .. 0.97, 28 %, and 1.84 (8 of 248
// rows of 1920 and the others of 1, 26.7 / 14.5).
bool pieces_pay(int64_t rows, int64_t positions, int64_t cus) {
  if (rows > cus - cus / 8) return false;
  return rows * positions <= (rows <= 64 ? 1 << 20 : rows <= 128 ? 1 << 19 : 1 << 18);
}

// Whether pieces are what a launch of that many rows takes if its table is not one of short rows.
bool pieces_take(int64_t batch, int head_dim, int64_t rows, int64_t positions, int64_t cus) {
  return head_dim == 128 && batch <= 64 && pieces_pay(rows, positions, cus);
}

// Whether the table rules out rows (of at most one per CU) that are not short: up to three
// rounds of the 8 waves of a workgroup, which take 1.2 (head_dim 64) to 2.8 us each, what one
// CU draws; such rows are finished inside one workgroup by the kernel without a split.  us,
// without a split / by the balanced kernel, at 768 positions, equal or ragged: head_dim 64, 1 ..
// 16 rows 7.6 .. 8.7 / 12.1 .. 13.2, 24 .. 64 rows 7.7 .. 9.3 / 12.1 .. 13.5, 65 .. 128 rows 8.3 ..
// 9.9 / 12.4 .. 13.9; head_dim 128, 65 .. 128 sequences of one row 10.4 .. 11.6 / 13.2 .. 14.6.
// (At 1024 equal lengths the balanced kernel is still 2 .. 5 us behind; lengths that differ
// have not been measured there.)
// Where pieces are the other choice, up to 128 rows, the third round is theirs: without a
// split / by pieces, at 288 positions 1 .. 64 rows 7.1 .. 8.3 / 6.8 .. 8.8, at 512 1 .. 32 rows 7.7
// .. 9.0 / 7.0 .. 9.5 (the more, the more query heads share a KV head), 64 rows 8.3 .. 8.5 / 8.7 ..
// 9.4, 128 rows 9.4 .. 10.7 / 10.3 .. 11.1; at 768 1 .. 16 rows 9.0 .. 10.1 / 7.1 .. 9.6, 64 rows 9.8 ..
// 10.5 / 9.2 .. 10.0, 128 rows 13.7 .. 14.0 / 13.3 .. 14.2, 192 rows 15.4 .. 15.7 / 16.0 .. 16.3, 256
// rows 18.1 .. 18.4 / 18.8 .. 19.3.
bool table_of_short_rows(int64_t rows, int64_t positions, bool pieces) {
  return positions <= (pieces && rows <= 128 ? 2 : 3) * 8 * kStep;
}

// Waves per workgroup of the fixed split = KV heads a workgroup covers: the
// largest of 8, 4, 2, 1 that divides the number of KV heads.
int waves_per_workgroup(int num_kv_heads) {
  return num_kv_heads % 8 == 0 ? 8 : num_kv_heads % 4 == 0 ? 4 : num_kv_heads % 2 == 0 ? 2 : 1;
}

// The counter region of the balanced split: word 0 is the stale flag, then one
// int32 per (sequence, KV head as the kernels walk them); padded to 256 bytes.
size_t counter_region_bytes(int64_t batch, int64_t kv_heads) {
  return ((size_t)(batch * kv_heads + 1) * sizeof(int32_t) + 255) / 256 * 256;
}

// Workspace layout.  Fixed chunks: partials of batch * max_chunks slots, every
// slot holding all query heads.  Balanced: first the counters, one int32 per
// (sequence, KV head), padded to 256 bytes; then the partials of slots =
// sub-runs + rows, a slot holding the query heads of hpw KV heads.
struct WorkspacePlan {
  int64_t records;  // partial records (one query head each)
  int max_chunks;   // fixed-chunk mode only
  int num_wgs, hpw, wr_hpw, wr_hpw_alt, shift;  // balanced mode only
  size_t counter_bytes;
  size_t bytes;
};

bool plan_workspace(int64_t batch, int64_t num_heads, int64_t head_dim, int64_t max_blocks,
                    int64_t block_size, int num_kv_heads, int chunk, WorkspacePlan* plan) {
  if (chunk == 0) {
    const int64_t max_steps = (max_blocks * block_size + kStep - 1) / kStep;
    const int hpw = balanced_heads_per_workgroup(batch, num_kv_heads, max_steps);
    const int parts = 8 / hpw;
    const int64_t rows_per_seq = num_kv_heads / hpw;
    const int64_t axis = rows_per_seq * batch * max_steps;
    if (axis > INT32_MAX / 2) return false;
    int64_t wgs = (axis + (int64_t)parts * kMinBalancedSteps - 1) / (parts * kMinBalancedSteps);
    const int64_t cus = compute_units();
    wgs = wgs < 1 ? 1 : wgs > cus ? cus : wgs;
    plan->num_wgs = (int)wgs;
    plan->hpw = hpw;
    // (units + 1) * sub-runs must fit 31 bits (Cut): coarser units for a very long axis
    plan->shift = 0;
    while ((((axis >> plan->shift) + 2) * wgs * parts) >> 31) ++plan->shift;
    // The whole-row layout of the kernel (no partials at all) is offered when the
    // kernel keeps every length in registers and there is a row for every
    // workgroup: with as many heads per workgroup as still give that, 2 at least
    // (rows of 1 head are only worth it as the second choice: 32 equal sequences
    // of 8192 positions take 167 us that way against 164 with the equal cut), and
    // as a second choice with half as many heads, which gives the kernel another
    // round or more of rows to pair long ones with short ones (64 sequences of
    // 2048..6144 positions: 175 us with 1 head per workgroup, by length, against
    // 180 with the equal cut; 128 of 2000..6000: 321 with 2 heads against 329).
    // The layout needs no workspace of its own.
    plan->wr_hpw = plan->wr_hpw_alt = 0;
    const auto whole_rows_can_use = [&](int h) {
      const int rps = h > 0 && num_kv_heads % h == 0 ? num_kv_heads / h : 0;
      return rps > 0 && (rps & (rps - 1)) == 0 &&   // the kernel divides by shifting
             batch * rps >= wgs;
    };
    if (batch <= kKeptSequences && wgs <= kMaxWholeRowWorkgroups)
      for (int h = hpw; h >= 2; h /= 2)
        if (num_kv_heads % h == 0 && batch * (num_kv_heads / h) >= wgs) {
          if (whole_rows_can_use(h)) {
            plan->wr_hpw = h;
            if (whole_rows_can_use(h / 2)) plan->wr_hpw_alt = h / 2;
          }
          break;
        }
    plan->max_chunks = 0;
    const int64_t slots = wgs * parts + batch * rows_per_seq;
    plan->records = slots * hpw * (num_heads / num_kv_heads);
    plan->counter_bytes = counter_region_bytes(batch, num_kv_heads);
    plan->bytes = plan->counter_bytes + (size_t)plan->records * (head_dim + 2) * sizeof(float);
    return true;
  }
  const int64_t mc = (max_blocks * block_size + chunk - 1) / chunk;
  if (batch * mc > INT32_MAX) return false;
  plan->num_wgs = plan->hpw = plan->wr_hpw = plan->wr_hpw_alt = plan->shift = 0;
  plan->max_chunks = (int)mc;
  plan->records = batch * mc * num_heads;
  plan->counter_bytes = 0;
  plan->bytes = (size_t)plan->records * (head_dim + 2) * sizeof(float);
  return true;
}

}  // namespace

extern "C" int32_t nvj_paged_decode_default_chunk(int32_t batch, int32_t num_kv_heads,
                                                  int32_t max_blocks, int32_t block_size) {
  if (batch <= 0 || num_kv_heads <= 0 || max_blocks <= 0 || block_size <= 0) return 256;
  // One 8-wave workgroup is resident per CU and a launch is fastest at exactly
  // one workgroup per CU (256 on MI355X): the chunk that gives that when every
  // sequence is at full length, if it is at most 2048 positions; else 1024,
  // which keeps ragged batches balanced; never below 128.
  const int64_t positions = (int64_t)batch * max_blocks * block_size;
  int64_t chunk = (positions + 255) / 256;
  if (chunk < 128) chunk = 128;
  if (chunk > 2048) chunk = 1024;
  return round_up((int)chunk, kStep);
}

extern "C" int32_t nvj_paged_decode_whole_sequence_workgroups(int32_t batch, int32_t num_heads,
                                                               int32_t num_kv_heads) {
  if (batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0) return 0;
  const int64_t heads =
      (int64_t)num_kv_heads * virtual_heads_per_cache_head(num_heads / num_kv_heads);
  if (batch * heads > INT32_MAX) return 0;
  return batch * ((int)heads / heads_per_workgroup(batch, (int)heads));
}

extern "C" size_t nvj_paged_decode_workspace_bytes(int32_t batch, int32_t num_heads,
                                                   int32_t head_dim, int32_t max_blocks,
                                                   int32_t block_size, int32_t num_kv_heads,
                                                   int32_t chunk) {
  if (chunk == NVJ_CHUNK_WHOLE_SEQUENCE) return 0;   // finished inside the workgroups
  if (batch <= 0 || num_heads <= 0 || (head_dim != 128 && head_dim != 64) || max_blocks <= 0 ||
      block_size <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0 || chunk < 0 ||
      chunk % kStep != 0)
    return 0;
  num_kv_heads *= virtual_heads_per_cache_head(num_heads / num_kv_heads);
  WorkspacePlan plan;
  if (!plan_workspace(batch, num_heads, head_dim, max_blocks, block_size, num_kv_heads, chunk,
                      &plan))
    return 0;
  return plan.bytes;
}

namespace {
// What a kernel gets to know of the new rows, and its grid: a workgroup of its own stores a
// row if that leaves one workgroup per CU, else one of the `wgs` that attend does.
NewRows rows_behind(const NewRows* rows, int wgs, int batch, dim3* grid) {
  NewRows n = rows ? *rows : NewRows{};
  n.main_wgs = rows && wgs + batch <= compute_units() ? wgs : 0;
  *grid = dim3((unsigned)(n.main_wgs > 0 ? wgs + batch : rows && batch > wgs ? batch : wgs));
  return n;
}

// The launch behind every decode entry point.  `ext_counters` != NULL: the
// counters of the balanced split live there and `workspace` holds the partials
// only (no counter header in front of them).
int launch_decode(void* stream, const void* q, const void* k_cache, const void* v_cache,
                  const int32_t* block_tables, const int32_t* context_lens, void* out,
                  void* workspace, size_t workspace_bytes, int32_t* ext_counters, int32_t batch,
                  int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                  int32_t max_blocks, int32_t num_blocks, float scale, int32_t chunk,
                  int32_t dtype, uint32_t phases, const NewRows* new_rows = nullptr,
                  const nvj::ReadAhead* ahead = nullptr) {
  if (dtype != NVJ_DTYPE_BF16 && dtype != NVJ_DTYPE_F16) return NVJ_ERR_BAD_DTYPE;
  const bool f16 = dtype == NVJ_DTYPE_F16;
  const bool whole = chunk == NVJ_CHUNK_WHOLE_SEQUENCE;
  if (batch < 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 ||
      max_blocks < 0 || num_blocks <= 0 || (chunk < 0 && !whole))
    return NVJ_ERR_BAD_SHAPE;
  if (num_heads % num_kv_heads != 0) return NVJ_ERR_BAD_SHAPE;
  if ((head_dim != 128 && head_dim != 64) || block_size % kStep != 0 ||
      (!whole && chunk % kStep != 0))
    return NVJ_ERR_UNSUPPORTED;
  const int cache_kv_heads = num_kv_heads;
  const int kv_rep = virtual_heads_per_cache_head(num_heads / num_kv_heads);
  if ((int64_t)num_kv_heads * kv_rep > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  num_kv_heads *= kv_rep;   // from here on: the heads as the kernels walk them
  const int group = num_heads / num_kv_heads;
  if ((int64_t)max_blocks * block_size > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  if (!(scale >= 0.f)) return NVJ_ERR_BAD_SHAPE;   // the running max assumes a non-negative scale
  if (batch == 0) return NVJ_OK;
  if (!q || !k_cache || !v_cache || !context_lens || !out) return NVJ_ERR_NULL_POINTER;
  if (max_blocks > 0 && !block_tables) return NVJ_ERR_NULL_POINTER;
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_cache) |
       reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(out) |
       (whole ? 0 : reinterpret_cast<uintptr_t>(workspace))) & 15u)   // unused in whole mode
    return NVJ_ERR_ALIGNMENT;
  // the vector-ALU measurement variant exists for one shape family only
  const bool valu = (phases & NVJ_PHASE_VALU_PRODUCTS) != 0;
  if (valu && (head_dim != 128 || f16 || kv_rep != 1 || (group != 4 && group != 8) ||
               num_kv_heads % 8 != 0 || chunk > 0))
    return NVJ_ERR_UNSUPPORTED;
  // the loads-only measurement variant: head_dim 128, bf16, not with a fixed chunk
  const bool loads_only = (phases & NVJ_PHASE_LOADS_ONLY) != 0;
  if (loads_only && (valu || head_dim != 128 || f16 || chunk > 0)) return NVJ_ERR_UNSUPPORTED;
  hipStream_t s = static_cast<hipStream_t>(stream);

  DecodeArgs a;
  a.q = static_cast<const uint4*>(q);
  a.k_cache = static_cast<const char*>(k_cache);
  a.v_cache = static_cast<const char*>(v_cache);
  a.block_tables = block_tables;
  a.context_lens = context_lens;
  a.out = static_cast<uint4*>(out);
  a.part_o = nullptr;
  a.part_ml = nullptr;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.group = group;
  a.kv_rep = kv_rep;
  a.cache_kv_heads = cache_kv_heads;
  a.block_size = block_size;
  a.page = nvj::Divisor(block_size);
  a.max_blocks = max_blocks;
  a.num_blocks = num_blocks;
  a.scale_log2e = scale * kLog2e;

  // Short rows: a workgroup per (sequence, KV head) or several, if the CUs and the lengths
  // a wave keeps allow it.  Where the table itself rules longer rows out, no length needs to
  // be looked at and the kernel without a split does it (64 / 256 / 512 positions 5.2 / 5.8
  // / 7.5 us); else small launches go by pieces, and in others the balanced kernel
  // decides on the device.
  const int64_t all_rows = (int64_t)batch * num_kv_heads;
  const int64_t cus = chunk == 0 && (phases & NVJ_PHASE_SHORT_ROWS) &&
                              !(phases & NVJ_PHASE_SHARED_ROWS) && batch <= kKeptSequences
                          ? compute_units()
                          : 0;
  const int short_rows = all_rows <= cus ? (int)all_rows : 0;
  const int64_t positions = (int64_t)max_blocks * block_size;
  const bool by_pieces = short_rows > 0 && !valu && !loads_only &&
                         pieces_take(batch, head_dim, all_rows, positions, cus);
  const bool all_short = short_rows > 0 && table_of_short_rows(all_rows, positions, by_pieces) &&
                         !(phases & NVJ_PHASE_CLEAR_COUNTERS);
  if ((whole || all_short) && max_blocks > 0) {
    if (all_rows > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
    if (!(phases & NVJ_PHASE_SPLITK)) return NVJ_OK;   // there is no second pass
    const int hpw = all_short ? 1 : heads_per_workgroup(batch, num_kv_heads);
    dim3 grid;
    const dim3 block(512);
    const NewRows fresh = rows_behind(new_rows, batch * (num_kv_heads / hpw), batch, &grid);
    hipError_t rc;
#define NVJ_LAUNCH_WHOLE(...) \
  rc = nvj::launch(paged_decode_whole_kernel<8, __VA_ARGS__>, grid, block, s, a, hpw,     \
                   nvj::Divisor(num_kv_heads / hpw), fresh, batch)
    if (new_rows && f16) NVJ_LAUNCH_WHOLE(128, true, 0, true);
    else if (new_rows) NVJ_LAUNCH_WHOLE(128, false, 0, true);
    else if (loads_only) NVJ_LAUNCH_WHOLE(128, false, -1);
    else if (valu && group == 4) NVJ_LAUNCH_WHOLE(128, false, 4);
    else if (valu) NVJ_LAUNCH_WHOLE(128, false, 8);
    else if (head_dim == 128 && !f16) NVJ_LAUNCH_WHOLE(128, false);
    else if (head_dim == 128) NVJ_LAUNCH_WHOLE(128, true);
    else if (!f16) NVJ_LAUNCH_WHOLE(64, false);
    else NVJ_LAUNCH_WHOLE(64, true);
#undef NVJ_LAUNCH_WHOLE
    return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
  }

  WorkspacePlan plan = {0, 1, 0, 0, 0, 0, 0, 0, 0};
  if (max_blocks > 0) {
    if (!plan_workspace(batch, num_heads, head_dim, max_blocks, block_size, num_kv_heads, chunk,
                        &plan))
      return NVJ_ERR_BAD_SHAPE;
    const size_t header = ext_counters ? 0 : plan.counter_bytes;
    if (!workspace || workspace_bytes < plan.bytes - plan.counter_bytes + header)
      return NVJ_ERR_WORKSPACE;
    int32_t* counters = ext_counters ? ext_counters : static_cast<int32_t*>(workspace);
    a.part_o = reinterpret_cast<float*>(static_cast<char*>(workspace) + header);
    a.part_ml = a.part_o + plan.records * head_dim;

    if (chunk == 0) {
      // one launch: the workgroup that completes a sequence merges it
      if (phases & NVJ_PHASE_CLEAR_COUNTERS) {
        const int n = (int)(plan.counter_bytes / sizeof(int32_t));   // stale flag, counters, padding
        if (nvj::launch(zero_int32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), s,
                        counters, n) != hipSuccess)
          return NVJ_ERR_LAUNCH;
      }
      if (!(phases & NVJ_PHASE_SPLITK)) return NVJ_OK;
      dim3 grid;
      if (by_pieces) {
        const int64_t per_row =
            (positions + kShortestPiece * kStep - 1) / (kShortestPiece * kStep);
        const int most = (int)std::min<int64_t>(batch * per_row, cus / num_kv_heads);
        const NewRows fresh = rows_behind(new_rows, most * num_kv_heads, batch, &grid);
        hipError_t rc;
#define NVJ_LAUNCH_PIECES(...)                                                                \
  rc = nvj::launch(paged_decode_pieces_kernel<__VA_ARGS__>, grid, dim3(512), s, a, batch,     \
                   most, counters, fresh)
        if (new_rows && f16) NVJ_LAUNCH_PIECES(true, true);
        else if (new_rows) NVJ_LAUNCH_PIECES(false, true);
        else if (f16) NVJ_LAUNCH_PIECES(true, false);
        else NVJ_LAUNCH_PIECES(false, false);
#undef NVJ_LAUNCH_PIECES
        return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
      }
      if (!new_rows && short_rows == 0 && head_dim == 128 && !valu && !loads_only && batch <= 64 &&
          (plan.wr_hpw == 0 || (phases & NVJ_PHASE_SHARED_ROWS))) {
        // nothing but the equal cut on offer
        const nvj::ReadAhead more = ahead ? *ahead : nvj::ReadAhead{};
        const dim3 shared_grid((unsigned)plan.num_wgs + more.chunks());
        hipError_t rc;
#define NVJ_LAUNCH_SHARED(N)                                                                   \
  rc = f16 ? nvj::launch(paged_decode_shared_kernel<true, N>, shared_grid, dim3(512), s, a,     \
                         batch, plan.num_wgs, kMinBalancedSteps, plan.shift, counters, more)   \
           : nvj::launch(paged_decode_shared_kernel<false, N>, shared_grid, dim3(512), s, a,    \
                         batch, plan.num_wgs, kMinBalancedSteps, plan.shift, counters, more)
        if (plan.hpw == 1) NVJ_LAUNCH_SHARED(1);
        else if (plan.hpw == 2) NVJ_LAUNCH_SHARED(2);
        else NVJ_LAUNCH_SHARED(4);
#undef NVJ_LAUNCH_SHARED
        return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
      }
      const NewRows fresh =
          rows_behind(new_rows, short_rows > plan.num_wgs ? short_rows : plan.num_wgs, batch, &grid);
      hipError_t rc;
#define NVJ_LAUNCH_BALANCED(...)                                                               \
  rc = nvj::launch(paged_decode_balanced_kernel<__VA_ARGS__>, grid, dim3(512), s, a, batch,   \
                   plan.num_wgs, kMinBalancedSteps, plan.hpw,                      \
                   (phases & NVJ_PHASE_SHARED_ROWS) ? 0 : plan.wr_hpw, plan.wr_hpw_alt,       \
                   kWholeRowTolerance, plan.shift, short_rows, counters, fresh)
      if (new_rows && f16) NVJ_LAUNCH_BALANCED(128, true, 0, true);
      else if (new_rows) NVJ_LAUNCH_BALANCED(128, false, 0, true);
      else if (loads_only) NVJ_LAUNCH_BALANCED(128, false, -1);
      else if (valu && group == 4) NVJ_LAUNCH_BALANCED(128, false, 4);
      else if (valu) NVJ_LAUNCH_BALANCED(128, false, 8);
      else if (head_dim == 128 && !f16) NVJ_LAUNCH_BALANCED(128, false, 0);
      else if (head_dim == 128) NVJ_LAUNCH_BALANCED(128, true, 0);
      else if (!f16) NVJ_LAUNCH_BALANCED(64, false, 0);
      else NVJ_LAUNCH_BALANCED(64, true, 0);
#undef NVJ_LAUNCH_BALANCED
      return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
    }

    if (phases & NVJ_PHASE_SPLITK) {
      const int nw = waves_per_workgroup(num_kv_heads);
      const dim3 grid((unsigned)(batch * plan.max_chunks), (unsigned)(num_kv_heads / nw));
      // one instantiation per (waves per workgroup, head_dim, element type)
      hipError_t rc;
#define NVJ_LAUNCH_FIXED(NWV, DV)                                                              \
  rc = f16 ? nvj::launch(paged_decode_splitk_kernel<NWV, DV, true>, grid, dim3(NWV * 64), s, a, \
                         chunk, plan.max_chunks)                                               \
           : nvj::launch(paged_decode_splitk_kernel<NWV, DV, false>, grid, dim3(NWV * 64), s, a, \
                         chunk, plan.max_chunks)
      switch (nw * 1000 + head_dim) {
        case 8128: NVJ_LAUNCH_FIXED(8, 128); break;
        case 4128: NVJ_LAUNCH_FIXED(4, 128); break;
        case 2128: NVJ_LAUNCH_FIXED(2, 128); break;
        case 1128: NVJ_LAUNCH_FIXED(1, 128); break;
        case 8064: NVJ_LAUNCH_FIXED(8, 64); break;
        case 4064: NVJ_LAUNCH_FIXED(4, 64); break;
        case 2064: NVJ_LAUNCH_FIXED(2, 64); break;
        default: NVJ_LAUNCH_FIXED(1, 64); break;
      }
#undef NVJ_LAUNCH_FIXED
      if (rc != hipSuccess) return NVJ_ERR_LAUNCH;
    }
  } else {
    chunk = kStep;  // no pages at all: every sequence is empty, the second pass writes zeros
  }
  if (!(phases & NVJ_PHASE_COMBINE)) return NVJ_OK;
  const hipError_t rc = nvj::launch(
      paged_decode_combine_kernel, dim3((unsigned)batch, (unsigned)num_heads), dim3(head_dim), s,
      a.part_o, a.part_ml, context_lens, static_cast<uint16_t*>(out), num_heads, chunk,
      plan.max_chunks, max_blocks * block_size, a.scale_log2e, f16);
  return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
}

}  // namespace

extern "C" int nvj_paged_decode_launch_phases(void* stream, const void* q, const void* k_cache,
                                              const void* v_cache, const int32_t* block_tables,
                                              const int32_t* context_lens, void* out,
                                              void* workspace, size_t workspace_bytes,
                                              int32_t batch, int32_t num_heads,
                                              int32_t num_kv_heads, int32_t head_dim,
                                              int32_t block_size, int32_t max_blocks,
                                              int32_t num_blocks, float scale, int32_t chunk,
                                              int32_t dtype, uint32_t phases) {
  return launch_decode(stream, q, k_cache, v_cache, block_tables, context_lens, out, workspace,
                       workspace_bytes, nullptr, batch, num_heads, num_kv_heads, head_dim,
                       block_size, max_blocks, num_blocks, scale, chunk, dtype, phases);
}

extern "C" size_t nvj_paged_decode_counter_bytes(int32_t batch, int32_t num_heads,
                                                 int32_t num_kv_heads) {
  if (batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0) return 0;
  const size_t heads =
      (size_t)num_kv_heads * virtual_heads_per_cache_head(num_heads / num_kv_heads);
  return counter_region_bytes(batch, (int64_t)heads);
}

extern "C" int nvj_paged_decode_launch(void* stream, const void* q, const void* k_cache,
                                       const void* v_cache, const int32_t* block_tables,
                                       const int32_t* context_lens, void* out, void* workspace,
                                       size_t workspace_bytes, int32_t batch, int32_t num_heads,
                                       int32_t num_kv_heads, int32_t head_dim,
                                       int32_t block_size, int32_t max_blocks,
                                       int32_t num_blocks, float scale, int32_t chunk,
                                       int32_t dtype) {
  return nvj_paged_decode_launch_phases(stream, q, k_cache, v_cache, block_tables, context_lens,
                                        out, workspace, workspace_bytes, batch, num_heads,
                                        num_kv_heads, head_dim, block_size, max_blocks,
                                        num_blocks, scale, chunk, dtype,
                                        NVJ_PHASE_SPLITK | NVJ_PHASE_COMBINE |
                                            NVJ_PHASE_CLEAR_COUNTERS);
}

// ---------------------------------------------------------------------------
// The library's own device array.  Its first kCounterRegion bytes are a counter
// region of the balanced split that belongs to no caller (the same words
// whatever the shape of a call: zero when the library is loaded, put back to
// zero by every launch); the rest is the workspace of the entry point that
// allocates nothing.  The array's name is a host-side stand-in; its device
// address is looked up once per device (hipGetSymbolAddress) and only that
// address is ever handed to a kernel.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[NVJ_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
constexpr size_t kCounterRegion = 64u << 10;
std::atomic<void*> g_scratch_ptr[kMaxDevices];   // per device: address of its copy of `scratch`

// Device address of the current device's copy of `scratch`.
int static_scratch_of_current_device(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return NVJ_ERR_LAUNCH;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    // every thread that races here gets the same address from the runtime
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr)
      return NVJ_ERR_LAUNCH;
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return NVJ_OK;
}
}  // namespace

extern "C" int nvj_paged_decode_library_counters(void** counters, size_t* bytes) {
  if (!counters) return NVJ_ERR_NULL_POINTER;
  if (bytes) *bytes = kCounterRegion;
  return static_scratch_of_current_device(counters);
}

extern "C" int nvj_paged_decode_counters_reset(void* stream, void* counters,
                                               size_t counter_bytes) {
  if (!counters) {
    const int rc = static_scratch_of_current_device(&counters);
    if (rc != NVJ_OK) return rc;
    counter_bytes = kCounterRegion;
  }
  if (reinterpret_cast<uintptr_t>(counters) & 3u) return NVJ_ERR_ALIGNMENT;
  if (counter_bytes / sizeof(int32_t) > (size_t)INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  const int n = (int)(counter_bytes / sizeof(int32_t));
  if (n == 0) return NVJ_OK;
  return nvj::launch(zero_int32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256),
                     static_cast<hipStream_t>(stream), static_cast<int32_t*>(counters),
                     n) == hipSuccess
             ? NVJ_OK
             : NVJ_ERR_LAUNCH;
}

// Counters of the store-and-attend calls that bring none, on the null stream only: its
// launches follow each other, and it is never recorded into a graph that another stream
// replays.  Two regions that such calls use in turn: each launch also zeroes the region of
// the next one, so that a call begins on cleared counters without a clearing launch in front
// of it, and a count left wrong by one launch (lengths rewritten under it, say) ends with it.
static __device__ __align__(256) int32_t null_stream_counters[2][kNullStreamWords];

namespace {
struct NullStreamCounters {
  std::mutex lock;   // held over a launch: the order of the launches is the order of the turns
  int32_t* base = nullptr;
  int next = 0;      // the region of the next launch
};
// Of the current device; null if there is none.
NullStreamCounters* null_stream_counters_of_current_device() {
  static NullStreamCounters of_device[kMaxDevices];
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  return &of_device[dev];
}
// With the lock held.
bool find_base(NullStreamCounters* c) {
  void* p = nullptr;
  if (c->base == nullptr) {
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(null_stream_counters)) != hipSuccess) return false;
    c->base = static_cast<int32_t*>(p);
  }
  return c->base != nullptr;
}
}  // namespace

extern "C" int nvj_paged_decode_null_stream_counters(void** counters, size_t* bytes) {
  if (!counters) return NVJ_ERR_NULL_POINTER;
  if (bytes) *bytes = kNullStreamWords * sizeof(int32_t);
  NullStreamCounters* c = null_stream_counters_of_current_device();
  if (!c) return NVJ_ERR_LAUNCH;
  std::lock_guard<std::mutex> hold(c->lock);
  if (!find_base(c)) return NVJ_ERR_LAUNCH;
  *counters = c->base + (1 - c->next) * kNullStreamWords;
  return NVJ_OK;
}

int nvj::paged_decode_launch_ahead(void* stream, const void* q, const void* k_cache,
                                                const void* v_cache, const int32_t* block_tables,
                                                const int32_t* context_lens, void* out,
                                                void* partials, size_t partial_bytes,
                                                void* counters, size_t counter_bytes,
                                                int32_t batch, int32_t num_heads,
                                                int32_t num_kv_heads, int32_t head_dim,
                                                int32_t block_size, int32_t max_blocks,
                                                int32_t num_blocks, float scale, int32_t dtype,
                                                uint32_t phases, const ReadAhead* ahead) {
  if (batch > 0 && max_blocks > 0) {
    const size_t need = nvj_paged_decode_counter_bytes(batch, num_heads, num_kv_heads);
    if (!counters) {
      // need == 0: invalid arguments, which the launch below reports by name
      if (need > kCounterRegion) return NVJ_ERR_SCRATCH_LIMIT;
      if (need > 0) {
        const int rc = static_scratch_of_current_device(&counters);
        if (rc != NVJ_OK) return rc;
      }
    } else {
      if (reinterpret_cast<uintptr_t>(counters) & 3u) return NVJ_ERR_ALIGNMENT;
      if (need > 0 && counter_bytes < need) return NVJ_ERR_WORKSPACE;
    }
  }
  return launch_decode(stream, q, k_cache, v_cache, block_tables, context_lens, out, partials,
                       partial_bytes, static_cast<int32_t*>(counters), batch, num_heads,
                       num_kv_heads, head_dim, block_size, max_blocks, num_blocks, scale, 0, dtype,
                       phases, nullptr, ahead);
}

extern "C" int nvj_paged_decode_launch_counters(void* stream, const void* q, const void* k_cache,
                                                const void* v_cache, const int32_t* block_tables,
                                                const int32_t* context_lens, void* out,
                                                void* partials, size_t partial_bytes,
                                                void* counters, size_t counter_bytes,
                                                int32_t batch, int32_t num_heads,
                                                int32_t num_kv_heads, int32_t head_dim,
                                                int32_t block_size, int32_t max_blocks,
                                                int32_t num_blocks, float scale, int32_t dtype,
                                                uint32_t phases) {
  return nvj::paged_decode_launch_ahead(stream, q, k_cache, v_cache, block_tables, context_lens,
                                        out, partials, partial_bytes, counters, counter_bytes,
                                        batch, num_heads, num_kv_heads, head_dim, block_size,
                                        max_blocks, num_blocks, scale, dtype, phases, nullptr);
}

// Up to one (sequence, KV head) per CU.  With more, the comparison in every step costs the
// stream as much as the store kernel in front of it: 1 / 8 / 16 sequences of 8 KV heads
// (700, 128 .. 2048, 32768 positions) take 12.3 / 16.1 / 319.1 us instead of 13.6 / 17.2 /
// 321.6, 64 of 4096 159.8 instead of 158.6.  The length sets no line: over 1 .. 64 sequences
// of 1024 .. 32768 positions, 2 / 8 / 32 KV heads, up to one row per CU, one launch is 0.5 ..
// 2.0 us less than two, at the longest even (32 of 16384 321.9 / 321.7).
extern "C" int32_t nvj_paged_decode_store_takes(int32_t batch, int32_t num_heads,
                                                int32_t num_kv_heads, int32_t head_dim,
                                                int32_t block_size, int32_t max_blocks,
                                                int32_t num_blocks, int32_t chunk) {
  if (batch <= 0 || batch > kMaxNewRows || head_dim != 128 || max_blocks <= 0 || block_size <= 0 ||
      num_blocks <= 0 || num_kv_heads <= 0 || num_heads <= 0 || num_heads % num_kv_heads != 0 ||
      (int64_t)num_blocks * block_size > INT32_MAX)
    return 0;
  const int64_t rows =
      (int64_t)batch * num_kv_heads * virtual_heads_per_cache_head(num_heads / num_kv_heads);
  const int64_t cus = compute_units();
  if (rows > cus) return 0;
  if (chunk == NVJ_CHUNK_WHOLE_SEQUENCE) return 1;
  if (chunk != 0 || nvj_paged_decode_counter_bytes(batch, num_heads, num_kv_heads) >
                        kNullStreamWords * sizeof(int32_t))
    return 0;
  const int64_t positions = (int64_t)max_blocks * block_size;
  return table_of_short_rows(rows, positions, pieces_take(batch, head_dim, rows, positions, cus)) ? 1
                                                                                                  : 2;
}

extern "C" int nvj_paged_decode_store_launch(
    void* stream, const void* q, const void* key, const void* value, const int32_t* slot_mapping,
    void* k_cache, void* v_cache, const int32_t* block_tables, const int32_t* context_lens,
    void* out, void* partials, size_t partial_bytes, void* counters, size_t counter_bytes,
    int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
    int32_t max_blocks, int32_t num_blocks, float scale, int32_t chunk, int32_t dtype,
    int32_t k_dtype, int32_t v_dtype) {
  const int takes = nvj_paged_decode_store_takes(batch, num_heads, num_kv_heads, head_dim,
                                                 block_size, max_blocks, num_blocks, chunk);
  if (takes == 0) return NVJ_ERR_UNSUPPORTED;
  if ((k_dtype != dtype && k_dtype != NVJ_DTYPE_F32) || (v_dtype != dtype && v_dtype != NVJ_DTYPE_F32))
    return NVJ_ERR_BAD_DTYPE;
  if (!key || !value || !slot_mapping) return NVJ_ERR_NULL_POINTER;
  if ((reinterpret_cast<uintptr_t>(key) | reinterpret_cast<uintptr_t>(value)) & 15u)
    return NVJ_ERR_ALIGNMENT;
  NewRows n = {};
  NullStreamCounters* own = nullptr;
  std::unique_lock<std::mutex> turn;
  if (takes == 2) {
    if (!counters && stream) return NVJ_ERR_NULL_POINTER;
    if (!counters) {
      own = null_stream_counters_of_current_device();
      if (!own) return NVJ_ERR_LAUNCH;
      turn = std::unique_lock<std::mutex>(own->lock);
      if (!find_base(own)) return NVJ_ERR_LAUNCH;
      counters = own->base + own->next * kNullStreamWords;
      n.clear = own->base + (1 - own->next) * kNullStreamWords;
    } else {
      if (reinterpret_cast<uintptr_t>(counters) & 3u) return NVJ_ERR_ALIGNMENT;
      if (counter_bytes < nvj_paged_decode_counter_bytes(batch, num_heads, num_kv_heads))
        return NVJ_ERR_WORKSPACE;
    }
  }
  n.key = key;
  n.value = value;
  n.slots = slot_mapping;
  n.num_slots = num_blocks * block_size;
  n.key_f32 = k_dtype == NVJ_DTYPE_F32;
  n.value_f32 = v_dtype == NVJ_DTYPE_F32;
  const int rc = launch_decode(
      stream, q, k_cache, v_cache, block_tables, context_lens, out, partials, partial_bytes,
      static_cast<int32_t*>(counters), batch, num_heads, num_kv_heads, head_dim, block_size,
      max_blocks, num_blocks, scale, chunk, dtype,
      NVJ_PHASE_SPLITK | NVJ_PHASE_COMBINE | NVJ_PHASE_SHORT_ROWS, &n);
  if (own && rc == NVJ_OK) own->next = 1 - own->next;   // (an error has launched nothing)
  return rc;
}

extern "C" int nvj_paged_decode_static_launch(void* stream, const void* q, const void* k_cache,
                                              const void* v_cache, const int32_t* block_tables,
                                              const int32_t* context_lens, void* out,
                                              int32_t batch, int32_t num_heads,
                                              int32_t num_kv_heads, int32_t head_dim,
                                              int32_t block_size, int32_t max_blocks,
                                              int32_t num_blocks, float scale, int32_t dtype) {
  void* base = nullptr;
  if (batch > 0 && max_blocks > 0) {
    const size_t need = nvj_paged_decode_workspace_bytes(batch, num_heads, head_dim, max_blocks,
                                                         block_size, num_kv_heads, 0);
    const size_t counters = nvj_paged_decode_counter_bytes(batch, num_heads, num_kv_heads);
    // need == 0: invalid arguments, which the launch below reports by name
    if (need > 0 && (counters > kCounterRegion ||
                     need - counters > NVJ_STATIC_SCRATCH_BYTES - kCounterRegion))
      return NVJ_ERR_SCRATCH_LIMIT;
    if (need > 0) {
      const int rc = static_scratch_of_current_device(&base);
      if (rc != NVJ_OK) return rc;
    }
  }
  char* partials = base ? static_cast<char*>(base) + kCounterRegion : nullptr;
  return launch_decode(stream, q, k_cache, v_cache, block_tables, context_lens, out, partials,
                       base ? (size_t)NVJ_STATIC_SCRATCH_BYTES - kCounterRegion : 0,
                       static_cast<int32_t*>(base), batch, num_heads, num_kv_heads, head_dim,
                       block_size, max_blocks, num_blocks, scale, 0, dtype,
                       NVJ_PHASE_SPLITK | NVJ_PHASE_COMBINE);
}

extern "C" const char* nvj_error_string(int code) {
  switch (code) {
    case NVJ_OK: return "ok";
    case NVJ_ERR_NULL_POINTER: return "a required pointer is NULL";
    case NVJ_ERR_BAD_SHAPE: return "invalid shape or size argument";
    case NVJ_ERR_UNSUPPORTED: return "unsupported head_dim / group size / block size / chunk";
    case NVJ_ERR_WORKSPACE: return "workspace missing or too small";
    case NVJ_ERR_ALIGNMENT: return "a pointer is not 16-byte aligned";
    case NVJ_ERR_LAUNCH: return "kernel launch failed";
    case NVJ_ERR_BAD_DTYPE: return "unknown element type code";
    case NVJ_ERR_SCRATCH_LIMIT:
      return "problem needs more than the library's static scratch (NVJ_STATIC_SCRATCH_BYTES)";
    default: return "unknown error code";
  }
}

extern "C" int nvj_abi_version(void) { return NVJ_ABI_VERSION; }
