// Variable-length causal prefill attention for gfx950 (CDNA4, wave64).
//
// Stands in for variable_length_attention_prefill (layers/attention.py:135-279
// of the reference) as called from Attention._prefill_attention (:331-364): q,
// k, v are the packed rows of the prompts being prefilled, sequence i owning q
// rows [cu_q[i], cu_q[i+1]) and k/v rows [cu_k[i], cu_k[i+1]).  Query position
// p of a sequence attends key positions <= p of the same sequence (the
// reference's mask `q_pos >= k_pos`, both counted from the start of the
// sequence, :232-243).  GQA maps query head h to kv head h / G.  Nothing is
// padded and nothing of size max_len^2 is materialised.
//
// MFMA-bound.  One workgroup = 4 waves = 8 column groups of one (sequence, kv head),
// a column group being 16 consecutive tokens of one query head (16 MFMA columns);
// the groups of a sequence are numbered head first, so a workgroup takes 128 / G
// tokens with all G heads that share their K/V, and a wave two column groups.  (128
// tokens of one query head did about as well for long prompts, 1051 against 1011 us
// for 8 x 4096, but a prompt of 30 tokens then fills a quarter of the columns, and
// a tile walks keys that its first tokens do not see: 128 prompts of 16..300
// tokens 177 against 134 us.)  Keys are walked 32 at a time.  The K rows and the V rows of a tile go from global memory
// straight into LDS (global_load_lds_dwordx4: no staging registers, no LDS
// write instructions), row-major with the 16-byte pieces of a row permuted so
// that the reads below are free of bank conflicts, in rings of 4 tiles each,
// fetched two tiles ahead; one barrier per tile:
//   * K is read back with ds_read_b128 as the A operand of
//     S^T[key, q] = K . Q^T  (v_mfma_f32_16x16x32_bf16, Q^T of both groups in
//     registers for the whole tile);
//   * V is read back with the transposing LDS read (ds_read_b64_tr_b16), which
//     hands each lane four keys of one head dimension: the A operand of
//     O^T[dim, q] += V^T . P^T.
// Softmax is the fp32 online form on the accumulator layout; P^T comes out of
// the S^T accumulators already in B-operand layout (same reduction-slot <-> key
// map as the decode kernel).  Only tiles that touch the diagonal are masked.
// The loop is software-pipelined: the scores of tile i are issued to the matrix
// core, then tile i-1 is accumulated while the vector ALU turns the scores of
// tile i into probabilities.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "bf16.h"
#include "device.h"
#include "divisor.h"
#include "launch.h"
#include "lds_copy.h"
#include "nvj_paged_attn.h"
#include "past_l2.h"
#include "wave_ops.h"

namespace {

using nvj::bf16x8;
using nvj::Divisor;
using nvj::f16x8;
using nvj::f32x4;
using nvj::store_past_l2;
using nvj::wave_combine;
using nvj::wave_inclusive_scan;   // (with shuffles the sequence lookup took 5 us of a short prompt)
using nvj::wave_max;

constexpr int kD = 128;
constexpr int kPieces = 16;          // 16-byte pieces per (position, head) row
// NG: column groups of 16 query rows per wave.  2 x 4 waves (128 query rows, two
// workgroups per CU) measured fastest: 4 groups x 4 waves (one wave per SIMD,
// accumulators in AGPRs) and 8-wave workgroups (1 or 2 groups) were 5-20 % slower.
// 1 x 4 waves for launches too small to give every CU a workgroup of 2 x 4.
constexpr int kWaves = 4;
constexpr int kKeys = 32;            // keys per step
constexpr int kTileBytes = kKeys * kD * 2;   // one K or V tile in LDS: 32 rows of 256 bytes
// RING: tiles of K and of V in LDS.  4, tile t in slot t % 4: iteration i reads K of tile i and
// V of tile i-1 while tiles i+1 (landing) and i+2 (just issued) are on their way.
// A ring of 3 would do for K; 4 makes the slot of every tile of an iteration a
// function of i % 4, so that a loop unrolled 4 times has every LDS offset as an
// instruction immediate.
// 3, fetched one tile ahead, with one column group per wave: three workgroups to a CU, for prompts
// whose workgroups have little but their head and tail (tile_form).
constexpr float kNegBig = -1.0e30f;
constexpr int kShortestPart = 8;     // tiles, a multiple of the ring's 4 (the last part may be shorter)
constexpr float kLazyLog2 = 8.0f;    // running max moves only for gains above 2^8
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// The element type of q, k, v and out: bf16 (F16 = false) or IEEE half.  The
// kernel moves 16-bit patterns (held as bf16x8 whatever they mean); only the
// matrix instruction, the rounding of probabilities and output and the
// constant 1 depend on the type.
template <bool F16> struct Elem;
template <> struct Elem<false> {
  static constexpr uint32_t kOnes = 0x3F803F80u;   // two bf16 ones
  static __device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    return nvj::pack2_bf16(lo, hi);
  }
};
template <> struct Elem<true> {
  static constexpr uint32_t kOnes = 0x3C003C00u;   // two half ones
  static __device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    return nvj::pack2_f16(lo, hi);
  }
};

typedef const __attribute__((address_space(4))) int32_t* const_i32_ptr;

// reduction slot j of key group kg stands for this key of the 32-key step
__device__ __forceinline__ int slot_key(int kg, int j) {
  return j < 4 ? 4 * kg + j : 16 + 4 * kg + (j - 4);
}

typedef __attribute__((address_space(3))) char* lds_ptr;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

// LDS layout of a tile: row R (key R of the tile) at byte 256 * R, its 16-byte
// piece p at position p ^ (R & 15) for K and p ^ (2 * (R & 7)) for V.
//   K read (ds_read_b128): the 16 lanes of a key group read one piece of 16
//     different rows -> 16 different positions.
//   V read (ds_read_b64_tr_b16): the 16 lanes of a key group read four 8-byte
//     chunks of each of 4 rows -> 16 different 8-byte slots modulo 128 bytes.
__device__ __forceinline__ int k_position(int row, int piece) { return piece ^ (row & 15); }
__device__ __forceinline__ int v_position(int row, int piece) { return piece ^ (2 * (row & 7)); }

using nvj::copy16_to_lds;   // waits: wait_tiles_in_flight

// Cooperative tile copies of a workgroup.  A tile is 512 pieces of K and 512 of
// V; each wave copies its share of the rows of both (8 rows with 4 waves), 4
// rows = 1024 contiguous LDS bytes per instruction.  Lane l of instruction j of
// wave w writes position l % 16 of row 8w + 4j + l / 16 and fetches the piece
// that belongs there.  Rows are clamped to the last visible key, so nothing at or beyond
// k_end is read.
constexpr int kCopyRowsPerWave = kKeys / kWaves;   // rows of a tile one wave copies
static_assert(kCopyRowsPerWave % 4 == 0, "one copy instruction covers 4 rows");
// Packed rows: key s of the sequence is row s behind k_head / v_head.  Paged
// (PAGED): k_head / v_head point at this kv head inside row 0 of the caches and
// key s is row table[s / block_size] * block_size + s % block_size; a tile of 32
// keys never leaves its page (block_size is a multiple of 32), so one scalar
// table lookup per tile gives the base and the lanes keep their row offsets.
template <bool PAGED>
struct TileCopier {
  const char* k_head;   // first key row of the sequence for this kv head
  const char* v_head;
  uint32_t row_bytes;   // bytes between consecutive keys; < 2^24 (checked by the host)
  uint32_t k_lds, v_lds;   // LDS byte addresses of the two rings
  int last_key, last_tile, wave, lane;
  const_i32_ptr table;  // PAGED: this sequence's row of the block tables
  Divisor page;         // block_size
  int num_blocks;
  int entry;            // PAGED: the table's entry for the next tile

  // Asks for the entry of the tile to come, so that its way is behind a tile's work (with that and
  // without a division per tile, us: 16 of 30..600 behind 100..5000 211 -> 209, 1 of 500 behind 5000
  // 83.6 -> 80.4, of 4000 behind 4000 343 -> 338, 8 of 30..200 behind 500..4000 65.6 -> 63.3).
  __device__ __forceinline__ void look_up(int tile) {
    if (PAGED) entry = table[page.divide(min(tile, last_tile) * kKeys)];
  }
  __device__ __forceinline__ size_t first_row_of(int tile) {
    const int ks = tile * kKeys;
    if (!PAGED) return (size_t)ks;
    const int phys = min(max(entry, 0), num_blocks - 1);
    look_up(tile + 1);
    return (size_t)phys * page.d + (ks - page.divide(ks) * page.d);
  }

  __device__ __forceinline__ void issue(int tile, int k_stage, int v_stage) {
    tile = min(tile, last_tile);   // past the end: fetch the last tile again (same instruction count)
    const int cap = last_key - tile * kKeys;   // >= 0: a tile starts at a visible key
    const size_t first_row = first_row_of(tile);
    const char* kb = k_head + first_row * row_bytes;
    const char* vb = v_head + first_row * row_bytes;
#pragma unroll
    for (int j = 0; j < kCopyRowsPerWave / 4; ++j) {
      const int row = kCopyRowsPerWave * wave + 4 * j + (lane >> 4);
      const uint32_t row_off = __umul24(min(row, cap), row_bytes);
      const uint32_t dst = (uint32_t)(kCopyRowsPerWave / 4 * wave + j) * 1024u;
      copy16_to_lds(kb, row_off + 16u * k_position(row, lane & 15),
                    k_lds + (uint32_t)k_stage * kTileBytes + dst);
      copy16_to_lds(vb, row_off + 16u * v_position(row, lane & 15),
                    v_lds + (uint32_t)v_stage * kTileBytes + dst);
    }
  }

  // The same for a tile all of whose 32 keys exist (tile < last_tile): the
  // lanes' offsets do not depend on the tile and are computed once (lane_offsets).
  __device__ __forceinline__ void lane_offsets(uint32_t (&koff)[kCopyRowsPerWave / 4],
                                               uint32_t (&voff)[kCopyRowsPerWave / 4]) const {
#pragma unroll
    for (int j = 0; j < kCopyRowsPerWave / 4; ++j) {
      const int row = kCopyRowsPerWave * wave + 4 * j + (lane >> 4);
      const uint32_t row_off = __umul24(row, row_bytes);
      koff[j] = row_off + 16u * k_position(row, lane & 15);
      voff[j] = row_off + 16u * v_position(row, lane & 15);
    }
  }
  template <int STAGE>
  __device__ __forceinline__ void issue_full(int tile, const uint32_t (&koff)[kCopyRowsPerWave / 4],
                                             const uint32_t (&voff)[kCopyRowsPerWave / 4]) {
    const size_t first_row = first_row_of(tile);
    const char* kb = k_head + first_row * row_bytes;
    const char* vb = v_head + first_row * row_bytes;
#pragma unroll
    for (int j = 0; j < kCopyRowsPerWave / 4; ++j) {
      const uint32_t dst = (uint32_t)(kCopyRowsPerWave / 4 * wave + j) * 1024u;
      copy16_to_lds(kb, koff[j], k_lds + (uint32_t)STAGE * kTileBytes + dst);
      copy16_to_lds(vb, voff[j], v_lds + (uint32_t)STAGE * kTileBytes + dst);
    }
  }
};
constexpr int kCopiesPerTile = 2 * (kCopyRowsPerWave / 4);   // copy16_to_lds calls of one lane per tile

// Blocks until at most `tiles` of this lane's most recent tile copies are still
// in flight (vmcnt counts the copies in order).
template <int TILES>
__device__ __forceinline__ void wait_tiles_in_flight() {
  static_assert(TILES == 0 || TILES == 1, "vmcnt immediates below");
  static_assert(kCopiesPerTile == 4 || kCopiesPerTile == 2, "vmcnt immediates below");
  if (TILES == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else if (kCopiesPerTile == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
}

// NaN-propagating maximum: one v_maximum3_f32 per three values, no
// canonicalising moves on MFMA results.
__device__ __forceinline__ float max2(float a, float b) {
  return __builtin_elementwise_maximum(a, b);
}
__device__ __forceinline__ float max_of8(const f32x4& a, const f32x4& b) {
  const float t1 = max2(max2(a[0], a[1]), a[2]);
  const float t2 = max2(max2(a[3], b[0]), b[1]);
  return max2(max2(max2(b[2], b[3]), t1), t2);
}

// S^T of one 32-key tile against both column groups (16 query rows each):
// sc[g][h] holds keys 16*h + 4*kg + e of the tile for query row r of group g.
// kaddr[s] is the lane's LDS address of its piece 4*s + kg of row r of ring slot
// 0 (k_read_addresses); `slot_bytes` selects the ring slot.
template <bool F16, int NG>
__device__ __forceinline__ void scores_of_tile(const lds_ptr (&kaddr)[4], int slot_bytes,
                                               const bf16x8 (&qreg)[NG][4],
                                               f32x4 (&sc)[NG][2]) {
  bf16x8 ka[2][4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    // rows r and 16 + r share a position: (16 + r) & 15 == r
    ka[0][s] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>(
        kaddr[s] + slot_bytes);
    ka[1][s] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>(
        kaddr[s] + slot_bytes + 16 * 256);
  }
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    sc[g][0] = sc[g][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      sc[g][0] = Elem<F16>::mfma(ka[0][s], qreg[g][s], sc[g][0]);
      sc[g][1] = Elem<F16>::mfma(ka[1][s], qreg[g][s], sc[g][1]);
    }
  }
}
__device__ __forceinline__ void k_read_addresses(lds_ptr k_lds, int r, int kg, lds_ptr (&kaddr)[4]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) kaddr[s] = k_lds + 256 * r + 16 * k_position(r, 4 * s + kg);
}

// O^T += V^T . P^T and l += 1 . P^T for the probabilities `pb` of one tile whose
// V rows are at `vt`.  Operand jd covers head dimensions 16*jd .. 16*jd + 15.
// ds_read_b64_tr_b16 works on groups of 16 lanes: source lane s = 4a + b of a
// group points at 4 consecutive bf16 (b selects which 4 of the 16 dimensions)
// of row a; result lane 4b + j receives, as element a, the j-th of those from
// source lane 4a + b.  With row a = key 4*kg + a of the tile (then 16 + 4*kg + a
// for the second read) lane i of the group ends up with keys of reduction
// slots 0..3 (then 4..7) of dimension 16*jd + i: the A operand.
// Every element of lacc[g] of a lane is the sum over all 32 keys of the tile for
// the lane's query row: a ones-row times P^T on the matrix core, from the same
// bf16 probabilities as the numerator.
// vaddr[jd] is the lane's LDS address for operand jd in ring slot 0
// (v_read_addresses); `slot_bytes` selects the ring slot.
template <bool F16, int NG>
__device__ __forceinline__ void accumulate_tile(const lds_ptr (&vaddr)[8], int slot_bytes,
                                                const bf16x8 (&pb)[NG],
                                                f32x4 (&acc)[NG][8], f32x4 (&lacc)[NG]) {
  bf16x8 va[8];
#pragma unroll
  for (int jd = 0; jd < 8; ++jd) {
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        reinterpret_cast<__attribute__((address_space(3))) bf16x4*>(vaddr[jd] + slot_bytes));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        reinterpret_cast<__attribute__((address_space(3))) bf16x4*>(vaddr[jd] + slot_bytes +
                                                                      16 * 256));
    va[jd] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  const uint32_t one2 = Elem<F16>::kOnes;
  const bf16x8 ones = as_bf16x8(make_uint4(one2, one2, one2, one2));
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    lacc[g] = Elem<F16>::mfma(ones, pb[g], lacc[g]);
#pragma unroll
    for (int jd = 0; jd < 8; ++jd)
      acc[g][jd] = Elem<F16>::mfma(va[jd], pb[g], acc[g][jd]);
  }
}
__device__ __forceinline__ void v_read_addresses(lds_ptr v_lds, int r, int kg, lds_ptr (&vaddr)[8]) {
  const int row = 4 * kg + (r >> 2);   // (16 + row) & 7 == row & 7: both reads share positions
  const int chunk = r & 3;             // 8-byte chunk of the 32 bytes of a dimension group
#pragma unroll
  for (int jd = 0; jd < 8; ++jd)
    vaddr[jd] = v_lds + 256 * row + 16 * v_position(row, 2 * jd + (chunk >> 1)) + 8 * (chunk & 1);
}

// Probabilities of one tile from its scores (fp32 online softmax on the
// accumulator layout), already in B-operand layout.
//   m_run[g]  reference point of the exponentials, mneg[g] = -m_run * sl2.
// MASK: entries beyond `row_limit + token[g]` (causal) or `key_limit` (end of the
// sequence), both relative to the first key of the tile, weigh exactly 0.
// Must run after the previous tile has been accumulated: moving the reference
// point rescales acc and lacc.
template <bool MASK, bool F16, int NG>
__device__ __forceinline__ void probabilities_of_tile(f32x4 (&sc)[NG][2], bf16x8 (&pb)[NG],
                                                      f32x4 (&acc)[NG][8], f32x4 (&lacc)[NG],
                                                      float (&m_run)[NG], float (&mneg)[NG],
                                                      float sl2, int kg, const int (&token)[NG],
                                                      int row_limit, int key_limit) {
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    f32x4& s0 = sc[g][0];
    f32x4& s1 = sc[g][1];
    // lane = (query row r of the group, key group kg): keys 4*kg + e and
    // 16 + 4*kg + e of the tile; `limit` = last key of the tile the row may see
    const int limit = MASK ? min(row_limit + token[g], key_limit) : 0;
    if (MASK) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (4 * kg + e > limit) s0[e] = kNegBig;
        if (16 + 4 * kg + e > limit) s1[e] = kNegBig;
      }
    }
    // Lazy running max: the reference point of the exponentials only moves
    // when some lane's maximum exceeds it by more than 2^kLazyLog2 (a
    // wave-uniform decision taken on each lane's own 8 keys, so most tiles need
    // neither a cross-lane reduction nor a rescale of O^T and l).
    // Probabilities may then exceed 1 (by at most that factor); the final O / l
    // is unchanged because both carry the same reference.
    float mx = max_of8(s0, s1);
    if (__any(fmaf(mx, sl2, mneg[g]) > kLazyLog2)) {
      mx = wave_combine<16>(mx, max2);
      mx = wave_combine<32>(mx, max2);
      const float m_new = max2(m_run[g], mx);
      const float alpha = __builtin_amdgcn_exp2f((m_run[g] - m_new) * sl2);
      m_run[g] = m_new;
      mneg[g] = -m_new * sl2;
      lacc[g] *= alpha;
#pragma unroll
      for (int jd = 0; jd < 8; ++jd) acc[g][jd] *= alpha;
    }
    float p0[4], p1[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p0[e] = __builtin_amdgcn_exp2f(fmaf(s0[e], sl2, mneg[g]));
      p1[e] = __builtin_amdgcn_exp2f(fmaf(s1[e], sl2, mneg[g]));
    }
    if (MASK) {
      // masked entries weigh exactly 0 whatever the scale and even for a row
      // whose reference point is still the initial one
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (4 * kg + e > limit) p0[e] = 0.f;
        if (16 + 4 * kg + e > limit) p1[e] = 0.f;
      }
    }
    uint4 pbits;
    pbits.x = Elem<F16>::pack2(p0[0], p0[1]);
    pbits.y = Elem<F16>::pack2(p0[2], p0[3]);
    pbits.z = Elem<F16>::pack2(p1[0], p1[1]);
    pbits.w = Elem<F16>::pack2(p1[2], p1[3]);
    pb[g] = as_bf16x8(pbits);
  }
}

struct PrefillArgs {
  const uint4* q;       // Tq rows of Hq * 16 pieces, q_stride pieces apart
  const uint4* k;       // Tk rows of Hkv * 16 pieces, kv_row_bytes apart
  const uint4* v;
  uint4* out;           // [Tq, Hq, 16] pieces
  const int32_t* cu_q;  // [B + 1]
  const int32_t* cu_k;  // [B + 1]; paged: the keys of a sequence, cached and new together
  int64_t q_stride;
  uint32_t kv_row_bytes;   // < 2^24 (checked by the host)
  int batch, num_heads, num_kv_heads;
  Divisor group;        // num_heads / num_kv_heads
  Divisor tiles;        // query tiles per KV head, at most
  float scale_log2e;
  // paged only: k and v are the caches [num_blocks, block_size, Hkv, 16] pieces
  const int32_t* block_tables;   // [B, max_blocks]
  Divisor page;         // block_size
  int max_blocks, num_blocks;
  // STORE: row t of k and v also goes to slot slots[t] of the caches
  const int32_t* slots;          // < 0 or >= num_slots: not stored
  uint4* k_cache;
  uint4* v_cache;
  int64_t num_slots;
  Divisor row_pieces;                // of a row
  uint32_t new_pieces, share_pieces; // of all rows, of a workgroup
  // SPLIT: the parts that the keys of a query tile may be cut into, and where those leave theirs
  Divisor splits;
  float* part_o;     // [workgroups of a part, splits, column group, 8, 64 lanes, 4]
  float2* part_ml;   // [workgroups of a part, splits, column group, 16 rows]: reference point, sum
};

// A workgroup's share of the new rows on their way into the caches.  The attention reads the
// packed rows and never the caches, so the store needs no place in front of it: a workgroup
// fetches two pieces of K and V per thread before its tiles and writes them behind, then what
// is left of its share.  The store's own launch takes 25 us for 156 MB; in here it hides under
// the tiles' round trips: 128 prompts of 16..300 tokens (32 / 8 heads) 143 -> 130 us, and 117
// with rows stored past the L2s (inputs of the call before; 140 -> 123 with fresh ones).
struct StoreShare {
  static constexpr uint32_t kBatch = 2 * kWaves * 64;
  uint32_t at, end;
  uint4 k0, k1, v0, v1;
  int slot0, slot1;

  // The share is counted from the end, as the tiles are walked: its rows are those that the
  // tiles of the same time read, and come out of a cache.  Whole heads, so that no two
  // workgroups write to one cache line (shares of 16 .. 64 pieces: 2 % of the launch).
  __device__ __forceinline__ StoreShare(const PrefillArgs& a) {
    const uint64_t from = (uint64_t)a.share_pieces * (gridDim.x - 1 - blockIdx.x);
    at = (uint32_t)min(from, (uint64_t)a.new_pieces);
    end = (uint32_t)min(from + a.share_pieces, (uint64_t)a.new_pieces);
    k0 = k1 = v0 = v1 = make_uint4(0u, 0u, 0u, 0u);
    slot0 = slot1 = -1;
  }
  __device__ __forceinline__ void fetch(const PrefillArgs& a) {
    if (at >= end) return;
    const uint32_t p0 = min(at + threadIdx.x, end - 1);   // (past the end: the last one again)
    const uint32_t p1 = min(at + threadIdx.x + kBatch / 2, end - 1);
    slot0 = a.slots[a.row_pieces.divide(p0)];
    slot1 = a.slots[a.row_pieces.divide(p1)];
    k0 = a.k[p0];
    v0 = a.v[p0];
    k1 = a.k[p1];
    v1 = a.v[p1];
  }
  static __device__ __forceinline__ int64_t place(const PrefillArgs& a, int slot, uint32_t p) {
    return (int64_t)slot * a.row_pieces.d + (p - a.row_pieces.divide(p) * a.row_pieces.d);
  }
  // (Nothing is stored past the end: hundreds of stores of one piece cost a workgroup with few
  // pieces 1 .. 2 us.)
  __device__ __forceinline__ void put(const PrefillArgs& a) {
    if (at >= end) return;
    const uint32_t p0 = at + threadIdx.x, p1 = p0 + kBatch / 2;
    if (p0 < end && slot0 >= 0 && slot0 < a.num_slots) {
      const int64_t dst = place(a, slot0, p0);
      store_past_l2(a.k_cache + dst, k0);
      store_past_l2(a.v_cache + dst, v0);
    }
    if (p1 < end && slot1 >= 0 && slot1 < a.num_slots) {
      const int64_t dst = place(a, slot1, p1);
      store_past_l2(a.k_cache + dst, k1);
      store_past_l2(a.v_cache + dst, v1);
    }
    at = at + min(kBatch, end - at);
  }
  __device__ __forceinline__ void finish(const PrefillArgs& a) {
    while (at < end) {
      fetch(a);
      put(a);
    }
  }
};
struct NoShare {
  __device__ __forceinline__ NoShare(const PrefillArgs&) {}
  __device__ __forceinline__ void fetch(const PrefillArgs&) const {}
  __device__ __forceinline__ void put(const PrefillArgs&) const {}
  __device__ __forceinline__ void finish(const PrefillArgs&) const {}
};

// The query tile of a workgroup and its sequence.
struct QueryTile {
  int seq, kvh;
  int c0;                                // its first column group of the sequence's
  int q_base, len_q, k_first, k_count;   // of that sequence, from the loads of the search
};

// Query tiles are numbered sequence by sequence.  A wave looks at 64 * K sequences at a time, a
// lane for each K neighbours, their offsets fetched in one round trip (a loop over the sequences
// one by one cost a batch of 128 short prompts more than its tiles).  What a workgroup does in
// front of its first tile is a chain of dependent instructions that nothing covers.  With a lane
// for every fourth group of 64 instead, fetched and scanned group by group, and divisions as
// divisions: 128 prompts of 16..300 tokens 122.9 us, now 115.2, 128 of 128 (32 / 8 heads) 87.1 / 79.2,
// 300 of 4 (64 / 8) 44.9 / 38.3, one of 200 7.6 / 7.1, 8 of 4096 971 / 946.
template <bool PAGED, int kColumnGroups, int K>
struct SequenceTiles {
  const PrefillArgs& a;
  int first;            // sequence of this lane
  int cq[K + 1], ck[K + 1];
  int nt[K], mine;      // tiles of each, of all
  int upto, total;      // tiles up to and including this lane's, of all lanes

  __device__ __forceinline__ SequenceTiles(const PrefillArgs& args, int base, int lane)
      : a(args), first(base + K * lane) {
#pragma unroll
    for (int j = 0; j <= K; ++j) {   // (behind the last sequence: empty ones)
      const int s = min(first + j, a.batch);
      cq[j] = a.cu_q[s];
      ck[j] = a.cu_k[s];
    }
    mine = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const uint32_t blocks = (uint32_t)(max(cq[j + 1] - cq[j], 0) + 15) / 16;
      nt[j] = (int)((blocks * a.group.d + kColumnGroups - 1) / kColumnGroups);
      mine += nt[j];
    }
    upto = wave_inclusive_scan(mine);
    total = __builtin_amdgcn_readlane(upto, 63);
  }
  // Tile `tile` of sequence j of lane `src`.
  __device__ __forceinline__ void take(int src, int j, int tile, QueryTile* t) const {
    int q0 = cq[0], q1 = cq[1], k0 = ck[0], k1 = ck[1];
#pragma unroll
    for (int i = 1; i < K; ++i) {
      if (j == i) {
        q0 = cq[i];
        q1 = cq[i + 1];
        k0 = ck[i];
        k1 = ck[i + 1];
      }
    }
    t->seq = __builtin_amdgcn_readlane(first, src) + j;
    t->c0 = tile * kColumnGroups;
    t->q_base = __builtin_amdgcn_readlane(q0, src);
    t->len_q = __builtin_amdgcn_readlane(q1, src) - t->q_base;
    t->k_first = __builtin_amdgcn_readlane(k0, src);
    t->k_count = __builtin_amdgcn_readlane(k1, src) - t->k_first;
  }
  // tile `id`, counted from `base` on; 0 <= id < total
  __device__ __forceinline__ void by_sequence(int id, QueryTile* t) const {
    const int src = __popcll(__ballot(upto <= id));   // lanes whose sequences end in front of it
    int tile = id - __builtin_amdgcn_readlane(upto - mine, src), j = 0;
#pragma unroll
    for (int i = 0; i < K - 1; ++i) {
      const int n = __builtin_amdgcn_readlane(nt[i], src);
      if (j == i && tile >= n) {
        tile -= n;
        ++j;
      }
    }
    take(src, j, tile, t);
  }
  // With few rounds of workgroups a long tile that starts late is what the launch waits for: tiles
  // are then walked by the keys they have, most first.  Behind cached prefixes where those are of
  // very different lengths (16 sequences of 130..5600 keys 239 -> 222 us; where they are alike
  // the order by sequence is the better one, as the search costs 0.5 us per workgroup and
  // neighbours no longer share their keys in L2: 12 prompts of 853..1475 tokens 170 -> 177 us),
  // packed prompts always (few tiles: launch_prefill).
  __device__ __forceinline__ int keys_of(int j) const {
    const int keys = max(ck[j + 1] - ck[j], 0);
    return PAGED ? min(keys, a.max_blocks * a.page.d) : keys;
  }
  static constexpr int kLevel = 128;   // keys: tiles this close in length count as equal
  __device__ __forceinline__ bool by_length(int* longest) const {
    int keys = 0, most = 0;
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (nt[j] > 0) {
        const int n = keys_of(j);
        most = max(most, max(n, cq[j + 1] - cq[j]));
        keys += n >> 5;
      }
    *longest = wave_max(most);
    if (!PAGED) return *longest > kLevel;
    keys = __builtin_amdgcn_readlane(wave_inclusive_scan(keys), 63);
    return *longest >= 1024 && (int64_t)*longest * a.batch * 3 > (int64_t)keys * 128;
  }
  // No sort: the number of tiles that walk more than T keys is a sum over the sequences
  // of a closed form, so item i is found by bisection of T.
  __device__ __forceinline__ int beyond(int j, int T) const {   // tiles that walk more, of sequence j
    const int len_q = cq[j + 1] - cq[j];
    // the first tile past token x - 1 of the sequence
    const int x = T - (PAGED ? max(keys_of(j) - len_q, 0) : 0);
    const int past = x < 0 ? 0 : x >= len_q ? nt[j] : (x >> 4) * a.group.d / kColumnGroups;
    return max(nt[j] - past, 0);
  }
  __device__ __forceinline__ int count_beyond(int T) const {
    int n = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) n += beyond(j, T);
    return __builtin_amdgcn_readlane(wave_inclusive_scan(n), 63);
  }
  __device__ __forceinline__ void longest_first(int item, int longest, QueryTile* t) const {
    // smallest level L with at most `item` tiles beyond (L + 1) * kLevel keys
    int lo = 0, hi = longest / kLevel;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (count_beyond((mid + 1) * kLevel) <= item) hi = mid;
      else lo = mid + 1;
    }
    const int before = count_beyond((lo + 1) * kLevel);
    int above[K], level[K], sum = 0;   // tiles beyond the level and in it
#pragma unroll
    for (int j = 0; j < K; ++j) {
      above[j] = beyond(j, (lo + 1) * kLevel);
      // level 0 takes everything that is left, tiles without any key included
      level[j] = (lo == 0 ? nt[j] : beyond(j, lo * kLevel)) - above[j];
      sum += level[j];
    }
    const int end = before + wave_inclusive_scan(sum);
    const int src = __popcll(__ballot(end <= item));
    int at = item - __builtin_amdgcn_readlane(end - sum, src), j = 0;
    int last = __builtin_amdgcn_readlane(nt[0] - above[0], src) - 1;
#pragma unroll
    for (int i = 0; i < K - 1; ++i) {
      const int n = __builtin_amdgcn_readlane(level[i], src);
      if (j == i && at >= n) {
        at -= n;
        ++j;
        last = __builtin_amdgcn_readlane(nt[i + 1] - above[i + 1], src) - 1;
      }
    }
    take(src, j, last - at, t);   // the later tiles of a sequence walk more keys
  }
  // Item `item` of a KV head's list, all sequences being here; false beyond the real tiles.
  __device__ __forceinline__ bool find(int item, bool may_sort, QueryTile* t) const {
    if (item >= total) return false;
    int longest;
    // (packed prompts only with the larger workgroups, launch_prefill: the rest is shorter without)
    if ((PAGED || kColumnGroups == 2 * kWaves) && may_sort && by_length(&longest))
      longest_first(item, longest, t);
    else
      by_sequence(total - 1 - item, t);
    return true;
  }
};

// False when the workgroup has no tile.
template <bool PAGED, int kColumnGroups>
__device__ __forceinline__ bool find_query_tile(const PrefillArgs& a, bool may_sort, int lane,
                                                QueryTile* t) {
  // Work item -> workgroup, XCD-aware.  Consecutive workgroup ids land on
  // different XCDs (8 of them, each with its own L2), so the work list is cut
  // into 8 contiguous parts and workgroup id L takes item (L % 8) * part + L / 8:
  // one XCD then walks neighbouring items.  Items are ordered (kv head, query
  // tile): neighbours share the K/V rows of one (sequence, kv head), which stay
  // in that XCD's L2 instead of being fetched by all eight.  Later tiles of a
  // sequence have more keys to walk and come first.
  // The work list is sized for a bound on the tiles, and the items beyond the real ones sit at its
  // end, where they delay nothing.  The real tiles are walked from the last one down.
  const int total_items = a.tiles.d * a.num_kv_heads;
  const int part = (total_items + 7) / 8;
  const int place = ((int)blockIdx.x % 8) * part + (int)blockIdx.x / 8;
  if (place >= total_items) return false;
  t->kvh = a.tiles.divide(place);
  const int item = place - t->kvh * a.tiles.d;
  if (a.batch <= 64)
    return SequenceTiles<PAGED, kColumnGroups, 1>(a, 0, lane).find(item, may_sort, t);
  if (a.batch <= 128)
    return SequenceTiles<PAGED, kColumnGroups, 2>(a, 0, lane).find(item, may_sort, t);
  if (a.batch <= 256)
    return SequenceTiles<PAGED, kColumnGroups, 4>(a, 0, lane).find(item, may_sort, t);
  int real_tiles = 0;
  for (int base = 0; base < a.batch; base += 256)
    real_tiles += SequenceTiles<PAGED, kColumnGroups, 4>(a, base, lane).total;
  if (item >= real_tiles) return false;
  int id = real_tiles - 1 - item;
  for (int base = 0; base < a.batch; base += 256) {
    const SequenceTiles<PAGED, kColumnGroups, 4> tiles(a, base, lane);
    if (id < tiles.total) {
      tiles.by_sequence(id, t);
      return true;
    }
    id -= tiles.total;
  }
  return false;   // (cannot happen: the item is a real tile)
}

// The keys that the rows of a query tile see.
template <bool PAGED, int kColumnGroups>
struct VisibleKeys {
  int off;      // key position of the first token: the new tokens are the tail when paged
  int k_end;    // keys [0, k_end) are visible to some row
  int nsteps;   // in tiles
  __device__ __forceinline__ VisibleKeys(const PrefillArgs& a, const QueryTile& tile) {
    const int len_k =
        PAGED ? min(max(tile.k_count, 0), a.max_blocks * a.page.d) : max(tile.k_count, 0);
    off = PAGED ? max(len_k - tile.len_q, 0) : 0;
    const int token_end =   // of the tile
        min(a.group.divide(tile.c0 + kColumnGroups - 1) * 16 + 16, tile.len_q);
    k_end = min(len_k, off + token_end);
    nsteps = (k_end + kKeys - 1) / kKeys;
  }
};

// The tiles [first, end) of part `part` of a query tile's keys: whole rounds of the ring, and none so
// short that its head and tail are most of it but for the last, which takes what is left over.
struct KeyPart {
  int first, end, count;   // count: parts that have keys
  __device__ __forceinline__ KeyPart(const PrefillArgs& a, int nsteps, int part) {
    const int each = nsteps <= 2 * kShortestPart
                         ? 2 * kShortestPart
                         : max((a.splits.divide(nsteps + a.splits.d - 1) + 3) & ~3, kShortestPart);
    count = (int)nvj::quotient(nsteps + each - 1, nvj::reciprocal(each));
    first = part * each;
    end = min(first + each, nsteps);
  }
};

// grid.x = 8 * ceil(tile bound * Hkv / 8) workgroups (see the work-item mapping below).
// PAGED: keys and values come from the block-paged cache through block_tables,
// sequence i has len_k = cu_k[i+1] - cu_k[i] keys, and its len_q query rows are the
// LAST len_q positions of the sequence (row j sees keys <= len_k - len_q + j):
// prompt rows behind a cached prefix.  Otherwise: packed rows, both counted
// from the start of the sequence as the reference's mask does.
// STORE (packed only): the rows of k and v also go into the caches (StoreShare).
// STREAM: the output goes past the L2s.
// SPLIT (paged only): workgroup (x, y) takes part y of the keys and leaves what it has for
// prefill_merge_kernel, unless the tile has no other part.
template <bool F16, bool PAGED, int NG, bool STORE, bool STREAM, int RING, bool SPLIT = false>
__global__ __launch_bounds__(kWaves * 64, RING == 3 ? 3 : 2) void prefill_attention_kernel(
    PrefillArgs a, bool may_sort) {
  static_assert(RING == 4 || (RING == 3 && NG == 1), "tiles in LDS");
  constexpr int kAhead = RING - 2;             // tiles fetched ahead
  constexpr int kColumnGroups = NG * kWaves;   // per workgroup
  __shared__ uint4 k_ring[RING * kTileBytes / 16];
  __shared__ uint4 v_ring[RING * kTileBytes / 16];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r = lane & 15;
  const int kg = lane >> 4;

  std::conditional_t<STORE, StoreShare, NoShare> share(a);
  QueryTile tile;
  if (!find_query_tile<PAGED, kColumnGroups>(a, may_sort, lane, &tile)) {
    share.finish(a);
    return;
  }
  const int seq = tile.seq, kvh = tile.kvh, c0 = tile.c0, q_base = tile.q_base, len_q = tile.len_q;
  share.fetch(a);
  const int k_base = PAGED ? 0 : tile.k_first;
  const VisibleKeys<PAGED, kColumnGroups> keys(a, tile);
  const int off = keys.off, k_end = keys.k_end;
  int first_tile = 0, nsteps = keys.nsteps;   // this workgroup's tiles, up to nsteps
  bool whole = true;
  if constexpr (SPLIT) {
    const KeyPart part(a, keys.nsteps, blockIdx.y);
    if (blockIdx.y > 0 && part.first >= keys.nsteps) return;
    first_tile = part.first;
    nsteps = part.end;
    whole = part.count <= 1;
  }

  // ---- Q^T of both column groups as B operands: column r of group g is token
  // block0[g] + r of head[g]; tokens beyond the sequence are zero ----
  int block0[NG], token[NG], head[NG];
  bf16x8 qreg[NG][4];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int c = c0 + NG * wave + g;
    const int block = a.group.divide(c);
    block0[g] = block * 16;
    head[g] = kvh * a.group.d + (c - block * a.group.d);
    token[g] = block0[g] + r;
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    const uint4* qrow = a.q + (int64_t)(q_base + min(token[g], len_q - 1)) * a.q_stride +
                        (int64_t)head[g] * kPieces;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint4 t = qrow[4 * s + kg];
      qreg[g][s] = as_bf16x8(token[g] < len_q ? t : zero);
    }
  }

  const uint32_t row_bytes = a.kv_row_bytes;
  const char* k_head =
      reinterpret_cast<const char*>(a.k + kvh * kPieces) + (int64_t)k_base * row_bytes;
  const char* v_head =
      reinterpret_cast<const char*>(a.v + kvh * kPieces) + (int64_t)k_base * row_bytes;
  const const_i32_ptr table =
      (const_i32_ptr)(uintptr_t)(PAGED ? a.block_tables + (int64_t)seq * a.max_blocks : a.cu_q);

  const lds_ptr k_lds = (lds_ptr)k_ring;
  const lds_ptr v_lds = (lds_ptr)v_ring;
  TileCopier<PAGED> copier = {k_head, v_head, row_bytes, (uint32_t)(uintptr_t)k_lds,
                                    (uint32_t)(uintptr_t)v_lds, k_end - 1, nsteps - 1, wave, lane,
                                    table, a.page, a.num_blocks, 0};

  const float sl2 = a.scale_log2e;
  f32x4 acc[NG][8], lacc[NG];
  float m_run[NG], mneg[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    m_run[g] = kNegBig;
    mneg[g] = -kNegBig * sl2;
    lacc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int jd = 0; jd < 8; ++jd) acc[g][jd] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // Software pipeline over the tiles: iteration i issues the scores of tile i to
  // the matrix core, then accumulates tile i-1 (probabilities kept from the
  // previous iteration) while the vector ALU turns the scores of tile i into
  // probabilities.  Iteration i therefore reads K of tile i and V of tile i-1,
  // and starts the copies of a tile to come: with a ring of 4 those of tile i+2 at its end, into
  // the ring slots last read in iteration i-1 (V of tile i-2); with a ring of 3 those of
  // tile i+1 at its start, into the slot of tile i-2, which nothing reads any more.  Before the barrier
  // that ends it, every lane waits for its copies of tile i+1.
  if (nsteps > first_tile) {
    // V "of tile -1" (probabilities are zero there, but 0 * NaN is not 0)
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    uint4* v_before = v_ring + (RING - 1) * (kTileBytes / 16);
    for (int p = tid; p < kTileBytes / 16; p += kWaves * 64) v_before[p] = zero;
    copier.look_up(first_tile);
    copier.issue(first_tile, 0, 0);
    if (kAhead > 1) copier.issue(first_tile + 1, 1, 1);
    wait_tiles_in_flight<kAhead - 1>();
  }
  __syncthreads();

  // Tiles of this wave, in order: plain ones (every key visible to every row),
  // masked ones (the diagonal tile, or one that reaches past the last key),
  // then tiles whose keys no row of the wave sees, where it only helps to copy.
  // Separate loops rather than a branch inside one keep the accumulators in place.
  // A wave without a real row only helps to copy.
  const int n_active =
      block0[0] >= len_q ? 0 : min(nsteps, (off + block0[NG - 1] + 15) / kKeys + 1);
  const int n_plain = min(min(off + block0[0] + 1, k_end) / kKeys, n_active);

  // Tile t lives in ring slot t % RING (K and V alike).  Iteration i: (a ring of 3: copies of
  // tile i+1,) scores of tile i, accumulation of tile i-1, probabilities of tile i, (a ring of 4: copies
  // of tile i+2,) wait for this lane's copies of tile i+1, barrier.
  lds_ptr kaddr[4], vaddr[8];
  k_read_addresses(k_lds, r, kg, kaddr);
  v_read_addresses(v_lds, r, kg, vaddr);
  uint32_t koff[kCopyRowsPerWave / 4], voff[kCopyRowsPerWave / 4];
  copier.lane_offsets(koff, voff);

  f32x4 sc[NG][2];
  bf16x8 pb[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) pb[g] = as_bf16x8(make_uint4(0u, 0u, 0u, 0u));
  // Waves that issue matrix instructions go first: a wave lowers its priority
  // only while it turns scores into probabilities (vector ALU work that the
  // other wave of the SIMD can overlap with its own matrix instructions).
  __builtin_amdgcn_s_setprio(1);
#define NVJ_END_OF_TILE()               \
  do {                                  \
    wait_tiles_in_flight<kAhead - 1>(); \
    __syncthreads();                    \
  } while (0)
  // a plain tile whose ring slots are known when the code is written: every LDS
  // offset is an immediate, the copies use the lanes' precomputed offsets
#define NVJ_PLAIN_TILE_AT(S, i)                                                              \
  do {                                                                                       \
    scores_of_tile<F16, NG>(kaddr, (S) * kTileBytes, qreg, sc);                                  \
    accumulate_tile<F16, NG>(vaddr, (((S) + 3) & 3) * kTileBytes, pb, acc, lacc);                \
    __builtin_amdgcn_s_setprio(0);                                                           \
    probabilities_of_tile<false, F16, NG>(sc, pb, acc, lacc, m_run, mneg, sl2, kg, token, 0, 0); \
    __builtin_amdgcn_s_setprio(1);                                                           \
    copier.template issue_full<((S) + 2) & 3>((i) + 2, koff, voff);                          \
    NVJ_END_OF_TILE();                                                                       \
  } while (0)
  // any tile, ring slots computed at run time
#define NVJ_TILE(MASKED, i, row_limit, key_limit)                                            \
  do {                                                                                       \
    if (RING == 3) copier.issue((i) + 1, slot(i, 1), slot(i, 1));                            \
    scores_of_tile<F16, NG>(kaddr, slot(i, 0) * kTileBytes, qreg, sc);                       \
    accumulate_tile<F16, NG>(vaddr, slot(i, RING - 1) * kTileBytes, pb, acc, lacc);          \
    __builtin_amdgcn_s_setprio(0);                                                           \
    probabilities_of_tile<MASKED, F16, NG>(sc, pb, acc, lacc, m_run, mneg, sl2, kg, token,   \
                                           row_limit, key_limit);                            \
    __builtin_amdgcn_s_setprio(1);                                                           \
    if (RING == 4) copier.issue((i) + 2, slot(i, 2), slot(i, 2));                            \
    third = slot(i, 1);                                                                      \
    NVJ_END_OF_TILE();                                                                       \
  } while (0)

  int third = 0;   // a ring of 3: the slot of tile i
  const auto slot = [&](int i, int ahead) {   // of tile i + ahead (of tile i - 1: ahead = RING - 1)
    if (RING == 4) return (i + ahead) & 3;
    return third + ahead < 3 ? third + ahead : third + ahead - 3;
  };
  int i = first_tile;
  // four plain tiles at a time while the tiles they fetch (up to i + 5) are full ones
  for (; RING == 4 && i + 4 <= n_plain && i + 5 < nsteps - 1; i += 4) {
    NVJ_PLAIN_TILE_AT(0, i);
    NVJ_PLAIN_TILE_AT(1, i + 1);
    NVJ_PLAIN_TILE_AT(2, i + 2);
    NVJ_PLAIN_TILE_AT(3, i + 3);
  }
  for (; i < n_plain; ++i) NVJ_TILE(false, i, 0, 0);
  for (; i < n_active; ++i) {
    const int ks = i * kKeys;
    NVJ_TILE(true, i, off - ks, k_end - 1 - ks);
  }
  // the last tile of the wave is still to be accumulated; its V stays in place
  // until the copies of two iterations from now
  if (n_active > first_tile)
    accumulate_tile<F16, NG>(vaddr, slot(i, RING - 1) * kTileBytes, pb, acc, lacc);
  for (; i < nsteps; ++i) {
    copier.issue(i + kAhead, slot(i, kAhead), slot(i, kAhead));
    third = slot(i, 1);
    NVJ_END_OF_TILE();
  }
  wait_tiles_in_flight<0>();   // copies past the last tile are still landing in LDS
#undef NVJ_TILE
#undef NVJ_PLAIN_TILE_AT
#undef NVJ_END_OF_TILE

  if (SPLIT && !whole) {
    const int64_t rec =
        ((int64_t)blockIdx.x * a.splits.d + blockIdx.y) * kColumnGroups + NG * wave;
    float4* o = reinterpret_cast<float4*>(a.part_o) + rec * (8 * 64) + lane;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
#pragma unroll
      for (int jd = 0; jd < 8; ++jd)
        o[64 * (8 * g + jd)] =
            make_float4(acc[g][jd][0], acc[g][jd][1], acc[g][jd][2], acc[g][jd][3]);
      if (kg == 0) a.part_ml[(rec + g) * 16 + r] = make_float2(m_run[g], lacc[g][0]);
    }
    return;
  }

  // ---- epilogue: acc[g][jd][e] is O[token][dim = 16*jd + 4*kg + e].  The rows are
  // turned in LDS (16-byte pieces permuted by the row as for K) so that every
  // store writes four whole 256-byte rows instead of 32 bytes of 16 of them ----
  __syncthreads();   // every wave is done with the rings, every copy has landed
  char* stage = reinterpret_cast<char*>(k_ring) + wave * (NG * 16 * 256);
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const float l = lacc[g][0];   // already summed over every key of the row
    const float inv = l > 0.f ? 1.0f / l : 0.f;   // no visible key at all -> zeros
#pragma unroll
    for (int jd = 0; jd < 8; ++jd) {
      uint2 o;
      o.x = Elem<F16>::pack2(acc[g][jd][0] * inv, acc[g][jd][1] * inv);
      o.y = Elem<F16>::pack2(acc[g][jd][2] * inv, acc[g][jd][3] * inv);
      *reinterpret_cast<uint2*>(stage + (16 * g + r) * 256 +
                                16 * k_position(r, 2 * jd + (kg >> 1)) + 8 * (kg & 1)) = o;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // rows of this wave only
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * i + kg, t = block0[g] + row;
      const uint4 o = *reinterpret_cast<const uint4*>(stage + (16 * g + row) * 256 +
                                                      16 * k_position(row, r));
      uint4* to = a.out + ((int64_t)(q_base + t) * a.num_heads + head[g]) * kPieces + r;
      if (t < len_q) {
        if constexpr (STREAM) store_past_l2(to, o);
        else *to = o;
      }
    }
  share.put(a);
  share.finish(a);
}

// Puts the parts of every query tile together, in their order.  grid.x as in the launch of the parts,
// grid.y = the eighths of the head dimension, block = a wave for each of the GROUPS column groups.
// Bound by the launch and its round trips: eight workgroups to a tile, so that all partials of a wave,
// up to 16, are on their way at once (by eights: +0.2 .. +1 us).
template <bool F16, int GROUPS>
__global__ __launch_bounds__(GROUPS * 64) void prefill_merge_kernel(PrefillArgs a, bool may_sort) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4, jd = blockIdx.y;
  QueryTile tile;
  if (!find_query_tile<true, GROUPS>(a, may_sort, lane, &tile)) return;
  const VisibleKeys<true, GROUPS> keys(a, tile);
  const int count = KeyPart(a, keys.nsteps, 0).count;
  const int c = tile.c0 + wave, block = a.group.divide(c);
  if (count <= 1 || block * 16 >= tile.len_q) return;
  const int64_t rec = (int64_t)blockIdx.x * a.splits.d * GROUPS + wave;
  const f32x4* o = reinterpret_cast<const f32x4*>(a.part_o) + rec * (8 * 64) + 64 * jd + lane;
  const float2* ml = a.part_ml + rec * 16 + r;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  float m_run = kNegBig, l = 0.f;
  // `batch` parts on their way together
  auto take = [&](auto batch) __attribute__((always_inline)) {
    constexpr int kBatch = decltype(batch)::value;
    for (int s = 0; s < count; s += kBatch) {
      f32x4 v[kBatch];
      float2 p[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        const int at = min(s + j, count - 1) * GROUPS;
        v[j] = o[(int64_t)at * (8 * 64)];
        p[j] = ml[at * 16];
      }
      float m_new = m_run;
#pragma unroll
      for (int j = 0; j < kBatch; ++j) m_new = max2(m_new, p[j].x);
      const float keep = __builtin_amdgcn_exp2f((m_run - m_new) * a.scale_log2e);
      m_run = m_new;
      acc *= keep;
      l *= keep;
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        if (s + j >= count) continue;
        const float w = __builtin_amdgcn_exp2f((p[j].x - m_new) * a.scale_log2e);
        l = fmaf(w, p[j].y, l);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(w, v[j][e], acc[e]);
      }
    }
  };
  if (count <= 4) take(std::integral_constant<int, 4>());
  else if (count <= 8) take(std::integral_constant<int, 8>());
  else take(std::integral_constant<int, 16>());
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  const int t = block * 16 + r, head = tile.kvh * a.group.d + (c - block * a.group.d);
  if (t >= tile.len_q) return;
  uint2* to = reinterpret_cast<uint2*>(
      a.out + ((int64_t)(tile.q_base + t) * a.num_heads + head) * kPieces + 2 * jd) + kg;
  *to = make_uint2(Elem<F16>::pack2(acc[0] * inv, acc[1] * inv),
                   Elem<F16>::pack2(acc[2] * inv, acc[3] * inv));
}

// Output rows that the L2s (32 MiB together) would not keep anyway are stored past them; left in
// the L2s they displace the K and V rows that other workgroups are about to read (128 prompts
// of 16..300 tokens, 166 MB of rows: 130 -> 117 us).  Smaller ones stay where the next launch
// can find them: an output projection behind 17 MB of rows takes 2.3 us longer than the
// attention saves (0.4).
constexpr int64_t kStreamOutBytes = 32 << 20;

// How a launch is cut: column groups per wave, tiles of K and V in LDS, and the most query tiles that
// it can have, per KV head.
struct TileForm {
  int groups, ring;
  int64_t tiles;
};
// Query tiles per KV head, at most: every sequence adds at most one partly filled token block and one
// partly filled tile.
int64_t most_tiles(int64_t tokens, int64_t batch, int64_t group, int64_t column_groups) {
  const int64_t blocks = (tokens + 15 * batch) / 16;
  return (blocks * group + (column_groups - 1) * batch) / column_groups;
}
// The same if the last block and the last tile of every sequence are half full.
int64_t half_full_tiles(int64_t tokens, int64_t batch, int64_t group, int64_t column_groups) {
  return ((2 * tokens + 15 * batch) * group + 16 * (column_groups - 1) * batch +
          16 * column_groups) /
         (32 * column_groups);
}
// And no less than sequences of a token or a few have.
int64_t expected_tiles(int64_t tokens, int64_t batch, int64_t group, int64_t column_groups) {
  return std::max(half_full_tiles(tokens, batch, group, column_groups),
                  std::min(tokens, batch) * ((group + column_groups - 1) / column_groups));
}
TileForm tile_form(int64_t tokens, int64_t batch, int64_t group, int64_t num_kv_heads, int64_t cus,
                   bool paged) {
  const int64_t wide = most_tiles(tokens, batch, group, 2 * kWaves);
  const int64_t narrow = most_tiles(tokens, batch, group, kWaves);
  const int64_t groups = (tokens + 16 * batch - 1) / (16 * batch) * group;   // of a mean prompt
  const bool xcds_even = num_kv_heads % 8 == 0;   // each takes whole KV heads
  // One column group per wave while the larger workgroups would leave CUs idle or start a second
  // round with little to do: one prompt of 700 tokens, 16 / 8 heads, 21.0 -> 16.2 us; 4 of
  // 70..90, 32 heads, 10.8 -> 9.1; up to 1.5 of them a CU, one prompt of 3000, 16 heads, 62 -> 50,
  // of 1500, 32 heads, 35 -> 29 (two a CU: 79 .. 111 %).
  if (wide * num_kv_heads <= cus) return {1, 4, narrow};
  if (paged) {
    // Behind cached prefixes, where the tiles of a sequence are equally long, up to two of the small
    // ones a CU: 4 of 55..268, at most 277 keys, 32 / 8 heads, 10.3 us in small ones, 12.0 in larger, 2
    // of 167..263, 557 keys, 64 / 8, 15.4 / 17.7; with 385 .. 512 of them behind more than 2048
    // positions 0.86 times as long in the mean (1100 drawn launches).  Unless the XCDs take whole KV
    // heads one of them gets nothing but real tiles, so there the bound counts: small ones in the
    // place of larger, by eighths of the bound, 449 .. 512 0.82 (2050 drawn launches, 1.5 % of them longer),
    // 513 .. 576 1.14 (14 of 3..243, up to 4424 keys, 28 / 4, 118 us / 94).
    const int64_t small = expected_tiles(tokens, batch, group, kWaves) * num_kv_heads;
    if ((xcds_even ? small : narrow * num_kv_heads) <= 2 * cus) return {1, 4, narrow};
    // Nor do the larger ones fit a round there once their bound is more than two a CU, so half-full
    // tiles count again: 0.89 (1400 drawn launches; 72 of 1..4 behind 1744, 28 / 4, 60.1 us / 82.0).
    const bool second_round = wide * num_kv_heads > 2 * cus;
    if (!xcds_even && second_round &&
        half_full_tiles(tokens, batch, group, kWaves) * num_kv_heads <= 2 * cus)
      return {1, 4, narrow};
    // More of them, but of sequences of a column group or two, or of up to 4 groups and a block of 16
    // tokens, few of which have a second: the larger workgroups are mostly empty (1 or 2 query heads a
    // KV head 0.88, 4 and 6 .. 12 tokens 0.89, 12 .. 16 tokens up to 8 a CU 0.92, one in seven longer
    // and at worst 1.46, where nearly all keys are long; more than 8 a CU 0.99, 31 % of them longer).
    if (small > 2 * cus &&
        (groups <= 2 || ((xcds_even || second_round) && groups <= 4 &&
                         tokens <= (small <= 8 * cus ? 16 : 12) * batch)))
      return {1, 4, narrow};
    return {2, 4, wide};
  }
  // Prompts that are longer than a block and whose KV heads do not fill the XCDs evenly keep the
  // larger ones, all of which run at once (8 / 1 heads, 6 of 186..1642 39 us, in small ones 45, 28 / 4,
  // one of 1731 42 / 47).
  if ((xcds_even || tokens <= 16 * batch) && wide * num_kv_heads * 2 <= cus * 3)
    return {1, 4, narrow};
  // Prompts of few column groups: the larger workgroups are mostly empty or mostly head and tail.
  // Three small ones to a CU instead, us with the store: 100 prompts of 4 tokens, 16 / 8 heads (2 groups)
  // 12.5 -> 8.2, 200 of 16, 32 / 8 (4) 31.0 -> 23.0, 100 of 60, 32 / 32 (4) 71 -> 57, 60 of 20..60, 32 / 8
  // (12) 17.9 -> 15.2, 16 / 8 (6) 12.1 -> 9.9, 40 of 100, 16 / 8 (14) 21.4 -> 18.0.  Larger against small
  // ones over drawn launches: up to 4 groups 1.37 in the mean (421 launches, at worst 0.965), 5 to 14
  // with up to 4 heads to a KV head 1.09 (200, 0.915, 4 % of them below 0.97); beyond the line, with 7 or 8
  // heads, 1.05 (150, 27 % of them below 0.97), 15 to 30 groups 1.05 (188, 18 %).
  if (groups <= 4 || (groups <= 14 && group <= 4)) return {1, 3, narrow};
  return {2, 4, wide};
}

// Whether the store of new rows rides in the attention launch.  A share costs its workgroup about
// 1 us: over more than three rounds of two workgroups per CU that is more than a launch of the
// store's own, unless the shares are large.  us in one launch / in two, 64 / 8 heads: 300
// prompts of 4 tokens 48.6 / 44.1, 200 of up to 17 34.8 / 32.4, 500 of 9 104.9 / 98.5 (31, 59 and 61
// pieces a share); from 80 pieces on -19 .. +2 %, with fewer rounds -22 .. -1 %.
bool store_rides(int64_t tokens, int64_t rows, int64_t batch, int64_t num_heads,
                 int64_t num_kv_heads, int64_t cus) {
  const int64_t tiles =
      tile_form(tokens, batch, num_heads / num_kv_heads, num_kv_heads, cus, false).tiles *
      num_kv_heads;
  return tiles <= 6 * cus || rows * num_kv_heads * kPieces >= 80 * tiles;
}

// Longest tiles first: behind cached prefixes, up to 8 rounds of two workgroups per CU.  Packed
// prompts of more than a round and at most 5 / 4: 8 of 500 tokens, 16 / 8 heads, 21.7 -> 19.7 us, 4
// of 1000 31.0 -> 28.4, 2 of 1000, 32 / 8, 30.0 -> 27.1, 8 of 165..945 27.1 -> 27.0; with 4 a CU and
// more -5 .. +12 %.  Each XCD takes an eighth of the list: unless that is whole KV heads, one gets
// the long tiles and another the short ones (8 / 1 heads, 11 of 624..775 30.8 -> 40.7, 28 / 4, 3 of
// 823..968 31.0 -> 39.4).
constexpr int64_t kLongestFirstPerCu = 16;

constexpr int64_t kMostSplits = 32;
constexpr int64_t kNeverCut = 2 * kKeys * kShortestPart;   // positions

// Parts that a query tile's keys may be cut into; 1: none.  Few rows behind a long prefix are a
// workgroup or two per KV head, each drawing 50 GB/s, 0.47 us a tile of keys, for thousands of keys,
// while the other CUs idle; in parts they fill one round of two workgroups a CU.  us, whole / in
// parts: 30 tokens behind 5000, 32 / 8 heads, 75 / 17, 13 behind 5300, 16 / 8, 79 / 14, 270 behind
// 4200, 32 / 8, 68 / 38, 8 of 13..16 behind 800..5000, 16 / 8, 78 / 26.  Against that the partials and
// the launch that merges them are 2 .. 10 us and more, whatever the lengths turn out to be, of which
// the host knows a bound: so the more workgroups there are, the longer the keys have to be.  us, whole / in
// parts, behind up to 512 positions 9 tokens behind 256, 10.6 / 12.3; 768: 21 sequences of 1 or 2 tokens,
// 8 / 1, 42 workgroups, 12.1 / 13.9; 1024: 49 of 1..6, 4 / 4, 196 of them, 14.4 / 19.7; 2048: 32 of 3 or
// 4, 28 / 4, 256 of them, 24.2 / 34.8, 90 of 7, 8 / 1, 197 of them, 29.1 / 42.0; beyond 8 of 1..7 behind
// 4400, 32 / 32, 256 of them, 96.7 / 120, 53 of 1..3 behind 6500, 4 / 4, 212 of them, 124 / 154.  Sequences of
// more than a block of tokens, whose tiles share their keys, gain up to a round (1 of 213 behind 1900, 64
// / 8, 224 of them, 33.9 / 31.7, 6 of 27 behind 3050 48 / 41); where every query head has keys of its own
// HBM is the bound earlier.  4206 launches drawn from 1..260 sequences of 1..700 tokens behind up to
// 12000 positions, where the bound is known, against a workgroup for every tile: 1.21 times as fast in
// the mean, 0.3 % of them more than 5 % slower, at worst 0.85.
// More than a round of parts is slower (4 of 100..300 behind
// 1000..4000, 34.7 / 40.2 at twice as many), three quarters of one better where there are many to put
// together (30 behind 5000 18.5 / 16.9, 20 behind 4000, 32 / 32, 28 / 22.5).  Parts of 4 tiles or of 12
// instead of 8: +3 .. -1 and -0.7 .. +1.4 us.
struct SplitForm {
  TileForm form;
  int64_t splits;
};
// The most workgroups whose keys are cut.  `streams`: sequences times KV heads, the keys that are not
// shared.  Where most workgroups have keys of their own HBM is the bound earlier than where several walk
// the same ones, so the lines lie higher for few streams.  In parts / whole, means of 51000 launches drawn
// from this side of the lines and beyond, by workgroups (and streams): up to 1024 positions 65 .. 72 0.96, 81
// .. 96 1.00 (0.88 and 0.90 where tables are as long as what is in them, 1.05 and 1.09 where they are
// longer); 2048, KV heads a multiple of 8, 129 .. 192 (up to 128) 0.94, (more) 1.07, 193 .. 224 (up to
// 128) 0.98; others 97 .. 128 0.88, 129 .. 160 (up to 32) 0.94, (more) 1.02, 161 .. 192 (up to 32) 0.97;
// 4096, a multiple of 8, 193 .. 256 (up to 160) 0.86, (more) 1.11; others 161 .. 192 (up to 64) 0.86, (more)
// 0.97 and now and then far longer (94 of 3..6 behind 2600, 6 / 2, 188 of them, 50.2 us whole, 66.7), 193 ..
// 224 (up to 32) 0.86, (more) 1.03, 225 .. 256 (up to 32) 0.99.
int64_t most_to_cut(int64_t tokens, int64_t batch, int64_t group, int64_t num_kv_heads, int64_t cus,
                    int64_t positions) {
  const bool xcds_even = num_kv_heads % 8 == 0;
  const int64_t streams = batch * num_kv_heads;
  if (positions <= kNeverCut) return 0;
  if (positions <= 768) return cus / 8;
  if (positions <= 1024) return cus * 9 / 32;
  if (positions <= 2048) {
    if (group == 1 || (xcds_even ? streams * 2 : streams * 8) > cus) return cus / 2;
    return cus * (xcds_even ? 6 : 5) / 8;
  }
  if (positions <= 4096) {
    if (group == 1) return cus * (xcds_even ? 6 : 5) / 8;
    if (xcds_even) return streams * 8 <= cus * 5 ? cus : cus * 6 / 8;
    return cus * (streams * 8 <= cus ? 7 : streams * 4 <= cus ? 6 : 5) / 8;
  }
  if (group == 1 || !xcds_even) return cus * 6 / 8;
  return tokens > 16 * batch ? cus : cus * 15 / 16;
}
int64_t key_splits(const TileForm& form, int64_t tokens, int64_t batch, int64_t group,
                   int64_t num_kv_heads, int64_t cus, int64_t positions) {
  const int64_t workgroups =
      std::max<int64_t>(expected_tiles(tokens, batch, group, kWaves) * num_kv_heads, 1);
  if (form.groups != 1 || batch > 256 ||
      workgroups > most_to_cut(tokens, batch, group, num_kv_heads, cus, positions))
    return 1;
  const bool few = workgroups * 4 <= cus;
  const int64_t shortest = kKeys * kShortestPart * (few ? 1 : workgroups * 2 <= cus ? 2 : 3);
  return std::max<int64_t>(std::min<int64_t>({(few ? 3 * cus / 2 : 2 * cus) / workgroups,
                                              positions / shortest, kMostSplits}),
                           1);
}

// The form of a launch in parts.  In the small workgroups every wave reads a whole tile of keys out of
// LDS for 16 rows, which is what bounds two of them to a CU (0.69 us a tile; the larger ones 1.2 for
// twice the rows).  Where the small ones would be cut into two or three parts or none at all the larger
// ones in parts, up to two a CU, are the shorter way behind more than 4096 positions.  us, before /
// so: 500 behind 5000, 32 / 8 heads, 69 / 60, 700 behind 5000 90 / 81, 512 behind 8000, 64 / 8, 157 /
// 133, 400 behind 4000, 32 / 32, 68 / 51, 6 of 23..44 behind 8555..10940, 64 / 8, 148 / 99.  Up to
// 4096 positions the partials cost more (1000 behind 2000 55 / 62), with fewer rows many small parts
// are as good (270 behind 4200 37.6 / 36.4, 150 behind 4000, 32 / 32, 29 / 33), with more large workgroups
// than CUs two parts each are not (4 of 244..494 behind 3357..5499, 368 of them, 125 / 151), and where the
// XCDs are not filled evenly earlier (193 .. 208 of them 0.94, 209 .. 224 0.96, 225 .. 256 1.02, where they are
// 241 .. 256 0.87; 168 of 5..18 behind 3500, 8 / 1, 250 of them, 119 / 160), and nor are they where they are
// hardly fewer than the small ones, half empty (55 of 2 behind 2500, 16 / 8, 126 / 153, 7 of 12 behind
// 7350, 32 / 32, 138 / 174).
SplitForm split_form(int64_t tokens, int64_t batch, int64_t group, int64_t num_kv_heads,
                     int64_t cus, int64_t positions) {
  const int64_t small = expected_tiles(tokens, batch, group, kWaves) * num_kv_heads;
  const int64_t large =
      std::max<int64_t>(expected_tiles(tokens, batch, group, 2 * kWaves) * num_kv_heads, 1);
  if (batch <= 256 && positions > 4096 && small * 4 > cus * 3 &&
      large * 16 <= cus * (num_kv_heads % 8 == 0 ? 16 : 13) && large * 4 <= small * 3)
    return {{2, 4, most_tiles(tokens, batch, group, 2 * kWaves)}, 2 * cus / large};
  const TileForm form = tile_form(tokens, batch, group, num_kv_heads, cus, true);
  return {form, key_splits(form, tokens, batch, group, num_kv_heads, cus, positions)};
}
int64_t most_keys(int64_t max_blocks, int64_t block_size, int64_t max_keys) {
  return max_keys > 0 ? std::min(max_keys, max_blocks * block_size) : max_blocks * block_size;
}
// Bytes of the partials of a launch, 0 where its keys are not cut.
size_t part_bytes(const SplitForm& cut, int64_t num_kv_heads) {
  constexpr size_t kGroupBytes = 8 * 64 * sizeof(float4) + 16 * sizeof(float2);
  if (cut.splits <= 1) return 0;
  const int64_t workgroups = (cut.form.tiles * num_kv_heads + 7) / 8 * 8;
  return (size_t)(workgroups * cut.splits * cut.form.groups * kWaves) * kGroupBytes;
}

int launch_prefill(hipStream_t stream, PrefillArgs a, bool paged, const TileForm& form,
                   int32_t total_q_tokens, int32_t dtype, int64_t cus) {
  if (((int64_t)total_q_tokens + 15) * a.group.d > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  const int64_t tiles = form.tiles;
  if (tiles > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  const int64_t items = tiles * a.num_kv_heads;
  if (items > INT32_MAX - 8) return NVJ_ERR_BAD_SHAPE;
  const dim3 grid((unsigned)((items + 7) / 8 * 8)), block(kWaves * 64);
  a.tiles = Divisor(tiles);
  if (a.slots) {   // whole heads, as many for each workgroup
    const int64_t heads = a.new_pieces / kPieces;
    a.share_pieces = (uint32_t)((heads + grid.x - 1) / grid.x * kPieces);
  }
  const bool may_sort =
      a.batch > 1 && a.batch <= 256 &&
      (paged ? items <= kLongestFirstPerCu * cus && (int64_t)a.max_blocks * a.page.d >= 1024
             : form.groups == 2 && items * 2 <= cus * 5 && a.num_kv_heads % 8 == 0);
  const bool f16 = dtype == NVJ_DTYPE_F16;
  if (a.part_o) {
    const dim3 parts(grid.x, (unsigned)a.splits.d), eighths(grid.x, 8);
    a.part_ml = reinterpret_cast<float2*>(a.part_o + (int64_t)grid.x * a.splits.d * form.groups *
                                                         kWaves * 8 * 64 * 4);
    const auto go = [&](auto groups) {
      constexpr int NG = decltype(groups)::value;
      const auto split = f16 ? prefill_attention_kernel<true, true, NG, false, false, 4, true>
                             : prefill_attention_kernel<false, true, NG, false, false, 4, true>;
      const auto merge =
          f16 ? prefill_merge_kernel<true, NG * kWaves> : prefill_merge_kernel<false, NG * kWaves>;
      const dim3 waves(NG * kWaves * 64);
      return nvj::launch(split, parts, block, stream, a, may_sort) == hipSuccess &&
             nvj::launch(merge, eighths, waves, stream, a, may_sort) == hipSuccess;
    };
    const bool ok = form.groups == 2 ? go(std::integral_constant<int, 2>())
                                     : go(std::integral_constant<int, 1>());
    return ok ? NVJ_OK : NVJ_ERR_LAUNCH;
  }
  const bool past_l2 = (int64_t)total_q_tokens * a.num_heads * (kD * 2) > kStreamOutBytes;
  hipError_t rc;
#define NVJ_LAUNCH(F, P, N, S, T, R)                                                              \
  rc = nvj::launch(prefill_attention_kernel<F, P, N, S, T, R>, grid, block, stream, a, may_sort)
#define NVJ_LAUNCH_STREAM(F, P, N, S, R)           \
  if (past_l2) NVJ_LAUNCH(F, P, N, S, true, R);    \
  else NVJ_LAUNCH(F, P, N, S, false, R)
#define NVJ_LAUNCH_PACKED(F, S)                       \
  if (form.groups == 2) {                             \
    NVJ_LAUNCH_STREAM(F, false, 2, S, 4);             \
  } else if (form.ring == 3) {                        \
    NVJ_LAUNCH_STREAM(F, false, 1, S, 3);             \
  } else {                                            \
    NVJ_LAUNCH(F, false, 1, S, false, 4);             \
  }
#define NVJ_LAUNCH_TYPE(F)                            \
  if (paged && form.groups == 1) {                    \
    NVJ_LAUNCH_STREAM(F, true, 1, false, 4);          \
  } else if (paged) {                                 \
    NVJ_LAUNCH_STREAM(F, true, 2, false, 4);          \
  } else if (a.slots) {                               \
    NVJ_LAUNCH_PACKED(F, true)                        \
  } else {                                            \
    NVJ_LAUNCH_PACKED(F, false)                       \
  }
  if (f16) {
    NVJ_LAUNCH_TYPE(true);
  } else {
    NVJ_LAUNCH_TYPE(false);
  }
#undef NVJ_LAUNCH_TYPE
#undef NVJ_LAUNCH_PACKED
#undef NVJ_LAUNCH_STREAM
#undef NVJ_LAUNCH
  return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
}

}  // namespace

namespace {
struct CacheRows {   // where new rows go: see PrefillArgs
  const int32_t* slots;
  void *k_cache, *v_cache;
  int64_t num_slots;
  int32_t rows;
};

int launch_packed(void* stream, const void* q, int64_t q_row_stride, const void* k, const void* v,
                  int64_t kv_row_stride, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                  void* out, int32_t total_q_tokens, int32_t batch, int32_t num_heads,
                  int32_t num_kv_heads, int32_t head_dim, float scale, int32_t dtype,
                  const CacheRows* store, int64_t cus) {
  if (dtype != NVJ_DTYPE_BF16 && dtype != NVJ_DTYPE_F16) return NVJ_ERR_BAD_DTYPE;
  if (total_q_tokens < 0 || batch < 0 || num_heads <= 0 || num_kv_heads <= 0)
    return NVJ_ERR_BAD_SHAPE;
  if (num_heads % num_kv_heads != 0) return NVJ_ERR_BAD_SHAPE;
  if (head_dim != kD) return NVJ_ERR_UNSUPPORTED;
  if (num_kv_heads > 32768) return NVJ_ERR_UNSUPPORTED;   // a key row stays below 2^24 bytes
  if (q_row_stride < (int64_t)num_heads * kD || kv_row_stride < (int64_t)num_kv_heads * kD)
    return NVJ_ERR_BAD_SHAPE;
  if (kv_row_stride > (1 << 22)) return NVJ_ERR_UNSUPPORTED;
  if (!(scale >= 0.f)) return NVJ_ERR_BAD_SHAPE;   // the running max assumes a non-negative scale
  if (total_q_tokens == 0 || batch == 0) return NVJ_OK;
  if (!q || !k || !v || !cu_seqlens_q || !cu_seqlens_k || !out) return NVJ_ERR_NULL_POINTER;
  if (((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
        reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(out)) & 15u) ||
      ((q_row_stride | kv_row_stride) & 7))
    return NVJ_ERR_ALIGNMENT;
  PrefillArgs a = {};
  a.q = static_cast<const uint4*>(q);
  a.k = static_cast<const uint4*>(k);
  a.v = static_cast<const uint4*>(v);
  a.out = static_cast<uint4*>(out);
  a.cu_q = cu_seqlens_q;
  a.cu_k = cu_seqlens_k;
  a.q_stride = q_row_stride / 8;
  a.kv_row_bytes = (uint32_t)kv_row_stride * 2;
  a.batch = batch;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.group = Divisor(num_heads / num_kv_heads);
  a.scale_log2e = scale * kLog2e;
  if (store) {
    a.slots = store->slots;
    a.k_cache = static_cast<uint4*>(store->k_cache);
    a.v_cache = static_cast<uint4*>(store->v_cache);
    a.num_slots = store->num_slots;
    a.row_pieces = Divisor((int64_t)num_kv_heads * kPieces);
    a.new_pieces = (uint32_t)store->rows * (uint32_t)a.row_pieces.d;
  }
  return launch_prefill(static_cast<hipStream_t>(stream), a, false,
                        tile_form(total_q_tokens, batch, a.group.d, num_kv_heads, cus, false),
                        total_q_tokens, dtype, cus);
}
}  // namespace

extern "C" int nvj_prefill_attention_rows_launch(
    void* stream, const void* q, int64_t q_row_stride, const void* k, const void* v,
    int64_t kv_row_stride, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, void* out,
    int32_t total_q_tokens, int32_t batch, int32_t num_heads, int32_t num_kv_heads,
    int32_t head_dim, float scale, int32_t dtype) {
  return launch_packed(stream, q, q_row_stride, k, v, kv_row_stride, cu_seqlens_q, cu_seqlens_k,
                       out, total_q_tokens, batch, num_heads, num_kv_heads, head_dim, scale, dtype,
                       nullptr, nvj::compute_units());
}

extern "C" int nvj_prefill_attention_store_launch(
    void* stream, const void* q, const void* k, const void* v, const int32_t* cu_seqlens_q,
    const int32_t* cu_seqlens_k, void* out, const int32_t* slot_mapping, void* k_cache,
    void* v_cache, int64_t num_slots, int32_t total_q_tokens, int32_t num_rows, int32_t batch,
    int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, float scale, int32_t dtype) {
  if (num_rows < 0 || num_slots < 0 || num_kv_heads <= 0 || head_dim <= 0)
    return NVJ_ERR_BAD_SHAPE;
  const auto store_alone = [&] {
    return nvj_store_kvcache_launch(stream, k, v, k_cache, v_cache, slot_mapping, num_rows,
                                    num_kv_heads, head_dim, num_slots, dtype, dtype, dtype);
  };
  if (num_rows > 0) {
    if (!slot_mapping || !k_cache || !v_cache) return NVJ_ERR_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) & 15u)
      return NVJ_ERR_ALIGNMENT;
  }
  const CacheRows rows = {slot_mapping, k_cache, v_cache, num_slots, num_rows};
  const int64_t cus = nvj::compute_units();   // (asked for once: 70 ns of a call of 5 us)
  // the kernel counts the pieces of all rows in 31 bits
  const bool together = num_rows > 0 && total_q_tokens > 0 && batch > 0 &&
                        (int64_t)num_rows * num_kv_heads * kPieces <= INT32_MAX - 4096 &&
                        store_rides(total_q_tokens, num_rows, batch, num_heads, num_kv_heads, cus);
  if (!together && num_rows > 0) {
    const int code = store_alone();
    if (code != NVJ_OK) return code;
  }
  return launch_packed(stream, q, (int64_t)num_heads * kD, k, v, (int64_t)num_kv_heads * kD,
                       cu_seqlens_q, cu_seqlens_k, out, total_q_tokens, batch, num_heads,
                       num_kv_heads, head_dim, scale, dtype, together ? &rows : nullptr, cus);
}

extern "C" int nvj_prefill_attention_launch(void* stream, const void* q, const void* k,
                                            const void* v, const int32_t* cu_seqlens_q,
                                            const int32_t* cu_seqlens_k, void* out,
                                            int32_t total_q_tokens, int32_t batch,
                                            int32_t num_heads, int32_t num_kv_heads,
                                            int32_t head_dim, float scale, int32_t dtype) {
  return nvj_prefill_attention_rows_launch(stream, q, (int64_t)num_heads * kD, k, v,
                                           (int64_t)num_kv_heads * kD, cu_seqlens_q, cu_seqlens_k,
                                           out, total_q_tokens, batch, num_heads, num_kv_heads,
                                           head_dim, scale, dtype);
}

namespace {
int launch_paged(void* stream, const void* q, const void* k_cache, const void* v_cache,
                 const int32_t* block_tables, const int32_t* cu_seqlens_q,
                 const int32_t* cu_seqlens_k, void* out, int32_t total_q_tokens, int32_t batch,
                 int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                 int32_t max_blocks, int32_t num_blocks, float scale, int32_t dtype,
                 bool may_split, int32_t max_keys, void* workspace, size_t workspace_bytes) {
  if (dtype != NVJ_DTYPE_BF16 && dtype != NVJ_DTYPE_F16) return NVJ_ERR_BAD_DTYPE;
  if (total_q_tokens < 0 || batch < 0 || num_heads <= 0 || num_kv_heads <= 0 || block_size <= 0 ||
      max_blocks < 0 || num_blocks <= 0)
    return NVJ_ERR_BAD_SHAPE;
  if (num_heads % num_kv_heads != 0) return NVJ_ERR_BAD_SHAPE;
  if (head_dim != kD || block_size % kKeys != 0) return NVJ_ERR_UNSUPPORTED;
  if (num_kv_heads > 32768) return NVJ_ERR_UNSUPPORTED;   // a key row stays below 2^24 bytes
  if ((int64_t)max_blocks * block_size > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  if (!(scale >= 0.f)) return NVJ_ERR_BAD_SHAPE;
  if (total_q_tokens == 0 || batch == 0) return NVJ_OK;
  if (!q || !k_cache || !v_cache || !cu_seqlens_q || !cu_seqlens_k || !out)
    return NVJ_ERR_NULL_POINTER;
  if (max_blocks > 0 && !block_tables) return NVJ_ERR_NULL_POINTER;
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_cache) |
       reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(out)) & 15u)
    return NVJ_ERR_ALIGNMENT;
  PrefillArgs a = {};
  a.q = static_cast<const uint4*>(q);
  a.k = static_cast<const uint4*>(k_cache);
  a.v = static_cast<const uint4*>(v_cache);
  a.out = static_cast<uint4*>(out);
  a.cu_q = cu_seqlens_q;
  a.cu_k = cu_seqlens_k;
  a.q_stride = (int64_t)num_heads * kPieces;
  a.kv_row_bytes = (uint32_t)num_kv_heads * (kD * 2);
  a.batch = batch;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.group = Divisor(num_heads / num_kv_heads);
  a.scale_log2e = scale * kLog2e;
  a.block_tables = block_tables;
  a.page = Divisor(block_size);
  a.max_blocks = max_blocks;
  a.num_blocks = num_blocks;
  const int64_t cus = nvj::compute_units();
  const int64_t positions = most_keys(max_blocks, block_size, max_keys);
  const SplitForm cut =
      may_split ? split_form(total_q_tokens, batch, a.group.d, num_kv_heads, cus, positions)
                : SplitForm{tile_form(total_q_tokens, batch, a.group.d, num_kv_heads, cus, true),
                            1};
  if (const size_t need = part_bytes(cut, num_kv_heads)) {
    if (!workspace || workspace_bytes < need) return NVJ_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(workspace) & 15u) return NVJ_ERR_ALIGNMENT;
    a.splits = Divisor(cut.splits);
    a.part_o = static_cast<float*>(workspace);
  }
  return launch_prefill(static_cast<hipStream_t>(stream), a, true, cut.form, total_q_tokens, dtype,
                        cus);
}
}  // namespace

extern "C" int nvj_paged_prefill_attention_launch(
    void* stream, const void* q, const void* k_cache, const void* v_cache,
    const int32_t* block_tables, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
    void* out, int32_t total_q_tokens, int32_t batch, int32_t num_heads, int32_t num_kv_heads,
    int32_t head_dim, int32_t block_size, int32_t max_blocks, int32_t num_blocks, float scale,
    int32_t dtype) {
  return launch_paged(stream, q, k_cache, v_cache, block_tables, cu_seqlens_q, cu_seqlens_k, out,
                      total_q_tokens, batch, num_heads, num_kv_heads, head_dim, block_size,
                      max_blocks, num_blocks, scale, dtype, false, 0, nullptr, 0);
}

extern "C" size_t nvj_paged_prefill_split_workspace_bytes(int32_t total_q_tokens, int32_t batch,
                                                          int32_t num_heads, int32_t num_kv_heads,
                                                          int32_t block_size, int32_t max_blocks,
                                                          int32_t max_keys) {
  if (total_q_tokens <= 0 || batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 ||
      num_heads % num_kv_heads != 0 || block_size <= 0 || max_blocks <= 0)
    return 0;
  const int64_t positions = most_keys(max_blocks, block_size, max_keys);
  if (positions <= kNeverCut) return 0;   // (without asking for the CUs, 70 ns)
  return part_bytes(split_form(total_q_tokens, batch, num_heads / num_kv_heads, num_kv_heads,
                               nvj::compute_units(), positions),
                    num_kv_heads);
}

extern "C" int nvj_paged_prefill_split_launch(
    void* stream, const void* q, const void* k_cache, const void* v_cache,
    const int32_t* block_tables, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
    void* out, void* workspace, size_t workspace_bytes, int32_t total_q_tokens, int32_t batch,
    int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
    int32_t max_blocks, int32_t num_blocks, int32_t max_keys, float scale, int32_t dtype) {
  return launch_paged(stream, q, k_cache, v_cache, block_tables, cu_seqlens_q, cu_seqlens_k, out,
                      total_q_tokens, batch, num_heads, num_kv_heads, head_dim, block_size,
                      max_blocks, num_blocks, scale, dtype, true, max_keys, workspace,
                      workspace_bytes);
}
