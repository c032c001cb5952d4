// Products of activation rows with bf16 weights, C[m][n] = x[m][:] . w[n][:], for
// prompts (hundreds to thousands of rows) on gfx950, with the element-wise stage that
// follows a projection of the decoder layer in the epilogue:
//   kPlain    bf16 rows (kRowsPastL2: the same, stored past the L2)
//   kSiluMul  SiLU(gate) * up of the fused gate/up projection (layers/activation.py:22-33
//             of the reference), half the columns
//   kQkRope   QK-RMSNorm, RoPE and KV-cache store of the fused QKV projection
//             (models/qwen3.py:147-166)
//
// MFMA-bound, if the operands arrive: a workgroup of 4 waves (2 x 2) computes BM x BN
// outputs, K in steps of 64.  Rows go global -> LDS directly (16 bytes per lane, whole
// 128-byte rows, pieces XOR-permuted by the row: no bank conflicts on the operand reads),
// in a ring of two to four stages, one barrier per step, which stands in the middle of it
// so that operand reads, copies and matrix instructions run under each other throughout.
// Measured, 4400 rows, alone: QKV (4096 x 1024) without its epilogue 40.9 us, O (1024 x 2048)
// 21.9, gate/up (6144 x 1024) with SiLU * up 62.2, down (1024 x 3072) 29.8; library 46.4, 27.6,
// 56.4 + 16.7, 35.2.  In a step of 4268: QKV with norm, RoPE and store 50.6, O 19.8, gate/up
// 64.0 (beside the workgroups that read ahead), down 27.2, the matrix pipe 38 % (QKV) to 52 %
// (O, down) busy.  LDS is the next limit: operand reads
// and arriving copies take 75 % (256 x 256) to 150 % (128 x 128) of the matrix cycles.
// Weights straight into registers instead (as in decoder_step.hip) were no way out: 64-byte
// pieces of 16 rows per load made it 1 us per step whatever the tile.
//
// Rows go past the writing XCD's L2 where that was measured to help the step: 4 .. 24 MB of plain
// rows (a norm on all XCDs reads them once), q and the cache rows: 4268 rows in 8 prompts 6310 ->
// 6184 us with the norm's residual (layer_glue.hip), 128 rows of decode 3517 -> 3492; not SiLU *
// up and the packed K and V, which the next launch reads several times.
//
// Every output is one chain of v_mfma_f32_16x16x32_bf16 over K in order, whatever the tile
// and the rows beside it (decoder_step.hip says where the library GEMMs sum likewise).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bf16.h"
#include "device.h"
#include "divisor.h"
#include "launch.h"
#include "lds_copy.h"
#include "linear.h"
#include "nvj_paged_attn.h"
#include "past_l2.h"
#include "qk_norm_rope.h"

namespace {

typedef __attribute__((address_space(3))) char* lds_ptr;

constexpr int kBK = 64;        // reduction per step: rows of 128 bytes, 8 pieces

using nvj::bf16_to_f32;
using nvj::bf16x8;
using nvj::copy16_to_lds;
using nvj::f32x4;
using nvj::f32_to_bf16_rne;
using nvj::LinearArgs;
using nvj::pack2_bf16;
using nvj::store_past_l2;
enum Epilogue { kPlain, kRowsPastL2, kSiluMul, kQkRope };

template <int N>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// QK-RMSNorm, RoPE and KV store of a tile of kHeads heads, in LDS as bf16 rows of `stride`
// bytes.  16 lanes per (row, head): unit u of a workgroup is row (16 * u + its group of 16
// lanes) / kHeads; N units at a time.  Bound by round trips where a workgroup is alone on its
// CU: positions and slots come with the first copies into LDS, table rows a batch ahead (4300
// rows of 4096 x 1024, us: 256 x 256 tiles 89.7 -> 79.1, 160 x 256 61.1 -> 56.3; 160 x 128, two
// to a CU, which cover for each other, 50.3 -> 49.5, where 39 are the product's; 128 rows
// 7.7 -> 7.4 of 5.5).
//
// A group of lanes works on the same head in every unit, so the norm's weights are fetched
// once: behind a store of the unit before they would be fetched again, a round trip a unit.
template <int kHeads>
struct RopeHead {
  int h, head;                 // of the tile, of all
  bool is_q, is_k, norm;
  float4 wl, wh;
  __device__ __forceinline__ RopeHead(const LinearArgs& a, int n_tile) {
    static_assert(16 % kHeads == 0, "one head per group of lanes");
    h = (int)(threadIdx.x >> 4) % kHeads;
    head = n_tile * kHeads + h;
    is_q = head < a.num_heads;
    is_k = !is_q && head < a.num_heads + a.num_kv_heads;
    norm = a.q_norm != nullptr;
    wl = wh = make_float4(0.f, 0.f, 0.f, 0.f);
    if (norm && (is_q || is_k)) {
      const float* w = (is_q ? a.q_norm : a.k_norm) + 4 * (threadIdx.x & 15);
      wl = nvj::load4<true>(w);
      wh = nvj::load4<true>(w + 64);
    }
  }
};
template <int N, int kHeads>
struct RopeUnits {
  int slot[N];
  float4 c4[N], s4[N];

  // places: positions of the tile's rows, then (from place `slots`) their slots, in LDS
  __device__ __forceinline__ void fetch(const LinearArgs& a, const int* places, int slots, int u0) {
    const int i = threadIdx.x & 15;
#pragma unroll
    for (int b = 0; b < N; ++b) {
      const int m = ((u0 + b) * 16 + (int)(threadIdx.x >> 4)) / kHeads;
      slot[b] = places[slots + m];
      const float* cs =
          a.cos_sin + (int64_t)min(max(places[m], 0), a.max_position - 1) * 128 + 4 * i;
      c4[b] = nvj::load4<true>(cs);
      s4[b] = nvj::load4<true>(cs + 64);
    }
  }
  // The tile of 32 x 128: positions and slots through scalar loads of the four rows that a wave
  // has in each unit.  In LDS, where the others have them, their 512 bytes beside its ring would
  // leave one workgroup to a CU: a prompt of 400 tokens 1898 us instead of 1827.  (The tile of
  // 64 x 128 has the room: 200 and 700 tokens 1535 and 2094 us, like this 1548 and 2115.)
  struct Places {
    int position[N], slot[N];
    __device__ __forceinline__ Places(const LinearArgs& a, int m0, int wave) {
      typedef const __attribute__((address_space(4))) int* const_int_ptr;
      const const_int_ptr positions = (const_int_ptr)(uintptr_t)a.positions;
      const const_int_ptr slots = (const_int_ptr)(uintptr_t)a.slot_mapping;
      const int group = (threadIdx.x >> 4) & 3;
#pragma unroll
      for (int b = 0; b < N; ++b) {
        position[b] = slot[b] = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int token = min(m0 + 16 * b + 4 * wave + j, a.M - 1);
          const int p = positions[token], s = slots[token];
          position[b] = group == j ? p : position[b];
          slot[b] = group == j ? s : slot[b];
        }
      }
    }
  };
  __device__ __forceinline__ void fetch(const LinearArgs& a, const Places& places) {
    const int i = threadIdx.x & 15;
#pragma unroll
    for (int b = 0; b < N; ++b) {
      slot[b] = places.slot[b];
      const float* cs =
          a.cos_sin + (int64_t)min(max(places.position[b], 0), a.max_position - 1) * 128 + 4 * i;
      c4[b] = nvj::load4<true>(cs);
      s4[b] = nvj::load4<true>(cs + 64);
    }
  }
  __device__ __forceinline__ void rows(const LinearArgs& a, const RopeHead<kHeads>& t,
                                       const char* lds, int stride, int m0, int u0) const {
    const int i = threadIdx.x & 15;
#pragma unroll
    for (int b = 0; b < N; ++b) {
      const int m = ((u0 + b) * 16 + (int)(threadIdx.x >> 4)) / kHeads, token = m0 + m;
      if (token >= a.M) continue;
      const uint2* src = reinterpret_cast<const uint2*>(lds + m * stride + 256 * t.h);
      uint2 lo = src[i], hi = src[16 + i];
      if (t.is_q || t.is_k)
        nvj::qk_norm_rope(lo, hi, t.norm, t.wl, t.wh, a.eps, c4[b], s4[b]);
      if (t.is_q || a.keep_kv) {
        uint2* dst = reinterpret_cast<uint2*>(
            t.is_q ? a.q_out + ((int64_t)token * a.num_heads + t.head) * 128
                   : a.out + (int64_t)token * a.N + t.head * 128);
        if (t.is_q) {
          store_past_l2(dst + i, lo);
          store_past_l2(dst + 16 + i, hi);
        } else {
          dst[i] = lo;
          dst[16 + i] = hi;
        }
      }
      if (!t.is_q && slot[b] >= 0 && slot[b] < a.num_slots) {
        const int kvh = t.head - a.num_heads - (t.is_k ? 0 : a.num_kv_heads);
        uint2* row = reinterpret_cast<uint2*>((t.is_k ? a.k_cache : a.v_cache) +
                                              ((int64_t)slot[b] * a.num_kv_heads + kvh) * 128);
        store_past_l2(row + i, lo);
        store_past_l2(row + 16 + i, hi);
      }
    }
  }
};

// Row tiles that are walked side by side: 8 x 4 tiles at a time per XCD (51 -> 42 us for 160 x 256
// tiles at 4400 rows).
constexpr int kGroupM = 8;

template <int BM, int BN, int kStages, Epilogue EPI>
__global__ __launch_bounds__(256) void linear_kernel(LinearArgs a) {
  constexpr int WM = BM / 2, WN = BN / 2;          // per wave
  constexpr int TM = WM / 16, TN = WN / 16;
  constexpr int kRows = BM + BN;                   // rows of one stage: x, then w
  constexpr int kStageBytes = kRows * 128;
  constexpr int kCopies = kRows / 8 / 4;           // per wave and stage, 8 rows each
  static_assert(kRows % 32 == 0, "copies are dealt to four waves");
  constexpr int kOut = EPI == kSiluMul ? BN / 2 : BN;   // columns of the output tile
  constexpr int kOutStride = kOut * 2 + 16;             // bytes per row of the tile in LDS
  constexpr int kLds = kStages * kStageBytes > BM * kOutStride ? kStages * kStageBytes
                                                               : BM * kOutStride;
  __shared__ __align__(128) char lds[kLds];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;

  // tiles of one weight column block are neighbours, and each XCD (workgroup id % 8)
  // walks a contiguous part of the list, so a weight tile is fetched by one L2
  const int total = a.m_tiles * a.n_tiles;
  const int part = (total + 7) / 8;
  if ((int)blockIdx.x >= 8 * part) {
    nvj::read_chunk<256>(a.ahead, (int)blockIdx.x - 8 * part);
    return;
  }
  const int tile = ((int)blockIdx.x % 8) * part + (int)blockIdx.x / 8;
  if (tile >= total) return;
  const int per_group = kGroupM * a.n_tiles;
  // (two divisions in front of the first copy: 18.0 -> 17.8 us for gate/up of 1000 rows)
  const int grp = (int)nvj::quotient(tile, nvj::reciprocal(per_group));
  const int in_group = tile - grp * per_group;
  const int gm = min(kGroupM, a.m_tiles - grp * kGroupM);
  const int n_tile = gm == kGroupM ? in_group / kGroupM
                                   : (int)nvj::quotient(in_group, nvj::reciprocal(gm));
  const int m_tile = grp * kGroupM + (in_group - n_tile * gm);
  const int m0 = m_tile * BM;
  const int row_bytes = a.K * 2;

  // kQkRope: positions and slots of the rows first of all, so that nothing waits for them
  constexpr int kHeads = BN >= 128 ? BN / 128 : 1, kUnits = BM * kHeads / 16;
  constexpr int kBatch = kUnits % 5 == 0 ? 5 : kUnits % 4 == 0 ? 4 : 2;
  static_assert(EPI != kQkRope || kUnits % kBatch == 0, "whole batches");
  constexpr int kPlaces = (BM + 63) / 64 * 64;
  constexpr bool kFewUnits = EPI == kQkRope && kUnits == 2 && kHeads == 1;
  __shared__ int places[EPI == kQkRope && !kFewUnits ? 2 * kPlaces : 1];
  RopeUnits<kBatch, kHeads> units;
  if constexpr (EPI == kQkRope && !kFewUnits) {
    if (64 * wave < kPlaces) {
      const uint32_t at = (uint32_t)(uintptr_t)(lds_ptr)places + 256u * wave;
      const uint32_t from = 4u * (uint32_t)min(m0 + 64 * wave + lane, a.M - 1);
      nvj::copy4_to_lds(a.positions, from, at);
      nvj::copy4_to_lds(a.slot_mapping, from, at + 4u * kPlaces);
    }
  }

  // what this wave copies: instruction j moves LDS rows 8 * (4 * j + wave) .. + 7; lane
  // l fetches the piece that belongs at position l % 8 of row l / 8
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds;
  const char* base[kCopies];
  uint32_t offset[kCopies];
  {
    const int row = lane >> 3, piece = (lane & 7) ^ row;
#pragma unroll
    for (int j = 0; j < kCopies; ++j) {
      const int first = 8 * (4 * j + wave);   // a multiple of 8: a block of x or of w rows
      if (first < BM) {
        base[j] = a.x;
        offset[j] = (uint32_t)min(m0 + first + row, a.M - 1) * (uint32_t)row_bytes + 16 * piece;
      } else {
        const int c = first - BM + row;       // column of the tile
        int n;
        if (EPI == kSiluMul)   // blocks of 16 columns: gate, then the same of up, in turn
          n = min(n_tile * (BN / 2) + (c >> 5) * 16 + (c & 15), a.N / 2 - 1) +
              ((c >> 4) & 1 ? a.N / 2 : 0);
        else
          n = min(n_tile * BN + c, a.N - 1);
        base[j] = a.w;
        offset[j] = (uint32_t)n * (uint32_t)row_bytes + 16 * piece;
      }
    }
  }
  const int steps = a.K / kBK;
  auto issue = [&](int step, int stage) {
    // past the end: the last step again, so that the count of copies in flight holds
    const uint32_t k = (uint32_t)min(step, steps - 1) * (kBK * 2);
#pragma unroll
    for (int j = 0; j < kCopies; ++j)
      copy16_to_lds(base[j], offset[j] + k,
                    lds0 + (uint32_t)stage * kStageBytes + (uint32_t)(4 * j + wave) * 1024u);
  };

  f32x4 acc[TM][TN];   // D[n][m]: lane holds n = 4 * kg + e of column m = r
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Software pipeline over halves of a step (32 of the reduction): while the matrix core
  // works on the operands of one half, those of the next are read from LDS, and
  // behind the barrier in the middle of a step the copies of a later one are issued,
  // one every few matrix instructions.
  const int x_row = wm * WM + r, w_row = BM + wn * WN + r;
  bf16x8 xf[2][TM], wf[2][TN];
  auto read = [&](int stage, int s, int i) {   // operand i of half s of a stage
    const char* at = lds + stage * kStageBytes + 16 * ((4 * s + kg) ^ (r & 7));
    if (i < TN) wf[s][i] = *reinterpret_cast<const bf16x8*>(at + (w_row + 16 * i) * 128);
    else xf[s][i - TN] = *reinterpret_cast<const bf16x8*>(at + (x_row + 16 * (i - TN)) * 128);
  };
  auto multiply = [&](int s, int i) {          // matrix instruction i of half s
    const int mi = i / TN, j = i % TN;
    acc[mi][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s][j], xf[s][mi], acc[mi][j], 0, 0, 0);
  };
  constexpr int kMul = TM * TN, kRead = TM + TN;
#pragma unroll
  for (int t = 0; t < kStages; ++t) issue(t, t);
  wait_copies<(kStages - 1) * kCopies>();
  __syncthreads();
  // few units: the table rows too, under the whole reduction
  if constexpr (kFewUnits)
    units.fetch(a, typename RopeUnits<kBatch, kHeads>::Places(a, m0, wave));
  else if constexpr (EPI == kQkRope && kUnits == kBatch)
    units.fetch(a, places, kPlaces, 0);
#pragma unroll
  for (int i = 0; i < kRead; ++i) read(0, 0, i);
  int stage = 0;
  for (int step = 0; step < steps; ++step) {
    int done = 0;
#pragma unroll
    for (int i = 0; i < kRead; ++i) {
      read(stage, 1, i);
#pragma unroll
      for (; done < (i + 1) * kMul / kRead; ++done) multiply(0, done);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int next = stage + 1 == kStages ? 0 : stage + 1;
    wait_copies<(kStages - 2) * kCopies>();   // the next step's rows of this wave are there
    __syncthreads();   // and everybody's; nobody reads this step's stage any more
    const uint32_t k = (uint32_t)min(step + kStages, steps - 1) * (kBK * 2);
    constexpr int kSlots = kRead > kCopies ? kRead : kCopies;
    done = 0;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      if (i < kRead) read(next, 0, i);
      if (i < kCopies)
        copy16_to_lds(base[i], offset[i] + k,
                      lds0 + (uint32_t)stage * kStageBytes + (uint32_t)(4 * i + wave) * 1024u);
#pragma unroll
      for (; done < (i + 1) * kMul / kSlots; ++done) multiply(1, done);
      __builtin_amdgcn_sched_barrier(0);
    }
    stage = next;
  }
  wait_copies<0>();   // copies past the last step are still landing
  if constexpr (EPI == kQkRope && kUnits > kBatch) units.fetch(a, places, kPlaces, 0);
  __syncthreads();

  // ---- the tile as bf16 rows in LDS, then out in whole pieces ----
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    char* row = lds + (wm * WM + 16 * i + r) * kOutStride;
    if constexpr (EPI == kSiluMul) {
#pragma unroll
      for (int j = 0; j < TN; j += 2) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = bf16_to_f32(f32_to_bf16_rne(acc[i][j][e]));
          const float u = bf16_to_f32(f32_to_bf16_rne(acc[i][j + 1][e]));
          o[e] = g / (1.0f + expf(-g)) * u;
        }
        *reinterpret_cast<uint2*>(row + (wn * (WN / 2) + 8 * j + 4 * kg) * 2) =
            make_uint2(pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3]));
      }
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j)
        *reinterpret_cast<uint2*>(row + (wn * WN + 16 * j + 4 * kg) * 2) =
            make_uint2(pack2_bf16(acc[i][j][0], acc[i][j][1]),
                       pack2_bf16(acc[i][j][2], acc[i][j][3]));
    }
  }
  __syncthreads();
  if constexpr (EPI == kQkRope) {
    // the table rows of a batch of units are on their way while the one before is worked on
    const RopeHead<kHeads> head(a, n_tile);
    for (int u0 = 0; u0 < kUnits; u0 += kBatch) {
      RopeUnits<kBatch, kHeads> next;
      if constexpr (!kFewUnits)
        if (u0 + kBatch < kUnits) next.fetch(a, places, kPlaces, u0 + kBatch);
      units.rows(a, head, lds, kOutStride, m0, u0);
      units = next;
    }
  } else {
    constexpr int kPieces = kOut / 8;
    const int n_out = EPI == kSiluMul ? a.N / 2 : a.N;
    for (int p = threadIdx.x; p < BM * kPieces; p += 256) {
      const int m = p / kPieces, piece = p % kPieces, n = n_tile * kOut + 8 * piece;
      if (m0 + m < a.M && n < n_out) {
        uint4* to = reinterpret_cast<uint4*>(a.out + (int64_t)(m0 + m) * n_out + n);
        const uint4 v = *reinterpret_cast<const uint4*>(lds + m * kOutStride + 16 * piece);
        if constexpr (EPI == kRowsPastL2) store_past_l2(to, v);
        else *to = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The same for up to 128 rows where the reduction is cut into chains (the output and
// down projections: few outputs, long reductions; decoder_step.hip on the orders): 4 waves =
// CHAINS chains x 4 / CHAINS row halves of a BM x BN tile; chain c takes every
// CHAINS-th run of RUN steps of 32.  Each operand of a stage is read by one wave, so a
// stage is a whole round of the chains (32 * CHAINS * RUN of the reduction) and the
// waves meet once per round.  Latency-bound: the ring is as deep as LDS allows.
// ---------------------------------------------------------------------------
template <int BM, int BN, int CHAINS, int RUN, int kStages>
__global__ __launch_bounds__(256) void chained_linear_kernel(LinearArgs a) {
  constexpr int kSubs = CHAINS * RUN / 2;          // 64-wide blocks of a round
  constexpr int kRows = BM + BN;
  constexpr int kSubBytes = kRows * 128, kStageBytes = kSubs * kSubBytes;
  constexpr int kCopies = kSubs * kRows / 8 / 4;   // per wave and stage, 8 rows each
  static_assert(kSubs * kRows % 32 == 0 && CHAINS * RUN % 2 == 0, "whole blocks, dealt to four waves");
  constexpr int kSplit = 4 / CHAINS;
  constexpr int WM = BM / kSplit, TM = WM / 16, TN = BN / 16;
  constexpr int kRedStride = BN + 4;
  constexpr int kRed = CHAINS * BM * kRedStride * 4;
  __shared__ __align__(128) char
      lds[kStages * kStageBytes > kRed ? kStages * kStageBytes : kRed];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, kg = lane >> 4;
  const int chain = wave % CHAINS, half = wave / CHAINS;
  const int n_tile = blockIdx.x, m0 = blockIdx.y * BM;
  const int row_bytes = a.K * 2;
  const int rounds = a.K / (32 * CHAINS * RUN);

  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds;
  const char* base[kCopies];
  uint32_t offset[kCopies];
#pragma unroll
  for (int j = 0; j < kCopies; ++j) {
    const int group = 4 * j + wave, sub = group / (kRows / 8), first = 8 * (group % (kRows / 8));
    const int row = lane >> 3, piece = (lane & 7) ^ row;
    base[j] = first < BM ? a.x : a.w;
    const int at = first < BM ? min(m0 + first + row, a.M - 1)
                              : min(n_tile * BN + first - BM + row, a.N - 1);
    offset[j] = (uint32_t)at * (uint32_t)row_bytes + 128 * sub + 16 * piece;
  }
  auto issue = [&](int round, int stage) {
    const uint32_t k = (uint32_t)min(round, rounds - 1) * (64 * CHAINS * RUN);
#pragma unroll
    for (int j = 0; j < kCopies; ++j)
      copy16_to_lds(base[j], offset[j] + k,
                    lds0 + (uint32_t)stage * kStageBytes + (uint32_t)(4 * j + wave) * 1024u);
  };
  f32x4 acc[TM][TN];   // D[n][m]: lane holds n = 4 * kg + e of column m = r
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < kStages - 1; ++t) issue(t, t);
  int stage = 0;
  for (int round = 0; round < rounds; ++round) {
    wait_copies<(kStages - 2) * kCopies>();   // this round's rows of this wave are there
    __syncthreads();                          // and everybody's; the stage read last is free
    issue(round + kStages - 1, stage == 0 ? kStages - 1 : stage - 1);
    const char* at = lds + stage * kStageBytes;
    stage = stage + 1 == kStages ? 0 : stage + 1;
#pragma unroll
    for (int u = 0; u < RUN; ++u) {
      const int step = chain * RUN + u;   // of the round
      const char* block = at + (step >> 1) * kSubBytes + 16 * ((4 * (step & 1) + kg) ^ (r & 7));
      bf16x8 xf[TM], wf[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j)
        wf[j] = *reinterpret_cast<const bf16x8*>(block + (BM + 16 * j + r) * 128);
#pragma unroll
      for (int i = 0; i < TM; ++i)
        xf[i] = *reinterpret_cast<const bf16x8*>(block + (half * WM + 16 * i + r) * 128);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[i], acc[i][j], 0, 0, 0);
    }
  }
  wait_copies<0>();
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *reinterpret_cast<f32x4*>(red + (chain * BM + half * WM + 16 * i + r) * kRedStride + 16 * j +
                                4 * kg) = acc[i][j];
  __syncthreads();
  for (int p = threadIdx.x; p < BM * BN / 4; p += 256) {
    const int m = p / (BN / 4), n = 4 * (p % (BN / 4));
    f32x4 v = *reinterpret_cast<const f32x4*>(red + m * kRedStride + n);
#pragma unroll
    for (int c = 1; c < CHAINS; ++c)
      v += *reinterpret_cast<const f32x4*>(red + (c * BM + m) * kRedStride + n);
    if (m0 + m < a.M && n_tile * BN + n < a.N)
      *reinterpret_cast<uint2*>(a.out + (int64_t)(m0 + m) * a.N + n_tile * BN + n) =
          make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
  }
}

template <int BM, int BN, int CHAINS, int RUN, int ST>
hipError_t launch_chained(hipStream_t s, const LinearArgs& a) {
  const dim3 grid((unsigned)((a.N + BN - 1) / BN), (unsigned)((a.M + BM - 1) / BM));
  return nvj::launch(chained_linear_kernel<BM, BN, CHAINS, RUN, ST>, grid, dim3(256), s, a);
}

template <int BM, int BN, int ST, Epilogue EPI>
hipError_t launch_tiles(hipStream_t s, LinearArgs a) {
  constexpr int kOut = EPI == kSiluMul ? BN / 2 : BN;
  const int outs = EPI == kSiluMul ? a.N / 2 : a.N;
  a.m_tiles = (a.M + BM - 1) / BM;
  a.n_tiles = (outs + kOut - 1) / kOut;
  const int total = a.m_tiles * a.n_tiles;
  const dim3 grid((unsigned)((total + 7) / 8 * 8) + a.ahead.chunks());
  return nvj::launch(linear_kernel<BM, BN, ST, EPI>, grid, dim3(256), s, a);
}

// Tile sizes.  A launch of T tiles takes rounds of one workgroup per CU (or two, where they
// share one), each round a fixed 3 us and per step of 64 a time between `low` (few CUs busy)
// and `full` (all of them: the L2s and the power limit share out).  Measured on an
// MI355X over 300 .. 4400 rows and the four projections of a 1024-wide layer, us
// (other widths: _native_step_pays in engine/decode_step.py has them against the library's):
struct TileShape {
  int bm, bn, per_cu;
  float low, full;
};
constexpr TileShape kShapes[] = {
    {64, 64, 2, 0.156f, 0.32f},  {32, 128, 2, 0.19f, 0.38f},  {64, 128, 2, 0.24f, 0.50f},
    {128, 128, 1, 0.356f, 0.46f}, {160, 128, 1, 0.43f, 0.60f}, {160, 128, 2, 0.60f, 1.09f},
    {192, 128, 1, 0.475f, 0.68f}, {128, 256, 1, 0.62f, 0.90f}, {160, 256, 1, 0.76f, 1.12f},
    {224, 256, 1, 1.00f, 1.52f}, {256, 256, 1, 1.21f, 1.75f}};

constexpr int kNumShapes = (int)(sizeof(kShapes) / sizeof(kShapes[0]));

int best_shape(int64_t m, int64_t n, int k, int min_bn) {
  int best = 0;
  float best_cost = 0.f;
  const int64_t cus = nvj::compute_units();
  for (int i = 0; i < kNumShapes; ++i) {
    const TileShape& t = kShapes[i];
    if (t.bn < min_bn) continue;
    const int64_t tiles = ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
    const int64_t slots = cus * t.per_cu, whole = tiles / slots, rest = tiles % slots;
    const float step_full = t.full, per_step = (float)(k / kBK);
    float cost = (float)whole * (per_step * step_full + 3.f);
    if (rest > 0)
      cost += per_step * (t.low + (t.full - t.low) * (float)rest / (float)slots) + 3.f;
    if (best_cost == 0.f || cost < best_cost) {
      best_cost = cost;
      best = i;
    }
  }
  return best;
}

// Plain rows that go past the L2s.  Smaller outputs stay where a norm behind them finds them, larger
// ones are written more slowly that way.  us with the norm behind, past the L2s / not: 1000 rows of
// 1024 (2 MB) 13.0 / 12.7, 200 of 4096 16.2 / 15.6, 2048 of 1024 20.2 / 20.3, 2048 of 4096 34.9 /
// 35.9, 3000 of 4096 44.7 / 45.3, 4268 of 4096 (35 MB) 65.1 / 61.7, 8192 of 4096 114 / 102.  Logits
// always do, and the next step's weights stay where they are instead: a graph of 106 rows (32 MB
// of them) 1849 / 1853, of 128 3389 / 3393.
// (A flag of the kernel instead of a kernel of its own costs registers, and 1 .. 3 % of a large
// product.)
constexpr int64_t kPastL2From = 4 << 20, kPastL2To = 24 << 20;

template <Epilogue EPI>
hipError_t launch_shape(int shape, hipStream_t s, const LinearArgs& a) {
  switch (shape) {
    case 0:
      if constexpr (EPI == kQkRope) return hipErrorInvalidValue;   // tiles hold whole heads
      else return launch_tiles<64, 64, 4, EPI>(s, a);
    case 1: return launch_tiles<32, 128, 4, EPI>(s, a);
    case 2: return launch_tiles<64, 128, 3, EPI>(s, a);
    case 3: return launch_tiles<128, 128, 4, EPI>(s, a);
    case 4: return launch_tiles<160, 128, 4, EPI>(s, a);
    case 5: return launch_tiles<160, 128, 2, EPI>(s, a);
    case 6: return launch_tiles<192, 128, 3, EPI>(s, a);
    case 7: return launch_tiles<128, 256, 3, EPI>(s, a);
    case 8: return launch_tiles<160, 256, 3, EPI>(s, a);
    case 9: return launch_tiles<224, 256, 2, EPI>(s, a);
    default: return launch_tiles<256, 256, 2, EPI>(s, a);
  }
}

}  // namespace

namespace nvj {

bool linear_takes(int64_t m, int64_t n, int64_t k) {
  // 32-bit lane offsets into both operands; whole steps; 16-byte pieces of output
  return m >= 1 && n >= 8 && n % 8 == 0 && k >= kBK && k % kBK == 0 && m * k * 2 < (1ll << 32) &&
         n * k * 2 < (1ll << 32) && m * n < (1ll << 40);
}

hipError_t linear(hipStream_t s, LinearArgs a, bool for_later) {
  const int shape = a.tile > 0 ? a.tile - 1 : best_shape(a.M, a.N, a.K, 0);
  const int64_t bytes = (int64_t)a.M * a.N * 2;
  const bool past_l2 = for_later || (bytes >= kPastL2From && bytes <= kPastL2To);
  return past_l2 ? launch_shape<kRowsPastL2>(shape, s, a) : launch_shape<kPlain>(shape, s, a);
}
hipError_t linear_silu_mul(hipStream_t s, LinearArgs a) {
  return launch_shape<kSiluMul>(a.tile > 0 ? a.tile - 1 : best_shape(a.M, a.N, a.K, 0), s, a);
}
hipError_t linear_qk_rope(hipStream_t s, LinearArgs a) {
  int shape = a.tile > 0 ? a.tile - 1 : best_shape(a.M, a.N, a.K, 128);
  // columns beyond the last head would be taken for one: 256-wide tiles for an even count only
  if (a.N % kShapes[shape].bn != 0) shape = 4;
  return launch_shape<kQkRope>(shape, s, a);
}

hipError_t linear_chained(hipStream_t s, const LinearArgs& a, int chains, int run) {
  if (chains == 4 && run == 1) return launch_chained<32, 16, 4, 1, 6>(s, a);
  if (chains == 4 && run == 2) return launch_chained<32, 16, 4, 2, 4>(s, a);
  if (chains == 2 && run == 4) return launch_chained<32, 16, 2, 4, 4>(s, a);
  return hipErrorInvalidValue;
}

}  // namespace nvj

namespace {
// What every product asks of its operands.
int check_product(const void* x, const void* w, const void* out, int64_t rows, int64_t outputs,
                  int64_t reduction, int32_t tile) {
  if (rows < 0 || outputs <= 0 || reduction <= 0 || tile < -1 || tile >= kNumShapes)
    return NVJ_ERR_BAD_SHAPE;
  if (!nvj::linear_takes(rows > 0 ? rows : 1, outputs, reduction)) return NVJ_ERR_UNSUPPORTED;
  if (rows == 0) return NVJ_OK;
  if (!x || !w || !out) return NVJ_ERR_NULL_POINTER;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) |
       reinterpret_cast<uintptr_t>(out)) & 15u)
    return NVJ_ERR_ALIGNMENT;
  return NVJ_OK;
}
}  // namespace

extern "C" int nvj_linear_launch(void* stream, const void* x, const void* w, void* out,
                                 int32_t rows, int32_t outputs, int32_t reduction, int32_t form,
                                 int32_t tile) {
  const int bad = check_product(x, w, out, rows, outputs, reduction, tile);
  if (bad != NVJ_OK) return bad;
  const int chains = form == NVJ_LINEAR_CHAINS_2_4 ? 2 : 4;
  const int run = form == NVJ_LINEAR_CHAINS_4_1 ? 1 : form == NVJ_LINEAR_CHAINS_4_2 ? 2 : 4;
  switch (form) {
    case NVJ_LINEAR_ROWS: break;
    case NVJ_LINEAR_SILU_MUL:
      if (outputs % 32 != 0) return NVJ_ERR_UNSUPPORTED;
      break;
    case NVJ_LINEAR_CHAINS_4_1:
    case NVJ_LINEAR_CHAINS_4_2:
    case NVJ_LINEAR_CHAINS_2_4:
      if (tile >= 0 || reduction % (32 * chains * run) != 0) return NVJ_ERR_UNSUPPORTED;
      break;
    default: return NVJ_ERR_BAD_SHAPE;
  }
  if (rows == 0) return NVJ_OK;
  LinearArgs a = {};
  a.x = static_cast<const char*>(x);
  a.w = static_cast<const char*>(w);
  a.out = static_cast<uint16_t*>(out);
  a.M = rows;
  a.N = outputs;
  a.K = reduction;
  a.tile = tile + 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const hipError_t rc = form == NVJ_LINEAR_ROWS       ? nvj::linear(s, a)
                        : form == NVJ_LINEAR_SILU_MUL ? nvj::linear_silu_mul(s, a)
                                                      : nvj::linear_chained(s, a, chains, run);
  return rc == hipSuccess ? NVJ_OK : NVJ_ERR_LAUNCH;
}

extern "C" int nvj_qkv_linear_launch(void* stream, const void* x, const void* w, int32_t rows,
                                     int32_t reduction, const int32_t* positions,
                                     const float* cos_sin_cache, int32_t max_position,
                                     const float* q_norm_weight, const float* k_norm_weight,
                                     float eps, const int32_t* slot_mapping, void* k_cache,
                                     void* v_cache, void* q_out, void* qkv_out, int32_t num_heads,
                                     int32_t num_kv_heads, int64_t num_slots, int32_t tile) {
  if (num_heads <= 0 || num_kv_heads <= 0 || max_position <= 0 || num_slots < 0)
    return NVJ_ERR_BAD_SHAPE;
  const int64_t outputs = ((int64_t)num_heads + 2 * (int64_t)num_kv_heads) * 128;
  if (outputs > INT32_MAX) return NVJ_ERR_BAD_SHAPE;
  const int bad = check_product(x, w, q_out, rows, outputs, reduction, tile);
  if (bad != NVJ_OK) return bad;
  if (tile >= 0 && (kShapes[tile].bn < 128 || outputs % kShapes[tile].bn != 0))
    return NVJ_ERR_UNSUPPORTED;   // tiles hold whole heads
  if (rows == 0) return NVJ_OK;
  if (!positions || !cos_sin_cache || !slot_mapping || !k_cache || !v_cache ||
      (q_norm_weight == nullptr) != (k_norm_weight == nullptr))
    return NVJ_ERR_NULL_POINTER;
  if ((reinterpret_cast<uintptr_t>(cos_sin_cache) | reinterpret_cast<uintptr_t>(q_norm_weight) |
       reinterpret_cast<uintptr_t>(k_norm_weight) | reinterpret_cast<uintptr_t>(k_cache) |
       reinterpret_cast<uintptr_t>(v_cache) | reinterpret_cast<uintptr_t>(qkv_out)) & 15u)
    return NVJ_ERR_ALIGNMENT;
  LinearArgs a = {};
  a.x = static_cast<const char*>(x);
  a.w = static_cast<const char*>(w);
  a.out = static_cast<uint16_t*>(qkv_out);
  a.M = rows;
  a.N = (int)outputs;
  a.K = reduction;
  a.q_out = static_cast<uint16_t*>(q_out);
  a.keep_kv = qkv_out != nullptr;
  a.positions = positions;
  a.cos_sin = cos_sin_cache;
  a.q_norm = q_norm_weight;
  a.k_norm = k_norm_weight;
  a.slot_mapping = slot_mapping;
  a.k_cache = static_cast<uint16_t*>(k_cache);
  a.v_cache = static_cast<uint16_t*>(v_cache);
  a.eps = eps;
  a.max_position = max_position;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.num_slots = num_slots;
  a.tile = tile + 1;
  return nvj::linear_qk_rope(static_cast<hipStream_t>(stream), a) == hipSuccess ? NVJ_OK
                                                                                 : NVJ_ERR_LAUNCH;
}
