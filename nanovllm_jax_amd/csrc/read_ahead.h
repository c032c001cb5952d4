// Memory that a launch reads on behalf of the launches behind it.
//
// The products of a decoder layer wait for their weights: a layer's 31 MB (hidden 1024) come
// from HBM on every step, and a launch asks for them only when it starts.  Workgroups
// behind a launch's own read the weights of the next products meanwhile, into the Infinity
// Cache and the L2s, while HBM has nothing else to do.  Nothing depends on it: what has not
// arrived, or has been displaced, is fetched as before.
#ifndef NVJ_READ_AHEAD_H_
#define NVJ_READ_AHEAD_H_

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "lds_copy.h"

namespace nvj {

// Up to kRegions regions of count[i] chunks of bytes[i] bytes each (a multiple of 16), a
// workgroup per chunk.
struct ReadAhead {
  static constexpr int kRegions = 5;
  const char* base[kRegions];
  int bytes[kRegions], count[kRegions];
  int used;

  int64_t total() const {
    int64_t n = 0;
    for (int i = 0; i < used; ++i) n += (int64_t)bytes[i] * count[i];
    return n;
  }
  unsigned chunks() const {
    unsigned n = 0;
    for (int i = 0; i < used; ++i) n += (unsigned)count[i];
    return n;
  }
  // The rows of a bf16 matrix, `rows_per_chunk` to a chunk; nothing where they do not divide.
  void add_matrix(const void* w, int64_t rows, int64_t columns, int rows_per_chunk) {
    if (used == kRegions || rows % rows_per_chunk != 0 || columns % 8 != 0) return;
    base[used] = static_cast<const char*>(w);
    bytes[used] = (int)(columns * 2 * rows_per_chunk);
    count[used++] = (int)(rows / rows_per_chunk);
  }
};

// One chunk, by a workgroup of THREADS; `chunk` counts through the regions.
template <int THREADS>
__device__ __forceinline__ void read_chunk(const ReadAhead& ahead, int chunk) {
#pragma unroll
  for (int i = 0; i < ReadAhead::kRegions; ++i) {
    if (chunk >= 0 && chunk < ahead.count[i]) {
      const char* from = ahead.base[i] + (int64_t)chunk * ahead.bytes[i];
      for (int at = 16 * threadIdx.x; at < ahead.bytes[i]; at += 4 * 16 * THREADS) {
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          v[u] = *reinterpret_cast<const uint4*>(from +
                                                 min(at + u * 16 * THREADS, ahead.bytes[i] - 16));
#pragma unroll
        for (int u = 0; u < 4; ++u)   // (the values are needed by nobody, the reads are)
          asm volatile("" ::"v"(v[u].x), "v"(v[u].y), "v"(v[u].z), "v"(v[u].w));
      }
    }
    chunk -= ahead.count[i];
  }
}

// The same by way of LDS (1 KB a wave, from `lds`), for kernels whose registers leave a CU one such
// workgroup at a time: nothing waits between the reads of a chunk.  us a step with registers / LDS
// in the attention of a layer of 1024 (3072), a graph: 1 sequence of 100 positions 916 / 882, 4 of
// 100 .. 900 1009 / 991, 2 of 2000 1057 / 1037, 6 of 900 1194 / 1161, 8 of 1000 1280 / 1258, and 1
// of 500, 16 of 100 .. 400, 4 of 3000 938 / 940, 1186 / 1182, 1206 / 1212.  (Fewer workgroups with
// several chunks each: 80 .. 256 of them within 2 % either way.)  In the norms, whose chunks are
// two batches of registers: 24 of 100 .. 900 1451 / 1440, 100 of 200 .. 400 1848 / 1828, 128 of 1024
// 3325 / 3310, a prompt of 200 tokens 1571 / 1550.  (Not in the products: 4268 tokens -0.3 %, 24 rows
// +1 %.)
template <int THREADS>
__device__ __forceinline__ void read_chunk_by_lds(const ReadAhead& ahead, int chunk, uint32_t lds) {
  lds += (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 1024u;
#pragma unroll
  for (int i = 0; i < ReadAhead::kRegions; ++i) {
    if (chunk >= 0 && chunk < ahead.count[i]) {
      const char* from = ahead.base[i] + (int64_t)chunk * ahead.bytes[i];
      for (int at = 16 * threadIdx.x; at < ahead.bytes[i]; at += 16 * THREADS)
        copy16_to_lds(from, (uint32_t)at, lds);
    }
    chunk -= ahead.count[i];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing may land in LDS that is another's
}

// nvj_paged_decode_launch_counters; where the launch takes the kernel for few sequences, with
// memory to read by workgroups behind its own.
int paged_decode_launch_ahead(void* stream, const void* q, const void* k_cache,
                              const void* v_cache, const int32_t* block_tables,
                              const int32_t* context_lens, void* out, void* partials,
                              size_t partial_bytes, void* counters, size_t counter_bytes,
                              int32_t batch, int32_t num_heads, int32_t num_kv_heads,
                              int32_t head_dim, int32_t block_size, int32_t max_blocks,
                              int32_t num_blocks, float scale, int32_t dtype, uint32_t phases,
                              const ReadAhead* ahead);

// nvj_add_rms_norm_launch, with memory to read by workgroups behind its own.
int add_rms_norm(void* stream, const void* x, const void* residual, const float* weight, float eps,
                 void* y, void* residual_out, int32_t num_tokens, int32_t hidden,
                 const ReadAhead& ahead);

}  // namespace nvj

#endif  // NVJ_READ_AHEAD_H_
