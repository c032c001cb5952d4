// Reductions over the 64 lanes of a wave with DPP moves and lane swaps (through LDS, as shuffles do
// it, each step is a round trip).
#ifndef NVJ_WAVE_OPS_H_
#define NVJ_WAVE_OPS_H_

#include <hip/hip_runtime.h>

namespace nvj {

// Inclusive prefix sum over the 64 lanes of a wave with DPP moves: a
// Hillis-Steele scan inside each row of 16 lanes (a lane without a source in
// its row adds 0), then the last lane of row 0 / row 2 is added to rows 1 / 3
// (row_bcast:15) and the last lane of row 1 to rows 2 and 3 (row_bcast:31).
__device__ __forceinline__ int wave_inclusive_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 -> rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 -> rows 2, 3
  return x;
}

// Maximum over the 64 lanes of a wave, wave-uniform, with the same DPP moves (a
// lane without a source keeps its own value).
__device__ __forceinline__ int wave_max(int x) {
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x111, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x112, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x114, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x118, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x142, 0xA, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(x, x, 0x143, 0xC, 0xF, false));
  return __builtin_amdgcn_readlane(x, 63);
}

// combine(x, x of the lane MASK = 16 or 32 away), for a combine whose operands may change places: the
// halves of a swap of x with itself are the two.  (A shuffle is a round trip through LDS: decode of one
// sequence of 768 positions 7.67 -> 7.53 us, of 8 of 100 .. 1500 11.0 -> 10.8.)
template <int MASK, typename Combine>
__device__ __forceinline__ float wave_combine(float x, Combine combine) {
  static_assert(MASK == 16 || MASK == 32, "rows of 16 lanes or halves of the wave");
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto halves = MASK == 32 ? __builtin_amdgcn_permlane32_swap(u, u, false, false)
                                 : __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned lower = halves[0], upper = halves[1];   // (a bit cast of halves[1] takes halves[0])
  return combine(__builtin_bit_cast(float, lower), __builtin_bit_cast(float, upper));
}
template <int MASK> __device__ __forceinline__ float wave_xor_add(float x) {
  return wave_combine<MASK>(x, [](float a, float b) { return a + b; });
}
template <int MASK> __device__ __forceinline__ float wave_xor_max(float x) {
  return wave_combine<MASK>(x, [](float a, float b) { return fmaxf(a, b); });
}

// x of another lane of the row of 16 (a DPP control)
template <int CTRL> __device__ __forceinline__ float row_move(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL,
                                                               0xF, 0xF, false));
}

// Sum over the 64 lanes, in every lane, by a butterfly over the masks 32, 16, .. 1.  (Once lanes i
// and i ^ 8 are equal, i ^ 4 is the lane 4 places on.)
__device__ __forceinline__ float wave_sum(float x) {
  x = wave_xor_add<32>(x);
  x = wave_xor_add<16>(x);
  x += row_move<0x128>(x);   // row_ror:8
  x += row_move<0x124>(x);   // row_ror:4
  x += row_move<0x4E>(x);    // i ^ 2
  x += row_move<0xB1>(x);    // i ^ 1
  return x;
}

}  // namespace nvj

#endif  // NVJ_WAVE_OPS_H_
