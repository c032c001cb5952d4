// Copies from global memory straight into LDS, without staging registers.
#ifndef NVJ_LDS_COPY_H_
#define NVJ_LDS_COPY_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvj {

// One 16-byte copy per lane: lane l's piece lands at lds_base + 16 * l (lds_base
// wave-uniform), fetched from base + offset.  Counts in vmcnt like any load; the compiler
// does not see it as one, so the waits are written out by hand.
//
// m0 is named as overwritten, so that nothing the compiler may keep there is set in front of
// this and used behind it.  It warns that m0 is a reserved register, whose value it will not
// restore; nothing here relies on that.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void copy16_to_lds(const char* base, uint32_t offset,
                                              uint32_t lds_base) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(lds_base), "v"(offset), "s"(base)
      : "memory", "m0");
}
// The same with 4 bytes per lane: lane l's lands at lds_base + 4 * l.
__device__ __forceinline__ void copy4_to_lds(const void* base, uint32_t offset,
                                             uint32_t lds_base) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %1, %2"
      :
      : "s"(lds_base), "v"(offset), "s"(base)
      : "memory", "m0");
}
#pragma clang diagnostic pop

}  // namespace nvj

#endif  // NVJ_LDS_COPY_H_
