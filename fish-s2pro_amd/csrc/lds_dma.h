// lds_dma.h -- loads from memory straight to LDS (global_load_lds) and the waits
// for them, for the pipelined products and convolutions.
//
// Written as inline assembly so that the compiler does not treat every later LDS
// read as dependent on a load (it would wait for all loads in flight first); the
// kernels wait for these loads themselves (vmcnt) before the barrier that publishes
// a stage.  The destination goes through m0, which the statements clobber.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace s2 {

// s_waitcnt immediate: at most `v` vector memory loads in flight, LDS reads
// drained if `lgkm0`
constexpr int wait_imm(int v, bool lgkm0) { return (v & 15) | ((v >> 4) << 14) | 0x70 | (lgkm0 ? 0 : 0xF00); }

// (the compiler reserves m0 and says so for every instance of a clobber list that
// names it; it has to be named for the compiler's own writes of m0 to be kept apart)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"

// 16 bytes per lane from `base` (wave-uniform) + `off` into the wave's 1 KiB at LDS
// byte `lds` (lane i at byte 16 i).
__device__ __forceinline__ void dma16(const uint8_t* base, uint32_t off, uint32_t lds) {
  asm volatile("s_nop 1\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds), "v"(off), "s"(base)
               : "memory", "m0");
}

// The same with an address per lane (W bytes: 16 or 4 per lane).
template <int W>
__device__ __forceinline__ void dma_lane(const uint8_t* src, uint32_t lds) {
  if constexpr (W == 16)
    asm volatile("s_nop 1\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(lds), "v"(src)
                 : "memory", "m0");
  else
    asm volatile("s_nop 1\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
                 :
                 : "s"(lds), "v"(src)
                 : "memory", "m0");
}

#pragma clang diagnostic pop

}  // namespace s2
