// qfrag.h -- Q8_0 / Q4_0 values in MFMA fragment order (tile_q_kernel) to f16.
//
// The integers are exact in f16: an unsigned byte or nibble u placed in the low
// bits of 0x6400 is the f16 value 1024 + u, and one packed subtraction leaves
// u - 128 or u - 8 (Q8_0: 2 byte permutes and 2 subtractions per 4 values).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace s2 {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t f16_from_1024(uint32_t bits, _Float16 off) {
  const half2v o = {off, off};
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, bits) - o);
}

// 8 values from 8 bytes q + 128 (value e in byte e)
__device__ __forceinline__ half8v q8_frag(uint32_t x, uint32_t y) {
  const _Float16 off = _Float16(1152.0f);
  uint4 r;
  // byte i of the result from the selector's byte i: 0..3 pick x, 4..7 the 0x64s
  r.x = f16_from_1024(__builtin_amdgcn_perm(0x64646464u, x, 0x04010400u), off);
  r.y = f16_from_1024(__builtin_amdgcn_perm(0x64646464u, x, 0x04030402u), off);
  r.z = f16_from_1024(__builtin_amdgcn_perm(0x64646464u, y, 0x04010400u), off);
  r.w = f16_from_1024(__builtin_amdgcn_perm(0x64646464u, y, 0x04030402u), off);
  return __builtin_bit_cast(half8v, r);
}

// 8 values from 8 nibbles (value 2 j in nibble j, value 2 j + 1 in nibble j + 4)
__device__ __forceinline__ half8v q4_frag(uint32_t x) {
  const _Float16 off = _Float16(1032.0f);
  uint4 r;
  r.x = f16_from_1024((x & 0x000f000fu) | 0x64006400u, off);
  r.y = f16_from_1024(((x >> 4) & 0x000f000fu) | 0x64006400u, off);
  r.z = f16_from_1024(((x >> 8) & 0x000f000fu) | 0x64006400u, off);
  r.w = f16_from_1024(((x >> 12) & 0x000f000fu) | 0x64006400u, off);
  return __builtin_bit_cast(half8v, r);
}

}  // namespace s2
