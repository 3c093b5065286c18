// The 6-bit (e3m2) encoding of int4 codes used by the operands of the 6-bit matrix instruction.
#pragma once
#include "lane_ops.h"

namespace flh {

constexpr int kF6BlockBytes = 96;   // encoded bytes of 128 codes of one row

// Eight int4 nibbles of one dword (two's complement; nibble j in bits 4 j) -> 48 bits of e3m2 codes, code j at
// bit 6 j.  A code is sign << 5 | {0, 12, 16, 18, 20, 21, 22, 23, 24}[magnitude]: a 16-entry byte table, looked up
// four nibbles at a time with two byte permutes (entries 0..7 and 8..15) and a bit select on the nibble's top bit.
__device__ __forceinline__ unsigned long long bf6_of_nibbles(unsigned w) {
  constexpr unsigned kPosLo = 0x12100C00u, kPosHi = 0x17161514u;   //  0 ..  7
  constexpr unsigned kNegLo = 0x35363738u, kNegHi = 0x2C303234u;   // -8 .. -1
  auto lut = [&](unsigned x) {                         // four nibbles, one per byte
    const unsigned sel = x & 0x07070707u;
    const unsigned pos = __builtin_amdgcn_perm(kPosHi, kPosLo, sel), neg = __builtin_amdgcn_perm(kNegHi, kNegLo, sel);
    const unsigned mask = ((x >> 3) & 0x01010101u) * 0xFFu;
    return (neg & mask) | (pos & ~mask);
  };
  const unsigned L = lut(w & 0x0F0F0F0Fu), H = lut((w >> 4) & 0x0F0F0F0Fu);   // codes 0,2,4,6 and 1,3,5,7
  // pairs p_i = code(2 i) | code(2 i + 1) << 6 in 16-bit lanes
  const unsigned X = (L & 0x00FF00FFu) | ((H & 0x00FF00FFu) << 6);           // p0, p2
  const unsigned Y = ((L >> 8) & 0x00FF00FFu) | (((H >> 8) & 0x00FF00FFu) << 6);   // p1, p3
  const unsigned long long p0 = X & 0xFFFu, p2 = X >> 16, p1 = Y & 0xFFFu, p3 = Y >> 16;
  return p0 | (p1 << 12) | (p2 << 24) | (p3 << 36);
}

// 32 whole numbers in -8 .. 7 as fp16 pairs -> their 6-bit codes, code k at bits 6 k of 192 (one instruction, 64 clocks; the table
// above takes 35 instructions for eight)
typedef unsigned u6 __attribute__((ext_vector_type(6)));
__device__ __forceinline__ u6 bf6_of_wholes(const unsigned (&h)[16]) {
  typedef unsigned u16 __attribute__((ext_vector_type(16)));
  typedef _Float16 h32 __attribute__((ext_vector_type(32)));
  u16 v;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = h[i];
  return __builtin_amdgcn_cvt_scalef32_pk32_bf6_f16(__builtin_bit_cast(h32, v), 1.0f);
}
// bytes from a block's start to the six of its chunk of eight codes c16 = 0 .. 15
__device__ __forceinline__ int f6_chunk_at(int c16) { return 48 * ((c16 >> 2) & 1) + 24 * (c16 >> 3) + 6 * (c16 & 3); }
typedef unsigned u32_at2 __attribute__((aligned(2)));
// chunk k = 0 .. 3 of what bf6_of_wholes gave
template <int K>
__device__ __forceinline__ void f6_store_six(const u6& r, uint8_t* dst) {
  constexpr int w = K / 2 * 3;
  if constexpr (K % 2 == 0) {
    *(u32_at2*)dst = r[w];
    *(unsigned short*)(dst + 4) = (unsigned short)r[w + 1];
  } else {
    *(u32_at2*)dst = __builtin_amdgcn_alignbit(r[w + 2], r[w + 1], 16);
    *(unsigned short*)(dst + 4) = (unsigned short)(r[w + 2] >> 16);
  }
}
// The eight codes of a chunk from their nibbles.  For rows that are not finite throughout: the quotient of a NaN, or of an infinity,
// is a NaN, of which the nibble packer makes some code (and, by carries, something of its neighbours) and the conversion
// another one.  By way of the nibbles both formats hold the same codes.
__device__ __forceinline__ void f6_store_nibbles(unsigned w, uint8_t* dst) {
  const unsigned long long codes = bf6_of_nibbles(w);
  *(u32_at2*)dst = (unsigned)codes;
  *(unsigned short*)(dst + 4) = (unsigned short)(codes >> 32);
}

}  // namespace flh
