// Scale of a group of G fp16 values held by G / 8 adjacent lanes, eight each: shared by the group quantisers and by the GEMM
// that quantises its own activations.
#pragma once
#include "lane_ops.h"
#include "quant_pack.h"

namespace flh {
namespace {

// which 16-byte chunk of its group a lane owns, by its position among the group's lanes: a relabelling with which every cross-lane
// stride is one DPP pattern (chunk bits b1, b2 flip with quad xor 1 / 2, b3 with the mirror inside 8 lanes, b4 with that inside 16)
template <int LPR>
__device__ __forceinline__ int group_chunk(int pos) {
  if constexpr (LPR <= 4) return pos;
  const int b1 = (pos ^ (pos >> 2)) & 1, b2 = ((pos >> 1) ^ (pos >> 2)) & 1;
  if constexpr (LPR == 8) return b1 | (b2 << 1) | (pos & 4);
  const int b3 = ((pos >> 2) ^ (pos >> 3)) & 1;
  return b1 | (b2 << 1) | (b3 << 2) | (pos & 8);
}

// max |v| over a lane's eight halves, as float: sign bits masked, three packed maxima, one across the pair
// (written out so that no canonicalising copies are added; NaNs are ignored as fmaxf ignores them)
__device__ __forceinline__ float lane_abs_max(const h2 (&v)[4]) {
  unsigned a[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = __builtin_bit_cast(unsigned, v[i]) & 0x7FFF7FFFu;
  unsigned m01, m23, m;
  asm("v_pk_max_f16 %0, %1, %2" : "=v"(m01) : "v"(a[0]), "v"(a[1]));
  asm("v_pk_max_f16 %0, %1, %2" : "=v"(m23) : "v"(a[2]), "v"(a[3]));
  asm("v_pk_max_f16 %0, %1, %2" : "=v"(m) : "v"(m01), "v"(m23));
  const h2 p = __builtin_bit_cast(h2, m);
  float lo = (float)p.x, hi = (float)p.y, r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}

// max(m, m of the partner lane) in one instruction (the DPP operand feeds the maximum directly; the two wait
// states a DPP read needs after the write of its source are spelled out, the assembler does not add them here)
template <int CTRL>
__device__ __forceinline__ float max_across(float m) {
  float r;
  if constexpr (CTRL == kDppQuadXor1)
    asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(m));
  else if constexpr (CTRL == kDppQuadXor2)
    asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(m));
  else if constexpr (CTRL == kDppRowHalfMirror)
    asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(m));
  else
    asm volatile("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 row_mirror row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(m));
  return r;
}

struct GroupScale {
  _Float16 s;
  float r;          // its reciprocal
  bool careful;     // the quotients of this wave have to be clamped
};
// m: the largest |value| of the lane
template <int LPR>
__device__ __forceinline__ GroupScale group_scale(float m) {
  m = max_across<kDppQuadXor1>(m);
  m = max_across<kDppQuadXor2>(m);
  if constexpr (LPR >= 8) m = max_across<kDppRowHalfMirror>(m);
  if constexpr (LPR >= 16) m = max_across<kDppRowMirror>(m);
  // no division sequences (see scale_of_max): a lane has only eight values to spread them over
  GroupScale g;
  g.s = scale_of_max(m);
  if (g.s <= (_Float16)1e-6f) g.s = (_Float16)1.0f;
  g.r = reciprocal_of_scale(g.s);
  // |y / s| <= 7.004 unless the scale is subnormal: only then (any row of this wave) clamp the quotients
  g.careful = __builtin_amdgcn_ballot_w64((float)g.s < 6.2e-5f) != 0;
  return g;
}

}  // namespace
}  // namespace flh
