// Mixed-precision one-instruction helpers and the nibble packer shared by the rotate+quantise
// kernels (gfx950 only).
#pragma once
#include "common.h"

namespace flh {

typedef unsigned short us2 __attribute__((ext_vector_type(2)));

// The scale of a row whose maximum is m (an fp16 value held as float), s = fp16(m / 7), and the float32 reciprocal
// the codes are computed with.  fp16(m * fl32(1/7)) equals fp16(m / 7) for every fp16 m, and the codes do not depend
// on the last bit of the reciprocal (both checked exhaustively on the host), so neither needs a division sequence.
__device__ __forceinline__ _Float16 scale_of_max(float m) { return (_Float16)(m * (1.0f / 7.0f)); }
__device__ __forceinline__ float reciprocal_of_scale(_Float16 s) { return __builtin_amdgcn_rcpf((float)s); }

// ---- mixed-precision helpers (one instruction each) ---------------------------------
// z - float(half `sel` of packed), float32
template <int SEL>
__device__ __forceinline__ float sub_half(float z, unsigned packed) {
  float d;
  if constexpr (SEL == 0) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(packed), "v"(z));
  else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(packed), "v"(z));
  return d;
}
// {fp16(float(y.lo) * r), fp16(float(y.hi) * r)}: the product is rounded once, to fp16
__device__ __forceinline__ unsigned mul_halves(unsigned y, float r) {
  unsigned d;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(y), "v"(r));
  asm("v_fma_mixhi_f16 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(d) : "v"(y), "v"(r));
  return d;
}
// {fp16(a * c), fp16(b * c)}: each product is rounded once, straight to fp16
__device__ __forceinline__ unsigned scale_pack_f16(float a, float b, float c) {
  unsigned d;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(c));
  asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(d) : "v"(b), "v"(c));
  return d;
}
__device__ __forceinline__ unsigned pack_f16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{a, b}, h2));
}

// Four fp16 quotients h (two packed registers) -> 16 bits of two's-complement nibbles, plus a
// known constant in the upper bits.  h + 1544 rounds to 1544 + rint(h) (fp16 spacing is 1
// there), whose bit pattern is 0x6608 + code; a dot product with (1, 16) / (256, 4096)
// lines the four low nibbles up.  Needs |rint(h)| <= 8, i.e. the caller's scale is not
// degenerate.  Returns sum (0x6600 + code_i + 8) 16^i.
__device__ __forceinline__ unsigned quad_nibbles(unsigned h01, unsigned h23) {
  const h2 magic = {(_Float16)1544.0f, (_Float16)1544.0f};
  const us2 a = __builtin_bit_cast(us2, __builtin_bit_cast(h2, h01) + magic);
  const us2 b = __builtin_bit_cast(us2, __builtin_bit_cast(h2, h23) + magic);
  unsigned t = __builtin_amdgcn_udot2(a, us2{1, 16}, 0u, false);
  return __builtin_amdgcn_udot2(b, us2{256, 4096}, t, false);
}
constexpr unsigned kQuadBias = 0x6600u * 0x1111u;                 // what quad_nibbles adds
constexpr unsigned kPairBias = kQuadBias + (kQuadBias << 16);     // for two quads, low | high << 16


// Eight fp16 values (four packed registers, ascending element order) -> one dword of eight
// two's-complement nibbles, element 0 in bits 0-3: rint(fp16(y * rinv)) per element.
// CAREFUL also clamps the values to +-bound and the quotients to [-8, 7]; it is needed only
// for clipping (clip_ratio < 1) or a subnormal scale, chosen once per row.
template <bool CAREFUL>
__device__ __forceinline__ unsigned quotients2(unsigned y, float rinv, h2 hb) {
  if constexpr (CAREFUL)
    y = __builtin_bit_cast(unsigned, __builtin_elementwise_min(__builtin_elementwise_max(__builtin_bit_cast(h2, y), -hb), hb));
  unsigned h = mul_halves(y, rinv);
  if constexpr (CAREFUL) {
    const h2 lo8 = {(_Float16)-8.0f, (_Float16)-8.0f}, hi7 = {(_Float16)7.0f, (_Float16)7.0f};
    h = __builtin_bit_cast(unsigned, __builtin_elementwise_min(__builtin_elementwise_max(__builtin_bit_cast(h2, h), lo8), hi7));
  }
  return h;
}
template <bool CAREFUL>
__device__ __forceinline__ unsigned nibbles8(unsigned y01, unsigned y23, unsigned y45, unsigned y67, float rinv, h2 hb) {
  unsigned t[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    t[u] = quad_nibbles(quotients2<CAREFUL>(u == 0 ? y01 : y45, rinv, hb), quotients2<CAREFUL>(u == 0 ? y23 : y67, rinv, hb));
  return ((t[1] << 16) + t[0] - kPairBias) ^ 0x88888888u;
}
// The largest |half| of N packed registers by the order of the bit patterns, in which a NaN is the largest: below infinity only if
// every value is finite (fmaxf and v_pk_max_f16 pass NaNs over).
template <int N>
__device__ __forceinline__ float abs_max_or_nan(const unsigned (&y)[N]) {
  us2 m = __builtin_bit_cast(us2, y[0] & 0x7FFF7FFFu);
#pragma unroll
  for (int i = 1; i < N; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(us2, y[i] & 0x7FFF7FFFu));
  return (float)__builtin_bit_cast(_Float16, m.x > m.y ? m.x : m.y);
}
// whether the lanes of a wave hold nothing but finite values, of which each gives its abs_max_or_nan
__device__ __forceinline__ bool all_finite(float m) { return __builtin_amdgcn_ballot_w64(!(m < INFINITY)) == 0; }
// rint of two fp16 quotients, as fp16 (zeros are +0): for the hardware's conversion to the 6-bit format
__device__ __forceinline__ unsigned whole2(unsigned h) {
  const h2 magic = {(_Float16)1544.0f, (_Float16)1544.0f};
  return __builtin_bit_cast(unsigned, (__builtin_bit_cast(h2, h) + magic) - magic);
}

}  // namespace flh
