// Walsh-Hadamard rotation, symmetric int4 quantisation and nibble packing of fp16 rows.
//
// Three families of kernels live here:
//
//  1. group kernels (rows of G = 32 / 64 / 128 fp16) with the arithmetic of the
//     reference's CUDA kernels: every butterfly rounded to fp16, s = fp16(max / 7),
//     s <= fp16(1e-6) -> 1, q = clamp(rint(fp16(y / s)), -8, 7)
//     (flh/kernels/had_and_quant.cu:13-155, quant_and_pack.cu:8-97, cuda_had_kernel.cu:190-354);
//  2. the wave-per-row kernel for whole rows of K = 512 * J fp16 (J = 1 .. 16): butterflies
//     in float32 in ascending stride order, so that the fp16 result equals the float32
//     restatement of had_transform (flh/nn/quantization.py:42-74) bit for bit; strides
//     1, 2, 4 and >= 512 are register-to-register, strides 8 .. 256 cross lanes with DPP
//     (quad permutes, row mirrors) and v_permlane16/32_swap -- no LDS, no barrier;
//  3. a generic workgroup-per-row kernel (any K = Kd * 2^m, Kd one of the literal
//     Hadamard sizes, grouped rotation, grouped scales), staged in LDS.
//
// Quantisation (all kernels): the fp16 quotient y / s is needed only through
// rint(fp16(y / s)).  For every pair of fp16 values the code obtained from
// fp16(float(y) * r), r = the float32 reciprocal of s (even when r is off by one ulp),
// equals the code from the correctly rounded fp16 quotient -- verified exhaustively over
// all 6.3e8 (y, s) pairs with |y / s| <= 20 on the host (tests/native/divcheck.c).
#include <atomic>
#include <cstdlib>
#include <type_traits>
#include "lane_ops.h"
#include "quant_pack.h"
#include "group_codes.h"
#include "encode_f6.h"
#include "f6_codes.h"
#include "rotate_row.h"

namespace flh {
namespace {

#include "hadk_tables.inc"

__device__ __forceinline__ const uint8_t* hadk_bits(int kd) {
  switch (kd) {
    case 12: return kHad12Bits;
    case 20: return kHad20Bits;
    case 28: return kHad28Bits;
    case 36: return kHad36Bits;
    case 40: return kHad40Bits;
    case 52: return kHad52Bits;
    case 60: return kHad60Bits;
    case 108: return kHad108Bits;
    case 140: return kHad140Bits;
    case 156: return kHad156Bits;
    case 172: return kHad172Bits;
    default: return nullptr;
  }
}

// code in [-8, 7] of an fp16 value y for reciprocal scale r, as a nibble
__device__ __forceinline__ unsigned quant_nibble(_Float16 y, float r) {
  const _Float16 h = (_Float16)((float)y * r);
  float c = __builtin_rintf((float)h);
  c = fminf(fmaxf(c, -8.f), 7.f);
  return (unsigned)(int)c & 0xFu;
}

// ------------------------------------------------------------------------------------
// 1. group kernels, fp16 butterflies.  One lane owns 8 consecutive values (16 bytes), G/8
//    adjacent lanes own a row.  Which chunk of the row a lane owns is a relabelling of its
//    position, chosen so that every cross-lane stride is ONE DPP pattern: chunk bits b1, b2
//    flip with quad xor 1 / 2, b3 with the mirror inside 8 lanes, b4 with the mirror inside 16:
//    position = b1*0001 ^ b2*0010 ^ b3*0111 ^ b4*1111.
// ------------------------------------------------------------------------------------
// butterfly with the partner lane of pattern CTRL: lower lane v + o, upper lane o - v, both as one
// packed fused multiply-add v * (+-1) + o (the product is exact, so the rounding is that of the sum)
template <int CTRL>
__device__ __forceinline__ void group_cross(h2 (&v)[4], bool upper) {
  const _Float16 sg = upper ? (_Float16)-1.0f : (_Float16)1.0f;
  const h2 sgn = {sg, sg};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const h2 o = __builtin_bit_cast(h2, dpp_i<CTRL>(__builtin_bit_cast(int, v[i])));
    v[i] = __builtin_elementwise_fma(v[i], sgn, o);
  }
}

template <int G>
__device__ __forceinline__ void fwht_group_f16(h2 (&v)[4], int chunk) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = h2{(_Float16)(v[i].x + v[i].y), (_Float16)(v[i].x - v[i].y)};
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const h2 a = v[i], b = v[i + 1];
    v[i] = a + b;
    v[i + 1] = a - b;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const h2 a = v[i], b = v[i + 2];
    v[i] = a + b;
    v[i + 2] = a - b;
  }
  group_cross<kDppQuadXor1>(v, chunk & 1);
  group_cross<kDppQuadXor2>(v, chunk & 2);
  if constexpr (G >= 64) group_cross<kDppRowHalfMirror>(v, chunk & 4);
  if constexpr (G >= 128) group_cross<kDppRowMirror>(v, chunk & 8);
}

// scale, codes and stores of one row of G values held by LPR = G / 8 adjacent lanes (this lane: chunk `lir`)
//
// F6 (G = 128 only): the codes leave in the operand format of the 6-bit matrix instruction instead -- 6 bits per
// code, the 96-byte block of this group at ((row % groups_per_token) * tokens + row / groups_per_token) * 96
// (K-slab-major, see gemm_f6.hip), a lane's eight as six bytes.  The conversion is the hardware's, a quarter full (18432 groups
// rotated 4.28 -> 4.03 us against a table and eight-byte stores behind an exchange between lanes).
//
// FINITE (F6): every value in this wave is.  m: the largest one of the lane.
template <int G, bool F6, bool OFF32, bool FINITE>
__device__ __forceinline__ void group_finish_from(float m, const h2 (&v)[4], int lir, bool valid, uint32_t row, uint8_t* __restrict__ q,
                                                  __half* __restrict__ scales, float scale_mul, uint32_t tokens,
                                                  uint32_t groups_per_token) {
  static_assert(!F6 || G == 128, "one 6-bit block is 128 codes");
  constexpr int LPR = G / 8;
  const GroupScale scale = group_scale<LPR>(m);
  const _Float16 s = scale.s;
  const float r = scale.r;
  const bool careful = scale.careful;
  const h2 hb = {(_Float16)65504.0f, (_Float16)65504.0f};   // no clipping in the group kernels
  const unsigned y01 = __builtin_bit_cast(unsigned, v[0]), y23 = __builtin_bit_cast(unsigned, v[1]),
                 y45 = __builtin_bit_cast(unsigned, v[2]), y67 = __builtin_bit_cast(unsigned, v[3]);
  unsigned w = 0;
  u6 six;
  if constexpr (F6 && FINITE) {
    unsigned h[16] = {};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned y = __builtin_bit_cast(unsigned, v[i]);
      h[i] = whole2(careful ? quotients2<true>(y, r, hb) : quotients2<false>(y, r, hb));
    }
    six = bf6_of_wholes(h);
  } else {
    w = careful ? nibbles8<true>(y01, y23, y45, y67, r, hb) : nibbles8<false>(y01, y23, y45, y67, r, hb);
  }
  if (valid) {
    using offset_t = std::conditional_t<OFF32, uint32_t, size_t>;
    if constexpr (F6) {
      const size_t block = (size_t)(row % groups_per_token) * tokens + row / groups_per_token;
      uint8_t* dst = q + block * kF6BlockBytes + f6_chunk_at(lir);
      if constexpr (FINITE) f6_store_six<0>(six, dst);
      else f6_store_nibbles(w, dst);
    } else {
      *(unsigned*)(q + ((offset_t)row * (LPR * 4) + (offset_t)lir * 4)) = w;
    }
    // the stored scale may carry a constant factor (the reference divides its scales by sqrt(G) in a
    // second kernel after the unnormalised transform): float32 product, then fp16; the codes above use s
    if (lir == 0) *(__half*)((char*)scales + (offset_t)row * 2) = scale_mul == 1.0f ? __builtin_bit_cast(__half, s) : __float2half(round_here((float)s * scale_mul));
  }
}

template <int G, bool F6 = false, bool OFF32 = false>
__device__ __forceinline__ void group_finish(const h2 (&v)[4], int lir, bool valid, uint32_t row, uint8_t* __restrict__ q,
                                             __half* __restrict__ scales, float scale_mul, uint32_t tokens = 0,
                                             uint32_t groups_per_token = 1) {
  if constexpr (F6) {
    unsigned y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = __builtin_bit_cast(unsigned, v[i]);
    const float m = abs_max_or_nan(y);
    if (__builtin_expect(all_finite(m), 1)) {
      group_finish_from<G, F6, OFF32, true>(m, v, lir, valid, row, q, scales, scale_mul, tokens, groups_per_token);
      return;
    }
  }
  group_finish_from<G, F6, OFF32, false>(lane_abs_max(v), v, lir, valid, row, q, scales, scale_mul, tokens, groups_per_token);
}

template <int G, bool OFF32>
__device__ __forceinline__ void load_chunk(const __half* src, uint32_t row, int lir, h2 (&v)[4]) {
  using offset_t = std::conditional_t<OFF32, uint32_t, size_t>;
  const h8 raw = *(const h8*)((const char*)src + ((offset_t)row * (G * 2) + (offset_t)lir * 16));
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = h2{raw[2 * i], raw[2 * i + 1]};
}
// one group by its G / 8 lanes (every lane of the wave has to call it; rows past the end work on the last one and store nothing)
template <int G, bool HAD, bool F6, bool OFF32 = false>
__device__ __forceinline__ void quantise_group(const __half* x, uint8_t* q, __half* scales, uint32_t row, int lir, uint32_t R,
                                               float scale_mul, uint32_t tokens, uint32_t groups_per_token) {
  const bool valid = row < R;
  h2 v[4];
  load_chunk<G, OFF32>(x, valid ? row : R - 1, lir, v);
  if constexpr (HAD) fwht_group_f16<G>(v, lir);
  group_finish<G, F6, OFF32>(v, lir, valid, row, q, scales, scale_mul, tokens, groups_per_token);
}

// OFF32: every byte offset of the launch fits 32 bits, so that the addresses are a scalar base plus a 32-bit lane
// offset (the instruction count of these kernels is what bounds them: eight values per lane, ~170 instructions).
template <int G, bool HAD, bool QUANT, bool F6 = false, bool OFF32 = false>
__global__ __launch_bounds__(256) void group_kernel(const __half* __restrict__ x, uint8_t* __restrict__ q,
                                                    __half* __restrict__ scales, __half* __restrict__ y_inplace,
                                                    uint32_t R, float scale_mul, uint32_t tokens = 0,
                                                    uint32_t groups_per_token = 1) {
  constexpr int LPR = G / 8;
  using offset_t = std::conditional_t<OFF32, uint32_t, size_t>;
  const uint32_t gl = blockIdx.x * 256u + threadIdx.x;
  const uint32_t row = gl / LPR;
  const int lir = group_chunk<LPR>(gl % LPR);         // the chunk of the row this lane owns
  if constexpr (!QUANT) {
    const bool valid = row < R;
    h2 v[4];
    load_chunk<G, OFF32>(y_inplace, valid ? row : R - 1, lir, v);
    fwht_group_f16<G>(v, lir);
    h8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = v[i].x;
      o[2 * i + 1] = v[i].y;
    }
    if (valid) *(h8*)((char*)y_inplace + ((offset_t)row * (G * 2) + (offset_t)lir * 16)) = o;
  } else {
    quantise_group<G, HAD, F6, OFF32>(x, q, scales, row, lir, R, scale_mul, tokens, groups_per_token);
  }
}

// SwiGLU in front of the group kernel: x = fp16( float(fp16(silu(gate))) * float(up) ) -- the two roundings
// of torch's fp16 silu and fp16 multiply (flh/quantized_model/modeling_llama.py:522-526 feeds exactly this
// product to the quantiser of down_proj) -- then transform + quantise as group_kernel<G, HAD, true>.
template <int G, bool HAD, bool F6 = false>
__global__ __launch_bounds__(256) void silu_mul_group_kernel(const __half* __restrict__ gate,
                                                             const __half* __restrict__ up, uint8_t* __restrict__ q,
                                                             __half* __restrict__ scales, uint32_t R, float scale_mul,
                                                             uint32_t tokens = 0, uint32_t groups_per_token = 1) {
  constexpr int LPR = G / 8;
  const uint32_t gl = blockIdx.x * 256u + threadIdx.x;
  const uint32_t row = gl / LPR;
  const int lir = group_chunk<LPR>(gl % LPR);
  const bool valid = row < R;
  const uint32_t rr = valid ? row : R - 1;
  const h8 g8 = *(const h8*)(gate + (size_t)rr * G + lir * 8);
  const h8 u8 = *(const h8*)(up + (size_t)rr * G + lir * 8);
  h2 v[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const _Float16 prod = silu_mul_f16(g8[i], u8[i]);
    if (i & 1) v[i >> 1].y = prod;
    else v[i >> 1].x = prod;
  }
  if constexpr (HAD) fwht_group_f16<G>(v, lir);
  group_finish<G, F6>(v, lir, valid, row, q, scales, scale_mul, tokens, groups_per_token);
}

// The group kernels for groups of 128 and launches that fill the chip: FOUR lanes own a group, 32 values each (lane p the
// chunks p, p + 4, p + 8, p + 12), so that of the seven butterfly strides only 8 and 16 cross lanes, and the row's maximum,
// scale and reciprocal are computed by four lanes instead of sixteen.  A lane's four code words are turned inside its wave
// through LDS, so that it stores sixteen consecutive bytes (32 codes; 6-bit output: the whole numbers are, and a lane converts
// and stores one 24-byte piece).  Same operations in the same order as group_kernel, the same bytes.
// What bounds it: memory.  4096-wide rows rotated and quantised, us, sixteen lanes -> four, replayed over inputs that together
// don't fit the last-level cache: 16384 rows 34.9 -> 31.8 (5.3 TB/s read + write), 8192 19.2 -> 17.1, 4096 11.2 -> 10.0; 6-bit output
// 524288 groups 52 -> 41, 65536 9.2 -> 7.2 (of which a table in the conversion's place takes 7 and 0.9, six-byte stores without the
// turn through LDS 17).  The sixteen-lane form is bound by its 165 instructions per eight values, 80 here.  Non-temporal loads and
// stores: equal or slower.  The SwiGLU product in front of it: 55.6 against 51.4 us, its exponentials want the sixteen lanes'
// parallelism; not here.
constexpr uint32_t kQuadRows = 64;                    // groups per workgroup of four waves
template <int CTRL>
__device__ __forceinline__ void quad_cross(h2 (&v)[4][4], _Float16 sg) {
  const h2 sgn = {sg, sg};
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const h2 o = __builtin_bit_cast(h2, dpp_i<CTRL>(__builtin_bit_cast(int, v[j][i])));
      v[j][i] = __builtin_elementwise_fma(v[j][i], sgn, o);
    }
}
__device__ __forceinline__ void butterfly(h2& a, h2& b) {
  const h2 s = a + b, d = a - b;
  a = s, b = d;
}
template <bool F6>
constexpr int kQuadWords = 256 * (F6 ? 16 : 4);          // LDS of a workgroup
template <bool HAD, bool F6>
__device__ __forceinline__ void group_quad_block(uint32_t block, const __half* __restrict__ x, uint8_t* __restrict__ q,
                                                 __half* __restrict__ scales, uint32_t R, float scale_mul, uint32_t tokens,
                                                 uint32_t groups_per_token, unsigned* turned) {
  const int tid = threadIdx.x, p = tid & 3;
  const uint32_t row0 = block * kQuadRows, row = row0 + (tid >> 2);
  const bool valid = row < R;
  const uint32_t at = ((valid ? row : R - 1) - row0) * 256 + p * 16;   // bytes from the workgroup's first group
  const char* xb = (const char*)x + (size_t)row0 * 256;
  h2 v[4][4];                                          // [chunk][pair]
  h8 raw[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) raw[j] = *(const h8*)(xb + (at + j * 64));
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[j][i] = h2{raw[j][2 * i], raw[j][2 * i + 1]};
  if constexpr (HAD) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {                    // {a + b, a - b} of a pair, one instruction
        unsigned d;
        asm("v_pk_add_f16 %0, %1, %1 op_sel:[0,1] op_sel_hi:[0,1] neg_hi:[0,1]" : "=v"(d) : "v"(__builtin_bit_cast(unsigned, v[j][i])));
        v[j][i] = __builtin_bit_cast(h2, d);
      }
      butterfly(v[j][0], v[j][1]), butterfly(v[j][2], v[j][3]);
      butterfly(v[j][0], v[j][2]), butterfly(v[j][1], v[j][3]);
    }
    quad_cross<kDppQuadXor1>(v, p & 1 ? (_Float16)-1.0f : (_Float16)1.0f);
    quad_cross<kDppQuadXor2>(v, p & 2 ? (_Float16)-1.0f : (_Float16)1.0f);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      butterfly(v[0][i], v[1][i]), butterfly(v[2][i], v[3][i]);
      butterfly(v[0][i], v[2][i]), butterfly(v[1][i], v[3][i]);
    }
  }
  unsigned y[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) y[i] = __builtin_bit_cast(unsigned, v[i >> 2][i & 3]);
  float m = abs_max_or_nan(y);
  if (__builtin_expect(!all_finite(m), 0)) {
    // What becomes of NaNs and infinities depends on the operand order of every addition and on which groups share a wave (see
    // `careful`): the wave's sixteen groups once more, as the sixteen-lane kernel takes them.
    const int lane = tid & 63;
    for (int i = 0; i < 16; i += 4)
      quantise_group<128, HAD, F6>(x, q, scales, row0 + (tid >> 6) * 16 + i + (lane >> 4), group_chunk<16>(lane & 15), R, scale_mul, tokens,
                                   groups_per_token);
    return;
  }
  m = max_across<kDppQuadXor1>(m);
  m = max_across<kDppQuadXor2>(m);
  _Float16 s = scale_of_max(m);
  if (s <= (_Float16)1e-6f) s = (_Float16)1.0f;
  const float r = reciprocal_of_scale(s);
  const bool careful = __builtin_amdgcn_ballot_w64((float)s < 6.2e-5f) != 0;   // as in group_finish
  const h2 hb = {(_Float16)65504.0f, (_Float16)65504.0f};
  if constexpr (F6) {
    unsigned h[16];
    auto wholes = [&](auto careful_tag) {
#pragma unroll
      for (int i = 0; i < 16; ++i) h[i] = whole2(quotients2<decltype(careful_tag)::value>(y[i], r, hb));
    };
    if (careful) wholes(std::true_type{});
    else wholes(std::false_type{});
    // the group's sixteen chunks, places of row and column XORed by the group: no bank conflicts either way
    const int g = (tid >> 2) & 3;
    v4i* const line = (v4i*)turned + (tid >> 2) * 16;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      line[4 * (j ^ g) + (p ^ g)] = v4i{(int)h[4 * j], (int)h[4 * j + 1], (int)h[4 * j + 2], (int)h[4 * j + 3]};
    __builtin_amdgcn_wave_barrier();                   // (the wave's own, LDS operations of a wave complete in order)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const v4i o = line[4 * (p ^ g) + (k ^ g)];
#pragma unroll
      for (int i = 0; i < 4; ++i) h[4 * k + i] = (unsigned)o[i];
    }
    if (!valid) return;
    const u6 six = bf6_of_wholes(h);
    const size_t block = (size_t)(row % groups_per_token) * tokens + row / groups_per_token;
    v2i* dst = (v2i*)(q + block * kF6BlockBytes + 48 * (p & 1) + 24 * (p >> 1));
#pragma unroll
    for (int i = 0; i < 3; ++i) dst[i] = v2i{(int)six[2 * i], (int)six[2 * i + 1]};
    if (p == 0) scales[row] = scale_mul == 1.0f ? __builtin_bit_cast(__half, s) : __float2half(round_here((float)s * scale_mul));
    return;
  }
  unsigned w[4];
  auto codes = [&](auto careful_tag) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = nibbles8<decltype(careful_tag)::value>(y[4 * j], y[4 * j + 1], y[4 * j + 2], y[4 * j + 3], r, hb);
  };
  if (careful) codes(std::true_type{});
  else codes(std::false_type{});
  // the group's sixteen words, blocks of four swapped by the group's place in the wave: no bank conflicts
  const int swap = (tid >> 4) & 3;
  unsigned* const line = turned + (tid >> 2) * 16;
#pragma unroll
  for (int j = 0; j < 4; ++j) line[4 * (j ^ swap) + p] = w[j];
  __builtin_amdgcn_wave_barrier();                     // (the wave's own words, LDS operations of a wave complete in order)
  const v4i o = *(const v4i*)(line + 4 * (p ^ swap));
  if (!valid) return;
  *(v4i*)(q + (size_t)row0 * 64 + tid * 16) = o;
  if (p == 0) scales[row] = scale_mul == 1.0f ? __builtin_bit_cast(__half, s) : __float2half(round_here((float)s * scale_mul));
}
template <bool HAD, bool F6>
__global__ __launch_bounds__(256) void group_quad_kernel(const __half* __restrict__ x, uint8_t* __restrict__ q,
                                                         __half* __restrict__ scales, uint32_t R, float scale_mul,
                                                         uint32_t tokens, uint32_t groups_per_token) {
  __shared__ __align__(16) unsigned turned[kQuadWords<F6>];
  group_quad_block<HAD, F6>(blockIdx.x, x, q, scales, R, scale_mul, tokens, groups_per_token, turned);
}

// the SwiGLU product alone, eight values per thread
__global__ __launch_bounds__(256) void silu_mul_kernel(const __half* __restrict__ gate, const __half* __restrict__ up,
                                                       __half* __restrict__ out, uint64_t chunks) {
  const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (i >= chunks) return;
  const h8 g = *(const h8*)(gate + i * 8), u = *(const h8*)(up + i * 8);
  h8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = silu_mul_f16(g[e], u[e]);
  *(h8*)(out + i * 8) = o;
}

// A model step's look-ups in one launch: the embedding rows of `ids`, for the group configuration with every 128 channels
// rotated (fp16 butterflies, then float32 1 / sqrt(128) and one rounding, as flh_fwht_f16_inplace and torch's division round
// them), and the rows of the rotary tables at `positions`.  One 16-byte chunk per lane: first `rows` x hidden, then T x dim
// of cos and of sin.  An index outside its table gives a row of NaNs.
// What bounds it is the launch: three to six kernels of 4-5 us each (one of them 12 us for 16 rows of a large table) -> 5 us.
template <bool HAD>
__global__ __launch_bounds__(256) void embed_kernel(const long long* __restrict__ ids, const __half* __restrict__ table,
                                                    __half* __restrict__ out, uint32_t rows, uint32_t vocab, uint32_t hidden,
                                                    const long long* __restrict__ positions, const __half* __restrict__ cos_table,
                                                    const __half* __restrict__ sin_table, __half* __restrict__ cos,
                                                    __half* __restrict__ sin, uint32_t T, uint32_t max_len, uint32_t dim) {
  const uint32_t per_row = hidden / 8, per_pos = dim / 8, blocks = (rows * per_row + 255) / 256;   // blocks of the first part
  const _Float16 bad = (_Float16)__builtin_nanf("");
  const h8 nans = {bad, bad, bad, bad, bad, bad, bad, bad};
  if (blockIdx.x < blocks) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= rows * per_row) return;                  // (whole groups of 16 lanes when HAD: hidden is a multiple of 128)
    const uint32_t row = i / per_row, pos = i % per_row;
    const int lir = HAD ? group_chunk<16>(pos % 16) : 0;
    const uint32_t chunk = HAD ? pos / 16 * 16 + lir : pos;
    const long long id = ids[row];
    const bool known = id >= 0 && id < (long long)vocab;
    h8 x = known ? *(const h8*)(table + (size_t)id * hidden + chunk * 8) : nans;
    if constexpr (HAD) {
      h2 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = h2{x[2 * e], x[2 * e + 1]};
      fwht_group_f16<128>(v, lir);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[2 * e] = (_Float16)round_here((float)v[e].x * 0.08838834764831845f);
        x[2 * e + 1] = (_Float16)round_here((float)v[e].y * 0.08838834764831845f);
      }
    }
    *(h8*)(out + (size_t)row * hidden + chunk * 8) = x;
    return;
  }
  uint32_t i = (blockIdx.x - blocks) * 256u + threadIdx.x;
  const bool second = i >= T * per_pos;
  if (second) i -= T * per_pos;
  if (i >= T * per_pos) return;
  const uint32_t t = i / per_pos, chunk = i % per_pos;
  const long long pos = positions[t];
  const bool known = pos >= 0 && pos < (long long)max_len;
  const h8 x = known ? *(const h8*)((second ? sin_table : cos_table) + (size_t)pos * dim + chunk * 8) : nans;
  *(h8*)((second ? sin : cos) + (size_t)t * dim + chunk * 8) = x;
}

// RMSNorm in front of the group kernel, one workgroup per token row of K = 8 * chunks values (K <= 16384):
// y = fp16( float(x) * rsqrt(sum(x^2) / K + eps) [* float(weight)] ) with the statistics in float32
// (flh/nn/normalization.py:12-20), then transform + quantise per group of G as group_kernel<G, HAD, true>.
template <int G, bool HAD, bool F6>
__device__ __forceinline__ void rmsnorm_group_block(uint32_t token, uint32_t tokens, const __half* __restrict__ x,
                                                    const __half* __restrict__ weight, uint8_t* __restrict__ q,
                                                    __half* __restrict__ scales, uint32_t K, float eps, float scale_mul) {
  constexpr int LPR = G / 8, MAXC = 8;
  __shared__ float part[4];
  const int tid = threadIdx.x;
  const uint32_t chunks = K / 8;
  const int lir = group_chunk<LPR>(tid % LPR);
  const uint32_t c0 = (tid / LPR) * LPR + lir;        // chunk of pass 0; pass i adds 256 i
  const __half* xr = x + (size_t)token * K;
  h8 raw[MAXC];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXC; ++i) {
    const uint32_t c = c0 + 256u * i;
    if (c < chunks) {
      raw[i] = *(const h8*)(xr + (size_t)c * 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = __builtin_fmaf((float)raw[i][e], (float)raw[i][e], ss);
    }
  }
  // workgroup sum: across the wave with DPP / swaps, across the four waves through LDS
  ss += dpp_f<kDppQuadXor1>(ss);
  ss += dpp_f<kDppQuadXor2>(ss);
  ss += dpp_f<kDppRowHalfMirror>(ss);
  ss += dpp_f<kDppRowMirror>(ss);
  ss += lane_xor_f<16>(ss);
  ss += lane_xor_f<32>(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  const float total = (part[0] + part[1]) + (part[2] + part[3]);
  const float inv = 1.0f / __builtin_sqrtf(total / (float)K + eps);
#pragma unroll
  for (int i = 0; i < MAXC; ++i) {
    const uint32_t c = c0 + 256u * i;
    if (c < chunks) {                                 // whole groups of LPR lanes take this branch together
      h8 w8;
      if (weight) w8 = *(const h8*)(weight + (size_t)c * 8);
      h2 v[4];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float t = round_here((float)raw[i][e] * inv);
        if (weight) t = round_here(t * (float)w8[e]);
        if (e & 1) v[e >> 1].y = (_Float16)t;
        else v[e >> 1].x = (_Float16)t;
      }
      if constexpr (HAD) fwht_group_f16<G>(v, lir);
      const uint32_t row = token * (K / G) + c / LPR;
      group_finish<G, F6>(v, lir, true, row, q, scales, scale_mul, tokens, K / G);   // (a quad is inside one group)
    }
  }
}
template <int G, bool HAD, bool F6 = false>
__global__ __launch_bounds__(256) void rmsnorm_group_kernel(const __half* __restrict__ x,
                                                            const __half* __restrict__ weight, uint8_t* __restrict__ q,
                                                            __half* __restrict__ scales, uint32_t K, float eps,
                                                            float scale_mul) {
  rmsnorm_group_block<G, HAD, F6>(blockIdx.x, gridDim.x, x, weight, q, scales, K, eps, scale_mul);
}

// RMSNorm on its own (a model's final norm, in front of an fp16 head), optionally behind the residual addition: one
// workgroup per row of K = 8 * chunks values (K <= 16384), the statistics and roundings of rmsnorm_group_kernel;
// with `add` the row is fp16(x + add), one rounding per value, stored to sum_out as well when that is given.
__global__ __launch_bounds__(256) void add_rmsnorm_kernel(const __half* __restrict__ x, const __half* __restrict__ add,
                                                          const __half* __restrict__ weight, __half* __restrict__ out,
                                                          __half* __restrict__ sum_out, uint32_t K, float eps) {
  constexpr int MAXC = 8;
  __shared__ float part[4];
  const int tid = threadIdx.x;
  const uint32_t chunks = K / 8;
  const size_t row = (size_t)blockIdx.x * K;
  h8 raw[MAXC];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXC; ++i) {
    const uint32_t c = tid + 256u * i;
    if (c < chunks) {
      raw[i] = *(const h8*)(x + row + (size_t)c * 8);
      if (add) {
        raw[i] = __builtin_bit_cast(h8, add_h8(__builtin_bit_cast(v4i, raw[i]), *(const v4i*)(add + row + (size_t)c * 8)));
        if (sum_out) *(h8*)(sum_out + row + (size_t)c * 8) = raw[i];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = __builtin_fmaf((float)raw[i][e], (float)raw[i][e], ss);
    }
  }
  ss += dpp_f<kDppQuadXor1>(ss);
  ss += dpp_f<kDppQuadXor2>(ss);
  ss += dpp_f<kDppRowHalfMirror>(ss);
  ss += dpp_f<kDppRowMirror>(ss);
  ss += lane_xor_f<16>(ss);
  ss += lane_xor_f<32>(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  const float total = (part[0] + part[1]) + (part[2] + part[3]);
  const float inv = 1.0f / __builtin_sqrtf(total / (float)K + eps);
#pragma unroll
  for (int i = 0; i < MAXC; ++i) {
    const uint32_t c = tid + 256u * i;
    if (c < chunks) {
      h8 w8, y;
      if (weight) w8 = *(const h8*)(weight + (size_t)c * 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float t = round_here((float)raw[i][e] * inv);
        if (weight) t = round_here(t * (float)w8[e]);
        y[e] = (_Float16)t;
      }
      *(h8*)(out + row + (size_t)c * 8) = y;
    }
  }
}

// ------------------------------------------------------------------------------------
// 2. wave-per-row kernel, float32 butterflies, K = 512 * J: four rows per workgroup, rotate_quant_row (rotate_row.h)
// ------------------------------------------------------------------------------------
template <int J, bool HAD, bool EXACT_NORM, bool RMS, bool F6>
__device__ __forceinline__ void rotate_quant_wave_block(uint32_t block, const __half* __restrict__ x, uint8_t* __restrict__ q,
                                                                __half* __restrict__ scales,
                                                                __half* __restrict__ y_out, uint32_t M, float norm,
                                                                float clip, const __half* __restrict__ rms_weight = nullptr,
                                                                float rms_eps = 0.f, const __half* add = nullptr,
                                                                __half* sum_out = nullptr) {
  constexpr int K = 512 * J;
  const uint32_t row = block * 4u + (threadIdx.x >> 6);
  if (row >= M) return;  // wave-uniform
  // F6: q is the encoded matrix of M rows in the 6-bit operand format instead of [M, K / 2] nibbles
  rotate_quant_row<J, HAD, EXACT_NORM, RMS, F6>(x + (size_t)row * K, F6 ? q : q + (size_t)row * (K / 2), scales + row,
                                            y_out ? y_out + (size_t)row * K : nullptr, norm, clip, rms_weight, rms_eps,
                                            add ? add + (size_t)row * K : nullptr,
                                            add ? sum_out + (size_t)row * K : nullptr, M, row);
}
template <int J, bool HAD, bool EXACT_NORM, bool RMS, bool F6>
__global__ __launch_bounds__(256) void rotate_quant_wave_kernel(const __half* __restrict__ x, uint8_t* __restrict__ q,
                                                                __half* __restrict__ scales,
                                                                __half* __restrict__ y_out, uint32_t M, float norm,
                                                                float clip, const __half* __restrict__ rms_weight = nullptr,
                                                                float rms_eps = 0.f, const __half* add = nullptr,
                                                                __half* sum_out = nullptr) {
  rotate_quant_wave_block<J, HAD, EXACT_NORM, RMS, F6>(blockIdx.x, x, q, scales, y_out, M, norm, clip, rms_weight, rms_eps, add, sum_out);
}

// A quantiser and the encoding of the weights that its codes meet, which does not depend on it, in one launch: the quantiser's workgroups
// first, the encoding's as compute units have room.  Saves the drain between the two and most of the shorter one's time where that one
// does not fill the memory.  us, two launches -> one (replayed in a graph, weights from memory):
//   norm and groups, 531 x 4096 beside 28672 / 6144 rows of weights  34.3 -> 29.9 / 14.5 -> 11.4; 2048: 39.4 -> 33.8 / 20.0 -> 17.0;
//     8192: 58.6 -> 56.6 / 40.0 -> 37.1
//   groups, beside 4096 rows: 531 x 4096 10.0 -> 7.9, 531 x 14336 23.2 -> 19.1, 2048 35.6 -> 29.8, 4096 51.2 -> 44.2, 6144 66.8 -> 63.0
//   rotation, 531 x 4096 beside 4096 rows 12.1 -> 9.1, 8192 33.4 -> 30.4; with the norm beside 28672, 2048 41.8 -> 40.6, 8192 63.6 -> 60.2
// (The two kinds of workgroup share their LDS: 28 KB instead of 16 costs the group quantiser waves, 2048 x 14336 30.5 instead of 29.8.)
template <typename Quantise>
__global__ __launch_bounds__(256) void quantise_encode_kernel(const Quantise quantise, uint32_t quant_blocks, const EncodeArgs encode,
                                                              uint32_t encode_x) {
  __shared__ __align__(16) uint8_t lds[Quantise::kLds > kEncodeLds ? Quantise::kLds : kEncodeLds];
  if (blockIdx.x < quant_blocks) {
    quantise(blockIdx.x, lds);
  } else {
    const uint32_t i = blockIdx.x - quant_blocks;
    encode_f6_block(encode, i % encode_x, i / encode_x, lds);
  }
}
template <bool QUAD>
struct GroupQuantise {                               // groups of 128, 6-bit output
  const __half* x;
  uint8_t* q;
  __half* scales;
  uint32_t R;
  float scale_mul;
  uint32_t tokens, groups_per_token;
  static constexpr int kLds = QUAD ? 4 * kQuadWords<true> : 0;
  __device__ void operator()(uint32_t block, uint8_t* lds) const {
    if constexpr (QUAD) {
      group_quad_block<false, true>(block, x, q, scales, R, scale_mul, tokens, groups_per_token, (unsigned*)lds);
    } else {
      const uint32_t gl = block * 256u + threadIdx.x;
      quantise_group<128, false, true>(x, q, scales, gl / 16, group_chunk<16>(gl % 16), R, scale_mul, tokens, groups_per_token);
    }
  }
};
struct NormGroupQuantise {
  const __half *x, *weight;
  uint8_t* q;
  __half* scales;
  uint32_t K;
  float eps;
  uint32_t tokens;
  static constexpr int kLds = 0;
  __device__ void operator()(uint32_t block, uint8_t*) const {
    rmsnorm_group_block<128, false, true>(block, tokens, x, weight, q, scales, K, eps, 1.0f);
  }
};
template <bool RMS>
struct RotateQuantise {                              // rows of 4096 rotated, one scale each
  const __half* x;
  uint8_t* q;
  __half* scales;
  uint32_t M;
  float clip;
  const __half* weight;
  float eps;
  const __half* add;
  __half* sum_out;
  static constexpr int kLds = 0;
  __device__ void operator()(uint32_t block, uint8_t*) const {
    rotate_quant_wave_block<8, true, true, RMS, true>(block, x, q, scales, nullptr, M, 1.0f / 64.0f, clip, weight, eps, add, sum_out);
  }
};
// Whether the two take one launch.  A quantiser that fills the memory by itself gains nothing and, where its values no longer fit the
// caches, loses: 8192 x 11008 (90 M values) 63.4 -> 58.6, 8192 x 14336 (117 M) 83.8 -> 92.9, 32768 x 4096 (134 M) 134.7 -> 138.4 with the
// norm and 28672 rows, 117.3 -> 115.1 with 6144.
constexpr uint64_t kBesideValues = 100ull << 20;
inline bool beside(uint64_t quant_blocks, uint64_t values, const EncodeLaunch& e) {
  return e.x > 0 && values <= kBesideValues && quant_blocks + (uint64_t)e.x * e.y <= 0x7FFFFFFFull;
}
template <typename Quantise>
int launch_beside(const Quantise& q, uint32_t quant_blocks, const EncodeLaunch& e, hipStream_t stream) {
  hipLaunchKernelGGL(quantise_encode_kernel<Quantise>, dim3(quant_blocks + e.x * e.y), dim3(256), 0, stream, q, quant_blocks, e.args, e.x);
  return check_launch("quantise_encode");
}

constexpr int kGenericThreads = 1024;      // one workgroup per compute unit (LDS): two waves per SIMD hide latencies

// 2^LOGR-point butterflies (strides 2^shift .. 2^(shift + LOGR - 1), ascending) over a row of K floats in LDS
template <int LOGR>
__device__ __forceinline__ void fwht_pass(float* a, uint32_t K, int shift, int tid) {
  constexpr int R = 1 << LOGR;
  for (uint32_t p = tid; p < K / R; p += kGenericThreads) {
    const uint32_t base = ((p >> shift) << (shift + LOGR)) | (p & ((1u << shift) - 1));
    float v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = a[base + ((uint32_t)r << shift)];
#pragma unroll
    for (int h = 1; h < R; h <<= 1)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (!(r & h)) {
          const float u = v[r], w = v[r + h];
          v[r] = u + w;
          v[r + h] = u - w;
        }
#pragma unroll
    for (int r = 0; r < R; ++r) a[base + ((uint32_t)r << shift)] = v[r];
  }
  __syncthreads();
}

// ------------------------------------------------------------------------------------
// 3. generic kernel: one workgroup per row, data in LDS as float32.
//    K = Kd * P: float32 butterflies over each contiguous block of P (ascending strides),
//    then (Kd > 1) out[j][t] = sum_j' H[j][j'] * a[j'][t] with the +/-1 literal matrix
//    (matmul_hadU, flh/functional/hadamard.py:92-113), then / norm.
//    had_width == 0: no rotation.  Scales per contiguous scale_group (0 = whole row).
// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(kGenericThreads) void rotate_quant_generic_kernel(const __half* __restrict__ x, uint8_t* __restrict__ q,
                                                                   __half* __restrict__ scales,
                                                                   __half* __restrict__ y_out, uint32_t K, int P,
                                                                   int Kd, float norm, int scale_group, float clip) {
  extern __shared__ __align__(16) float smem[];
  float* a = smem;
  float* b = smem + K;                       // used only when Kd > 1
  __shared__ float red[kGenericThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const size_t row = blockIdx.x;
  const __half* xr = x + row * K;
  if (K % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0) {
    // 16-byte loads, four in flight per lane: a workgroup owns a whole compute unit's LDS here, so nothing
    // else hides the latency of this read
    const uint4* xv = reinterpret_cast<const uint4*>(xr);
    const uint32_t n = K / 8;
    for (uint32_t i0 = tid; i0 < n; i0 += 4 * kGenericThreads) {
      uint4 w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + kGenericThreads * u < n) w[u] = xv[i0 + kGenericThreads * u];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + kGenericThreads * u < n) {
          const __half2* h = reinterpret_cast<const __half2*>(&w[u]);
          const float2 f0 = __half22float2(h[0]), f1 = __half22float2(h[1]), f2 = __half22float2(h[2]),
                       f3 = __half22float2(h[3]);
          float4* dst = reinterpret_cast<float4*>(a + 8 * (size_t)(i0 + kGenericThreads * u));
          dst[0] = make_float4(f0.x, f0.y, f1.x, f1.y);
          dst[1] = make_float4(f2.x, f2.y, f3.x, f3.y);
        }
    }
  } else {
    for (uint32_t i = tid; i < K / 2; i += kGenericThreads) {       // K is even (two codes per output byte)
      const float2 v = __half22float2(reinterpret_cast<const __half2*>(xr)[i]);
      a[2 * i] = v.x;
      a[2 * i + 1] = v.y;
    }
  }
  __syncthreads();
  if (P > 1) {
    // three butterfly stages per pass over LDS (then what is left), each thread holding the 2^LOGR values that
    // those stages couple; every value still goes through the same additions in ascending stride order
    int shift = 0, stages = 0;
    while ((1 << stages) < P) ++stages;
    for (; shift + 3 <= stages; shift += 3) fwht_pass<3>(a, K, shift, tid);
    if (stages - shift == 2) fwht_pass<2>(a, K, shift, tid);
    if (stages - shift == 1) fwht_pass<1>(a, K, shift, tid);
    if (Kd > 1) {
      const uint8_t* bits = hadk_bits(Kd);
      if (P >= 16) {
        // Lanes hold 64 output blocks j, registers 16 positions t: a[jj * P + t] is then one address for the
        // whole wave (an LDS broadcast) and the sign of (j, jj) one value per lane, so that an accumulation is
        // a single FMA, acc = fma(+-1, a, acc) -- the same sum, in the same order, as the loop below.
        uint8_t* sign_bits = reinterpret_cast<uint8_t*>(smem + 2 * (size_t)K);
        for (int i = tid; i < (Kd * Kd + 7) >> 3; i += kGenericThreads) sign_bits[i] = bits[i];
        __syncthreads();
        const int jblocks = (Kd + 63) >> 6, units = jblocks * (P >> 4);
        for (int u = wave; u < units; u += kGenericThreads / 64) {
          const int j = (u % jblocks) * 64 + lane, t0 = (u / jblocks) << 4;
          // the signs of row j are Kd consecutive bits (most significant first) from bit j * Kd of the table:
          // a 16-bit window over two bytes covers the 8 columns of a chunk whatever the row's bit offset
          const uint32_t jbit = (uint32_t)(j < Kd ? j : Kd - 1) * Kd;
          const uint8_t* sb = sign_bits + (jbit >> 3);
          const uint32_t align = 16 + (jbit & 7);
          float acc[16] = {};
          auto four = [&](int jj, uint32_t minus, int e0) {     // columns jj .. jj + 3 are bits 31 - e0 .. of ~window
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float sgn = __uint_as_float(((minus << (e0 + e)) & 0x80000000u) | 0x3f800000u);
              const float4* av = reinterpret_cast<const float4*>(a + (jj + e) * P + t0);
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float4 v = av[i];
                acc[4 * i + 0] = fmaf(sgn, v.x, acc[4 * i + 0]);
                acc[4 * i + 1] = fmaf(sgn, v.y, acc[4 * i + 1]);
                acc[4 * i + 2] = fmaf(sgn, v.z, acc[4 * i + 2]);
                acc[4 * i + 3] = fmaf(sgn, v.w, acc[4 * i + 3]);
              }
            }
          };
          uint32_t cur = sb[0];
          for (int jj = 0; jj < Kd; jj += 8) {                  // every literal size is a multiple of 4
            const uint32_t next = sb[(jj >> 3) + 1];
            const uint32_t minus = ~(((cur << 8) | next) << align);
            cur = next;
            four(jj, minus, 0);
            if (jj + 4 < Kd) four(jj + 4, minus, 4);
          }
          if (j < Kd) {
            float4* bv = reinterpret_cast<float4*>(b + j * P + t0);
#pragma unroll
            for (int i = 0; i < 4; ++i) bv[i] = make_float4(acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]);
          }
        }
      } else {
        for (uint32_t o = tid; o < K; o += kGenericThreads) {
          const int j = o / P, t = o % P;
          float acc = 0.f;
          for (int jj = 0; jj < Kd; ++jj) {
            const int bit = j * Kd + jj;
            const bool plus = (bits[bit >> 3] >> (7 - (bit & 7))) & 1;
            const float val = a[jj * P + t];
            acc += plus ? val : -val;
          }
          b[o] = acc;
        }
      }
      __syncthreads();
      a = b;
    }
  }
  // normalise (norm = 1 without rotation), round to fp16 (kept as float in LDS), optional copy out, row maximum
  float m = 0.f;
  for (uint32_t i = tid; i < K / 2; i += kGenericThreads) {
    const __half2 h = __floats2half2_rn(a[2 * i] / norm, a[2 * i + 1] / norm);
    const float2 f = __half22float2(h);
    a[2 * i] = f.x;
    a[2 * i + 1] = f.y;
    m = fmaxf(m, fmaxf(fabsf(f.x), fabsf(f.y)));
    if (y_out) reinterpret_cast<__half2*>(y_out + row * K)[i] = h;
  }
  m = wave_max(m);
  if (lane == 0) red[wave] = m;
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int w = 1; w < kGenericThreads / 64; ++w) m = fmaxf(m, red[w]);
  if (clip < 1.0f) {
    const float bound = __half2float(__float2half(round_here(m * clip)));
    for (uint32_t i = tid; i < K; i += kGenericThreads) a[i] = fminf(fmaxf(a[i], -bound), bound);
    m = fminf(m, bound);
    __syncthreads();
  }
  const uint32_t G = scale_group > 0 ? (uint32_t)scale_group : K;
  const uint32_t ng = K / G;
  if (ng == 1) {                               // one scale for the row: the whole workgroup quantises it
    _Float16 s = (_Float16)(m / 7.0f);
    if (s == (_Float16)0.0f) s = (_Float16)1.0f;
    const float r = 1.0f / (float)s;
    uint8_t* qg = q + row * (K / 2);
    for (uint32_t i = tid; i < K / 2; i += kGenericThreads)
      qg[i] = (uint8_t)(quant_nibble((_Float16)a[2 * i], r) | (quant_nibble((_Float16)a[2 * i + 1], r) << 4));
    if (tid == 0) scales[row] = __builtin_bit_cast(__half, s);
    return;
  }
  // one wave per scale group at a time
  for (uint32_t g = wave; g < ng; g += kGenericThreads / 64) {
    const float* ag = a + g * G;
    float mg = 0.f;
    for (uint32_t i = lane; i < G; i += 64) mg = fmaxf(mg, fabsf(ag[i]));
    mg = wave_max(mg);
    _Float16 s = (_Float16)(mg / 7.0f);
    if (s == (_Float16)0.0f) s = (_Float16)1.0f;
    const float r = 1.0f / (float)s;
    uint8_t* qg = q + row * (K / 2) + g * (G / 2);
    for (uint32_t i = lane; i < G / 2; i += 64)
      qg[i] = (uint8_t)(quant_nibble((_Float16)ag[2 * i], r) | (quant_nibble((_Float16)ag[2 * i + 1], r) << 4));
    if (lane == 0) scales[row * ng + g] = __builtin_bit_cast(__half, s);
  }
}

bool is_pow2(uint32_t n) { return n && !(n & (n - 1)); }

// K = Kd * P with the reference's divisor order (flh/functional/hadamard.py:41-84)
bool factor_hadamard(uint32_t K, int* Kd, int* P) {
  static const int order[] = {172, 156, 140, 108, 60, 52, 36, 28, 40, 20, 12};
  for (int k : order)
    if (K % k == 0) {
      if (!is_pow2(K / k)) return false;
      *Kd = k;
      *P = (int)(K / k);
      return true;
    }
  if (!is_pow2(K)) return false;
  *Kd = 1;
  *P = (int)K;
  return true;
}

template <int J, bool F6 = false>
int launch_wave(const __half* x, uint8_t* q, __half* s, __half* y, uint32_t M, bool had, float clip,
                hipStream_t stream) {
  constexpr int K = 512 * J;
  int lg = 0;
  while ((1 << lg) < K) ++lg;
  const dim3 grid((M + 3) / 4), block(256);
  if (!had)
    hipLaunchKernelGGL((rotate_quant_wave_kernel<J, false, true, false, F6>), grid, block, 0, stream, x, q, s, y, M, 1.0f, clip);
  else if (lg % 2 == 0)
    hipLaunchKernelGGL((rotate_quant_wave_kernel<J, true, true, false, F6>), grid, block, 0, stream, x, q, s, y, M,
                       1.0f / (float)(1 << (lg / 2)), clip);
  else
    hipLaunchKernelGGL((rotate_quant_wave_kernel<J, true, false, false, F6>), grid, block, 0, stream, x, q, s, y, M, sqrtf((float)K),
                       clip);
  return check_launch("rotate_quant_wave");
}

// A few rows of 4096: one workgroup of eight waves per row (rotate_quant_rows_8waves: the same additions in the same
// order as the wave-per-row kernel, hence the same bytes), so that a decode-sized batch waits for an eighth of a
// row's arithmetic instead of a whole row's on a single wave.
__global__ __launch_bounds__(512) void rotate_quant_row8_kernel(const __half* __restrict__ x, uint8_t* __restrict__ q,
                                                                __half* __restrict__ scales, float norm) {
  __shared__ RowScratch<> lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t row = blockIdx.x;
  const v4i none = {0, 0, 0, 0};
  const RowPiece piece[1] = {{row_piece(x + row * 4096, wave), none, none}};
  rotate_quant_rows_8waves(piece, lds, q + row * 2048, 0, scales + row, norm, wave);
}
// ... and with RMSNorm in front (flh_rmsnorm_rotate_quant_i4), the same bytes as rotate_quant_wave_kernel<8, ..., RMS>
__global__ __launch_bounds__(512) void rmsnorm_rotate_quant_row8_kernel(const __half* __restrict__ x,
                                                                        const __half* __restrict__ weight, float eps,
                                                                        uint8_t* __restrict__ q,
                                                                        __half* __restrict__ scales, float norm) {
  __shared__ RowScratch<> lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t row = blockIdx.x;
  const v4i none = {0, 0, 0, 0};
  const RowPiece piece[1] = {{row_piece(x + row * 4096, wave), none, weight ? row_piece(weight, wave) : none}};
  rotate_quant_rows_8waves<true>(piece, lds, q + row * 2048, 0, scales + row, norm, wave, weight != nullptr, eps);
}
// ... and with the residual addition in front of that (flh_add_rmsnorm_rotate_quant_i4)
__global__ __launch_bounds__(512) void add_rmsnorm_rotate_quant_row8_kernel(const __half* __restrict__ x,
                                                                            const __half* __restrict__ add,
                                                                            __half* __restrict__ sum_out,
                                                                            const __half* __restrict__ weight, float eps,
                                                                            uint8_t* __restrict__ q,
                                                                            __half* __restrict__ scales, float norm) {
  __shared__ RowScratch<> lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t row = blockIdx.x;
  const v4i none = {0, 0, 0, 0};
  const RowPiece piece[1] = {{row_piece(x + row * 4096, wave), row_piece(add + row * 4096, wave), weight ? row_piece(weight, wave) : none}};
  rotate_quant_rows_8waves<true, true>(piece, lds, q + row * 2048, 0, scales + row, norm, wave, weight != nullptr, eps,
                                      sum_out + row * 4096);
}
// measured per launch inside a replayed graph: 2.7 against 4.4 us for one row, 3.2 against 4.9 us for 256 rows,
// 3.9 against 5.0 us for 512; from 1024 rows on the wave-per-row kernel is the faster one
constexpr uint32_t kRow8MaxRows = 512;

template <int J, bool F6 = false>
int launch_wave_rms(const __half* x, const __half* w, float eps, uint8_t* q, __half* s, __half* y, uint32_t M, bool had,
                    float clip, hipStream_t stream, const __half* add = nullptr, __half* sum_out = nullptr) {
  constexpr int K = 512 * J;
  int lg = 0;
  while ((1 << lg) < K) ++lg;
  const dim3 grid((M + 3) / 4), block(256);
  if (!had)
    hipLaunchKernelGGL((rotate_quant_wave_kernel<J, false, true, true, F6>), grid, block, 0, stream, x, q, s, y, M, 1.0f,
                       clip, w, eps, add, sum_out);
  else if (lg % 2 == 0)
    hipLaunchKernelGGL((rotate_quant_wave_kernel<J, true, true, true, F6>), grid, block, 0, stream, x, q, s, y, M,
                       1.0f / (float)(1 << (lg / 2)), clip, w, eps, add, sum_out);
  else
    hipLaunchKernelGGL((rotate_quant_wave_kernel<J, true, false, true, F6>), grid, block, 0, stream, x, q, s, y, M,
                       sqrtf((float)K), clip, w, eps, add, sum_out);
  return check_launch("rmsnorm_rotate_quant_wave");
}

// Groups of 128 from which four lanes per group are the faster form: below, a quarter of the wavefronts does not fill the chip,
// least of all just beyond a full round of it (us, inputs from HBM, sixteen lanes / four: rotated 18490 groups 3.40 / 3.82,
// 32768 4.10 / 4.28, 49152 5.70 / 5.73 and 4.35 / 3.96 from the caches, 65536 6.65 / 6.51; not rotated 49152 5.15 / 5.15, 65536
// 6.21 / 5.66; 6-bit output, rotated and not, 16384 3.83 / 3.41 and 3.42 / 3.14, 18432 4.07 / 4.03 and 3.62 / 3.53, 24576 4.55
// / 4.27 and 4.00 / 3.75).
constexpr uint32_t quad_min_rows(bool had, bool f6) { return f6 ? 16384 : had ? 49152 : 65536; }
template <bool HAD, bool F6>
int launch_group_quad(const __half* x, uint8_t* q, __half* s, uint32_t R, float scale_mul, uint32_t tokens,
                      uint32_t groups_per_token, hipStream_t stream) {
  hipLaunchKernelGGL((group_quad_kernel<HAD, F6>), dim3((unsigned)(((uint64_t)R + kQuadRows - 1) / kQuadRows)), dim3(256), 0,
                     stream, x, q, s, R, scale_mul, tokens, groups_per_token);
  return check_launch("group_quad_kernel");
}

template <int G>
int launch_group(const __half* x, uint8_t* q, __half* s, __half* y, uint32_t R, bool had, bool quant,
                 float scale_mul, hipStream_t stream) {
  constexpr int LPR = G / 8;
  if (G == 128 && quant && R >= quad_min_rows(had, false))
    return had ? launch_group_quad<true, false>(x, q, s, R, scale_mul, 0, 1, stream)
               : launch_group_quad<false, false>(x, q, s, R, scale_mul, 0, 1, stream);
  const dim3 grid((unsigned)(((uint64_t)R * LPR + 255) / 256)), block(256);
  auto go = [&](auto off32_tag) {
    constexpr bool OFF32 = decltype(off32_tag)::value;
    if (!quant) {
      hipLaunchKernelGGL((group_kernel<G, true, false, false, OFF32>), grid, block, 0, stream, x, q, s, y, R, scale_mul, 0u, 1u);
    } else if constexpr (G != 128 || OFF32) {           // (longer batches of 128 are the four-lane kernel's)
      if (had) hipLaunchKernelGGL((group_kernel<G, true, true, false, OFF32>), grid, block, 0, stream, x, q, s, y, R, scale_mul, 0u, 1u);
      else hipLaunchKernelGGL((group_kernel<G, false, true, false, OFF32>), grid, block, 0, stream, x, q, s, y, R, scale_mul, 0u, 1u);
    }
  };
  if ((uint64_t)R * G * 2 <= 0xFFFFFFFFull) go(std::true_type{});   // the largest array of the launch: the fp16 rows
  else go(std::false_type{});
  return check_launch("group_kernel");
}

int group_dispatch(const __half* x, uint8_t* q, __half* s, __half* y, uint32_t R, int group, bool had, bool quant,
                   float scale_mul, hipStream_t stream) {
  if (R == 0) return FLH_OK;
  switch (group) {
    case 32: return launch_group<32>(x, q, s, y, R, had, quant, scale_mul, stream);
    case 64: return launch_group<64>(x, q, s, y, R, had, quant, scale_mul, stream);
    case 128: return launch_group<128>(x, q, s, y, R, had, quant, scale_mul, stream);
    default: return fail(FLH_EINVAL, "group size must be 32, 64 or 128 (got %d)", group);
  }
}

template <int G>
int launch_silu_mul(const __half* gate, const __half* up, uint8_t* q, __half* s, uint32_t R, bool had, float scale_mul,
                    hipStream_t stream) {
  const dim3 grid((unsigned)(((uint64_t)R * (G / 8) + 255) / 256)), block(256);
  if (had)
    hipLaunchKernelGGL((silu_mul_group_kernel<G, true>), grid, block, 0, stream, gate, up, q, s, R, scale_mul);
  else
    hipLaunchKernelGGL((silu_mul_group_kernel<G, false>), grid, block, 0, stream, gate, up, q, s, R, scale_mul);
  return check_launch("silu_mul_group_kernel");
}

template <int G>
int launch_rmsnorm(const __half* x, const __half* w, uint8_t* q, __half* s, uint32_t M, uint32_t K, float eps, bool had,
                   float scale_mul, hipStream_t stream) {
  if (had)
    hipLaunchKernelGGL((rmsnorm_group_kernel<G, true>), dim3(M), dim3(256), 0, stream, x, w, q, s, K, eps, scale_mul);
  else
    hipLaunchKernelGGL((rmsnorm_group_kernel<G, false>), dim3(M), dim3(256), 0, stream, x, w, q, s, K, eps, scale_mul);
  return check_launch("rmsnorm_group_kernel");
}

}  // namespace

// matrix-core variant (fwht_mfma.hip)
int launch_rotate_quant_mfma(const __half* x, uint8_t* q, __half* scales, uint32_t M, uint32_t K, float clip,
                             hipStream_t stream);
bool rotate_quant_mfma_supports(uint32_t K);
int launch_silu_mul_rotate_quant_mfma(const __half* gate, const __half* up, uint8_t* q, __half* scales, uint32_t M,
                                      uint32_t K, hipStream_t stream);
int launch_rotate_quant_mfma4096(const __half* x, const __half* add, __half* sum_out, bool rms, const __half* weight,
                                 float eps, uint8_t* q, __half* scales, uint32_t M, float clip, bool f6,
                                 hipStream_t stream);
int launch_rotate_quant_mfma_f6(const __half* x, uint8_t* encoded, __half* scales, uint32_t M, uint32_t K, float clip,
                                hipStream_t stream);

}  // namespace flh

using namespace flh;

extern "C" int flh_group_quant_i4(const flh_half* x, uint8_t* q_packed, flh_half* scales, uint32_t R, int group,
                                  int hadamard, float scale_mul, void* stream) {
  if (!x || !q_packed || !scales) return fail(FLH_EINVAL, "group_quant: null pointer");
  if (misaligned16(x, q_packed)) return fail(FLH_EINVAL, "group_quant: x and q_packed must be 16-byte aligned");
  if (!(scale_mul > 0.f)) return fail(FLH_EINVAL, "group_quant: scale_mul must be positive");
  return group_dispatch((const __half*)x, q_packed, (__half*)scales, nullptr, R, group, hadamard != 0, true, scale_mul,
                        (hipStream_t)stream);
}

extern "C" int flh_silu_mul_group_quant_i4(const flh_half* gate, const flh_half* up, uint8_t* q_packed, flh_half* scales,
                                           uint32_t R, int group, int hadamard, float scale_mul, void* stream) {
  if (!gate || !up || !q_packed || !scales) return fail(FLH_EINVAL, "silu_mul_group_quant: null pointer");
  if (misaligned16(gate, up, q_packed)) return fail(FLH_EINVAL, "silu_mul_group_quant: gate, up and q_packed must be 16-byte aligned");
  if (!(scale_mul > 0.f)) return fail(FLH_EINVAL, "silu_mul_group_quant: scale_mul must be positive");
  if (R == 0) return FLH_OK;
  const __half *g = (const __half*)gate, *u = (const __half*)up;
  switch (group) {
    case 32: return launch_silu_mul<32>(g, u, q_packed, (__half*)scales, R, hadamard != 0, scale_mul, (hipStream_t)stream);
    case 64: return launch_silu_mul<64>(g, u, q_packed, (__half*)scales, R, hadamard != 0, scale_mul, (hipStream_t)stream);
    case 128: return launch_silu_mul<128>(g, u, q_packed, (__half*)scales, R, hadamard != 0, scale_mul, (hipStream_t)stream);
    default: return fail(FLH_EINVAL, "group size must be 32, 64 or 128 (got %d)", group);
  }
}

extern "C" int flh_rmsnorm_group_quant_i4(const flh_half* x, const flh_half* weight, uint8_t* q_packed, flh_half* scales,
                                          uint32_t M, uint32_t K, float eps, int group, int hadamard, float scale_mul,
                                          void* stream) {
  if (!x || !q_packed || !scales) return fail(FLH_EINVAL, "rmsnorm_group_quant: null pointer");
  if (misaligned16(x, q_packed)) return fail(FLH_EINVAL, "rmsnorm_group_quant: x and q_packed must be 16-byte aligned");
  if (!(scale_mul > 0.f)) return fail(FLH_EINVAL, "rmsnorm_group_quant: scale_mul must be positive");
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "rmsnorm_group_quant: eps must not be negative");
  if (group != 32 && group != 64 && group != 128)
    return fail(FLH_EINVAL, "group size must be 32, 64 or 128 (got %d)", group);
  if (K == 0 || K % (uint32_t)group || K > 16384u)
    return fail(FLH_EINVAL, "rmsnorm_group_quant: K (%u) must be a multiple of the group size, at most 16384", K);
  if (M == 0) return FLH_OK;
  const __half *xh = (const __half*)x, *wh = (const __half*)weight;
  switch (group) {
    case 32: return launch_rmsnorm<32>(xh, wh, q_packed, (__half*)scales, M, K, eps, hadamard != 0, scale_mul, (hipStream_t)stream);
    case 64: return launch_rmsnorm<64>(xh, wh, q_packed, (__half*)scales, M, K, eps, hadamard != 0, scale_mul, (hipStream_t)stream);
    default: return launch_rmsnorm<128>(xh, wh, q_packed, (__half*)scales, M, K, eps, hadamard != 0, scale_mul, (hipStream_t)stream);
  }
}

extern "C" int flh_rmsnorm_rotate_quant_i4(const flh_half* x, const flh_half* weight, float eps, uint8_t* q_packed,
                                           flh_half* scales, flh_half* y_out, uint32_t M, uint32_t K, int hadamard,
                                           float clip_ratio, void* stream) {
  if (!x || !q_packed || !scales) return fail(FLH_EINVAL, "rmsnorm_rotate_quant: null pointer");
  if (misaligned16(x, q_packed)) return fail(FLH_EINVAL, "rmsnorm_rotate_quant: x and q_packed must be 16-byte aligned");
  if (!(clip_ratio > 0.f)) return fail(FLH_EINVAL, "rmsnorm_rotate_quant: clip_ratio must be positive");
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "rmsnorm_rotate_quant: eps must not be negative");
  if (hadamard != FLH_HAD_NONE && hadamard != FLH_HAD_F32 && hadamard != FLH_HAD_MFMA)
    return fail(FLH_EINVAL, "rmsnorm_rotate_quant: unknown hadamard mode %d", hadamard);
  if (K % 512 || !is_pow2(K / 512) || K > 8192)
    return fail(FLH_EINVAL, "rmsnorm_rotate_quant: K (%u) must be 512, 1024, 2048, 4096 or 8192", K);
  if (M == 0) return FLH_OK;
  const __half *xh = (const __half*)x, *wh = (const __half*)weight;
  __half *sh = (__half*)scales, *yh = (__half*)y_out;
  if (hadamard == FLH_HAD_MFMA) {                      // matrix cores: K = 4096 without y_out, else the float32 butterflies
    if (K == 4096 && !yh && (!wh || !misaligned16(wh)))
      return launch_rotate_quant_mfma4096(xh, nullptr, nullptr, true, wh, eps, q_packed, sh, M, clip_ratio, false,
                                          (hipStream_t)stream);
    hadamard = FLH_HAD_F32;
  }
  const bool had = hadamard != FLH_HAD_NONE;
  hipStream_t st = (hipStream_t)stream;
  if (had && K == 4096 && !yh && clip_ratio >= 1.0f && M <= kRow8MaxRows && (!wh || !misaligned16(wh))) {
    hipLaunchKernelGGL(rmsnorm_rotate_quant_row8_kernel, dim3(M), dim3(512), 0, st, xh, wh, eps, q_packed, sh, 1.0f / 64.0f);
    return check_launch("rmsnorm_rotate_quant_row8");
  }
  switch (K / 512) {
    case 1: return launch_wave_rms<1>(xh, wh, eps, q_packed, sh, yh, M, had, clip_ratio, st);
    case 2: return launch_wave_rms<2>(xh, wh, eps, q_packed, sh, yh, M, had, clip_ratio, st);
    case 4: return launch_wave_rms<4>(xh, wh, eps, q_packed, sh, yh, M, had, clip_ratio, st);
    case 8: return launch_wave_rms<8>(xh, wh, eps, q_packed, sh, yh, M, had, clip_ratio, st);
    default: return launch_wave_rms<16>(xh, wh, eps, q_packed, sh, yh, M, had, clip_ratio, st);
  }
}

extern "C" int flh_add_rmsnorm_rotate_quant_i4(const flh_half* x, const flh_half* add, flh_half* sum_out,
                                               const flh_half* weight, float eps, uint8_t* q_packed, flh_half* scales,
                                               uint32_t M, uint32_t K, int hadamard, float clip_ratio, void* stream) {
  if (!x || !add || !sum_out || !q_packed || !scales) return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: null pointer");
  if (misaligned16(x, add, sum_out) || misaligned16(q_packed))
    return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: x, add, sum_out and q_packed must be 16-byte aligned");
  if (weight && misaligned16(weight)) return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: weight must be 16-byte aligned");
  if (!(clip_ratio > 0.f)) return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: clip_ratio must be positive");
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: eps must not be negative");
  if (hadamard != FLH_HAD_NONE && hadamard != FLH_HAD_F32 && hadamard != FLH_HAD_MFMA)
    return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: unknown hadamard mode %d", hadamard);
  if (K % 512 || !is_pow2(K / 512) || K > 8192)
    return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: K (%u) must be 512, 1024, 2048, 4096 or 8192", K);
  if (M == 0) return FLH_OK;
  const __half *xh = (const __half*)x, *ah = (const __half*)add, *wh = (const __half*)weight;
  __half *sh = (__half*)scales, *oh = (__half*)sum_out;
  hipStream_t st = (hipStream_t)stream;
  // (the eight-waves-per-row kernel lets other waves read x and add after one has stored its part of the sum)
  if ((const void*)sum_out == (const void*)x || (const void*)sum_out == (const void*)add)
    return fail(FLH_EINVAL, "add_rmsnorm_rotate_quant: sum_out must not be x or add");
  if (hadamard == FLH_HAD_MFMA) {                      // matrix cores: K = 4096, else the float32 butterflies
    if (K == 4096) return launch_rotate_quant_mfma4096(xh, ah, oh, true, wh, eps, q_packed, sh, M, clip_ratio, false, st);
    hadamard = FLH_HAD_F32;
  }
  const bool had = hadamard != FLH_HAD_NONE;
  if (had && K == 4096 && clip_ratio >= 1.0f && M <= kRow8MaxRows) {
    hipLaunchKernelGGL(add_rmsnorm_rotate_quant_row8_kernel, dim3(M), dim3(512), 0, st, xh, ah, oh, wh, eps, q_packed, sh,
                       1.0f / 64.0f);
    return check_launch("add_rmsnorm_rotate_quant_row8");
  }
  switch (K / 512) {
    case 1: return launch_wave_rms<1>(xh, wh, eps, q_packed, sh, nullptr, M, had, clip_ratio, st, ah, oh);
    case 2: return launch_wave_rms<2>(xh, wh, eps, q_packed, sh, nullptr, M, had, clip_ratio, st, ah, oh);
    case 4: return launch_wave_rms<4>(xh, wh, eps, q_packed, sh, nullptr, M, had, clip_ratio, st, ah, oh);
    case 8: return launch_wave_rms<8>(xh, wh, eps, q_packed, sh, nullptr, M, had, clip_ratio, st, ah, oh);
    default: return launch_wave_rms<16>(xh, wh, eps, q_packed, sh, nullptr, M, had, clip_ratio, st, ah, oh);
  }
}

namespace {
// what a call without weights to encode has, and what one that has launched them separately is left with
const EncodeLaunch kNoWeights{};

int rotate_quant_f6(const flh_half* x, const flh_half* add, flh_half* sum_out, int rmsnorm, const flh_half* weight, float eps,
                    uint8_t* encoded, flh_half* scales, uint32_t M, uint32_t K, int hadamard, float clip_ratio, const EncodeLaunch& e,
                    bool* taken, void* stream) {
  const char* who = "rotate_quant_f6";
  if (!x || !encoded || !scales) return fail(FLH_EINVAL, "%s: null pointer", who);
  if (misaligned16(x, encoded)) return fail(FLH_EINVAL, "%s: x and encoded must be 16-byte aligned", who);
  if ((add == nullptr) != (sum_out == nullptr)) return fail(FLH_EINVAL, "%s: add and sum_out come together or not at all", who);
  if (add && !rmsnorm) return fail(FLH_EINVAL, "%s: the residual addition comes with the RMSNorm prologue", who);
  if (add && misaligned16(add, sum_out)) return fail(FLH_EINVAL, "%s: add and sum_out must be 16-byte aligned", who);
  if (sum_out && ((const void*)sum_out == (const void*)x || (const void*)sum_out == (const void*)add))
    return fail(FLH_EINVAL, "%s: sum_out must not be x or add", who);
  if (weight && (!rmsnorm || misaligned16(weight))) return fail(FLH_EINVAL, "%s: weight needs rmsnorm != 0 and 16-byte alignment", who);
  if (!(clip_ratio > 0.f)) return fail(FLH_EINVAL, "%s: clip_ratio must be positive", who);
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "%s: eps must not be negative", who);
  if (M == 0) return FLH_OK;
  const __half *xh = (const __half*)x, *ah = (const __half*)add, *wh = (const __half*)weight;
  __half *sh = (__half*)scales, *oh = (__half*)sum_out;
  hipStream_t st = (hipStream_t)stream;
  if (hadamard == FLH_HAD_MFMA) {
    if (K == 4096) return launch_rotate_quant_mfma4096(xh, ah, oh, rmsnorm != 0, wh, eps, encoded, sh, M, clip_ratio, true, st);
    if (rmsnorm) return fail(FLH_EINVAL, "%s: the matrix-core rotation has an RMSNorm prologue for K = 4096 only", who);
    if (K != 11008 && K != 14336)
      return fail(FLH_EINVAL, "%s: matrix-core rotation with 6-bit output: K (%u) must be 4096, 11008 or 14336", who, K);
    return launch_rotate_quant_mfma_f6(xh, encoded, sh, M, K, clip_ratio, st);
  }
  if (hadamard != FLH_HAD_NONE && hadamard != FLH_HAD_F32) return fail(FLH_EINVAL, "%s: unknown hadamard mode %d", who, hadamard);
  if (K % 512 || !is_pow2(K / 512) || K > 8192)
    return fail(FLH_EINVAL, "%s: K (%u) must be 512, 1024, 2048, 4096 or 8192 (or 11008 / 14336 on the matrix cores)", who, K);
  const bool had = hadamard != FLH_HAD_NONE;
  if (K == 4096 && had && beside((M + 3ull) / 4, (uint64_t)M * K, e)) {
    *taken = true;
    const uint32_t blocks = (uint32_t)((M + 3ull) / 4);
    if (rmsnorm) return launch_beside(RotateQuantise<true>{xh, encoded, sh, M, clip_ratio, wh, eps, ah, oh}, blocks, e, st);
    return launch_beside(RotateQuantise<false>{xh, encoded, sh, M, clip_ratio, nullptr, 0.f, nullptr, nullptr}, blocks, e, st);
  }
  if (rmsnorm) {
    switch (K / 512) {
      case 1: return launch_wave_rms<1, true>(xh, wh, eps, encoded, sh, nullptr, M, had, clip_ratio, st, ah, oh);
      case 2: return launch_wave_rms<2, true>(xh, wh, eps, encoded, sh, nullptr, M, had, clip_ratio, st, ah, oh);
      case 4: return launch_wave_rms<4, true>(xh, wh, eps, encoded, sh, nullptr, M, had, clip_ratio, st, ah, oh);
      case 8: return launch_wave_rms<8, true>(xh, wh, eps, encoded, sh, nullptr, M, had, clip_ratio, st, ah, oh);
      default: return launch_wave_rms<16, true>(xh, wh, eps, encoded, sh, nullptr, M, had, clip_ratio, st, ah, oh);
    }
  }
  switch (K / 512) {
    case 1: return launch_wave<1, true>(xh, encoded, sh, nullptr, M, had, clip_ratio, st);
    case 2: return launch_wave<2, true>(xh, encoded, sh, nullptr, M, had, clip_ratio, st);
    case 4: return launch_wave<4, true>(xh, encoded, sh, nullptr, M, had, clip_ratio, st);
    case 8: return launch_wave<8, true>(xh, encoded, sh, nullptr, M, had, clip_ratio, st);
    default: return launch_wave<16, true>(xh, encoded, sh, nullptr, M, had, clip_ratio, st);
  }
}

// a quantiser's call, then the weights if it has not taken them into its launch
template <typename F>
int with_weights(const flh_encode_list* weights, uint32_t M, void* stream, F&& quantise) {
  EncodeLaunch e{};
  if (weights)
    if (int rc = encode_launch(weights->count, weights->packed, weights->encoded, weights->rows, weights->K, e)) return rc;
  bool taken = false;
  if (M > 0 || !weights)                             // (no rows: there may be no pointers either)
    if (int rc = quantise(e, &taken)) return rc;
  if (taken || e.x == 0) return FLH_OK;
  return flh_encode_f6_multi(weights->count, weights->packed, weights->encoded, weights->rows, weights->K, stream);
}
}  // namespace

extern "C" int flh_rotate_quant_f6(const flh_half* x, const flh_half* add, flh_half* sum_out, int rmsnorm,
                                   const flh_half* weight, float eps, uint8_t* encoded, flh_half* scales, uint32_t M,
                                   uint32_t K, int hadamard, float clip_ratio, void* stream) {
  return rotate_quant_f6(x, add, sum_out, rmsnorm, weight, eps, encoded, scales, M, K, hadamard, clip_ratio, kNoWeights, nullptr, stream);
}

extern "C" int flh_rotate_quant_encode_f6(const flh_half* x, const flh_half* add, flh_half* sum_out, int rmsnorm,
                                          const flh_half* weight, float eps, uint8_t* encoded, flh_half* scales, uint32_t M,
                                          uint32_t K, int hadamard, float clip_ratio, const flh_encode_list* weights, void* stream) {
  return with_weights(weights, M, stream, [&](const EncodeLaunch& e, bool* taken) {
    return rotate_quant_f6(x, add, sum_out, rmsnorm, weight, eps, encoded, scales, M, K, hadamard, clip_ratio, e, taken, stream);
  });
}

extern "C" int flh_silu_mul_f16(const flh_half* gate, const flh_half* up, flh_half* out, uint64_t n, void* stream) {
  if (!gate || !up || !out) return fail(FLH_EINVAL, "silu_mul: null pointer");
  if (misaligned16(gate, up, out)) return fail(FLH_EINVAL, "silu_mul: gate, up and out must be 16-byte aligned");
  if (n % 8) return fail(FLH_EINVAL, "silu_mul: the element count (%llu) must be a multiple of 8", (unsigned long long)n);
  if (n / 8 > 0x7fffffffull * 256) return fail(FLH_EINVAL, "silu_mul: too many elements");
  if (n == 0) return FLH_OK;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const __half*)gate, (const __half*)up, (__half*)out, n / 8);
  return check_launch("silu_mul_kernel");
}

// The two producers of the group configuration writing the 6-bit operand format: groups of 128, no rotation.  A pass that
// re-encodes the nibbles costs 4-6 us per 1000 tokens in front of every GEMM.
namespace {
int rmsnorm_group_quant_f6(const flh_half* x, const flh_half* weight, uint8_t* encoded, flh_half* scales, uint32_t M, uint32_t K, float eps,
                           const EncodeLaunch& e, bool* taken, void* stream) {
  if (!x || !encoded || !scales) return fail(FLH_EINVAL, "rmsnorm_group_quant_f6: null pointer");
  if (misaligned16(x, encoded) || (weight && misaligned16(weight)))
    return fail(FLH_EINVAL, "rmsnorm_group_quant_f6: x, weight and encoded must be 16-byte aligned");
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "rmsnorm_group_quant_f6: eps must not be negative");
  if (K == 0 || K % 128 || K > 16384u) return fail(FLH_EINVAL, "rmsnorm_group_quant_f6: K (%u) must be a multiple of 128, at most 16384", K);
  if ((uint64_t)M * (K / 128) > 0xFFFFFFFFull) return fail(FLH_EINVAL, "rmsnorm_group_quant_f6: too many groups");
  if (M == 0) return FLH_OK;
  const __half *xh = (const __half*)x, *wh = (const __half*)weight;
  if (beside(M, (uint64_t)M * K, e)) {
    *taken = true;
    return launch_beside(NormGroupQuantise{xh, wh, encoded, (__half*)scales, K, eps, M}, M, e, (hipStream_t)stream);
  }
  hipLaunchKernelGGL((rmsnorm_group_kernel<128, false, true>), dim3(M), dim3(256), 0, (hipStream_t)stream, xh, wh, encoded,
                     (__half*)scales, K, eps, 1.0f);
  return check_launch("rmsnorm_group_kernel (6-bit output)");
}
}  // namespace

extern "C" int flh_rmsnorm_group_quant_f6(const flh_half* x, const flh_half* weight, uint8_t* encoded, flh_half* scales,
                                          uint32_t M, uint32_t K, float eps, void* stream) {
  return rmsnorm_group_quant_f6(x, weight, encoded, scales, M, K, eps, kNoWeights, nullptr, stream);
}

extern "C" int flh_rmsnorm_group_quant_encode_f6(const flh_half* x, const flh_half* weight, uint8_t* encoded, flh_half* scales, uint32_t M,
                                                 uint32_t K, float eps, const flh_encode_list* weights, void* stream) {
  return with_weights(weights, M, stream, [&](const EncodeLaunch& e, bool* taken) {
    return rmsnorm_group_quant_f6(x, weight, encoded, scales, M, K, eps, e, taken, stream);
  });
}

extern "C" int flh_silu_mul_group_quant_f6(const flh_half* gate, const flh_half* up, uint8_t* encoded, flh_half* scales,
                                           uint32_t M, uint32_t K, void* stream) {
  if (!gate || !up || !encoded || !scales) return fail(FLH_EINVAL, "silu_mul_group_quant_f6: null pointer");
  if (misaligned16(gate, up, encoded)) return fail(FLH_EINVAL, "silu_mul_group_quant_f6: gate, up and encoded must be 16-byte aligned");
  if (K == 0 || K % 128) return fail(FLH_EINVAL, "silu_mul_group_quant_f6: K (%u) must be a positive multiple of 128", K);
  if ((uint64_t)M * (K / 128) > 0x0FFFFFFFull) return fail(FLH_EINVAL, "silu_mul_group_quant_f6: too many groups");
  if (M == 0) return FLH_OK;
  const uint32_t R = M * (K / 128);
  hipLaunchKernelGGL((silu_mul_group_kernel<128, false, true>), dim3((unsigned)(((uint64_t)R * 16 + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (const __half*)gate, (const __half*)up, encoded, (__half*)scales, R, 1.0f, M, K / 128);
  return check_launch("silu_mul_group_kernel (6-bit output)");
}

extern "C" int flh_embed_f16(const int64_t* ids, const flh_half* table, flh_half* out, uint32_t rows, uint32_t vocab,
                             uint32_t hidden, int hadamard, const int64_t* positions, const flh_half* cos_table,
                             const flh_half* sin_table, flh_half* cos, flh_half* sin, uint32_t T, uint32_t max_len,
                             uint32_t head_dim, void* stream) {
  if (!ids || !table || !out || !positions || !cos_table || !sin_table || !cos || !sin) return fail(FLH_EINVAL, "embed: null pointer");
  if (misaligned16(table, out) || misaligned16(cos_table, sin_table, cos, sin)) return fail(FLH_EINVAL, "embed: tables and outputs must be 16-byte aligned");
  if (vocab == 0 || max_len == 0) return fail(FLH_EINVAL, "embed: the tables must not be empty");
  if (hidden == 0 || hidden % (hadamard ? 128 : 8)) return fail(FLH_EINVAL, "embed: hidden (%u) must be a multiple of %d", hidden, hadamard ? 128 : 8);
  if (head_dim == 0 || head_dim % 8) return fail(FLH_EINVAL, "embed: head_dim (%u) must be a multiple of 8", head_dim);
  const uint64_t first = (uint64_t)rows * (hidden / 8), second = 2ull * T * (head_dim / 8);
  if (first + second > 0x7FFFFFFFull) return fail(FLH_EINVAL, "embed: too many elements for one launch");
  const unsigned blocks = (unsigned)((first + 255) / 256 + (second + 255) / 256);
  if (blocks == 0) return FLH_OK;
  auto kern = hadamard ? embed_kernel<true> : embed_kernel<false>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (const long long*)ids, (const __half*)table,
                     (__half*)out, rows, vocab, hidden, (const long long*)positions, (const __half*)cos_table,
                     (const __half*)sin_table, (__half*)cos, (__half*)sin, T, max_len, head_dim);
  return check_launch("embed_kernel");
}

extern "C" int flh_add_rmsnorm_f16(const flh_half* x, const flh_half* add, const flh_half* weight, float eps, flh_half* out,
                                   flh_half* sum_out, uint32_t M, uint32_t K, void* stream) {
  if (!x || !out) return fail(FLH_EINVAL, "add_rmsnorm: null pointer");
  if (sum_out && !add) return fail(FLH_EINVAL, "add_rmsnorm: sum_out is the stored sum x + add and needs add");
  if (misaligned16(x, add, weight, out, sum_out)) return fail(FLH_EINVAL, "add_rmsnorm: tensors must be 16-byte aligned");
  if (K == 0 || K % 8 || K > 16384) return fail(FLH_EINVAL, "add_rmsnorm: K (%u) must be a multiple of 8, at most 16384", K);
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "add_rmsnorm: eps must not be negative");
  if (M == 0) return FLH_OK;
  hipLaunchKernelGGL(add_rmsnorm_kernel, dim3(M), dim3(256), 0, (hipStream_t)stream, (const __half*)x, (const __half*)add,
                     (const __half*)weight, (__half*)out, (__half*)sum_out, K, eps);
  return check_launch("add_rmsnorm_kernel");
}

extern "C" int flh_silu_mul_rotate_quant_i4(const flh_half* gate, const flh_half* up, uint8_t* q_packed, flh_half* scales,
                                            uint32_t M, uint32_t K, void* stream) {
  if (!gate || !up || !q_packed || !scales) return fail(FLH_EINVAL, "silu_mul_rotate_quant: null pointer");
  if (misaligned16(gate, up, q_packed)) return fail(FLH_EINVAL, "silu_mul_rotate_quant: gate, up and q_packed must be 16-byte aligned");
  if (K != 11008 && K != 14336) return fail(FLH_EINVAL, "silu_mul_rotate_quant: K (%u) must be 11008 or 14336", K);
  if (M > 256) return fail(FLH_EINVAL, "silu_mul_rotate_quant: at most 256 rows (%u given); longer batches take the gate / up GEMM that stores the product", M);
  if (M == 0) return FLH_OK;
  return launch_silu_mul_rotate_quant_mfma((const __half*)gate, (const __half*)up, q_packed, (__half*)scales, M, K,
                                           (hipStream_t)stream);
}

namespace {
int group_quant_f6(const flh_half* x, uint8_t* encoded, flh_half* scales, uint32_t M, uint32_t K, int hadamard, float scale_mul,
                   const EncodeLaunch& e, bool* taken, void* stream) {
  if (!x || !encoded || !scales) return fail(FLH_EINVAL, "group_quant_f6: null pointer");
  if (misaligned16(x, encoded)) return fail(FLH_EINVAL, "group_quant_f6: x and encoded must be 16-byte aligned");
  if (!(scale_mul > 0.f)) return fail(FLH_EINVAL, "group_quant_f6: scale_mul must be positive");
  if (K == 0 || K % 128) return fail(FLH_EINVAL, "group_quant_f6: K (%u) must be a positive multiple of 128", K);
  if ((uint64_t)M * (K / 128) > 0xFFFFFFFFull) return fail(FLH_EINVAL, "group_quant_f6: too many groups");
  if (M == 0) return FLH_OK;
  const uint32_t R = M * (K / 128);
  const dim3 grid((unsigned)(((uint64_t)R * 16 + 255) / 256)), block(256);
  const __half* xh = (const __half*)x;
  const bool quad = R >= quad_min_rows(hadamard != 0, true);
  const uint64_t quad_blocks = ((uint64_t)R + kQuadRows - 1) / kQuadRows;
  if (!hadamard && beside(quad ? quad_blocks : grid.x, (uint64_t)M * K, e)) {
    *taken = true;
    __half* sh = (__half*)scales;
    const hipStream_t st = (hipStream_t)stream;
    if (quad) return launch_beside(GroupQuantise<true>{xh, encoded, sh, R, scale_mul, M, K / 128}, (uint32_t)quad_blocks, e, st);
    return launch_beside(GroupQuantise<false>{xh, encoded, sh, R, scale_mul, M, K / 128}, grid.x, e, st);
  }
  if (quad)
    return hadamard ? launch_group_quad<true, true>(xh, encoded, (__half*)scales, R, scale_mul, M, K / 128, (hipStream_t)stream)
                    : launch_group_quad<false, true>(xh, encoded, (__half*)scales, R, scale_mul, M, K / 128, (hipStream_t)stream);
  if (hadamard)
    hipLaunchKernelGGL((group_kernel<128, true, true, true>), grid, block, 0, (hipStream_t)stream, xh, encoded,
                       (__half*)scales, nullptr, R, scale_mul, M, K / 128);
  else
    hipLaunchKernelGGL((group_kernel<128, false, true, true>), grid, block, 0, (hipStream_t)stream, xh, encoded,
                       (__half*)scales, nullptr, R, scale_mul, M, K / 128);
  return check_launch("group_kernel (6-bit output)");
}
}  // namespace

extern "C" int flh_group_quant_f6(const flh_half* x, uint8_t* encoded, flh_half* scales, uint32_t M, uint32_t K,
                                  int hadamard, float scale_mul, void* stream) {
  return group_quant_f6(x, encoded, scales, M, K, hadamard, scale_mul, kNoWeights, nullptr, stream);
}

extern "C" int flh_group_quant_encode_f6(const flh_half* x, uint8_t* encoded, flh_half* scales, uint32_t M, uint32_t K, int hadamard,
                                         float scale_mul, const flh_encode_list* weights, void* stream) {
  return with_weights(weights, M, stream, [&](const EncodeLaunch& e, bool* taken) {
    return group_quant_f6(x, encoded, scales, M, K, hadamard, scale_mul, e, taken, stream);
  });
}

extern "C" int flh_fwht_f16_inplace(flh_half* x, uint32_t R, int group, void* stream) {
  if (!x) return fail(FLH_EINVAL, "fwht: null pointer");
  if (misaligned16(x)) return fail(FLH_EINVAL, "fwht: x must be 16-byte aligned");
  return group_dispatch(nullptr, nullptr, nullptr, (__half*)x, R, group, true, false, 1.0f, (hipStream_t)stream);
}

extern "C" int flh_rotate_quant_i4(const flh_half* x, uint8_t* q_packed, flh_half* scales, flh_half* y_out, uint32_t M,
                                   uint32_t K, int hadamard, int had_group, int scale_group, float clip_ratio,
                                   void* stream) {
  if (!x || !q_packed || !scales) return fail(FLH_EINVAL, "rotate_quant: null pointer");
  if (misaligned16(x, q_packed, y_out)) return fail(FLH_EINVAL, "rotate_quant: x, q_packed and y_out must be 16-byte aligned");
  if (K == 0 || K % 16) return fail(FLH_EINVAL, "rotate_quant: K (%u) must be a positive multiple of 16", K);
  if (!(clip_ratio > 0.f)) return fail(FLH_EINVAL, "rotate_quant: clip_ratio must be positive");
  if (scale_group < 0) scale_group = 0;
  if (scale_group > 0 && (K % scale_group || scale_group % 2))
    return fail(FLH_EINVAL, "rotate_quant: scale group %d must be even and divide K = %u", scale_group, K);
  if (M == 0) return FLH_OK;
  hipStream_t st = (hipStream_t)stream;
  const __half* xh = (const __half*)x;
  __half* sh = (__half*)scales;
  __half* yh = (__half*)y_out;

  if (hadamard == FLH_HAD_MFMA) {
    if (had_group <= 0 && scale_group == 0 && !y_out && rotate_quant_mfma_supports(K))
      return launch_rotate_quant_mfma(xh, q_packed, sh, M, K, clip_ratio, st);
    hadamard = FLH_HAD_F32;  // shapes / options the matrix-core kernels do not cover
  }
  int Kd = 1, P = 1;
  float norm = 1.f;
  if (hadamard == FLH_HAD_F32) {
    if (had_group > 0 && (uint32_t)had_group != K) {
      if (!is_pow2(had_group) || K % had_group)
        return fail(FLH_EINVAL, "rotate_quant: hadamard group %d must be a power of two dividing K = %u", had_group, K);
      P = had_group;
      norm = sqrtf((float)had_group);
    } else {
      if (!factor_hadamard(K, &Kd, &P))
        return fail(FLH_EINVAL, "rotate_quant: no Hadamard factorisation for K = %u", K);
      norm = sqrtf((float)K);
    }
  } else if (hadamard != FLH_HAD_NONE) {
    return fail(FLH_EINVAL, "rotate_quant: unknown hadamard mode %d", hadamard);
  }

  const bool whole_row_pow2 = (hadamard == FLH_HAD_NONE || (Kd == 1 && (uint32_t)P == K));
  if (whole_row_pow2 && scale_group == 0 && K % 512 == 0 && is_pow2(K / 512) && K <= 8192) {
    const bool had = hadamard != FLH_HAD_NONE;
    if (had && K == 4096 && !yh && clip_ratio >= 1.0f && M <= kRow8MaxRows) {
      hipLaunchKernelGGL(rotate_quant_row8_kernel, dim3(M), dim3(512), 0, st, xh, q_packed, sh, 1.0f / 64.0f);
      return check_launch("rotate_quant_row8");
    }
    switch (K / 512) {
      case 1: return launch_wave<1>(xh, q_packed, sh, yh, M, had, clip_ratio, st);
      case 2: return launch_wave<2>(xh, q_packed, sh, yh, M, had, clip_ratio, st);
      case 4: return launch_wave<4>(xh, q_packed, sh, yh, M, had, clip_ratio, st);
      case 8: return launch_wave<8>(xh, q_packed, sh, yh, M, had, clip_ratio, st);
      case 16: return launch_wave<16>(xh, q_packed, sh, yh, M, had, clip_ratio, st);
    }
  }
  // the row in float32, a second copy for the dense factor's output and that factor's sign bits
  const size_t smem = (size_t)K * sizeof(float) * (Kd > 1 ? 2 : 1) + (Kd > 1 ? (((size_t)Kd * Kd + 7) / 8 / 16 + 2) * 16 : 0);   // + the byte after the last row's window
  if (smem > 160 * 1024 - 64) return fail(FLH_EINVAL, "rotate_quant: K = %u does not fit the LDS staging", K);
  static LdsGrant grant;                               // grows to the largest row asked for
  if (int rc = reserve_lds((const void*)rotate_quant_generic_kernel, smem, grant, "rotate_quant")) return rc;
  hipLaunchKernelGGL(rotate_quant_generic_kernel, dim3(M), dim3(kGenericThreads), smem, st, xh, q_packed, sh, yh, K,
                     hadamard == FLH_HAD_NONE ? 0 : P, Kd, norm, scale_group, clip_ratio);
  return check_launch("rotate_quant_generic");
}
