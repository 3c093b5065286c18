// The 6-bit-instruction GEMM for launches with enough work to fill the chip with large tiles (operand format, arithmetic
// and epilogues: gemm_f6.hip).
//
// Persistent workgroups walk over the launch's tiles.  One scale per row: four waves, one per SIMD with up to 512 registers, a
// wave 128 x 128 outputs (workgroup tile 256 x 256, accumulators in the 256 accumulation registers) or 64 x 128 (256 x 128).
// Group scales: eight waves, two per SIMD, on tiles of 256 x 128 or 128 x 128 (gemm_f6_large_group.hip).  K advances by 128
// codes per step through a ring of LDS stages that direct-to-LDS loads fill a whole ring ahead; the ring does not know about
// tiles: while the last steps of one tile are multiplied, the first stages of the next are already on their way, and a
// tile's outputs leave as stores that nobody waits for.
//
// What bounds it.  A compute unit loads 64 bytes per clock into LDS and reads 256 (16-byte reads; 8-byte ones 128), its SIMD needs
// 32 clocks per MFMA.  A step of a 128 x 128 tile (four waves of 64 x 64) is 384 clocks of loads for 256 of MFMAs, a step of the
// 256 x 256 tile 768 for 1024.  In-kernel timestamps at 8192 x 14336 x 4096: 1450-1580 clocks per step of the 256 x 256 tile (1150
// without its loads, 1050 without its fragment reads as well), 9700 per tile for the outputs.  The part is at its power limit:
// 1.6 GHz under the 256 x 256 tile, 1.95 under the group-scale kernel, where light kernels run at 2.4; launches back to back take
// 296 us instead of 262.  Prefetching the slabs into L2 changed nothing.
// us per launch, weights from HBM, alone - back to back where they differ, against the 128 x 128 tiles of gemm_f6.hip and the
// int8 kernel:
//   one scale per row, 8192 x 14336 x 4096:  262 - 296 (3.67 - 3.25 POP/s) against 372 and 378;  4096 x 4096 x 11008: 88 against 118, 136
//   token scales,      8192 x 14336 x 4096:  361 - 372 (2.66 - 2.58) against 429 and 599;  2048 x 28672 x 4096: 188 against 221, 304
//   group scales,      8192 x 14336 x 4096:  395 - 400 (2.43 - 2.40) against 575 and 701;  2048 x 28672 x 4096: 202 against 289, 356
#pragma once
#include "gemm_i4.h"
#include "lane_ops.h"

namespace flh {
namespace f6l {

typedef int v8i __attribute__((ext_vector_type(8)));


enum Out { kPlain = 0, kSwiglu = 1, kRope = 2, kResidual = 3 };

constexpr int kPitch = 256 + 16;    // bytes per row of a wave's staging tile (128 fp16 channels)
constexpr int kBlock = 96;          // encoded bytes of K per row per step
constexpr int kBf6 = 3;             // e3m2
constexpr int kRowBlock = 32 * kBlock + 16;   // LDS bytes of 32 rows of a stage: the 16 bytes keep the compiler from
                                              // merging the 8-byte fragment reads of two row blocks

// where a tile's operands and outputs are
struct Tile {
  const uint8_t *B, *B2;
  const __half *Bs, *Bs2;
  void* D;
  int N, m0, n0, seg, head0;
};

template <int BN, int OUT, int BM = 256>
__device__ __forceinline__ Tile tile_of(const GemmArgs& p, unsigned L) {
  constexpr int BNC = OUT == kSwiglu ? BN / 2 : BN;
  const unsigned band = p.group_m * p.tiles_n;
  const unsigned first_m = (L / band) * p.group_m;
  const unsigned gsz = min((unsigned)p.tiles_m - first_m, (unsigned)p.group_m);
  const int tile_m = first_m + (L % band) % gsz;
  const int tile_n = (L % band) / gsz;
  Tile t{p.B, p.B2, p.Bs, p.Bs2, p.D, p.N, tile_m * BM, tile_n * BNC, 0, 0};
  for (int s = 1; s < p.n_seg; ++s)
    if (tile_n >= p.seg_tile0[s]) {
      t.B = p.seg_B[s];
      t.Bs = p.seg_Bs[s];
      t.D = p.seg_D[s];
      t.N = p.seg_N[s];
      t.n0 = (tile_n - p.seg_tile0[s]) * BNC;
      t.seg = s;
    }
  t.head0 = t.n0 / 128;
  return t;
}

// ---- operand loads through buffer descriptors
// 3 KiB in three instructions: lane i's 16 bytes at voff, + 1024, + 2048 go to lds_base + 16 i, + 1024, + 2048
__device__ __forceinline__ void load_block_to_lds(const v4i& d, unsigned voff, unsigned lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen offset:1024 lds\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen offset:2048 lds" ::"s"(lds_base), "v"(voff), "s"(d) : "memory", "m0");
}

// ... the first 2 KiB of it, and the third
__device__ __forceinline__ void load_two_thirds_to_lds(const v4i& d, unsigned voff, unsigned lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen offset:1024 lds" ::"s"(lds_base), "v"(voff), "s"(d) : "memory", "m0");
}
__device__ __forceinline__ void load_last_third_to_lds(const v4i& d, unsigned voff, unsigned lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen offset:2048 lds" ::"s"(lds_base), "v"(voff), "s"(d) : "memory", "m0");
}

// The last step of the outputs: ROWS rows of 128 fp16 values, staged in LDS by this wave (kPitch bytes apart, the first
// row being row m_first of the launch), leave as whole row segments.  wcol: which 128 of the tile's weight rows the values belong to.
template <int ROWS, int OUT>
__device__ __forceinline__ void store_rows(const GemmArgs& p, const Tile& cur, const uint8_t* ep, int m_first, int wcol, int lane) {
  if constexpr (OUT == kPlain || OUT == kResidual) {
    const int r4 = lane >> 4, n = cur.n0 + wcol * 128 + (lane & 15) * 8;
    const unsigned off = ((unsigned)r4 * (unsigned)cur.N + (unsigned)n) * 2;   // from the block's first row
    v4i v[ROWS / 4], add[OUT == kResidual ? ROWS / 4 : 1];
#pragma unroll
    for (int it = 0; it < ROWS / 4; ++it) {
      v[it] = *(const v4i*)(ep + (it * 4 + r4) * kPitch + (lane & 15) * 16);
      if constexpr (OUT == kResidual)   // (may be the output itself: read before the store)
        if (m_first + it * 4 + r4 < p.M && n < cur.N)
          add[it] = *(const v4i*)((const uint8_t*)p.R + (size_t)(m_first + it * 4) * cur.N * 2 + off);
    }
#pragma unroll
    for (int it = 0; it < ROWS / 4; ++it) {
      if constexpr (OUT == kResidual) v[it] = add_h8(v[it], add[it]);
      if (m_first + it * 4 + r4 < p.M && n < cur.N)   // (N is a multiple of 8)
        *(v4i*)((uint8_t*)cur.D + (size_t)(m_first + it * 4) * cur.N * 2 + off) = v[it];
    }
  } else {
    // the two halves of a row, 64 channels apart: gate and up of the same channels, or the halves of a head
    const int c = lane & 7;
    h8 x1[ROWS / 8], x2[ROWS / 8];
#pragma unroll
    for (int it = 0; it < ROWS / 8; ++it) {
      const uint8_t* row = ep + (it * 8 + (lane >> 3)) * kPitch + c * 16;
      x1[it] = *(const h8*)row, x2[it] = *(const h8*)(row + 128);
    }
    if constexpr (OUT == kSwiglu) {
      const int n = cur.n0 + wcol * 64 + c * 8;
#pragma unroll
      for (int it = 0; it < ROWS / 8; ++it) {
        const int m = m_first + it * 8 + (lane >> 3);
        h8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = silu_mul_f16(x1[it][e], x2[it][e]);
        if (m < p.M && n < cur.N) *(h8*)((__half*)cur.D + (size_t)m * cur.N + n) = o;
      }
    } else {
      const int head = cur.head0 + wcol;
#pragma unroll
      for (int it = 0; it < ROWS / 8; ++it) {
        const int m = m_first + it * 8 + (lane >> 3);
        const bool live = m < p.M && head * 128 < cur.N;
        const int b = m / p.rope_T, t = live ? m - b * p.rope_T : 0;
        long long at_slot = 0;
        if (cur.seg > 0) at_slot = p.rope_pos[t];
        const bool in_range = at_slot >= 0 && (cur.seg == 0 || at_slot < (long long)p.rope_max_len);
        __half* dst = cur.seg == 0 ? (__half*)cur.D + (size_t)m * cur.N + head * 128
                                   : (__half*)cur.D + (((size_t)b * p.rope_hkv + head) * p.rope_max_len +
                                                       (size_t)(in_range ? at_slot : 0)) * 128;
        if (cur.seg < 2) {
          const __half *ct = p.rope_cos + (size_t)t * 128 + c * 8, *st = p.rope_sin + (size_t)t * 128 + c * 8;
          const h8 k1 = *(const h8*)ct, k2 = *(const h8*)(ct + 64), n1 = *(const h8*)st, n2 = *(const h8*)(st + 64);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            _Float16 y1 = x1[it][e], y2 = x2[it][e];
            rope_pair(y1, y2, k1[e], k2[e], n1[e], n2[e]);
            x1[it][e] = y1, x2[it][e] = y2;
          }
        }
        if (live && in_range) {
          *(h8*)(dst + c * 8) = x1[it];
          *(h8*)(dst + 64 + c * 8) = x2[it];
        }
      }
    }
  }
}

// The same for a wave of 64 channels (kHalfPitch bytes apart): channels wcol * 64 + 0 .. 63 of the tile, or, where pairs meet,
// wcol * 32 + 0 .. 31 of either half of it.
constexpr int kHalfPitch = 128 + 16;
template <int ROWS, int OUT>
__device__ __forceinline__ void store_half_rows(const GemmArgs& p, const Tile& cur, const uint8_t* ep, int m_first, int wcol, int lane) {
  if constexpr (OUT == kPlain || OUT == kResidual) {
    const int r8 = lane >> 3, n = cur.n0 + wcol * 64 + (lane & 7) * 8;
    const unsigned off = ((unsigned)r8 * (unsigned)cur.N + (unsigned)n) * 2;   // from the block's first row
    v4i v[ROWS / 8], add[OUT == kResidual ? ROWS / 8 : 1];
#pragma unroll
    for (int it = 0; it < ROWS / 8; ++it) {
      v[it] = *(const v4i*)(ep + (it * 8 + r8) * kHalfPitch + (lane & 7) * 16);
      if constexpr (OUT == kResidual)   // (may be the output itself: read before the store)
        if (m_first + it * 8 + r8 < p.M && n < cur.N)
          add[it] = *(const v4i*)((const uint8_t*)p.R + (size_t)(m_first + it * 8) * cur.N * 2 + off);
    }
#pragma unroll
    for (int it = 0; it < ROWS / 8; ++it) {
      if constexpr (OUT == kResidual) v[it] = add_h8(v[it], add[it]);
      if (m_first + it * 8 + r8 < p.M && n < cur.N)   // (N is a multiple of 8)
        *(v4i*)((uint8_t*)cur.D + (size_t)(m_first + it * 8) * cur.N * 2 + off) = v[it];
    }
  } else {
    static_assert(ROWS == 16, "one row per four lanes");
    const int c = lane & 3, m = m_first + (lane >> 2);
    const uint8_t* row = ep + (lane >> 2) * kHalfPitch + c * 16;
    h8 x1 = *(const h8*)row, x2 = *(const h8*)(row + 64);
    if constexpr (OUT == kSwiglu) {
      const int n = cur.n0 + wcol * 32 + c * 8;
      h8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = silu_mul_f16(x1[e], x2[e]);
      if (m < p.M && n < cur.N) *(h8*)((__half*)cur.D + (size_t)m * cur.N + n) = o;
    } else {
      const int head = cur.head0, ch = wcol * 32 + c * 8;   // a tile's 128 channels are one head
      const bool live = m < p.M && head * 128 < cur.N;
      const int b = m / p.rope_T, t = live ? m - b * p.rope_T : 0;
      long long at_slot = 0;
      if (cur.seg > 0) at_slot = p.rope_pos[t];
      const bool in_range = at_slot >= 0 && (cur.seg == 0 || at_slot < (long long)p.rope_max_len);
      __half* dst = cur.seg == 0 ? (__half*)cur.D + (size_t)m * cur.N + head * 128
                                 : (__half*)cur.D + (((size_t)b * p.rope_hkv + head) * p.rope_max_len +
                                                     (size_t)(in_range ? at_slot : 0)) * 128;
      if (cur.seg < 2) {
        const __half *ct = p.rope_cos + (size_t)t * 128 + ch, *st = p.rope_sin + (size_t)t * 128 + ch;
        const h8 k1 = *(const h8*)ct, k2 = *(const h8*)(ct + 64), n1 = *(const h8*)st, n2 = *(const h8*)(st + 64);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          _Float16 y1 = x1[e], y2 = x2[e];
          rope_pair(y1, y2, k1[e], k2[e], n1[e], n2[e]);
          x1[e] = y1, x2[e] = y2;
        }
      }
      if (live && in_range) {
        *(h8*)(dst + ch) = x1;
        *(h8*)(dst + 64 + ch) = x2;
      }
    }
  }
}

// Launches, for a.M x a.N x a.K and the operands of `a` (segments, B2, R and the rotary fields as `out` needs them).
int launch_large_row(const GemmArgs& a, bool wide, Out out, hipStream_t stream);
// tall: tiles of 256 x 128, else 128 x 128
int launch_large_group(const GemmArgs& a, bool token, bool tall, Out out, hipStream_t stream);

}  // namespace f6l
}  // namespace flh
