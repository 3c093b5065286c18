// int4 x int4 GEMM + dequant for a handful of tokens (decode, M <= 64): the weights are
// streamed from HBM exactly once and the contraction is split over K inside a workgroup.
//
// Same arithmetic as gemm_i4.hip (codes x 16 as int8 on the matrix cores, exact int32 sums,
// identical epilogue roundings); reference: flh/kernels/gemm_and_dequant_i4.cu:315-508.
//
// One workgroup of 8 waves owns 16 output channels and every token.  A wave takes every 8th
// "double step" of K (256 codes = one 128-byte line of each of the 16 weight rows): lane l
// loads 2 x 16 packed bytes of weight row l % 16 at chunk l / 16, the same of the activation
// row l % 16 of each 16-token tile, and issues v_mfma_i32_16x16x64_i8 on the low and the high
// nibbles.  With 256 workgroups x 8 waves x two double steps in flight the whole of a
// 4096 x 4096 weight matrix is requested at once, which is what a latency-bound stream needs.
// Partial sums meet in LDS:
//   * one scale per row: the eight waves' int32 tiles are added and dequantised;
//   * scale groups of 128: every group's tile is kept in LDS (as float32) and the fp32 result is built
//     by one fused multiply-add per group in ascending order, exactly as the prefill kernel does.
// What bounds it, beside the weights (in-kernel timestamps, 4096 x 14336 with group scales, 16 tokens, when it took 14.5 us):
// the scale tables took 3.4 us before the first weight was requested and the fold 2.4 at the end.  The scales now come as they
// are, by direct-to-LDS loads behind the first weights; tiles are stored as float32 by the waves that made them and folded
// without bank conflicts, two groups of scales per read, eight pairs of groups read ahead of their multiply-adds (a pair at a
// time the chain waits for LDS at every pair: one token 4096 x 14336 12.7 us with group scales where the eight take 10.9).
// us, weights from HBM, against scales as float tables and integer tiles (N x K), token scales / group scales:
//   16 tokens: 4096 x 14336 14.8 / 15.1 -> 11.4 / 11.5, 4096 x 11008 12.4 / 12.7 -> 9.9 / 9.8, 6144 x 4096 8.5 / 8.4 -> 7.4 /
//   7.4, 4096 x 4096 6.5 / 6.6 -> 5.5 / 5.6;  one token: 4096 x 14336 11.9 / 12.0 -> 10.3 / 10.9, 4096 x 4096 5.7 / 5.7 -> 5.1 / 5.2
#include <atomic>
#include "gemm_i4.h"
#include "rotate_row.h"

namespace flh {
namespace {

constexpr int kWaves = 8;
constexpr int kRotateGemmMaxTokens = 4;    // tokens of the GEMM that quantises its own activations
constexpr int kGroupMaxKT = 128;   // groups of 128 codes that fit the LDS tile store (K <= 16384)

__device__ __forceinline__ void unpack_lo_hi(const v4i w, v4i& lo, v4i& hi) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    lo[i] = (w[i] << 4) & (int)0xF0F0F0F0;
    hi[i] = w[i] & (int)0xF0F0F0F0;
  }
}

// The weight matrix a workgroup's block of 16 output channels belongs to (several may share the activations in
// one launch; segment starts are counted in blocks of 16 here) and the block's first channel inside it.
struct DecodeWeights {
  const uint8_t* B;
  const __half* Bs;
  void* D;
  int N, n0;
};
__device__ __forceinline__ DecodeWeights decode_weights(const GemmArgs& p, int block) {
  DecodeWeights w{p.B, p.Bs, p.D, p.N, block * 16};
  for (int s = 1; s < p.n_seg; ++s)
    if (block >= p.seg_tile0[s]) w = DecodeWeights{p.seg_B[s], p.seg_Bs[s], p.seg_D[s], p.seg_N[s], (block - p.seg_tile0[s]) * 16};
  return w;
}
// host side: segment starts in blocks of 16 channels; returns the number of blocks of the launch
int decode_blocks(GemmArgs& a) {
  int blocks = (a.N + 15) / 16;
  for (int s = 1; s < a.n_seg; ++s) {
    a.seg_tile0[s] = blocks;
    blocks += (a.seg_N[s] + 15) / 16;
  }
  return blocks;
}

// one fp16 output; with a residual (single weight matrix) the stored value is fp16(R + value)
__device__ __forceinline__ void store_f16(const GemmArgs& p, const DecodeWeights& w, int gm, int gn, _Float16 v) {
  const size_t at = (size_t)gm * w.N + gn;
  if (p.R) v = v + ((const _Float16*)p.R)[at];
  ((_Float16*)w.D)[at] = v;
}

// Group scales wait in LDS as they are: row after row (the tokens if they have group scales, then the 16 channels) of KT
// halves, an odd number of dwords apart.  They come by direct-to-LDS loads that are requested behind the first weights and waited for last;
// rows that dword loads cannot fetch (an odd number of groups, an odd element offset, one scale per channel) are filled half by half.
__host__ __device__ constexpr int scale_pitch(int KT) { return ((KT + 1) >> 1) | 1; }   // dwords per row

__device__ __forceinline__ void request_scales(const GemmArgs& p, const DecodeWeights& w, unsigned* table, int KT, int tid) {
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pitch = scale_pitch(KT), tokens = p.a_cols > 1 ? p.M : 0, rows = tokens + 16;   // (at most 16 tokens)
  auto row_of = [&](int row) {
    return row < tokens ? p.As + (size_t)row * KT : w.Bs + (size_t)min(w.n0 + row - tokens, w.N - 1) * p.b_cols;
  };
  if (p.b_cols > 1 && ((uintptr_t)w.Bs & 3) == 0 && (tokens == 0 || ((uintptr_t)p.As & 3) == 0) && KT % 2 == 0) {
    const float inv = 1.0f / (float)pitch;
    const int total = rows * pitch;
    const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned*)table;
    for (int f0 = wave * 64; f0 < total; f0 += kWaves * 64) {
      const int f = min(f0 + lane, total - 1);
      int row = (int)((float)f * inv);               // f < 2^12: off by one at most
      row += (f >= (row + 1) * pitch ? 1 : 0) - (f < row * pitch ? 1 : 0);
      load_to_lds4(row_of(row) + 2 * min(f - row * pitch, (KT >> 1) - 1), base + f0 * 4);
    }
  } else {
#pragma nounroll
    for (int i = tid; i < rows * KT; i += kWaves * 64) {
      const int row = i / KT, g = i - row * KT;
      ((__half*)(table + row * pitch))[g] = row_of(row)[row >= tokens && p.b_cols == 1 ? 0 : g];
    }
    if (KT % 2)
      for (int row = tid; row < rows; row += kWaves * 64) ((__half*)(table + row * pitch))[KT] = __half(0.f);
  }
}
// dwords of the table, rounded up to whole load instructions
__host__ __device__ constexpr size_t scale_table_dwords(int KT) { return ((size_t)32 * scale_pitch(KT) + 63) / 64 * 64; }

// The token's and, with one scale per row, the channel's scale of the value that thread `tid` finishes first: requested with the
// weights, one latency less at the end.
struct FirstScales {
  float a, b;
};
template <int EPI>
__device__ __forceinline__ FirstScales first_scales(const GemmArgs& p, const DecodeWeights& w, const __half* a_scales, int tid) {
  const int gm = min((tid >> 8) * 16 + ((tid >> 2) & 15), p.M - 1), gn = min(w.n0 + ((tid >> 6) & 3) * 4 + (tid & 3), w.N - 1);
  FirstScales f{0.f, 0.f};
  if (a_scales && EPI != kInt32 && (EPI == kRowScale || p.a_cols == 1)) f.a = __half2float(a_scales[gm]);
  if constexpr (EPI == kRowScale) f.b = __half2float(w.Bs[gn]);
  return f;
}

// out = fma(sum, scale, out) over the groups in ascending order: v[g * MT * 256] the sums, ra and rb the token's and the channel's
// scales, two to a dword (TOKEN: the channel's alone).  Eight pairs of groups are read ahead of their multiply-adds, by hand:
// a loop with inline assembly is not unrolled, and a pair at a time waits for LDS at every pair.
template <int MT, bool TOKEN>
__device__ __forceinline__ float fold_groups(const float* v, const unsigned* ra, const unsigned* rb, int KT) {
  constexpr int kAhead = 8;
  const int pairs = KT >> 1;
  float out = 0.f;
  auto fold = [&](float lo, float hi, unsigned a, unsigned b) {
    if constexpr (TOKEN) {
      out = fma_half<0>(lo, b, out);
      out = fma_half<1>(hi, b, out);
    } else {
      out = __builtin_fmaf(lo, mul_halves<0>(a, b), out);
      out = __builtin_fmaf(hi, mul_halves<1>(a, b), out);
    }
  };
  auto batch = [&](int g, auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
    float lo[kAhead], hi[kAhead];
    unsigned a[kAhead], b[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int at = WHOLE ? g + u : min(g + u, pairs - 1);
      lo[u] = v[2 * at * MT * 256], hi[u] = v[(2 * at + 1) * MT * 256];
      a[u] = TOKEN ? 0u : ra[at], b[u] = rb[at];
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (WHOLE || g + u < pairs) fold(lo[u], hi[u], a[u], b[u]);
  };
  int g = 0;
  for (; g + kAhead <= pairs; g += kAhead) batch(g, std::true_type{});
  if (g < pairs) batch(g, std::false_type{});
  if (KT & 1) {
    const float last = v[(KT - 1) * MT * 256];
    if constexpr (TOKEN) out = fma_half<0>(last, rb[pairs], out);
    else out = __builtin_fmaf(last, mul_halves<0>(ra[pairs], rb[pairs]), out);
  }
  return out;
}

// Partial sums in LDS -> outputs.  Lane l of a tile holds token l % 16 and channels 4 (l / 16) + i, i = 0..3; a thread
// finishes the value at its own place of the tile (reads without bank conflicts).
// Groups: float32 tiles of 256 x the sums, one fused multiply-add per group in ascending order, the exact 2^-8 at the end.
// KTC: the groups of a row where they are known (one scale per token then, and the channels' rows of the table without padding).
template <int MT, int EPI, int KTC = 0>
__device__ __forceinline__ void decode_finish(const GemmArgs& p, const DecodeWeights& w, const int* red, const unsigned* table,
                                              const __half* a_scales, const FirstScales& first, int tid) {
  const int KT = KTC ? KTC : p.K >> 7;
  for (int idx = tid; idx < MT * 256; idx += kWaves * 64) {
    const int mt = idx >> 8, pos = idx & 255, m = (pos >> 2) & 15, n = (pos >> 6) * 4 + (pos & 3);
    const int gm = mt * 16 + m, gn = w.n0 + n;
    if (gm >= p.M || gn >= w.N) continue;
    if constexpr (EPI == kGroupScale) {
      const int pitch = KTC ? KTC / 2 : scale_pitch(KT);
      const float* v = (const float*)red + mt * 256 + pos;
      float out;
      if (KTC || p.a_cols == 1) {                    // one scale per token: applied once, after the groups
        const float s_a = idx == tid ? first.a : __half2float(a_scales[gm]);
        out = fold_groups<MT, true>(v, nullptr, table + n * pitch, KT);
        out = round_here(out * 0.00390625f) * s_a;
      } else {
        out = fold_groups<MT, false>(v, table + m * pitch, table + (p.M + n) * pitch, KT);
        out *= 0.00390625f;
      }
      store_f16(p, w, gm, gn, (_Float16)round_here(out));
    } else {
      int sum = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) sum += red[(w * MT + mt) * 256 + pos];
      if constexpr (EPI == kInt32) {
        ((int32_t*)w.D)[(size_t)gm * w.N + gn] = sum >> 8;
      } else {
        // sum = 256 * (exact contraction); the weight scale carries the matching exact 2^-8
        const float sa = idx == tid ? first.a : __half2float(a_scales[gm]);
        const float sb = (idx == tid ? first.b : __half2float(w.Bs[gn])) * 0.00390625f;
        store_f16(p, w, gm, gn, (_Float16)round_here((float)sum * (sa * sb)));
      }
    }
  }
}

__device__ __forceinline__ v4f tile_as_float(const v4i& t) { return v4f{(float)t[0], (float)t[1], (float)t[2], (float)t[3]}; }

template <int MT, int EPI>
__global__ __launch_bounds__(kWaves * 64) void gemm_i4_decode_kernel(const GemmArgs p) {
  extern __shared__ __align__(16) int red[];   // tiles: [wave | group][MT][64 lanes][4], int32 | float32; then the scales
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const DecodeWeights w = decode_weights(p, blockIdx.x);
  const int n0 = w.n0;
  const int Kb = p.K >> 1, KT = p.K >> 7, ND = (KT + 1) >> 1;

  const uint8_t* bptr = w.B + (size_t)min(n0 + r, w.N - 1) * Kb + c * 16;
  const uint8_t* aptr[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) aptr[mt] = p.A + (size_t)min(mt * 16 + r, p.M - 1) * Kb + c * 16;

  unsigned* table = (unsigned*)(red + KT * MT * 256);   // group mode
  const FirstScales first = first_scales<EPI>(p, w, p.As, tid);
  v4i acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = v4i{0, 0, 0, 0};

  auto load = [&](int ds, v4i (&b)[2], v4i (&a)[MT][2]) {
    const size_t off = (size_t)ds * 128;
    const bool second = 2 * ds + 1 < KT;           // K = 128 * odd: the last double step is half empty
    b[0] = *(const v4i*)(bptr + off);
    b[1] = second ? *(const v4i*)(bptr + off + 64) : v4i{0, 0, 0, 0};
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      a[mt][0] = *(const v4i*)(aptr[mt] + off);
      a[mt][1] = second ? *(const v4i*)(aptr[mt] + off + 64) : v4i{0, 0, 0, 0};
    }
  };
  auto compute = [&](int ds, const v4i (&b)[2], const v4i (&a)[MT][2]) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      v4i blo, bhi;
      unpack_lo_hi(b[half], blo, bhi);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        v4i alo, ahi;
        unpack_lo_hi(a[mt][half], alo, ahi);
        acc[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(blo, alo, acc[mt], 0, 0, 0);
        acc[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bhi, ahi, acc[mt], 0, 0, 0);
        if constexpr (EPI == kGroupScale) {
          const int g = 2 * ds + half;
          if (g < KT) *(v4f*)(red + ((g * MT + mt) * 64 + lane) * 4) = tile_as_float(acc[mt]);
          acc[mt] = v4i{0, 0, 0, 0};
        }
      }
    }
  };

  // two double steps in flight per wave
  v4i b0[2], b1[2], a0[MT][2], a1[MT][2];
  int ds = wave;
  if (ds < ND) load(ds, b0, a0);
  if constexpr (EPI == kGroupScale) request_scales(p, w, table, KT, tid);
  for (; ds < ND; ds += 2 * kWaves) {
    const bool more = ds + kWaves < ND;
    if (more) load(ds + kWaves, b1, a1);
    compute(ds, b0, a0);
    if (more) {
      if (ds + 2 * kWaves < ND) load(ds + 2 * kWaves, b0, a0);
      compute(ds + kWaves, b1, a1);
    }
  }
  if constexpr (EPI != kGroupScale) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) *(v4i*)(red + ((wave * MT + mt) * 64 + lane) * 4) = acc[mt];
  }
  if constexpr (EPI == kGroupScale) wait_vmcnt<0>();     // the scales
  __syncthreads();

  decode_finish<MT, EPI>(p, w, red, table, p.As, first, tid);
}

template <int MT, int EPI>
int launch_decode(const GemmArgs& a, hipStream_t stream) {
  const int KT = a.K >> 7;
  const size_t smem = EPI == kGroupScale ? (size_t)KT * MT * 1024 + scale_table_dwords(KT) * 4 : (size_t)kWaves * MT * 1024;
  auto kern = gemm_i4_decode_kernel<MT, EPI>;
  if constexpr (EPI == kGroupScale) {
    static LdsGrant grant;                             // per instantiation; sized for the longest rows it takes
    if (int rc = reserve_lds((const void*)kern, (size_t)kGroupMaxKT * MT * 1024 + scale_table_dwords(kGroupMaxKT) * 4, grant, "gemm (decode)"))
      return rc;
  }
  GemmArgs g = a;
  const int blocks = decode_blocks(g);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kWaves * 64), smem, stream, g);
  return check_launch("gemm_i4_decode");
}

// The decode GEMM with the activation quantiser inside, for one to four tokens of K = 4096: every workgroup
// requests its share of the weights, then rotates, quantises and packs the tokens into LDS itself -- all eight
// waves on each row, rotate_quant_row_8waves: the additions of the stand-alone kernel in the same order, so the
// codes and scales are the same bits -- while the weights are still on their way from HBM.  The rotation is
// repeated by every workgroup (about a microsecond per token, two with the norm); what it saves is a whole launch
// in front of the GEMM, which is worth more than that for one or two tokens and outputs up to about 8 K channels
// (the callers' rules say where).
//
// T tiles of 16 channels per workgroup.  Two rotations that share a compute unit get in each other's way: with one
// tile each, what goes beyond 256 workgroups paid for a second rotation.  A workgroup that owns two tiles requests
// the weights of both, rotates once, and multiplies one tile after the other from the same codes in LDS.  One token,
// us, one tile / two: norm and residual 4096 x 5120 10.4 / 8.7, 6144 10.4 / 8.8, 8192 10.9 / 9.5 (group scales 11.6 /
// 10.4); two tokens, rotation only, 6144 9.2 / 8.5.
//
// NORM / ADD: the tokens are RMS-normalised first (NORM), after a residual addition x + add (ADD) -- the prologues of
// flh_rmsnorm_rotate_quant_i4 / flh_add_rmsnorm_rotate_quant_i4 with the same roundings, so again the same bits as the
// separate launches.  Every workgroup forms the sum for itself; workgroup 0 stores it (the new residual stream).
struct DecodePrologue {
  const __half* rms_weight;   // NORM: null = no weight
  float eps;
  const __half* add;          // ADD
  __half* sum_out;            // ADD
};

template <int EPI, int T, bool NORM, bool ADD>
__global__ __launch_bounds__(kWaves * 64) void rotate_gemm_i4_decode_kernel(const __half* __restrict__ x,
                                                                            const GemmArgs p, float norm,
                                                                            const DecodePrologue pro) {
  constexpr int K = 4096, Kb = K / 2, KT = K / 128, ND = KT / 2, NDW = ND / kWaves;
  constexpr int ROW = Kb + 16;                 // code rows 16 bytes apart in the banks
  constexpr int TILES = EPI == kGroupScale ? KT : 2 * kWaves;   // at least the 16 KB the rotation stages in
  extern __shared__ __align__(16) int red[];   // tiles [wave | group][64 lanes][4], channel scales, maxima, codes, token scales
  unsigned* table = (unsigned*)(red + TILES * 256);
  constexpr int TABLE = EPI == kGroupScale ? 16 * KT / 2 : 0;   // dwords of a tile's scales
  float* sA = (float*)(table + T * TABLE);     // scratch of the rotation
  uint8_t* codes = (uint8_t*)(sA + 16);
  __half* tok = (__half*)(codes + kRotateGemmMaxTokens * ROW);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  auto tile = [&](int t) { return decode_weights(p, min((int)blockIdx.x * T + t, p.tiles_n - 1)); };

  // this wave's weights first, of all its tiles: they are in flight while the tokens are rotated
  v4i b[T][NDW][2];
  FirstScales first[T];
  static_for<T>([&](auto t_tag) {
    constexpr int t = decltype(t_tag)::value;
    const DecodeWeights w = tile(t);
    const uint8_t* bptr = w.B + (size_t)min(w.n0 + r, w.N - 1) * Kb + c * 16;
#pragma unroll
    for (int i = 0; i < NDW; ++i) {
      const int ds = wave + i * kWaves;
      b[t][i][0] = *(const v4i*)(bptr + (size_t)ds * 128);
      b[t][i][1] = *(const v4i*)(bptr + (size_t)ds * 128 + 64);
    }
    // The scales, 16 rows of 64 bytes one behind the other: one load instruction of one wave (with the other kernel's request, its
    // divisions and its branch for rows of any kind, a token took 11.5 us through 6144 channels with the prologues; 10.9 with this).
    if constexpr (EPI == kGroupScale) {
      static_assert(kWaves * 64 == 16 * KT && KT == 32, "a load instruction, or a half per thread");
      if (((uintptr_t)w.Bs & 15) == 0) {
        if (wave == kWaves - 1 - t % kWaves)
          load_to_lds16(w.Bs + (size_t)min(w.n0 + (lane >> 2), w.N - 1) * KT + (lane & 3) * 8,
                        (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned*)(table + t * TABLE));
      } else {
        ((__half*)(table + t * TABLE))[tid] = w.Bs[(size_t)min(w.n0 + (tid >> 5), w.N - 1) * KT + (tid & 31)];
      }
    }
    first[t] = first_scales<EPI>(p, w, nullptr, tid);
  });
  for (int row = 0; row < p.M; ++row) {
    if constexpr (NORM || ADD)
      rotate_quant_row_8waves<NORM, ADD>(x + (size_t)row * K, (float*)red, sA, codes + row * ROW, tok + row, norm, wave,
                                         pro.rms_weight, pro.eps, ADD ? pro.add + (size_t)row * K : nullptr,
                                         ADD && blockIdx.x == 0 ? pro.sum_out + (size_t)row * K : nullptr);
    else
      rotate_quant_row_8waves(x + (size_t)row * K, (float*)red, sA, codes + row * ROW, tok + row, norm, wave);
  }
  __syncthreads();

  const uint8_t* arow = codes + min(r, p.M - 1) * ROW + c * 16;
  static_for<T>([&](auto t_tag) {
    constexpr int t = decltype(t_tag)::value;
    if (t > 0) __syncthreads();                          // the tile before is finished
    v4i acc = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NDW; ++i) {
      const int ds = wave + i * kWaves;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        v4i blo, bhi, alo, ahi;
        unpack_lo_hi(b[t][i][half], blo, bhi);
        unpack_lo_hi(*(const v4i*)(arow + ds * 128 + half * 64), alo, ahi);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(blo, alo, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(bhi, ahi, acc, 0, 0, 0);
        if constexpr (EPI == kGroupScale) {
          *(v4f*)(red + ((2 * ds + half) * 64 + lane) * 4) = tile_as_float(acc);
          acc = v4i{0, 0, 0, 0};
        }
      }
    }
    if constexpr (EPI != kGroupScale) *(v4i*)(red + (wave * 64 + lane) * 4) = acc;
    if constexpr (EPI == kGroupScale && t == 0) wait_vmcnt<0>();   // the scales, of every tile
    __syncthreads();
    first[t].a = __half2float(tok[min((tid >> 2) & 15, p.M - 1)]);
    if ((int)blockIdx.x * T + t < p.tiles_n)
      decode_finish<1, EPI, EPI == kGroupScale ? KT : 0>(p, tile(t), red, table + t * TABLE, tok, first[t], tid);
  });
}

template <int EPI, int T>
int launch_rotate_decode(const __half* x, const GemmArgs& g, hipStream_t stream, const DecodePrologue* pro) {
  constexpr int K = 4096, KT = K / 128;
  constexpr size_t smem = (size_t)(EPI == kGroupScale ? KT : 2 * kWaves) * 1024 + (EPI == kGroupScale ? T * 16 * KT * 2 : 0) + 64 +
                          kRotateGemmMaxTokens * (K / 2 + 16) + 32;
  static_assert(smem <= 64 * 1024, "fits the default dynamic LDS limit");
  const dim3 grid((g.tiles_n + T - 1) / T), block(kWaves * 64);
  const DecodePrologue none{nullptr, 0.f, nullptr, nullptr};
  if (!pro)
    hipLaunchKernelGGL((rotate_gemm_i4_decode_kernel<EPI, T, false, false>), grid, block, smem, stream, x, g, 1.0f / 64.0f, none);
  else if (pro->add)
    hipLaunchKernelGGL((rotate_gemm_i4_decode_kernel<EPI, T, true, true>), grid, block, smem, stream, x, g, 1.0f / 64.0f, *pro);
  else
    hipLaunchKernelGGL((rotate_gemm_i4_decode_kernel<EPI, T, true, false>), grid, block, smem, stream, x, g, 1.0f / 64.0f, *pro);
  return check_launch("rotate_gemm_i4_decode");
}

template <int EPI>
int launch_rotate_decode(const __half* x, const GemmArgs& a, hipStream_t stream, const DecodePrologue* pro = nullptr) {
  GemmArgs g = a;
  g.tiles_n = decode_blocks(g);
  // Two tiles per workgroup where one each would put several rotations on a compute unit and that costs more than the
  // tiles' turns: with the norm always; without it, two and more tokens while two tiles each still are one round (9.2 ->
  // 8.5 us at 6144 channels; 11.8 -> 12.1 at 12288), and beyond three and a half rounds (one token 22016 channels 13.2 ->
  // 12.8, group scales 15.2 -> 14.1; 14336 10.2 either way).  One token without the norm rotates fast enough beside
  // another workgroup's (8192 7.5 / 7.7, 12288 8.8 / 9.9).
  const int n = g.tiles_n;
  const bool two = n > 256 && (pro || n > 896 || (g.M > 1 && n <= 512));
  return two ? launch_rotate_decode<EPI, 2>(x, g, stream, pro) : launch_rotate_decode<EPI, 1>(x, g, stream, pro);
}

}  // namespace

bool gemm_decode_supports(const GemmArgs& a, int epi, int group) {
  if (a.M <= 0 || a.M > kDecodeMaxM) return false;
  if (epi == kGroupScale) return group == 128 && a.M <= 16 && (a.K >> 7) <= kGroupMaxKT;
  return true;
}

int gemm_decode_dispatch(const GemmArgs& a, int epi, hipStream_t stream) {
  const int mt = (a.M + 15) / 16;
  if (epi == kGroupScale) return launch_decode<1, kGroupScale>(a, stream);
  if (epi == kInt32) {
    if (mt == 1) return launch_decode<1, kInt32>(a, stream);
    if (mt == 2) return launch_decode<2, kInt32>(a, stream);
    return launch_decode<4, kInt32>(a, stream);
  }
  if (mt == 1) return launch_decode<1, kRowScale>(a, stream);
  if (mt == 2) return launch_decode<2, kRowScale>(a, stream);
  return launch_decode<4, kRowScale>(a, stream);
}

}  // namespace flh

namespace {
int rotate_gemm_checked(const char* who, const flh_half* x, const flh::DecodePrologue* pro, int count,
                        const uint8_t* const* B, const flh_half* const* b_scale, flh_half* const* D, const size_t* N,
                        size_t M, size_t K, int b_cols, void* stream) {
  using namespace flh;
  if (count < 1 || count > kMaxGemmSegments)
    return fail(FLH_EINVAL, "%s: count = %d, must be 1 .. %d", who, count, kMaxGemmSegments);
  if (!B || !b_scale || !D || !N) return fail(FLH_EINVAL, "%s: null array", who);
  if (M == 0) return FLH_OK;
  if (!x) return fail(FLH_EINVAL, "%s: null pointer", who);
  if (misaligned16(x)) return fail(FLH_EINVAL, "%s: x must be 16-byte aligned", who);
  if (M > (size_t)kRotateGemmMaxTokens)
    return fail(FLH_EINVAL, "%s: M = %zu, at most %d tokens (more tokens quantise once, in their own launch)", who, M,
                kRotateGemmMaxTokens);
  if (K != 4096) return fail(FLH_EINVAL, "%s: K = %zu is not supported (4096)", who, K);
  if (b_cols != 1 && (size_t)b_cols != K / 128)
    return fail(FLH_EINVAL, "%s: weight scale columns (%d) must be 1 or K / 128 = %zu", who, b_cols, K / 128);
  size_t n_all = 0;
  for (int s = 0; s < count; ++s) {
    if (N[s] == 0) return fail(FLH_EINVAL, "%s: N[%d] = 0", who, s);
    if (!B[s] || !b_scale[s] || !D[s]) return fail(FLH_EINVAL, "%s: null pointer", who);
    if (misaligned16(B[s], D[s])) return fail(FLH_EINVAL, "%s: B and D must be 16-byte aligned", who);
    n_all += N[s];
  }
  if (n_all > (1u << 30)) return fail(FLH_EINVAL, "%s: N too large", who);
  GemmArgs g{nullptr, B[0], nullptr, (const __half*)b_scale[0], D[0], (int)M, (int)N[0], (int)K, 1, b_cols, 0, 0, 0};
  g.n_seg = count;
  for (int s = 1; s < count; ++s) {
    g.seg_B[s] = B[s];
    g.seg_Bs[s] = (const __half*)b_scale[s];
    g.seg_D[s] = D[s];
    g.seg_N[s] = (int)N[s];
  }
  return b_cols == 1 ? launch_rotate_decode<kRowScale>((const __half*)x, g, (hipStream_t)stream, pro)
                     : launch_rotate_decode<kGroupScale>((const __half*)x, g, (hipStream_t)stream, pro);
}
}  // namespace

extern "C" int flh_rotate_quant_gemm_i4_o16_multi(const flh_half* x, int count, const uint8_t* const* B,
                                                  const flh_half* const* b_scale, flh_half* const* D, const size_t* N,
                                                  size_t M, size_t K, int b_cols, void* stream) {
  return rotate_gemm_checked("rotate_quant_gemm", x, nullptr, count, B, b_scale, D, N, M, K, b_cols, stream);
}

extern "C" int flh_rmsnorm_rotate_quant_gemm_i4_o16_multi(const flh_half* x, const flh_half* add, flh_half* sum_out,
                                                          const flh_half* weight, float eps, int count,
                                                          const uint8_t* const* B, const flh_half* const* b_scale,
                                                          flh_half* const* D, const size_t* N, size_t M, size_t K,
                                                          int b_cols, void* stream) {
  using namespace flh;
  const char* who = "rmsnorm_rotate_quant_gemm";
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "%s: eps must not be negative", who);
  if ((add == nullptr) != (sum_out == nullptr)) return fail(FLH_EINVAL, "%s: add and sum_out come together or not at all", who);
  if (add && (misaligned16(add, sum_out))) return fail(FLH_EINVAL, "%s: add and sum_out must be 16-byte aligned", who);
  if (weight && misaligned16(weight)) return fail(FLH_EINVAL, "%s: weight must be 16-byte aligned", who);
  if (sum_out && ((const void*)sum_out == (const void*)x || (const void*)sum_out == (const void*)add))
    return fail(FLH_EINVAL, "%s: sum_out must not be x or add", who);
  const DecodePrologue pro{(const __half*)weight, eps, (const __half*)add, (__half*)sum_out};
  return rotate_gemm_checked(who, x, &pro, count, B, b_scale, D, N, M, K, b_cols, stream);
}

extern "C" int flh_rotate_quant_gemm_i4_o16(const flh_half* x, const uint8_t* B, const flh_half* b_scale, flh_half* D,
                                            size_t M, size_t N, size_t K, int b_cols, void* stream) {
  if (N == 0) return FLH_OK;
  return flh_rotate_quant_gemm_i4_o16_multi(x, 1, &B, &b_scale, &D, &N, M, K, b_cols, stream);
}
