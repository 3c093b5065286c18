// int4 x int4 GEMM + dequant for a handful of tokens (decode, M <= 64; up to sixteen mostly take the kernels at the end): the weights are
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
// time the chain waits for LDS at every pair).  What still comes here is long rows with group scales, widths that the kernels at the
// end are not filled by, and integer output.  us, weights from HBM, against scales as float tables and integer tiles (N x K), token scales /
// group scales: 16 tokens 4096 x 14336 14.8 / 15.1 -> 11.4 / 11.5, 4096 x 11008 12.4 / 12.7 -> 9.9 / 9.8; now also 5 tokens 5120 x 5120
// 7.6 / 7.6, 16 tokens 8.7 / 8.6.
#include <atomic>
#include "gemm_i4.h"
#include "lane_ops.h"

namespace flh {
namespace {

constexpr int kWaves = 8;
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
template <typename Args>
__device__ __forceinline__ void store_f16(const Args& p, const DecodeWeights& w, int gm, int gn, _Float16 v) {
  const size_t at = (size_t)gm * w.N + gn;
  if (p.R) v = v + ((const _Float16*)p.R)[at];
  ((_Float16*)w.D)[at] = v;
}

// Group scales wait in LDS as they are: row after row (the tokens if they have group scales, then the 16 channels) of KT
// halves, an odd number of dwords apart.  They come by direct-to-LDS loads that are requested behind the first weights and waited for last;
// rows that dword loads cannot fetch (an odd number of groups, an odd element offset, one scale per channel) are filled half by half.
__host__ __device__ constexpr int scale_pitch(int KT) { return ((KT + 1) >> 1) | 1; }   // dwords per row

template <typename Args>
__device__ __forceinline__ void request_scales(const Args& p, const DecodeWeights& w, unsigned* table, int KT, int tid) {
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

// out = fma(sum, scale, out) over the groups in ascending order: v[g * STRIDE] the sums, ra and rb the token's and the channel's
// scales, two to a dword (TOKEN: the channel's alone).  Eight pairs of groups are read ahead of their multiply-adds, by hand:
// a loop with inline assembly is not unrolled, and a pair at a time waits for LDS at every pair.
template <int STRIDE, bool TOKEN>
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
      lo[u] = v[2 * at * STRIDE], hi[u] = v[(2 * at + 1) * STRIDE];
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
    const float last = v[(KT - 1) * STRIDE];
    if constexpr (TOKEN) out = fma_half<0>(last, rb[pairs], out);
    else out = __builtin_fmaf(last, mul_halves<0>(ra[pairs], rb[pairs]), out);
  }
  return out;
}

// Partial sums in LDS -> outputs.  Lane l of a tile holds token l % 16 and channels 4 (l / 16) + i, i = 0..3; a thread
// finishes the value at its own place of the tile (reads without bank conflicts).
// Groups: float32 tiles of 256 x the sums, one fused multiply-add per group in ascending order, the exact 2^-8 at the end.
template <int MT, int EPI>
__device__ __forceinline__ void decode_finish(const GemmArgs& p, const DecodeWeights& w, const int* red, const unsigned* table,
                                              const __half* a_scales, const FirstScales& first, int tid) {
  const int KT = p.K >> 7;
  for (int idx = tid; idx < MT * 256; idx += kWaves * 64) {
    const int mt = idx >> 8, pos = idx & 255, m = (pos >> 2) & 15, n = (pos >> 6) * 4 + (pos & 3);
    const int gm = mt * 16 + m, gn = w.n0 + n;
    if (gm >= p.M || gn >= w.N) continue;
    if constexpr (EPI == kGroupScale) {
      const int pitch = scale_pitch(KT);
      const float* v = (const float*)red + mt * 256 + pos;
      float out;
      if (p.a_cols == 1) {                    // one scale per token: applied once, after the groups
        const float s_a = idx == tid ? first.a : __half2float(a_scales[gm]);
        out = fold_groups<MT * 256, true>(v, nullptr, table + n * pitch, KT);
        out = round_here(out * 0.00390625f) * s_a;
      } else {
        out = fold_groups<MT * 256, false>(v, table + m * pitch, table + (p.M + n) * pitch, KT);
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

// Up to sixteen tokens (gemm_lines_supports): the kernel above with its weights by direct-to-LDS loads of whole lines, past the caches, that
// every wave stages for itself: 2 KiB per double step, all of them requested at once; a wave waits for its own loads only.  A
// step's sums (two groups of 1 KiB) take the place of its operands, so that the LDS of the tiles is that of the stages.
// 16-byte piece c of row r sits at slot c ^ (r % 8): written lane after lane, and read without bank conflicts.
// us, weights from HBM, half lines to registers -> this, one scale per row / token scales / group scales: five tokens 4096 x 4096 4.7 /
// 5.1 / 5.1 -> 3.8 / 4.6 / 4.6, x 6144 6.1 / 6.6 / 6.4 -> 4.8 / 5.9 / 5.7; sixteen x 4096 5.1 / 5.4 / 5.4 -> 3.9 / 4.7 / 4.9, x 6144 7.1 /
// 7.4 / 7.4 -> 5.5 / 6.2 / 6.3, 14336 x 4096 10.0 -> 9.5 with one scale per row.  Beyond 8192 channels the tokens' half lines, as many as
// the weights' from sixteen tokens on, are what bounds it.
template <int STEPS, int EPI>
__global__ __launch_bounds__(kWaves * 64) void gemm_i4_lines_kernel(const GemmArgs p) {
  extern __shared__ __align__(16) int red[];   // [wave][step][2 KiB]: operands, then the sums of two groups; then the scales
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const DecodeWeights w = decode_weights(p, blockIdx.x);
  const int Kb = p.K >> 1, KT = p.K >> 7, ND = (KT + 1) >> 1;
  const int mine = (ND - wave + kWaves - 1) / kWaves;      // double steps of this wave, at most STEPS

  unsigned* table = (unsigned*)red + kWaves * STEPS * 512;
  if constexpr (EPI == kGroupScale) request_scales(p, w, table, KT, tid);
  const FirstScales first = first_scales<EPI>(p, w, p.As, tid);
  // (steps that the row does not have: the last one again, neither half of which is used)
  v4i a[STEPS][2];
  const uint8_t* arow = p.A + (size_t)min(r, p.M - 1) * Kb + c * 16;
  auto step_at = [&](int i) { return min(wave + i * kWaves, ND - 1) * 128; };
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int at = step_at(i);
    a[i][0] = *(const v4i*)(arow + at);
    a[i][1] = *(const v4i*)(arow + (at + 64 < Kb ? at + 64 : at));
  }
  __builtin_amdgcn_sched_barrier(0);
  const unsigned stage = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int*)red + wave * STEPS * 2048;
  const int line_row = lane >> 3, piece = ((lane & 7) ^ line_row) * 16;
  const uint8_t* rows[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) rows[q] = w.B + (size_t)min(w.n0 + q * 8 + line_row, w.N - 1) * Kb;
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int at = step_at(i), byte = at + (at + piece < Kb ? piece : piece - 64);   // K = 128 * odd: the last line is half a line
    const uint8_t* g[2] = {rows[0] + byte, rows[1] + byte - 1024};
    load_kib_to_lds16_nt(g, stage + i * 2048);
  }

  v4i acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  static_for<STEPS>([&](auto index) {
    constexpr int i = decltype(index)::value;
    wait_vmcnt<2 * (STEPS - 1 - i)>();
    asm volatile("" ::: "memory");
    if (i < mine) {
      int* area = red + (wave * STEPS + i) * 512;
      const bool second = 2 * (wave + i * kWaves) + 1 < KT;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v4i b = *(const v4i*)((const uint8_t*)area + r * 128 + ((h * 4 + c) ^ (r & 7)) * 16);
        v4i blo, bhi, alo, ahi;
        unpack_lo_hi(b, blo, bhi);
        if (h == 1 && !second) a[i][1] = v4i{0, 0, 0, 0};
        unpack_lo_hi(a[i][h], alo, ahi);
        const v4i zero = {0, 0, 0, 0};
        acc[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(blo, alo, EPI == kGroupScale ? zero : acc[h], 0, 0, 0);
        acc[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bhi, ahi, acc[h], 0, 0, 0);
      }
      if constexpr (EPI == kGroupScale) {
        *(v4f*)(area + lane * 4) = tile_as_float(acc[0]);
        *(v4f*)(area + 256 + lane * 4) = tile_as_float(acc[1]);
      }
    }
  });
  if constexpr (EPI != kGroupScale) *(v4i*)(red + wave * STEPS * 512 + lane * 4) = acc[0] + acc[1];
  __syncthreads();

  const int m = (tid >> 2) & 15, n = (tid >> 6) * 4 + (tid & 3), gn = w.n0 + n;
  if (tid >= 256 || m >= p.M || gn >= w.N) return;
  if constexpr (EPI == kGroupScale) {
    const float* v = (const float*)red + tid;
    const int pitch = scale_pitch(KT);
    const unsigned *ra = table + m * pitch, *rb = table + ((p.a_cols > 1 ? p.M : 0) + n) * pitch;
    float out = 0.f;
    // eight pairs of groups, a step of every wave, read ahead of their multiply-adds
    auto fold = [&](auto token) {
      constexpr bool TOKEN = decltype(token)::value;
      for (int i = 0; i * 2 * kWaves < KT; ++i) {
        float lo[kWaves], hi[kWaves];
        unsigned sa[kWaves], sb[kWaves];
#pragma unroll
        for (int u = 0; u < kWaves; ++u) {
          const int pair = min(i * kWaves + u, ND - 1);
          lo[u] = v[(u * STEPS + i) * 512], hi[u] = v[(u * STEPS + i) * 512 + 256];
          sa[u] = TOKEN ? 0u : ra[pair], sb[u] = rb[pair];
        }
        auto pair = [&](int u) {                 // (an even number of groups: gemm_lines_supports)
          if constexpr (TOKEN) {
            out = fma_half<0>(lo[u], sb[u], out);
            out = fma_half<1>(hi[u], sb[u], out);
          } else {
            out = __builtin_fmaf(lo[u], mul_halves<0>(sa[u], sb[u]), out);
            out = __builtin_fmaf(hi[u], mul_halves<1>(sa[u], sb[u]), out);
          }
        };
        if ((i + 1) * 2 * kWaves <= KT) {
#pragma unroll
          for (int u = 0; u < kWaves; ++u) pair(u);
        } else {
#pragma unroll
          for (int u = 0; u < kWaves; ++u)
            if (2 * (i * kWaves + u) < KT) pair(u);
        }
      }
    };
    if (p.a_cols == 1) {
      fold(std::true_type{});
      out = round_here(out * 0.00390625f) * first.a;
    } else {
      fold(std::false_type{});
      out *= 0.00390625f;
    }
    store_f16(p, w, m, gn, (_Float16)round_here(out));
  } else {
    int sum = 0;
#pragma unroll
    for (int u = 0; u < kWaves; ++u) sum += red[u * STEPS * 512 + tid];
    store_f16(p, w, m, gn, (_Float16)round_here((float)sum * (first.a * (first.b * 0.00390625f))));
  }
}

template <int STEPS, int EPI>
int launch_lines(const GemmArgs& a, hipStream_t stream) {
  const auto lds = [](int kt) { return (size_t)kWaves * STEPS * 2048 + (EPI == kGroupScale ? scale_table_dwords(kt) * 4 : 0); };
  auto kern = gemm_i4_lines_kernel<STEPS, EPI>;
  static_assert((size_t)kWaves * STEPS * 2048 + scale_table_dwords(2 * STEPS * kWaves) * 4 <= 160 * 1024, "LDS of a compute unit");
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)kern, lds(2 * STEPS * kWaves), grant, "gemm (lines)")) return rc;
  GemmArgs g = a;
  const int blocks = decode_blocks(g);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kWaves * 64), lds(a.K >> 7), stream, g);
  return check_launch("gemm_i4_lines");
}
template <int EPI>
int launch_lines(const GemmArgs& a, hipStream_t stream) {
  const int steps = (a.K + 256 * kWaves - 1) / (256 * kWaves);
  if (steps <= 2) return launch_lines<2, EPI>(a, stream);
  if constexpr (EPI == kRowScale) {
    if (steps > 4) return steps <= 6 ? launch_lines<6, EPI>(a, stream) : launch_lines<8, EPI>(a, stream);
  }
  return launch_lines<4, EPI>(a, stream);
}

// One to four tokens: products by v_dot8_i32_i4 on the packed codes as they are, which need no fragment layout, so that a load takes
// whole lines of eight weight rows, past the caches (gemm_i4_online.hip has the same, and what it is worth there).  A workgroup of
// eight waves owns 16 channels; a wave requests all its double steps at once, DOUBLES of them, through buffer descriptors:
// what lies beyond the matrix or the row reads as zero, without a branch.  Lane l holds piece l % 8 (32 codes) of the lines of rows l / 8
// and 8 + l / 8; four adjacent lanes make a group.  Up to K = 4096 64 registers, four workgroups per compute unit.
// What bounds it: first access (3 us), then HBM (6 TB/s between 12288 and 28672 channels).  us, weights from HBM, the kernels above and
// gemm_i4_stream.hip -> this one, one scale per row / token scales / group scales:
//   one token   4096 x 1024 3.9 / 4.6 / 4.7 -> 2.8 / 3.2 / 3.3, x 4096 4.6 / 5.1 / 5.2 -> 3.4 / 3.8 / 3.8, x 12288 7.8 / 8.4 / 8.2 -> 6.2 /
//               6.7 / 6.5, x 28672 14.0 / 15.4 / 15.0 -> 11.4 / 11.9 / 11.9;  14336 x 4096 8.8 / 10.5 / 11.0 -> 7.6 / 8.7 / 8.8
//   four        4096 x 4096 4.7 / 5.2 / 5.1 -> 3.9 / 4.6 / 4.4, x 28672 13.3 / 14.1 / 14.4 -> 13.1 / 13.3 / 13.1
struct DotSegment {
  const uint8_t* B;
  const __half* Bs;
  __half* D;
  int N, tile0;                                // its first block of 16 channels (unused ones: beyond every block)
};
struct DotArgs {                               // (small and read without a loop: the arguments come by one round of loads)
  const uint8_t* A;
  const __half *As, *R;
  int M, K, a_cols, b_cols;
  DotSegment seg[kMaxGemmSegments];
};

template <int MAXM, int DOUBLES, int EPI>
__global__ __launch_bounds__(kWaves * 64, DOUBLES == 2 ? 8 : 2) void gemm_i4_dot_kernel(const DotArgs p) {
  extern __shared__ __align__(16) int red[];   // [group | wave][token][16 channels], float32 | int32; then the scales
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int line_row = lane >> 3, piece = lane & 7;
  const int block = blockIdx.x;
  // all of the arguments by one round of scalar loads, not segment after segment
  asm volatile("" ::"s"(p.A), "s"(p.As), "s"(p.M), "s"(p.K), "s"(p.a_cols), "s"(p.b_cols), "s"(p.seg[1].tile0), "s"(p.seg[2].tile0), "s"(p.seg[3].tile0), "s"(p.seg[0].N), "s"(p.seg[1].N),
               "s"(p.seg[2].N), "s"(p.seg[3].N), "s"(p.seg[0].B), "s"(p.seg[1].B), "s"(p.seg[2].B), "s"(p.seg[3].B), "s"(p.seg[0].Bs),
               "s"(p.seg[1].Bs), "s"(p.seg[2].Bs), "s"(p.seg[3].Bs));
  DecodeWeights w{p.seg[0].B, p.seg[0].Bs, p.seg[0].D, p.seg[0].N, block * 16};
#pragma unroll
  for (int s = 1; s < kMaxGemmSegments; ++s)
    if (block >= p.seg[s].tile0) w = DecodeWeights{p.seg[s].B, p.seg[s].Bs, p.seg[s].D, p.seg[s].N, (block - p.seg[s].tile0) * 16};
  const int Kb = p.K >> 1, KT = p.K >> 7;
  const auto rows_b = __builtin_amdgcn_make_buffer_rsrc((void*)(w.B + (size_t)w.n0 * Kb), 0, min(16, w.N - w.n0) * Kb, 0x00020000);
  const auto rows_a = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, p.M * Kb, 0x00020000);
  constexpr unsigned kBeyond = 0x80000000u;

  unsigned* table = (unsigned*)(red + KT * MAXM * 16);
  if constexpr (EPI == kGroupScale) request_scales(p, w, table, KT, tid);   // (first: behind the operands it takes too many registers)
  v4i a[MAXM][DOUBLES], b[DOUBLES][2];
  unsigned at[DOUBLES];                        // byte of the row
#pragma unroll
  for (int i = 0; i < DOUBLES; ++i) {
    at[i] = (wave + i * kWaves) * 128 + piece * 16;
    if ((int)at[i] >= Kb) at[i] = kBeyond;
  }
#pragma unroll
  for (int i = 0; i < DOUBLES; ++i)
#pragma unroll
    for (int m = 0; m < MAXM; ++m) a[m][i] = __builtin_amdgcn_raw_buffer_load_b128(rows_a, at[i] + m * Kb, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < DOUBLES; ++i)
#pragma unroll
    for (int q = 0; q < 2; ++q) b[i][q] = __builtin_amdgcn_raw_buffer_load_b128(rows_b, at[i] + (q * 8 + line_row) * Kb, 0, 2 /* nt */);
  __builtin_amdgcn_sched_barrier(0);
  const int fm = lane >> 4, fn = lane & 15;    // what the lane of wave 0 finishes
  float s_a = 0.f, s_b = 0.f;
  if (EPI == kRowScale || p.a_cols == 1) s_a = __half2float(p.As[min(fm, p.M - 1)]);
  if constexpr (EPI == kRowScale) s_b = __half2float(w.Bs[min(w.n0 + fn, w.N - 1)]);

  auto dot = [](const v4i& x, const v4i& y, int sum) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_sdot8(x[e], y[e], sum, false);
    return sum;
  };
  const bool odd = lane & 1, high = lane & 2;
  const int n = (lane & 1) * 8 + line_row;     // the lane's channel of a reduced pair of rows
  if constexpr (EPI == kRowScale) {
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      int p0 = 0, p1 = 0;
#pragma unroll
      for (int i = 0; i < DOUBLES; ++i) p0 = dot(b[i][0], a[m][i], p0), p1 = dot(b[i][1], a[m][i], p1);
      int sum = (odd ? p1 : p0) + dpp_i<kDppQuadXor1>(odd ? p0 : p1);
      sum += dpp_i<kDppQuadXor2>(sum);
      sum += dpp_i<kDppRowHalfMirror>(dpp_i<kDppQuadXor1>(sum));   // (lane ^ 6: the other four of the row)
      if ((lane & 6) == 0) red[(wave * MAXM + m) * 16 + n] = sum;
    }
  } else {
    static_assert(DOUBLES % 2 == 0, "two double steps at a time");
#pragma unroll
    for (int i = 0; i < DOUBLES; i += 2)
#pragma unroll
      for (int m = 0; m < MAXM; ++m) {
        // four parts of four lanes: lane k of them gets part k, rows line_row and 8 + line_row of either double step
        const int p0 = dot(b[i][0], a[m][i], 0), p1 = dot(b[i][1], a[m][i], 0), p2 = dot(b[i + 1][0], a[m][i + 1], 0),
                  p3 = dot(b[i + 1][1], a[m][i + 1], 0);
        const int x = (odd ? p1 : p0) + dpp_i<kDppQuadXor1>(odd ? p0 : p1), y = (odd ? p3 : p2) + dpp_i<kDppQuadXor1>(odd ? p2 : p3);
        const int sum = (high ? y : x) + dpp_i<kDppQuadXor2>(high ? x : y);
        const int g = 2 * (wave + (i + (high ? 1 : 0)) * kWaves) + (piece >> 2);
        if (g < KT) ((float*)red)[(g * MAXM + m) * 16 + n] = (float)sum;
      }
    wait_vmcnt<0>();                           // the scales
  }
  __syncthreads();

  const int gn = w.n0 + fn;
  if (wave > 0 || fm >= p.M || gn >= w.N) return;
  if constexpr (EPI == kRowScale) {
    int sum = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) sum += red[(v * MAXM + fm) * 16 + fn];
    store_f16(p, w, fm, gn, (_Float16)round_here((float)sum * (s_a * s_b)));
  } else {
    const float* v = (const float*)red + fm * 16 + fn;
    const int pitch = scale_pitch(KT);
    float out;
    if (p.a_cols == 1) out = round_here(fold_groups<MAXM * 16, true>(v, nullptr, table + fn * pitch, KT)) * s_a;
    else out = fold_groups<MAXM * 16, false>(v, table + fm * pitch, table + (p.M + fn) * pitch, KT);
    store_f16(p, w, fm, gn, (_Float16)round_here(out));
  }
}

template <int MAXM, int DOUBLES, int EPI>
int launch_dot(const GemmArgs& a, hipStream_t stream) {
  const int KT = a.K >> 7;
  const size_t smem = EPI == kGroupScale ? (size_t)KT * MAXM * 64 + scale_table_dwords(KT) * 4 : (size_t)kWaves * MAXM * 64;
  static_assert(EPI != kGroupScale || (2 * DOUBLES * kWaves) * MAXM * 64 + scale_table_dwords(2 * DOUBLES * kWaves) * 4 <= 64 * 1024,
                "fits the default dynamic LDS limit");
  DotArgs d{a.A, a.As, a.R, a.M, a.K, a.a_cols, a.b_cols, {}};
  int blocks = 0;
  for (int s = 0; s < kMaxGemmSegments; ++s) {
    d.seg[s].tile0 = 0x7FFFFFFF;
    if (s > 0 && s >= a.n_seg) continue;
    d.seg[s] = s == 0 ? DotSegment{a.B, a.Bs, (__half*)a.D, a.N, 0}
                      : DotSegment{a.seg_B[s], a.seg_Bs[s], (__half*)a.seg_D[s], a.seg_N[s], blocks};
    blocks += (d.seg[s].N + 15) / 16;
  }
  hipLaunchKernelGGL((gemm_i4_dot_kernel<MAXM, DOUBLES, EPI>), dim3(blocks), dim3(kWaves * 64), smem, stream, d);
  return check_launch("gemm_i4_dot");
}
template <int MAXM, int EPI>
int launch_dot(const GemmArgs& a, hipStream_t stream) {
  const int steps = (a.K + 256 * kWaves - 1) / (256 * kWaves);   // double steps of a wave
  if (steps <= 2) return launch_dot<MAXM, 2, EPI>(a, stream);
  if constexpr (MAXM <= 2) {                                     // (gemm_dot_supports: more tokens up to K = 8192)
    if (steps > 4) return steps <= 6 ? launch_dot<MAXM, 6, EPI>(a, stream) : launch_dot<MAXM, 8, EPI>(a, stream);
  }
  return launch_dot<MAXM, 4, EPI>(a, stream);
}
template <int EPI>
int launch_dot(const GemmArgs& a, hipStream_t stream) {
  return a.M == 1 ? launch_dot<1, EPI>(a, stream) : a.M == 2 ? launch_dot<2, EPI>(a, stream) : launch_dot<4, EPI>(a, stream);
}

}  // namespace

namespace {
// Double steps of K that the waves of the two kernels above have room for and the row does not have: a wave's share is two, four, six or
// eight.  They are multiplied, or another step is loaded again in their place, all the same.  What that costs sets the lines below.
int idle_steps(const GemmArgs& a) {
  const int filled = (a.K + 255) / 256, share = (filled + kWaves - 1) / kWaves;
  return (share + (share & 1)) * kWaves - filled;
}
long all_columns(const GemmArgs& a) {
  long columns = a.N;
  for (int s = 1; s < a.n_seg; ++s) columns += a.seg_N[s];
  return columns;
}
}  // namespace

// Up to four tokens (us, weights from HBM, one scale per row / token scales / group scales; this kernel against what takes the launch
// else: the kernels above, beyond 12288 channels gemm_i4_stream.hip).
//  * One token from K = 1280 on: 1280 x 18432 5.3 / 5.7 / 5.6 against 6.3 / 7.0 / 6.1, 768 x 13824 4.5 / 4.8 / 4.8 against 4.3 / 4.3 / 4.4.
//  * Two from 1792 on.  On many channels not where the codes of eight double steps take the registers of the weights in flight
//    (15360 x 13824 25.0 / 29.2 / 27.0 against 22.9 / 24.8 / 24.0), nor with eleven idle steps or more on less than a workgroup of the other
//    kernel per compute unit (4608 x 13824 9.7 / 9.9 / 9.8 against 9.3 / 9.5 / 9.6, 5376 x 18432 11.7 / 12.3 / 12.3 against 14.3 / 14.7 /
//    15.3).  It does not take an odd number of groups (group scales, 12416 x 16384 29.4 against 36.2 on half lines).
//  * Three and four up to K = 8192, for the codes' registers again (four tokens 11008 x 4096 7.8 / 9.3 / 9.1 against 7.2 / 8.8 / 8.8), with few
//    idle steps (four tokens 2048 x 8192 4.9 / 5.2 / 5.2 against 4.4 / 4.7 / 4.6, 5120 x 5120 6.9 / 8.0 / 7.9 against 6.9 / 7.5 / 7.5, 6656 x
//    5120 7.4 / 8.6 / 8.5 against 8.0 / 9.0 / 9.1).  Many channels with one scale per row go to the other kernels (4096 x 28672 13.1, whole
//    lines 12.5); group scales with as few idle steps, from a full round of the other kernel on (token / group scales 3456 x
//    28672 13.6 / 14.1 against 15.2 / 15.5, 7168 x 13824 15.1 / 14.7 against 13.0 / 13.1), token scales of long rows without (7936 x
//    16384 17.3 against 15.4).
bool gemm_dot_supports(const GemmArgs& a, int epi, int group) {
  if (a.M <= 0 || a.M > 4 || a.K > 16384 || !(epi == kRowScale || (epi == kGroupScale && group == 128))) return false;
  const int idle = idle_steps(a);
  const long columns = all_columns(a);
  const bool row = epi == kRowScale, two = a.K <= 4096;   // two: the share of a wave
  if (a.M == 1) return a.K >= 1280;
  if (a.M == 2)
    return a.K >= 1792 && (columns <= 12288 || (a.K <= 12288 && (idle <= 10 || columns >= 16384)) || (!row && a.K % 256));
  if (a.K > 8192 || idle > (two ? 4 : 6)) return false;
  if (columns <= 12288) return true;
  if (row) return false;
  return (idle == 0 && two) || (columns >= 16384 && idle <= 4 && (two || idle == 0 || a.a_cols > 1));
}

int gemm_dot_dispatch(const GemmArgs& a, int epi, hipStream_t stream) {
  return epi == kRowScale ? launch_dot<kRowScale>(a, stream) : launch_dot<kGroupScale>(a, stream);
}

// Whole lines through LDS instead of half lines to registers (us, five tokens unless stated, this against that).
//  * One scale per row: from K = 2048 on (2048 x 5120 4.2 against 4.3, 1536 x 5120 4.3 against 3.9).  Every other row of an odd number of
//    half lines starts inside a line: on many channels only (16 tokens 3200 x 4096 4.3 against 4.1; 3200 x 11008 6.5 against 7.2), and
//    not beyond K = 4096.  There up to eleven idle steps (5376 x 8192 7.2 against 7.6, 4608 x 5120 6.4 against 6.2).  Shares of six and
//    eight steps leave a compute unit one workgroup: few channels (9728 x 3072 6.2 against 6.6, x 10240 16.0 against 15.3; 12800 x
//    3072 7.3 against 7.6, x 8192 15.0 against 13.9; three tokens 14336 x 12288 22.0 against 21.0).
//  * Group scales wait for their table: an even number of groups, which dword loads fetch (16 tokens 3456 x 3072 5.7 against
//    5.0), few idle steps (3584 x 5120 5.7 against 6.0; token scales 3072 x 5120 5.9 against 5.5), with a share of four on enough channels
//    (8192 x 3072 6.8 against 7.1, x 2048 6.5 against 6.3; 6656 x 5120 8.7 against 9.0, 6400 x 3072 6.6 against 5.7), and no longer rows
//    (11008 x 4096 9.2 against 8.7).
bool gemm_lines_supports(const GemmArgs& a, int epi) {
  if (a.M > 16 || a.K > 16384) return false;
  const int idle = idle_steps(a);
  const long columns = all_columns(a);
  const bool even = a.K % 256 == 0;
  if (epi == kRowScale) {
    if (a.K <= 4096) return a.K >= 2048 && (even || columns >= 8192);
    if (!even || a.K <= 8192) return even && idle <= 11;
    return columns <= 4096 ? idle <= 14 : columns <= 10240 && idle <= (a.K > 12288 ? 12 : 8);
  }
  if (epi != kGroupScale || !even || a.K > 8192) return false;
  if (a.K <= 4096) return idle <= 3;
  return idle <= 1 ? a.a_cols == 1 || columns >= 3072 : idle <= 7 && columns >= 5120;
}

// Where whole lines have lines of their own against gemm_i4_stream.hip (takes_few_tokens there; elsewhere those of half lines hold): full
// shares, group scales of two steps only and token scales of four from a full round of that kernel on (token scales 8192 x 13824 16.0
// against 14.6, 8 tokens x 18432 20.5 against 23.4).  One scale per row also up to three idle steps of two (3840 x 13824 7.5 against
// 8.0, 3712 x 22016 11.2 against 12.7), some more where that kernel's only round is far from full or its last one short (7424 x 11008 10.9
// against 12.5, 7936 x 18432 17.0 against 19.8; 7168 x 13824 12.9 against 12.5, 8 tokens 6400 x 28672 23.4 against 20.6, 2048 x 11008
// 5.9 against 5.3).
bool gemm_lines_over_stream(const GemmArgs& a, int epi) {
  const int idle = idle_steps(a);
  const long columns = all_columns(a);
  if (!gemm_lines_supports(a, epi) || columns > 32768 || a.K > 8192) return false;
  const bool two = a.K <= 4096;
  if (epi != kRowScale) return idle == 0 && (two || (a.a_cols == 1 && columns >= 16384));
  return idle <= (two ? 3 : 0) || (idle <= (two ? 5 : 7) && (columns <= 12288 || (columns >= 16384 && columns <= 24576)));
}

bool gemm_decode_supports(const GemmArgs& a, int epi, int group) {
  if (a.M <= 0 || a.M > kDecodeMaxM) return false;
  if (epi == kGroupScale) return group == 128 && a.M <= 16 && (a.K >> 7) <= kGroupMaxKT;
  return true;
}

int gemm_decode_dispatch(const GemmArgs& a, int epi, hipStream_t stream) {
  const int mt = (a.M + 15) / 16;
  if (gemm_lines_supports(a, epi))
    return epi == kGroupScale ? launch_lines<kGroupScale>(a, stream) : launch_lines<kRowScale>(a, stream);
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
