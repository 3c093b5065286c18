// int4 x int4 GEMM that quantises its own activations: one to four tokens of K = 4096, so few that
// repeating the quantiser in every workgroup costs less than a launch of its own in front of the GEMM.
//
// A workgroup of eight waves owns T tiles of 16 channels, as many as put one workgroup on a compute unit, and every token.  A
// wave takes every eighth double step of K (256 codes = a 128-byte line of a weight row, gemm_i4_decode.hip) of all its tiles.
// Prologues, all with the arithmetic of the stand-alone quantisers, hence the same codes and scales:
//   rotate            the whole row rotated, one scale per token (rotate_quant_row_8waves)
//   norm + rotate     RMSNorm in front, with or without a residual addition in front of that (workgroup 0 stores the sum)
//   norm + groups     RMSNorm, then one scale per 128 channels, no rotation (rmsnorm_group_kernel)
// The sums, their folds and the epilogue are those of the other kernels: the same bits as quantiser and GEMM in two launches.
//
// What bounds it: first access, then the weight stream (one token 28672 x 4096 15.6 us, 58.7 MB).  The order of the requests is what
// hides the quantiser: loads come back in the order they were made, so the token's are made first, then those of all the workgroup's
// weights, and no barrier in between waits for more than LDS.  All sums of a workgroup's tokens (not of the sixteen that a tile
// of the matrix instruction has room for) fit LDS, so that one barrier separates the products of all tiles from their folds.
// The products are v_dot8_i32_i4 on the packed codes as they are: nothing to unpack, no idle columns, and no
// fragment layout, so that a load takes whole lines of eight weight rows, past the caches.  One token, token scales, us, weights from
// HBM: with the requests in the old order, 16 x 16 x 64 products and half lines -> these requests -> dot products -> whole lines
// past the caches (quantiser and GEMM in two launches):
//   rotation, 4096 x 4096 6.2 -> 5.3 -> 4.6 -> 3.7 (8.1);  norm and residual, 6144 x 4096 9.9 -> 7.6 -> 6.8 -> 6.2 (10.7);
//   the same, 28672 x 4096 26.3 -> 19.7 -> 17.6 -> 15.6 (18.7), 15.0 with tiles a round of workgroups apart instead of side by side
// Norm and groups, two launches -> one: 6144 x 4096 one token 9.7 -> 5.0, four 9.9 -> 7.2; 22016 x 4096 16.0 -> 11.5, 16.6 -> 14.6.
#include "gemm_i4.h"
#include "group_codes.h"
#include "rotate_row.h"

namespace flh {
namespace {

constexpr int kWaves = 8;
// The rotations are written for rows of 4096; norm and groups would do at any multiple of 2048 and is measured at this one only.
constexpr int kK = 4096, kRowB = kK / 2, kGroups = kK / 128;
constexpr int kDoubles = kGroups / 2 / kWaves;     // double steps per wave
constexpr int kCodePitch = kRowB + 16;             // code rows 16 bytes apart in the banks
constexpr int kMaxTokens = 4;

enum Prologue { kRotate = 0, kNormRotate = 1, kAddNormRotate = 2, kNormGroup = 3 };

struct OnlineSegment {
  const uint8_t* B;
  const __half* Bs;
  __half* D;
  int N, tile0;                                    // its first tile of 16 channels in the launch
};
struct OnlineArgs {
  const __half *x, *add, *weight;                  // add: kAddNormRotate; weight: of the norm, or null
  __half* sum_out;
  float eps;
  int M, tiles;                                    // tiles: of the launch
  OnlineSegment seg[kMaxGemmSegments];             // (unused ones: tile0 beyond every tile)
};

struct OnlineTile {
  const uint8_t* B;
  const __half* Bs;
  __half* D;
  int N, n0;
};


// dynamic LDS of M tokens: codes, their scales, the tiles' channel scales, then the quantiser's scratch or the sums
template <int EPI, int PRO, int T>
__host__ __device__ constexpr int lds_codes(int M) { return M * kCodePitch; }
template <int EPI, int PRO, int T>
__host__ __device__ constexpr int lds_tables(int M) { return (PRO == kNormGroup ? M * kGroups * 2 : 16) + (EPI == kRowScale ? 0 : T * 16 * kGroups * 2); }
template <int EPI, int PRO, int T>
__host__ __device__ constexpr int lds_bytes(int M) {
  const int sums = T * (EPI == kRowScale ? kWaves : kGroups) * (M == 3 ? 4 : M) * 64;
  const int scratch = PRO == kNormGroup ? 256 : (int)(M > 1 ? sizeof(RowScratch<2>) : sizeof(RowScratch<1>));
  return lds_codes<EPI, PRO, T>(M) + lds_tables<EPI, PRO, T>(M) + (sums > scratch ? sums : scratch);
}

// MAXM: tokens that the kernel takes, 1, 2 or 4.  A tile of a wave takes 16 dot products and nine instructions across lanes per
// token, and one four-byte LDS write without idle lanes, where the matrix instruction takes 96 instructions of unpacking and, per
// group, a 16-byte write of which a token fills a sixteenth.
template <int EPI, int PRO, int T, int MAXM>
__global__ __launch_bounds__(kWaves * 64) void gemm_i4_online_kernel(const OnlineArgs p) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;          // what the lane finishes: channel r, token c
  const int line_row = lane >> 3, line_piece = lane & 7;   // what it loads: whole lines of eight weight rows
  const int M = MAXM <= 2 ? MAXM : p.M;
  uint8_t* codes = lds;
  __half* tok = (__half*)(lds + lds_codes<EPI, PRO, T>(M));
  uint8_t* table = (uint8_t*)tok + (PRO == kNormGroup ? M * kGroups * 2 : 16);
  uint8_t* sums = lds + lds_codes<EPI, PRO, T>(M) + lds_tables<EPI, PRO, T>(M);

  // tile t of the workgroup: its weights
  auto tile = [&](int t) {
    const int block = min((int)(blockIdx.x + t * gridDim.x), p.tiles - 1);
    OnlineTile w{p.seg[0].B, p.seg[0].Bs, p.seg[0].D, p.seg[0].N, block * 16};
#pragma unroll
    for (int s = 1; s < kMaxGemmSegments; ++s)
      if (block >= p.seg[s].tile0) w = OnlineTile{p.seg[s].B, p.seg[s].Bs, p.seg[s].D, p.seg[s].N, (block - p.seg[s].tile0) * 16};
    return w;
  };

  // 1. the tokens (no branches around loads: what merges behind one is waited for there)
  constexpr int HALF = kWaves / 2;                 // kNormGroup: four waves per row, as the stand-alone kernel
  constexpr int ROWS = PRO == kNormGroup ? (MAXM + 1) / 2 : MAXM;
  v4i xr[ROWS][PRO == kNormGroup ? 2 : 1], ar[PRO == kAddNormRotate ? ROWS : 1], wr[PRO == kNormGroup ? 2 : 1];
  const int half = wave / HALF, t256 = tid & 255;
  const int chunk0 = (t256 & ~15) + group_chunk<16>(t256 & 15);   // kNormGroup: this thread's chunks of 8 are chunk0, chunk0 + 256
  const __half* const norm_weight = p.weight ? p.weight : p.x;
  if constexpr (PRO == kNormGroup) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const __half* row = p.x + (size_t)min(2 * i + half, M - 1) * kK + chunk0 * 8;
      xr[i][0] = *(const v4i*)row, xr[i][1] = *(const v4i*)(row + 2048);
    }
    wr[0] = *(const v4i*)(norm_weight + chunk0 * 8), wr[1] = *(const v4i*)(norm_weight + chunk0 * 8 + 2048);
  } else {
    wr[0] = ar[0] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      xr[i][0] = row_piece(p.x + (size_t)min(i, M - 1) * kK, wave);
      if constexpr (PRO == kAddNormRotate) ar[i] = row_piece(p.add + (size_t)min(i, M - 1) * kK, wave);
    }
    if constexpr (PRO != kRotate) wr[0] = row_piece(norm_weight, wave);
  }
  __builtin_amdgcn_sched_barrier(0);

  // 2. the channels' scales: group scales into LDS as they are, a tile's 16 rows of 64 bytes by one load of one wave (the 16-byte
  // pieces of row n in the order q ^ (n / 4): the fold reads them without bank conflicts); one per row: the lane's own
  float s_row = 0.f;
  if constexpr (EPI == kRowScale) {
    const OnlineTile w = tile(wave < T ? wave : 0);
    s_row = __half2float(w.Bs[min(w.n0 + r, w.N - 1)]);
  } else {
    static_assert(kWaves * 64 == 16 * kGroups && kGroups == 32, "a load instruction, or a half per thread");
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const OnlineTile w = tile(t);
      uint8_t* dst = table + t * 1024;
      if (((uintptr_t)w.Bs & 15) == 0) {
        if (wave == t)
          load_to_lds16(w.Bs + (size_t)min(w.n0 + (lane >> 2), w.N - 1) * kGroups + ((lane ^ (lane >> 4)) & 3) * 8,
                        (unsigned)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)dst);
      } else {
        const int n = tid >> 5, g = tid & 31;
        ((__half*)dst)[n * kGroups + (((g >> 3) ^ (n >> 2)) & 3) * 8 + (g & 7)] = w.Bs[(size_t)min(w.n0 + n, w.N - 1) * kGroups + g];
      }
    }
  }

  // 3. this wave's weights of all tiles, in the order of their use
  v4i b[T][kDoubles][2];
  static_for<T * kDoubles>([&](auto index) {
    constexpr int t = decltype(index)::value / kDoubles, i = decltype(index)::value % kDoubles;
    const OnlineTile w = tile(t);
    const uint8_t* base = w.B + (size_t)w.n0 * kRowB + i * (kWaves * 128);
    const int last = w.N - 1 - w.n0;
    b[t][i][0] = __builtin_nontemporal_load((const v4i*)(base + (unsigned)(min(line_row, last) * kRowB + wave * 128 + line_piece * 16)));
    b[t][i][1] = __builtin_nontemporal_load((const v4i*)(base + (unsigned)(min(8 + line_row, last) * kRowB + wave * 128 + line_piece * 16)));
  });
  __builtin_amdgcn_sched_barrier(0);

  // 4. the quantiser
  if constexpr (PRO == kNormGroup) {
    float* part = (float*)sums;                    // [token][wave of the half]
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
      if (2 * i + half < M) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const h2 v = __builtin_bit_cast(h2, (unsigned)xr[i][u][e]);
            ss = __builtin_fmaf((float)v[0], (float)v[0], ss);
            ss = __builtin_fmaf((float)v[1], (float)v[1], ss);
          }
        ss = wave_sum(ss);
        if (lane == 0) part[(2 * i + half) * HALF + wave % HALF] = ss;
      }
    barrier_after_lds();
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
      if (2 * i + half < M) {
        const int row = 2 * i + half;
        const v4f ps = *(const v4f*)(part + row * HALF);
        const float inv = 1.0f / __builtin_sqrtf(((ps[0] + ps[1]) + (ps[2] + ps[3])) / (float)kK + p.eps);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          h2 v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const h2 x = __builtin_bit_cast(h2, (unsigned)xr[i][u][e]);
            float a = round_here((float)x[0] * inv), d = round_here((float)x[1] * inv);
            if (p.weight) {
              const h2 g = __builtin_bit_cast(h2, (unsigned)wr[u][e]);
              a = round_here(a * (float)g[0]), d = round_here(d * (float)g[1]);
            }
            v[e] = h2{(_Float16)a, (_Float16)d};
          }
          const GroupScale s = group_scale<16>(lane_abs_max(v));
          const h2 hb = {(_Float16)65504.0f, (_Float16)65504.0f};
          unsigned y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = __builtin_bit_cast(unsigned, v[e]);
          const int chunk = chunk0 + 256 * u;
          *(unsigned*)(codes + row * kCodePitch + chunk * 4) =
              s.careful ? nibbles8<true>(y[0], y[1], y[2], y[3], s.r, hb) : nibbles8<false>(y[0], y[1], y[2], y[3], s.r, hb);
          if ((chunk & 15) == 0) tok[row * kGroups + (chunk >> 4)] = __builtin_bit_cast(__half, s.s);
        }
      }
  } else {
    constexpr int R = ROWS > 1 ? 2 : 1;             // rows at a time
    RowScratch<R>& scratch = *(RowScratch<R>*)sums;
#pragma unroll
    for (int i = 0; i < ROWS; i += R)
      if (i < M) {
        RowPiece in[R];
#pragma unroll
        for (int u = 0; u < R; ++u) in[u] = RowPiece{xr[i + u][0], ar[PRO == kAddNormRotate ? i + u : 0], wr[0]};
        rotate_quant_rows_8waves<PRO != kRotate, PRO == kAddNormRotate>(
            in, scratch, codes + i * kCodePitch, kCodePitch, tok + i, 1.0f / 64.0f, wave, p.weight != nullptr, p.eps,
            PRO == kAddNormRotate && blockIdx.x == 0 ? p.sum_out + (size_t)i * kK : nullptr, M - i);
      }
  }
  barrier_after_lds();

  // 5. products.  Sums: [tile][group | wave][token][16 channels]
  v4i a[MAXM][kDoubles];
#pragma unroll
  for (int m = 0; m < MAXM; ++m)
#pragma unroll
    for (int i = 0; i < kDoubles; ++i) a[m][i] = *(const v4i*)(codes + min(m, M - 1) * kCodePitch + (wave + i * kWaves) * 128 + line_piece * 16);
  auto dot = [](v4i x, v4i y, int sum) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_sdot8(x[e], y[e], sum, false);
    return sum;
  };
  // lane k of four adjacent ones: part k, summed over the four
  auto gather = [&](int p0, int p1, int p2, int p3) {
    const bool odd = lane & 1, high = lane & 2;
    const int x = (odd ? p1 : p0) + dpp_i<kDppQuadXor1>(odd ? p0 : p1), y = (odd ? p3 : p2) + dpp_i<kDppQuadXor1>(odd ? p2 : p3);
    return (high ? y : x) + dpp_i<kDppQuadXor2>(high ? x : y);
  };
  const int n = (lane & 1) * 8 + line_row, half_line = line_piece >> 2;
  static_for<T>([&](auto t_tag) {
    constexpr int t = decltype(t_tag)::value;
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      // parts: rows line_row and 8 + line_row of either double step
      if constexpr (EPI == kRowScale) {
        const int p0 = dot(b[t][1][0], a[m][1], dot(b[t][0][0], a[m][0], 0)), p1 = dot(b[t][1][1], a[m][1], dot(b[t][0][1], a[m][0], 0));
        const bool odd = lane & 1;
        int sum = (odd ? p1 : p0) + dpp_i<kDppQuadXor1>(odd ? p0 : p1);
        sum += dpp_i<kDppQuadXor2>(sum);
        sum += dpp_i<kDppRowHalfMirror>(dpp_i<kDppQuadXor1>(sum));   // (lane ^ 6: the other four)
        if ((lane & 6) == 0) ((int*)sums)[((t * kWaves + wave) * MAXM + m) * 16 + n] = sum;
      } else {
        const int sum = gather(dot(b[t][0][0], a[m][0], 0), dot(b[t][0][1], a[m][0], 0), dot(b[t][1][0], a[m][1], 0),
                               dot(b[t][1][1], a[m][1], 0));
        const int g = 2 * (wave + ((lane >> 1) & 1) * kWaves) + half_line;
        ((float*)sums)[((t * kGroups + g) * MAXM + m) * 16 + n] = (float)sum;
      }
    }
  });
  if constexpr (EPI != kRowScale) wait_vmcnt<0>();   // the channels' scales
  barrier_after_lds();

  // 6. folds: a wave finishes a tile, a lane token lane / 16, channel lane % 16
  if (wave < T) {
    const int t = wave, m = c;
    auto value = [&] {                             // before the rounding to fp16
      if constexpr (EPI == kRowScale) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) sum += ((const int*)sums)[((t * kWaves + w) * MAXM + m) * 16 + r];
        return (float)sum * (__half2float(tok[m]) * s_row);
      } else {
        const float* v = (const float*)sums + (t * kGroups * MAXM + m) * 16 + r;
        const uint8_t* sb = table + t * 1024 + r * 64;
        float out = 0.f;
#pragma unroll
        for (int q = 0; q < kGroups / 8; ++q) {
          const v4i bq = *(const v4i*)(sb + ((q ^ (r >> 2)) & 3) * 16);
          const v4i aq = PRO == kNormGroup ? *(const v4i*)(tok + m * kGroups + q * 8) : v4i{0, 0, 0, 0};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v0 = v[(q * 8 + 2 * e) * MAXM * 16], v1 = v[(q * 8 + 2 * e + 1) * MAXM * 16];
            if constexpr (PRO == kNormGroup) {
              out = __builtin_fmaf(v0, mul_halves<0>((unsigned)aq[e], (unsigned)bq[e]), out);
              out = __builtin_fmaf(v1, mul_halves<1>((unsigned)aq[e], (unsigned)bq[e]), out);
            } else {
              out = fma_half<0>(v0, (unsigned)bq[e], out);
              out = fma_half<1>(v1, (unsigned)bq[e], out);
            }
          }
        }
        return PRO == kNormGroup ? out : round_here(out) * __half2float(tok[m]);
      }
    };
    if (m < M && (int)(blockIdx.x + t * gridDim.x) < p.tiles) {
      const OnlineTile w = tile(t);
      const int n = w.n0 + r;
      if (n < w.N) ((_Float16*)w.D)[(size_t)m * w.N + n] = (_Float16)round_here(value());
    }
  }
}

template <int EPI, int PRO, int T, int MAXM>
int launch_kernel(const OnlineArgs& a, hipStream_t stream) {
  auto kern = gemm_i4_online_kernel<EPI, PRO, T, MAXM>;
  constexpr size_t most = lds_bytes<EPI, PRO, T>(MAXM);
  static_assert(T <= kWaves && most <= 160 * 1024, "LDS of a compute unit");
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)kern, most, grant, "gemm (online)")) return rc;
  const size_t bytes = lds_bytes<EPI, PRO, T>(a.M);
  hipLaunchKernelGGL(kern, dim3((a.tiles + T - 1) / T), dim3(kWaves * 64), bytes, stream, a);
  return check_launch("gemm_i4_online");
}

// As many tiles per workgroup as leave one workgroup to a compute unit; beyond eight, as many as leave every compute unit the same number
// (us, rotation, one scale per row, eight tiles always / so: one token x 33000 19.2 / 14.1, x 40960 21.0 / 15.8, two 24.6 / 20.1; norm and
// groups, one token x 36864 22.1 / 15.9).  The package's own rules stop at eight tiles and earlier with more tokens (torch_ext.cpp has
// them); the entry points take every width.
template <int EPI, int PRO, int MAXM>
int launch_by_tiles(const OnlineArgs& a, hipStream_t stream) {
  const int all = (a.tiles + 255) / 256, rounds = (all + 7) / 8, per = (all + rounds - 1) / rounds;
  if (per <= 1) return launch_kernel<EPI, PRO, 1, MAXM>(a, stream);
  if (per == 2) return launch_kernel<EPI, PRO, 2, MAXM>(a, stream);
  if constexpr (MAXM <= 2 || PRO == kNormGroup) {      // (more tokens to rotate than two: the callers' rules stop earlier)
    if (per == 3) return launch_kernel<EPI, PRO, 3, MAXM>(a, stream);
    if (per == 5) return launch_kernel<EPI, PRO, 5, MAXM>(a, stream);
    if (per == 6) return launch_kernel<EPI, PRO, 6, MAXM>(a, stream);
    if (per == 7) return launch_kernel<EPI, PRO, 7, MAXM>(a, stream);
  }
  return per <= 4 ? launch_kernel<EPI, PRO, 4, MAXM>(a, stream) : launch_kernel<EPI, PRO, 8, MAXM>(a, stream);
}
template <int EPI, int PRO>
int launch(const OnlineArgs& a, hipStream_t stream) {
  if (a.M == 1) return launch_by_tiles<EPI, PRO, 1>(a, stream);
  return a.M == 2 ? launch_by_tiles<EPI, PRO, 2>(a, stream) : launch_by_tiles<EPI, PRO, kMaxTokens>(a, stream);
}

struct OnlineCall {
  const flh_half *x, *add, *weight;
  flh_half* sum_out;
  float eps;
  bool norm, groups;
};

int online_checked(const char* who, const OnlineCall& call, int count, const uint8_t* const* B, const flh_half* const* b_scale,
                   flh_half* const* D, const size_t* N, size_t M, size_t K, int b_cols, void* stream) {
  if (count < 1 || count > kMaxGemmSegments)
    return fail(FLH_EINVAL, "%s: count = %d, must be 1 .. %d", who, count, kMaxGemmSegments);
  if (!B || !b_scale || !D || !N) return fail(FLH_EINVAL, "%s: null array", who);
  if (M == 0) return FLH_OK;
  if (!call.x) return fail(FLH_EINVAL, "%s: null pointer", who);
  if (misaligned16(call.x)) return fail(FLH_EINVAL, "%s: x must be 16-byte aligned", who);
  if (M > (size_t)kMaxTokens)
    return fail(FLH_EINVAL, "%s: M = %zu, at most %d tokens (more tokens quantise once, in their own launch)", who, M, kMaxTokens);
  if (K != kK) return fail(FLH_EINVAL, "%s: K = %zu is not supported (4096)", who, K);
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
  OnlineArgs a{(const __half*)call.x, (const __half*)call.add, (const __half*)call.weight, (__half*)call.sum_out, call.eps, (int)M, 0, {}};
  for (int s = 0; s < kMaxGemmSegments; ++s) {
    a.seg[s].tile0 = 0x7FFFFFFF;
    if (s >= count) continue;
    a.seg[s] = OnlineSegment{B[s], (const __half*)b_scale[s], (__half*)D[s], (int)N[s], a.tiles};
    a.tiles += ((int)N[s] + 15) / 16;
  }
  hipStream_t st = (hipStream_t)stream;
  if (call.groups) return launch<kGroupScale, kNormGroup>(a, st);
  if (b_cols == 1) {
    if (!call.norm) return launch<kRowScale, kRotate>(a, st);
    return call.add ? launch<kRowScale, kAddNormRotate>(a, st) : launch<kRowScale, kNormRotate>(a, st);
  }
  if (!call.norm) return launch<kTokenGroup, kRotate>(a, st);
  return call.add ? launch<kTokenGroup, kAddNormRotate>(a, st) : launch<kTokenGroup, kNormRotate>(a, st);
}

}  // namespace
}  // namespace flh

using namespace flh;

extern "C" int flh_rotate_quant_gemm_i4_o16_multi(const flh_half* x, int count, const uint8_t* const* B,
                                                  const flh_half* const* b_scale, flh_half* const* D, const size_t* N,
                                                  size_t M, size_t K, int b_cols, void* stream) {
  return online_checked("rotate_quant_gemm", OnlineCall{x, nullptr, nullptr, nullptr, 0.f, false, false}, count, B, b_scale, D, N, M, K,
                        b_cols, stream);
}

extern "C" int flh_rmsnorm_rotate_quant_gemm_i4_o16_multi(const flh_half* x, const flh_half* add, flh_half* sum_out,
                                                          const flh_half* weight, float eps, int count,
                                                          const uint8_t* const* B, const flh_half* const* b_scale,
                                                          flh_half* const* D, const size_t* N, size_t M, size_t K,
                                                          int b_cols, void* stream) {
  const char* who = "rmsnorm_rotate_quant_gemm";
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "%s: eps must not be negative", who);
  if ((add == nullptr) != (sum_out == nullptr)) return fail(FLH_EINVAL, "%s: add and sum_out come together or not at all", who);
  if (add && (misaligned16(add, sum_out))) return fail(FLH_EINVAL, "%s: add and sum_out must be 16-byte aligned", who);
  if (weight && misaligned16(weight)) return fail(FLH_EINVAL, "%s: weight must be 16-byte aligned", who);
  if (sum_out && ((const void*)sum_out == (const void*)x || (const void*)sum_out == (const void*)add))
    return fail(FLH_EINVAL, "%s: sum_out must not be x or add", who);
  return online_checked(who, OnlineCall{x, add, weight, sum_out, eps, true, false}, count, B, b_scale, D, N, M, K, b_cols, stream);
}

extern "C" int flh_rotate_quant_gemm_i4_o16(const flh_half* x, const uint8_t* B, const flh_half* b_scale, flh_half* D,
                                            size_t M, size_t N, size_t K, int b_cols, void* stream) {
  if (N == 0) return FLH_OK;
  return flh_rotate_quant_gemm_i4_o16_multi(x, 1, &B, &b_scale, &D, &N, M, K, b_cols, stream);
}

extern "C" int flh_rmsnorm_group_quant_gemm_i4_o16_multi(const flh_half* x, const flh_half* weight, float eps, int count,
                                                         const uint8_t* const* B, const flh_half* const* b_scale, flh_half* const* D,
                                                         const size_t* N, size_t M, size_t K, void* stream) {
  const char* who = "rmsnorm_group_quant_gemm";
  if (!(eps >= 0.f)) return fail(FLH_EINVAL, "%s: eps must not be negative", who);
  if (weight && misaligned16(weight)) return fail(FLH_EINVAL, "%s: weight must be 16-byte aligned", who);
  return online_checked(who, OnlineCall{x, nullptr, weight, nullptr, eps, true, true}, count, B, b_scale, D, N, M, K, (int)(K / 128), stream);
}
