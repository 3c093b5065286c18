// int4 x int4 GEMM + dequant for launches between decoding and prefill: up to a few hundred tokens, and a handful of tokens
// against many output channels.  Same arithmetic as gemm_i4.hip (codes x 16 as int8 on the matrix cores, exact int32 sums per
// group, one fused multiply-add per group in ascending order, identical epilogue roundings): same bits.
//
// Why.  The 64 x 64 tiles of gemm_i4.hip leave most of the chip idle here (4096 channels, 45 tokens: 64 workgroups), each
// with one latency per 128 codes of K; a K split (gemm_i4_decode.hip) needs every group's sums of a tile in LDS, which ends
// at 16 tokens.  Here a workgroup owns a small tile (BM x BN below) for the whole of K, so there is one per compute unit from
// 33 tokens x 4096 channels on, and each wave folds its own 16 x 16 tiles in order.  Operands come through a ring of LDS stages of
// four groups (256 bytes of every row) filled by direct-to-LDS loads two stages ahead; fragments, and the scales from a
// table in LDS, are read into registers one stage ahead of the products.  (Fragments straight from memory reach 16 bytes
// per clock and compute unit, sixteen half lines per load: 17-25 us where this kernel takes 11-17.)
//
// What bounds it: the vector ALU.  A 16 x 16 x 128 product is 32 clocks of MFMA next to 24 instructions of unpacking (12 more
// per further tile of the wave) and 12 of folding (8 with one scale per token), and the one or two waves of a SIMD overlap
// little.  Deeper rings (6 stages) changed nothing up to one workgroup per compute unit and cost the second resident beyond.
//
// us per launch, weights from HBM, group scales on both sides, before -> after (K x N):
//   17-64 tokens: 4096 x 4096 21.1 -> 8.2, 11008 x 4096 50 -> 17, 14336 x 4096 68 -> 21, 4096 x 28672 40 -> 20 (32), 31 (64)
//   128: 4096 x 4096 21.7 -> 10.9, 4096 x 6144 22.2 -> 14.3;  256: 4096 x 4096 21.8 -> 15.7;  512: 4096 x 1024 18.3 -> 10.3
//   16 tokens: 4096 x 28672 22.5 -> 15.7, 4096 x 14336 13.9 -> 9.8 (5 and 3.7 TB/s of weights)
// One scale per row has a kernel of its own below (gemm_i4_dealt_kernel).
#include "gemm_i4.h"

namespace flh {
namespace {

// What a launch does with its results: rows of D, or q / k / v with the rotary embedding (two tiles half a head apart)
enum StreamOut { kStreamPlain = 0, kStreamRope = 1 };

constexpr int kStageGroups = 4;                    // groups of 128 codes per stage: 256 bytes of every row
constexpr int kRowBytes = kStageGroups * 64;
constexpr int kStreamMaxGroups = 128;              // scales of a row that fit beside the ring (K <= 16384)

typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t lds_byte;
template <typename T>
__device__ __forceinline__ T from_lds(const lds_byte* q) { return *(const __attribute__((address_space(3))) T*)q; }

// channels n .. n + 3 of row m
__device__ __forceinline__ void store_four(const GemmArgs& p, void* Dp, int N, int m, int n, const _Float16 (&y)[4]) {
  const size_t at = (size_t)m * N + n;
  if (N % 4 == 0) {
    if (n >= N) return;
    h4 v = {y[0], y[1], y[2], y[3]};
    if (p.R) v = v + *(const h4*)((const _Float16*)p.R + at);   // (R may be D: read before the store)
    *(h4*)((_Float16*)Dp + at) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) ((_Float16*)Dp)[at + e] = p.R ? y[e] + ((const _Float16*)p.R)[at + e] : y[e];
  }
}

template <int TN>
struct StageRegs {                                 // a wave's operands of one stage
  v4i a[kStageGroups], b[TN][kStageGroups];
  v2u sa, sb[TN][4];                               // scales of the four groups: the lane's token, its four channels
};

template <int WM, int WN, int TN, int S, int EPI, int OUT>
__global__ __launch_bounds__(64 * WM * WN) void gemm_i4_stream_kernel(const GemmArgs p) {
  constexpr int WAVES = WM * WN, RA = 16 * WM, RB = 16 * TN * WN, ROWS = RA + RB;
  constexpr int STAGE = ROWS * kRowBytes;
  constexpr int NA = RA / 4 / WAVES, NB = RB / 4 / WAVES, NI = NA + NB;   // 1 KiB load instructions per wave and stage
  constexpr int SROWS = EPI == kGroupScale ? ROWS : RB;   // rows of the scale table: tokens, then channels
  static_assert(RA / 4 % WAVES == 0 && RB / 4 % WAVES == 0 && (S - 2) * NI < 64 && kRowBytes * 4 == 1024, "loads per stage");
  static_assert(OUT == kStreamPlain || (TN == 2 && WN == 1), "partner tiles");
  extern __shared__ __align__(16) uint8_t lds[];
  lds_byte* ring = (lds_byte*)lds;                 // (typed: a generic pointer would make the reads wait for all loads)
  lds_byte* scales = ring + S * STAGE;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, c = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const unsigned L = xcd_contiguous(blockIdx.x, gridDim.x);
  const int bn = L / p.tiles_m, bm = L % p.tiles_m;       // the blocks of one weight stripe sit next to each other on a die

  const uint8_t* B = p.B;
  const __half* Bs = p.Bs;
  void* Dp = p.D;
  int N = p.N, seg = 0, t = bn;
  for (int s = 1; s < p.n_seg; ++s)
    if (bn >= p.seg_tile0[s]) B = p.seg_B[s], Bs = p.seg_Bs[s], Dp = p.seg_D[s], N = p.seg_N[s], seg = s, t = bn - p.seg_tile0[s];
  const int Kb = p.K >> 1, KT = p.K >> 7;
  const int stages = (KT + kStageGroups - 1) / kStageGroups;
  const int m0 = bm * RA;
  // first channel of the block's tile j
  auto first = [&](int j) {
    return OUT == kStreamPlain ? (t * (TN * WN) + j) * 16 : (t >> 2) * 128 + (t & 3) * 16 + j * 64;
  };
  auto b_row = [&](int row) { return min(first(row >> 4) + (row & 15), N - 1); };      // row of B behind LDS row RA + row

  auto first_group = [&](int s) { return min(s * kStageGroups, KT - kStageGroups); };   // the last stage ends with the row

  const int pitch = (KT >> 1) | 1;                 // of the scale table
  // operands: a load instruction brings 256 bytes of four rows, chunk c of row r to slot c ^ (r % 16); a wave's share of either
  // operand is consecutive KiB of LDS (load_kib_to_lds16: addresses less 1024 i)
  const int lrow = lane >> 4;
  const uint8_t *src_a[NA], *src_b[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int row = (wave * NA + i) * 4 + lrow;
    src_a[i] = p.A + (size_t)min(m0 + row, p.M - 1) * Kb + ((lane & 15) ^ (row & 15)) * 16 - 1024 * i;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int row = (wave * NB + i) * 4 + lrow;
    src_b[i] = B + (size_t)b_row(row) * Kb + ((lane & 15) ^ (row & 15)) * 16 - 1024 * i;
  }
  const unsigned base = (unsigned)(uintptr_t)ring;
  auto request = [&](int s, int slot) {            // slot: byte offset of the ring slot
    const size_t off = (size_t)first_group(s) * 64;
    const uint8_t *a[NA], *b[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) a[i] = src_a[i] + off;
#pragma unroll
    for (int i = 0; i < NB; ++i) b[i] = src_b[i] + off;
    load_kib_to_lds16(a, base + slot + wave * NA * 1024);
    load_kib_to_lds16(b, base + slot + (RA * kRowBytes + wave * NB * 1024));
  };
  int chunk[kStageGroups];                         // of the lane's row
#pragma unroll
  for (int g = 0; g < kStageGroups; ++g) chunk[g] = r * kRowBytes + ((g * 4 + c) ^ r) * 16;
  auto read = [&](int s, int slot, StageRegs<TN>& q) {
    const lds_byte* st = ring + slot;
#pragma unroll
    for (int g = 0; g < kStageGroups; ++g) {
#pragma unroll
      for (int j = 0; j < TN; ++j) q.b[j][g] = from_lds<v4i>(st + chunk[g] + (RA + (wn * TN + j) * 16) * kRowBytes);
      q.a[g] = from_lds<v4i>(st + chunk[g] + wm * 16 * kRowBytes);
    }
    const int at = first_group(s) >> 1;
    auto two = [&](int row) {
      const __attribute__((address_space(3))) unsigned* e = (const __attribute__((address_space(3))) unsigned*)scales + row * pitch + at;
      return v2u{e[0], e[1]};
    };
    if constexpr (EPI == kGroupScale) q.sa = two(wm * 16 + r);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) q.sb[j][e] = two(SROWS - RB + (wn * TN + j) * 16 + 4 * c + e);
  };
  float out[TN][4];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) out[j][e] = 0.f;
  auto product = [&](const v4i& a, const v4i& b) {
    v4i d = {0, 0, 0, 0};
    v4i alo, ahi, blo, bhi;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      alo[e] = (a[e] << 4) & (int)0xF0F0F0F0, ahi[e] = a[e] & (int)0xF0F0F0F0;
      blo[e] = (b[e] << 4) & (int)0xF0F0F0F0, bhi[e] = b[e] & (int)0xF0F0F0F0;
    }
    d = __builtin_amdgcn_mfma_i32_16x16x64_i8(blo, alo, d, 0, 0, 0);
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(bhi, ahi, d, 0, 0, 0);
  };
  auto fold = [&](auto G, int j, const v4i& d, const StageRegs<TN>& q) {
    constexpr int g = decltype(G)::value, w = g / 2, h = g % 2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float v = (float)d[e];                 // 256 x the exact sum
      const unsigned sb = q.sb[j][e][w];
      if constexpr (EPI == kGroupScale) out[j][e] = __builtin_fmaf(v, mul_halves<h>(q.sa[w], sb), out[j][e]);
      else out[j][e] = fma_half<h>(v, sb, out[j][e]);
    }
  };
  auto multiply = [&](const StageRegs<TN>& q) {    // a whole stage: all products, then their folds in ascending order
    v4i d[kStageGroups][TN];
#pragma unroll
    for (int g = 0; g < kStageGroups; ++g)
#pragma unroll
      for (int j = 0; j < TN; ++j) d[g][j] = product(q.a[g], q.b[j][g]);
    static_for<kStageGroups>([&](auto G) {
#pragma unroll
      for (int j = 0; j < TN; ++j) fold(G, j, d[decltype(G)::value][j], q);
    });
  };

  request(0, 0);
  // scales behind the first stage (in front of it, their addresses took 0.6 us before the first operand was requested), as their rows
  // are: [row][KT / 2 pairs, an odd number of slots] in LDS, every wave a share of them
  {
    const float inv = 1.0f / (float)pitch;
    const int total = SROWS * pitch;
    for (int f0 = wave * 64; f0 < total; f0 += WAVES * 64) {
      const int f = min(f0 + lane, total - 1);
      int row = (int)((float)f * inv);             // f < 2^14: off by one at most
      row += (f >= (row + 1) * pitch ? 1 : 0) - (f < row * pitch ? 1 : 0);
      const int pair = min(f - row * pitch, (KT >> 1) - 1), chan = row - (SROWS - RB);
      const __half* q = chan < 0 ? p.As + (size_t)min(m0 + row, p.M - 1) * KT
                                 : Bs + (size_t)b_row(chan) * KT;
      load_to_lds4(q + 2 * pair, (unsigned)(uintptr_t)scales + f0 * 4);
    }
  }
#pragma unroll
  for (int s = 1; s < S - 1; ++s)
    if (s < stages) request(s, s * STAGE);
  const bool live = m0 + wm * 16 < p.M;
  // every wave's loads of the oldest stage but `newer` are in LDS, every wave has its last stage in registers
  auto arrive = [&](bool steady) {
    if (steady) wait_vmcnt<(S - 2) * NI>();
    else wait_vmcnt<0>();
    wait_lgkmcnt0();
    barrier_no_fence();
  };
  StageRegs<TN> q0, q1;
  int slot = 0;                                    // of stage s
  auto step = [&](int s, StageRegs<TN>& cur, StageRegs<TN>& next) {     // s + 1 < stages
    arrive(s + S - 1 < stages);
    if (s + S < stages) request(s + S, slot);
    slot = slot == (S - 1) * STAGE ? 0 : slot + STAGE;
    if (live) {
      read(s + 1, slot, next);
      __builtin_amdgcn_sched_barrier(0);           // (the reads have the products' time to arrive)
      multiply(cur);
    }
  };
  auto last = [&](const StageRegs<TN>& q) {
    if (!live) return;
    const int skip = (stages - 1) * kStageGroups - first_group(stages - 1);   // groups that the stage before has done
    static_for<kStageGroups>([&](auto G) {
      constexpr int g = decltype(G)::value;
      if (g < skip) return;
#pragma unroll
      for (int j = 0; j < TN; ++j) fold(G, j, product(q.a[g], q.b[j][g]), q);
    });
  };
  arrive(stages >= S);                             // stage 0; slot S - 1 is free
  if (S - 1 < stages) request(S - 1, (S - 1) * STAGE);
  if (live) read(0, 0, q0);
  int s = 0;
  for (; s + 2 < stages; s += 2) {
    step(s, q0, q1);
    step(s + 1, q1, q0);
  }
  if (s + 1 < stages) {
    step(s, q0, q1);
    last(q1);
  } else {
    last(q0);
  }

  // lane: token r, channels 4 c + e of each tile
  const int m = m0 + wm * 16 + r;
  if (m >= p.M) return;
  _Float16 y[TN][4];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v;
      if constexpr (EPI == kGroupScale) v = out[j][e] * 0.00390625f;
      else v = round_here(out[j][e] * 0.00390625f) * __half2float(p.As[m]);
      y[j][e] = (_Float16)round_here(v);
    }
  if constexpr (OUT == kStreamRope) {
    const int head = t >> 2, ch = (t & 3) * 16 + 4 * c;
    if (head * 128 >= N) return;
    const int b = m / p.rope_T, tok = m - b * p.rope_T;
    __half* dst = (__half*)Dp + (size_t)m * N + head * 128 + ch;
    if (seg > 0) {
      const long long slot = p.rope_pos[tok];
      if (slot < 0 || slot >= (long long)p.rope_max_len) return;
      dst = (__half*)Dp + (((size_t)b * p.rope_hkv + head) * p.rope_max_len + (size_t)slot) * 128 + ch;
    }
    if (seg < 2) {
      const __half *ct = p.rope_cos + (size_t)tok * 128 + ch, *st = p.rope_sin + (size_t)tok * 128 + ch;
      const h4 c1 = *(const h4*)ct, c2 = *(const h4*)(ct + 64), s1 = *(const h4*)st, s2 = *(const h4*)(st + 64);
#pragma unroll
      for (int e = 0; e < 4; ++e) rope_pair(y[0][e], y[1][e], c1[e], c2[e], s1[e], s2[e]);
    }
    *(h4*)dst = h4{y[0][0], y[0][1], y[0][2], y[0][3]};
    *(h4*)(dst + 64) = h4{y[1][0], y[1][1], y[1][2], y[1][3]};
  } else {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = first(wn * TN + j) + 4 * c;
      store_four(p, Dp, N, m, n, y[j]);
    }
  }
}

template <int RA, int RB, int OUT>
void set_stream_tiles(GemmArgs& a) {
  a.tiles_m = (a.M + RA - 1) / RA;
  auto tiles = [&](int n) { return OUT == kStreamRope ? (n + 127) / 128 * 4 : (n + RB - 1) / RB; };
  a.tiles_n = tiles(a.N);
  for (int s = 1; s < a.n_seg; ++s) {
    a.seg_tile0[s] = a.tiles_n;
    a.tiles_n += tiles(a.seg_N[s]);
  }
}

template <int WM, int WN, int TN, int S, int EPI, int OUT>
int launch_stream(GemmArgs a, hipStream_t stream) {
  constexpr int RA = 16 * WM, RB = 16 * TN * WN;
  set_stream_tiles<RA, RB, OUT>(a);
  constexpr size_t ring = (size_t)S * (RA + RB) * kRowBytes;
    // (rounded up to whole load instructions)
  auto table = [](int kt) { return ((size_t)((kt / 2) | 1) * (EPI == kGroupScale ? RA + RB : RB) * 4 + 255) / 256 * 256; };
  auto kern = gemm_i4_stream_kernel<WM, WN, TN, S, EPI, OUT>;
  static LdsGrant grant;                               // per instantiation; sized for the longest rows it takes
  if (int rc = reserve_lds((const void*)kern, ring + table(kStreamMaxGroups), grant, "gemm (stream)")) return rc;
  hipLaunchKernelGGL(kern, dim3(a.tiles_m * a.tiles_n), dim3(64 * WM * WN), ring + table(a.K >> 7), stream, a);
  return check_launch("gemm_i4_stream");
}

// One scale per row: a stage's four groups are dealt out to the four waves.  Wave w multiplies group w for the whole tile -- 16
// tokens x 64 channels as four 16 x 16 products, 32 or 64 tokens x 32 channels as one or two 32 x 32 ones -- so that an operand is
// unpacked once and not by every wave whose product it enters; the integer sums meet at the end, through the ring's LDS.
// (Group scales have to be folded in order: handing the sums over stage by stage costs what the unpacking saves, 45 x 4096 x
// 11008 15.8 -> 16.7.  Two waves per 16 x 16 tile, two groups each, the same: 16.0.)
template <int TOK, int S>
__global__ __launch_bounds__(256) void gemm_i4_dealt_kernel(const GemmArgs p) {
  constexpr bool SMALL = TOK == 16;
  constexpr int RA = TOK, RB = SMALL ? 64 : 32, STAGE = (RA + RB) * kRowBytes, NI = (RA + RB) / 16;
  constexpr int TT = SMALL ? 1 : TOK / 32, C = SMALL ? 1 : 2;   // token tiles; 16-byte pieces of a row's group per lane
  static_assert((RA + RB) % 16 == 0 && NI >= 4 && NI <= 6 && (S - 2) * NI < 64 && 12 * TT * 1024 <= S * STAGE, "loads per stage, exchange");
  extern __shared__ __align__(16) uint8_t lds[];
  lds_byte* ring = (lds_byte*)lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = lane % (SMALL ? 16 : 32), c = lane / (SMALL ? 16 : 32);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned L = xcd_contiguous(blockIdx.x, gridDim.x);
  const int bn = L / p.tiles_m, bm = L % p.tiles_m;

  const uint8_t* B = p.B;
  const __half* Bs = p.Bs;
  void* Dp = p.D;
  int N = p.N, t = bn;
  for (int s = 1; s < p.n_seg; ++s)
    if (bn >= p.seg_tile0[s]) B = p.seg_B[s], Bs = p.seg_Bs[s], Dp = p.seg_D[s], N = p.seg_N[s], t = bn - p.seg_tile0[s];
  const int Kb = p.K >> 1, KT = p.K >> 7;
  const int stages = (KT + kStageGroups - 1) / kStageGroups;
  const int m0 = bm * RA, n0 = t * RB;
  auto first_group = [&](int s) { return min(s * kStageGroups, KT - kStageGroups); };   // the last stage ends with the row

  // a load instruction brings 256 bytes of four rows, chunk c of row r to slot c ^ (r % 16); a wave's rows are consecutive KiB of
  // LDS (load_kib_to_lds16: addresses less 1024 i, four at a time)
  constexpr int N0 = 4, N1 = NI - N0;
  const uint8_t* src[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = (wave * NI + i) * 4 + (lane >> 4);
    src[i] = (row < RA ? p.A + (size_t)min(m0 + row, p.M - 1) * Kb : B + (size_t)min(n0 + max(row - RA, 0), N - 1) * Kb) +
             ((lane & 15) ^ (row & 15)) * 16 - 1024 * (i % 4);
  }
  const unsigned base = (unsigned)(uintptr_t)ring;
  auto request = [&](int s, int slot) {
    const size_t off = (size_t)first_group(s) * 64;
    const unsigned dst = base + slot + wave * NI * 1024;
    const uint8_t *g[N0], *rest[N1 ? N1 : 1];
#pragma unroll
    for (int i = 0; i < N0; ++i) g[i] = src[i] + off;
    load_kib_to_lds16(g, dst);
    if constexpr (N1 > 0) {
#pragma unroll
      for (int i = 0; i < N1; ++i) rest[i] = src[N0 + i] + off;
      load_kib_to_lds16(rest, dst + 4096);
    }
  };
  int piece[C];                                    // of the wave's group in the lane's row
#pragma unroll
  for (int i = 0; i < C; ++i) piece[i] = r * kRowBytes + ((wave * 4 + c + 2 * i) ^ (r & 15)) * 16;
  struct Operands { v4i a[TT][C], b[SMALL ? 4 : C]; };
  auto read = [&](int slot, Operands& q) {
    const lds_byte* st = ring + slot;
#pragma unroll
    for (int i = 0; i < (SMALL ? 4 : C); ++i)
      q.b[i] = from_lds<v4i>(st + (SMALL ? piece[0] + i * (16 * kRowBytes) : piece[SMALL ? 0 : i]) + RA * kRowBytes);
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int i = 0; i < C; ++i) q.a[j][i] = from_lds<v4i>(st + piece[i] + j * (32 * kRowBytes));
  };
  auto lo = [](v4i x) { return (x << 4) & (int)0xF0F0F0F0; };
  auto hi = [](v4i x) { return x & (int)0xF0F0F0F0; };
  v16i wide[TT];                                   // 32 x 32: quarter q (registers 4 q ..) is folded by wave q
  v4i part[4];                                     // 16 x 16: tile q
#pragma unroll
  for (int i = 0; i < 4; ++i) part[i] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < TT; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) wide[j][i] = 0;
  auto multiply = [&](const Operands& q) {
    if constexpr (SMALL) {
      const v4i al = lo(q.a[0][0]), ah = hi(q.a[0][0]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        part[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lo(q.b[i]), al, part[i], 0, 0, 0);
        part[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(hi(q.b[i]), ah, part[i], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const v4i bl = lo(q.b[i]), bh = hi(q.b[i]);
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          wide[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bl, lo(q.a[j][i]), wide[j], 0, 0, 0);
          wide[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bh, hi(q.a[j][i]), wide[j], 0, 0, 0);
        }
      }
    }
  };

#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < stages) request(s, s * STAGE);
  // every wave's loads of the oldest stage but `newer` are in LDS, every wave has its last stage in registers
  auto arrive = [&](bool steady) {
    if (steady) wait_vmcnt<(S - 2) * NI>();
    else wait_vmcnt<0>();
    wait_lgkmcnt0();
    barrier_no_fence();
  };
  Operands q0, q1;
  int slot = 0;                                    // of stage s
  auto step = [&](int s, Operands& cur, Operands& next) {   // s + 1 < stages
    arrive(s + S - 1 < stages);
    if (s + S < stages) request(s + S, slot);
    slot = slot == (S - 1) * STAGE ? 0 : slot + STAGE;
    read(slot, next);
    __builtin_amdgcn_sched_barrier(0);             // (the reads have the products' time to arrive)
    multiply(cur);
  };
  auto last = [&](const Operands& q) {             // without the groups that the stage before has done
    if (wave >= (stages - 1) * kStageGroups - first_group(stages - 1)) multiply(q);
  };
  arrive(stages >= S);                             // stage 0; slot S - 1 is free
  if (S - 1 < stages) request(S - 1, (S - 1) * STAGE);
  read(0, q0);
  int s = 0;
  for (; s + 2 < stages; s += 2) {
    step(s, q0, q1);
    step(s + 1, q1, q0);
  }
  if (s + 1 < stages) {
    step(s, q0, q1);
    last(q1);
  } else {
    last(q0);
  }

  // every wave's quarter of the sums: [token tile][receiver][sender after it][lane]
  wait_lgkmcnt0();
  barrier_no_fence();                              // nobody reads the ring any more
  v4i sum[TT];
#pragma unroll
  for (int j = 0; j < TT; ++j)
    static_for<4>([&](auto V) {
      constexpr int v = decltype(V)::value;
      const v4i d = SMALL ? part[v] : v4i{wide[j][4 * v], wide[j][4 * v + 1], wide[j][4 * v + 2], wide[j][4 * v + 3]};
      if (wave == v) sum[j] = d;
      else *(__attribute__((address_space(3))) v4i*)(ring + (j * 12 + v * 3 + ((wave - v + 3) & 3)) * 1024 + lane * 16) = d;
    });
  wait_lgkmcnt0();
  barrier_no_fence();
#pragma unroll
  for (int j = 0; j < TT; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i) sum[j] += from_lds<v4i>(ring + (j * 12 + wave * 3 + i) * 1024 + lane * 16);

  // lane: token r of each token tile, four channels
  const int n = n0 + wave * (SMALL ? 16 : 8) + 4 * c;
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    const int m = m0 + j * 32 + r;
    if (m >= p.M) return;
    const float s_a = __half2float(p.As[m]);
    _Float16 y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float s_b = __half2float(Bs[min(n + e, N - 1)]) * 0.00390625f;
      y[e] = (_Float16)round_here((float)sum[j][e] * (s_a * s_b));
    }
    store_four(p, Dp, N, m, n, y);
  }
}

template <int TOK, int S>
int launch_dealt(GemmArgs a, hipStream_t stream) {
  constexpr int RA = TOK, RB = TOK == 16 ? 64 : 32;
  set_stream_tiles<RA, RB, kStreamPlain>(a);
  constexpr size_t ring = (size_t)S * (RA + RB) * kRowBytes;
  auto kern = gemm_i4_dealt_kernel<TOK, S>;
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)kern, ring, grant, "gemm (stream)")) return rc;
  hipLaunchKernelGGL(kern, dim3(a.tiles_m * a.tiles_n), dim3(256), ring, stream, a);
  return check_launch("gemm_i4_stream");
}

long stream_columns(const GemmArgs& a) {
  long n = a.N;
  for (int s = 1; s < a.n_seg; ++s) n += a.seg_N[s];
  return n;
}

// Tiles with group scales, tokens x channels: 16 x 64 for up to 16 tokens, else 32 x 32, or 64 x 32 (half the weight traffic, a fifth less
// vector work) where nearly two of its workgroups per compute unit remain and the tokens fill it as well as the smaller tile
// (64 tokens: 4096 x 14336, 448 workgroups, 17.0 against 18.3 us; 256: 4096 x 4096, 512, 15.7 against 18.1; 128: 4096 x 6144,
// 384, 15.7 against 14.3).
template <int EPI>
int launch_grouped_by_shape(const GemmArgs& a, hipStream_t stream) {
  if (a.M <= 16) return launch_stream<1, 4, 1, 3, EPI, kStreamPlain>(a, stream);
  const long large = (long)((a.M + 63) / 64) * ((stream_columns(a) + 31) / 32);
  if (large >= 448 && (a.M + 31) / 32 % 2 == 0) return launch_stream<4, 1, 2, 3, EPI, kStreamPlain>(a, stream);
  return launch_stream<2, 2, 1, 3, EPI, kStreamPlain>(a, stream);
}

// ... and with one scale per row: 16 x 64 for up to 16 tokens, else 32 x 32 while three workgroups per compute unit hold all of
// them, with a longer ring where one does, and 64 x 32 beyond or where K is long.  us, 32 x 32 (ring of 3, of 5) / 64 x 32, K =
// 4096 unless stated:
//   45 x 4096 of K = 11008 (256 workgroups of 32 x 32) 11.2, 9.2 / 12.7;  45 x 11008 (688) 9.5, 10.8 / 10.3;  128 x 6144 (768)
//   9.3, 10.8 / 10.0;
//   64 x 14336 (896) 13.1 / 11.4;  64 x 28672 (1792) 21.4, 24.1 / 20.5;  128 x 4096 of K = 11008 (512) 15.2, 15.5 / 13.5
int launch_rows_by_shape(const GemmArgs& a, hipStream_t stream) {
  if (a.M <= 16) return launch_dealt<16, 3>(a, stream);
  const long columns = (stream_columns(a) + 31) / 32, small = (long)((a.M + 31) / 32) * columns, large = (long)((a.M + 63) / 64) * columns;
  if (small > 768 || (a.K > 8192 && small > 256 && large <= 256)) return launch_dealt<64, 3>(a, stream);
  return small <= 256 ? launch_dealt<32, 5>(a, stream) : launch_dealt<32, 3>(a, stream);
}

// what the kernel can take: whole stages, and group scales that dword loads can fetch two at a time
bool stream_takes(const GemmArgs& a, int epi, int group) {
  const int kt = a.K >> 7;
  if (epi == kInt32 || kt < kStageGroups) return false;
  if (epi == kRowScale) return true;
  auto off4 = [](const void* q) { return ((uintptr_t)q & 3) != 0; };
  if (group != 128 || a.b_cols == 1 || kt % 2 || kt > kStreamMaxGroups || off4(a.Bs) || (a.a_cols > 1 && off4(a.As))) return false;
  for (int s = 1; s < a.n_seg; ++s)
    if (off4(a.seg_Bs[s])) return false;
  return true;
}

// Up to 16 tokens against gemm_i4_decode.hip (us, K = 4096, this kernel / that one, one scale per row / token scales / group scales; one to
// four tokens come here only where the dot-product kernel does not take them).
//  * Against whole lines (gemm_lines_over_stream), up to 32768 channels: from nine tokens on from 172 workgroups of 64 channels on (16 x
//    11008 7.7 / 8.2 / 8.4 against 7.6 / 8.2 / 8.1, x 12288 7.9 / 8.4 / 8.5 against 7.9 / 8.4 / 8.4, x 14336 8.3 / 8.7 / 8.8 against 9.3 / 9.9 /
//    9.8; weights that the last-level cache holds x 12288 6.6 / 7.7 / 8.0 against 7.1 / 8.0 / 8.0), with fewer only token scales beyond
//    24576 (5 x 22016 12.6 / 12.7 / 12.8 against 10.6 / 12.0 / 11.3, x 28672 13.9 / 13.9 / 14.0 against 12.5 / 14.1 / 12.9).
//  * Else, up to 16384 channels, one workgroup of 64 per compute unit: with five or more tokens from 172 workgroups on, with fewer
//    beyond 12288 channels, where half lines have more than three workgroups on a compute unit.  Beyond, the compute units that get
//    one workgroup more set the time and the other kernel's grows with the channels: with few tokens only if the last round has
//    enough workgroups, and not where that kernel's tiles of every group leave a compute unit one workgroup.  (Drawn against half lines;
//    beyond 32768 channels, where whole lines may stand in for them, the launches that they get are as fast as on half lines: one
//    scale per row, 3 to 8 tokens, x 49152 0.99, x 65536 1.00, x 128256 1.01 of the time.)
bool takes_few_tokens(const GemmArgs& a, int epi, long columns) {
  const bool row = epi == kRowScale, token = a.a_cols == 1;
  if (gemm_lines_over_stream(a, epi)) return a.M > 8 ? columns >= 172 * 64 : !row && token && columns > 24576;
  if (columns <= 16384 || a.M > (row ? 4 : token ? 6 : 8) || (!row && a.K > 8192))
    return a.M >= 5 ? columns >= 172 * 64 : columns > 12288;
  const long last = (columns - 1) % 16384 + 1;             // channels of the last round
  return last * 3 >= 16384 && (row || token || a.M > 6 || last >= 9830);   // a third, or six tenths
}

}  // namespace

// Which launches are faster here than on the kernels on either side.  us, this kernel against the other (K = 4096 unless
// stated; "large" counts 64 x 32 tiles):
//  * up to 16 tokens, against the K split of the decode kernels: takes_few_tokens above.
//  * 17 .. 64 tokens: always (one scale per row, 32 x 4096 5.0 against 5.7, 17 x 4096 4.9 against 5.1).
//  * more, group-scaled weights, against 64 x 64 and 128 x 128 tiles: up to 768 large tiles, 512 if K is long (128 x 12288,
//    768: 24 against 27; 192 x 12288, 1152: 35 against 33; 384 x 4096, 768: 22.3 against 25.1, but 64 against 60 for K = 11008,
//    where 300 x 4096, 640, takes 69 against 59 on weights that are in the last-level cache).
//  * more, one scale per row, against the K-split tiles: up to 768 (256 x 6144, 768: 14.4 against 15.4; 320 x 6144, 960: 17.0 against
//    15.0; 300 x 4096, 640: 12.1 against 12.6; 400 x 4096, 896: 15.0 against 13.5; 128 x 22016, 1376: 26.5 against 24.5; K = 11008: 300 x
//    4096, 640, 27.5 against 34.5, 400 x 4096, 896, 33.1 against 33.6).
//  * and no more tokens than 1280: on 1024 channels the tiles fill the chip by then (1500 tokens, token scales, with their
//    quantiser: 31.6 against 29.5; one scale per row: 1000 8.8 against 10.1).
// (A forced tile goes to the tile kernels.)
bool gemm_stream_supports(const GemmArgs& a, int epi, int group) {
  if (!stream_takes(a, epi, group) || g_tune_tile.load(std::memory_order_relaxed) || g_tune_ks.load(std::memory_order_relaxed))
    return false;
  const long columns = stream_columns(a);
  if (a.M <= 16) return takes_few_tokens(a, epi, columns);
  if (a.M <= 64) return true;
  if (a.M > 1280) return false;
  const long large = (long)((a.M + 63) / 64) * ((columns + 31) / 32);
  return large <= (epi == kRowScale || a.K <= 8192 ? 768 : 512);
}

int gemm_stream_dispatch(const GemmArgs& a, int epi, hipStream_t stream) {
  if (epi == kRowScale) return launch_rows_by_shape(a, stream);
  return a.a_cols == 1 ? launch_grouped_by_shape<kTokenGroup>(a, stream) : launch_grouped_by_shape<kGroupScale>(a, stream);
}

// q / k / v with the rotary embedding and the cache write, group-scaled weights: the alternative is 128 x 128 tiles only
// (48 or 96 of them for the Llama widths).
bool gemm_stream_rope_supports(const GemmArgs& a, int epi) {
  return epi != kRowScale && stream_takes(a, kGroupScale, 128) && !g_tune_tile.load(std::memory_order_relaxed) &&
         (long)((a.M + 63) / 64) * (stream_columns(a) / 32) <= 768;
}

int gemm_stream_rope_dispatch(const GemmArgs& a, hipStream_t stream) {
  return a.a_cols == 1 ? launch_stream<4, 1, 2, 3, kTokenGroup, kStreamRope>(a, stream)
                       : launch_stream<4, 1, 2, 3, kGroupScale, kStreamRope>(a, stream);
}

}  // namespace flh
