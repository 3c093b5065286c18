// Group-scaled weights (groups of 128) with group-scaled or per-token activations: the large-tile kernel of
// gemm_f6_large.h in the form that the per-group fold needs.
//
// A step of K is one group.  Every 32 x 32 tile's two MFMAs start from zero and its exact sums are folded into float32
// results: out = fma(sum, a_g * b_g, out) (one scale per token: fma(sum, b_g, out), the token scale at the end) in
// ascending g -- the arithmetic of the int8 kernel.  The activations are the MFMA's first operand, so that a lane holds
// one channel and a group's weight scale is one register per column block; with group-scaled activations as well, the
// tile's scale products come from one more MFMA, an outer product of the two scale vectors (exact in float32, in the
// layout of the sums), instead of a conversion and a multiplication per output on the vector ALU.
//
// What bounds it: one wave per SIMD, which issues everything in turn.  Counters at 2048 x 28672 x 4096, per step of one group,
// outputs included: 1800 clocks with token scales, 1970 with group scales, of which vector instructions hold the issue port 712
// resp. 820 (128 of 178 are the fold's multiply-adds, 4 clocks each, with token scales), the matrix pipe is busy 512 resp. 770
// and LDS 500 resp. 530, a third of that in bank conflicts; with token scales some 570 clocks are in none of the first two.  A
// wave of 64 x 128 outputs has the fewest LDS reads and loads per MFMA; four of them, one per SIMD with up to 512 registers,
// were faster than eight of 32 x 128 (8192 x 14336 x 4096: 414 against 436 us with token scales, 444 against 479 with group scales).
#include "gemm_f6_large.h"

namespace flh {
namespace f6l {
namespace {

template <int EPI>
struct Shape {
  static constexpr int BM = 256, BN = 128, WAVES = 4, WM = BM / WAVES;
  static constexpr int BLK = (BM + BN) / 32, STAGES = 4, STAGE = BLK * kRowBlock;
  static constexpr int NI = BLK * 3 / WAVES;          // load instructions per wave and stage
  // behind the ring: two blocks of eight groups per channel [2][BN][8], the same per token or one scale per token
  static constexpr int SC_B = 2 * BN * 16, SC_A = EPI == kGroupScale ? 2 * BM * 16 : BM * 2;
  static constexpr int LDS = STAGES * STAGE + SC_B + SC_A;
  static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
};

template <int EPI, int OUT>
__global__ __launch_bounds__(256, 1) void gemm_f6_large_group_kernel(const GemmArgs p) {
  using S = Shape<EPI>;
  constexpr bool TOKEN = EPI == kTokenGroup;
  constexpr int BM = S::BM, BN = S::BN, STAGES = S::STAGES, STAGE = S::STAGE, NI = S::NI;
  constexpr int TM = S::WM / 32, TN = BN / 32, NT = TM * TN, ABLK = BM / 32, NB = NI / 3;
  static_assert(TM == 2 && TN == 4, "order of the fragment reads");
  extern __shared__ __align__(1024) uint8_t lds[];    // [STAGES][STAGE], weight scales, activation scales
  uint8_t* const sc_b = lds + STAGES * STAGE;
  uint8_t* const sc_a = sc_b + S::SC_B;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lds0 = (unsigned)(size_t)lds;
  const int wm = wave * S::WM;
  const int fr = lane & 31, fc = lane >> 5;

  // tiles of this workgroup, as in the row-scale kernel
  const unsigned total = p.tiles_m * p.tiles_n;
  const unsigned xcd = blockIdx.x % kNumXCD, slot = blockIdx.x / kNumXCD;
  const unsigned per = total / kNumXCD, rem = total % kNumXCD;
  const unsigned die_first = xcd * per + (xcd < rem ? xcd : rem), die_count = per + (xcd < rem ? 1 : 0);
  const unsigned die_wgs = (gridDim.x - xcd + kNumXCD - 1) / kNumXCD;
  unsigned at = slot;
  if (at >= die_count) return;
  const int KT = p.K / 128;                            // steps = groups

  // ---- operand loads, as in the row-scale kernel
  unsigned loff[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int s = q * 64 + lane, r = s / 6;
    loff[q] = (unsigned)r * kBlock + ((s % 6) ^ ((r >> 3) & 1)) * 16;
  }
  const uint8_t* lp[NB];
  unsigned lim[NB];
  unsigned b_step = 0;
  int kld = 0;
  auto set_loads = [&](const Tile& t) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int blk = wave * NB + b, wb = blk - ABLK;
      const bool isA = blk < ABLK, up = OUT == kSwiglu && wb >= 2;
      const int first = isA ? t.m0 + blk * 32 : t.n0 + (OUT == kSwiglu ? (wb & 1) * 32 : wb * 32);
      const int all = isA ? p.M : t.N, rows = all - first;
      lp[b] = wave_uniform((isA ? p.A : up ? t.B2 : t.B) + (rows > 0 ? (size_t)first * kBlock : 0));
      lim[b] = (unsigned)min(rows > 0 ? rows : all, 32) * kBlock - 16;
    }
    b_step = (unsigned)t.N * kBlock;
    kld = 0;
  };
  auto step_of = [&](int b) { return wave * NB + b < ABLK ? (unsigned)p.M * kBlock : b_step; };
  auto issue = [&](int stage, auto i_tag) __attribute__((always_inline)) {
    constexpr int b = decltype(i_tag)::value / 3, q = decltype(i_tag)::value % 3;
    load_to_lds16(lp[b], min(loff[q], lim[b]), lds0 + stage * STAGE + (wave * NB + b) * kRowBlock + q * 1024);
  };
  auto advance = [&]() __attribute__((always_inline)) {
    if (__builtin_expect(++kld == KT, 0)) {
      if (at + die_wgs < die_count) set_loads(tile_of<BN, OUT>(p, die_first + at + die_wgs));
      else kld = KT - 1;
#pragma unroll
      for (int b = 0; b < NB; ++b) lp[b] -= step_of(b);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) lp[b] += step_of(b);
  };

  // ---- scales: eight groups at a time, 16-byte pieces of the rows of scales straight to LDS ([row][8 groups]), double
  // buffered by blocks of eight steps.  A block is requested in the first step of the one before it (the next tile's
  // first block in the first step of a tile's last block); the last block of a row may start early.
  int sblk = 0;                                        // blocks requested so far
  auto sc_issue = [&](const Tile& t, int blk) __attribute__((always_inline)) {
    constexpr int PIECES = TOKEN ? 2 : 6, PER_WAVE = (PIECES + 3) / 4;
    const int g0 = min(8 * blk, KT - 8);
#pragma unroll
    for (int u = 0; u < PER_WAVE; ++u) {
      const int piece = (wave * PER_WAVE + u) % PIECES;   // (a wave without a piece of its own repeats another's)
      const bool isB = piece < 2, up = OUT == kSwiglu && piece == 1;
      const int r = (isB ? piece : piece - 2) * 64 + lane;
      const int row = isB ? min(t.n0 + (up ? r - 64 : r), t.N - 1) : min(t.m0 + r, p.M - 1);
      const __half* base = isB ? (up ? t.Bs2 : t.Bs) : p.As;
      const unsigned dst = lds0 + STAGES * STAGE + (isB ? (sblk & 1) * (BN * 16) + piece * 1024
                                                        : S::SC_B + (sblk & 1) * (BM * 16) + (piece - 2) * 1024);
      load_to_lds16(wave_uniform(base), (unsigned)(row * KT + g0) * 2, dst);
    }
    ++sblk;
  };
  __half parked = __float2half(1.f);                   // one scale per token: read in a tile's first step, parked after it
  // a pair of steps' scales as read: steps come in pairs (KT is even, and so is the first group of a block)
  unsigned raw_b[TN], raw_a[TM];
  auto read_scales = [&](int kt, int parity) __attribute__((always_inline)) {
    const int gi = kt - min(kt & ~7, KT - 8);
    const unsigned* tb = (const unsigned*)(sc_b + parity * (BN * 16) + gi * 2 + fr * 16);
#pragma unroll
    for (int j = 0; j < TN; ++j) raw_b[j] = tb[j * 32 * 4];
    if constexpr (!TOKEN) {
      const unsigned* ta = (const unsigned*)(sc_a + parity * (BM * 16) + gi * 2 + (wm + fr) * 16);
#pragma unroll
      for (int i = 0; i < TM; ++i) raw_a[i] = ta[i * 32 * 4];
    }
  };
  auto rank1 = [&](unsigned bits) __attribute__((always_inline)) {   // K element 0 of the lane's row / column
    const v2i d = {fc == 0 ? (int)bits : 0, 0};
    return __builtin_bit_cast(h4, d);
  };

  // ---- fragments: 24 bytes per lane and MFMA, as 16 + 8 and 8 + 16 bytes
  const int sw = (fr >> 3) & 1;
  const int c0 = ((3 * fc) ^ sw) * 16, c1 = ((3 * fc + 1) ^ sw) * 16, c2 = ((3 * fc + 2) ^ sw) * 16;
  const int a_base = wave * TM * kRowBlock + fr * kBlock, b_base = ABLK * kRowBlock + fr * kBlock;
  int ao[4] = {a_base + c0, a_base + c1, a_base + c1 + 8, a_base + c2};
  int bo[4] = {b_base + c0, b_base + c1, b_base + c1 + 8, b_base + c2};
  // (adjacent 8-byte reads would be merged into one of 16 bytes and taken apart with copies, if the compiler saw that
  // they are adjacent; three 16-byte reads into one tuple cost copies of the middle one, too)
  asm("" : "+v"(ao[2]), "+v"(bo[2]));
  v4i f4[2][TN + TM];                                  // [half of the step][B0 .. B3, A0, A1]
  v2i f2[2][TN + TM];
  auto read_fragment = [&](auto f_tag, int stage) __attribute__((always_inline)) {
    constexpr int f = decltype(f_tag)::value;
    const uint8_t* st = lds + stage * STAGE + (f < TN ? f : f - TN) * kRowBlock;
    const int* o = f < TN ? bo : ao;
    f4[0][f] = *(const v4i*)(st + o[0]);
    f2[0][f] = *(const v2i*)(st + o[1]);
    f2[1][f] = *(const v2i*)(st + o[2]);
    f4[1][f] = *(const v4i*)(st + o[3]);
  };
  auto operand = [&](auto m_tag, int f) __attribute__((always_inline)) {
    constexpr int m = decltype(m_tag)::value;
    const v4i a = f4[m][f];
    const v2i b = f2[m][f];
    return m == 0 ? v8i{a[0], a[1], a[2], a[3], b[0], b[1], 0, 0} : v8i{b[0], b[1], a[0], a[1], a[2], a[3], 0, 0};
  };

  // ---- prologue
  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  constexpr int SPLIT = NI / 2;
  int stage = 0;
  set_loads(tile_of<BN, OUT>(p, die_first + at));
  sc_issue(tile_of<BN, OUT>(p, die_first + at), 0);
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) {
    static_for<NI>([&](auto i) { issue(s, i); });
    advance();
  }
  static_for<SPLIT>([&](auto i) { issue(STAGES - 1, i); });
  wait_vmcnt<(STAGES - 2) * NI + SPLIT>();
  __syncthreads();

  // float32 results: scalars, not a matrix-instruction tuple, on whose registers the compiler forms multiply-adds of
  // eight bytes instead of four
  float res[NT][16];
  v16f sums[4], prod[TOKEN ? 1 : 4];
  float chan[TN], chan_last[2];                        // (one scale per token) this step's weight scales; the last pair's of the one before
  auto fold = [&](auto t_tag, auto h_tag, float sb) __attribute__((always_inline)) {
    constexpr int t = decltype(t_tag)::value, h = decltype(h_tag)::value;
#pragma unroll
    for (int r = 8 * h; r < 8 * h + 8; ++r) res[t][r] = __builtin_fmaf(sums[t % 4][r], TOKEN ? sb : prod[TOKEN ? 0 : t % 4][r], res[t][r]);
    float* q = &res[t][8 * h];                         // here, and not sunk past the branches half way through a step
    asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]), "+v"(q[4]), "+v"(q[5]), "+v"(q[6]), "+v"(q[7]));
  };
  const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // vector-memory operations that are certain to be younger than the next stage's loads in a tile's first step, besides
  // the stages behind it: the stores of the tile before, if it was a whole one
  constexpr int kBehind = (STAGES - 2) * NI, kStores = OUT == kSwiglu ? 8 : 16;
  static_assert(kBehind + kStores < 64, "vmcnt range");
  bool stored = false;
  int prev = STAGES - 1;
  // One step: four pairs of tiles.  The four slots of a pair issue the first MFMA of either tile, then the second (which
  // would wait for the first if it came right behind it), and the half folds of the pair before (the previous step's last
  // pair in the first).  The next step's fragments go into the registers of fragments that are done with.  ODD: the
  // second step of a pair, whose scales are the upper halves of what the first step's were read with.
  auto group_step = [&](auto first_tag, auto last_tag, auto odd_tag, int kt) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_tag)::value, LAST = decltype(last_tag)::value, ODD = decltype(odd_tag)::value;
    const int nx = stage + 1 == STAGES ? 0 : stage + 1;
    h4 sbv[TN], sav[TM];
    if constexpr (TOKEN) {
      chan_last[0] = chan[2], chan_last[1] = chan[3];
#pragma unroll
      for (int j = 0; j < TN; ++j)
        chan[j] = round_here((float)__builtin_bit_cast(_Float16, (unsigned short)(ODD ? raw_b[j] >> 16 : raw_b[j])));
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) sbv[j] = rank1(ODD ? raw_b[j] >> 16 : raw_b[j] & 0xFFFFu);
#pragma unroll
      for (int i = 0; i < TM; ++i) sav[i] = rank1(ODD ? raw_a[i] >> 16 : raw_a[i] & 0xFFFFu);
    }
    static_for<2 * NT>([&](auto s_tag) {
      constexpr int s = decltype(s_tag)::value, m = (s >> 1) & 1, t = 2 * (s >> 2) + (s & 1), i = t / TN, j = t % TN;
      if constexpr (s == NT) {                          // half way: the next stage is there, and nobody reads this one's A
        advance();
        if (FIRST && stored) wait_vmcnt<kBehind + kStores>();
        else wait_vmcnt<kBehind>();
        wait_lgkmcnt0();
        barrier_no_fence();
        if (!ODD && !(kt & 7)) {
          if (kt + 8 < KT) sc_issue(tile_of<BN, OUT>(p, die_first + at), (kt >> 3) + 1);
          else if (at + die_wgs < die_count) sc_issue(tile_of<BN, OUT>(p, die_first + at + die_wgs), 0);
          else ++sblk;
        }
      }
      if constexpr (m == 0)
        sums[t % 4] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(operand(I0, TN + i), operand(I0, j), zero, kBf6, kBf6, 0, 0, 0, 0);
      else
        sums[t % 4] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(operand(I1, TN + i), operand(I1, j), sums[t % 4], kBf6, kBf6,
                                                                     0, 0, 0, 0);
      if constexpr (!TOKEN && m == 1) prod[t % 4] = __builtin_amdgcn_mfma_f32_32x32x8f16(sav[i], sbv[j], zero, 0, 0, 0);
      constexpr std::integral_constant<int, (s & 1)> half{};
      constexpr int ft = (s < 4 ? NT : 2 * (s / 4)) - 2 + ((s >> 1) & 1);
      if constexpr (s >= 4) fold(std::integral_constant<int, ft>{}, half, chan[ft % TN]);
      else if constexpr (!FIRST) fold(std::integral_constant<int, ft>{}, half, chan_last[ft - (NT - 2)]);
      static_for<NI>([&](auto l) {
        constexpr int li = decltype(l)::value;
        if constexpr (li < SPLIT) {
          if constexpr (!LAST && s == NT + li * NT / SPLIT) issue(stage, l);
        } else {
          if constexpr (s == (li - SPLIT) * NT / (NI - SPLIT)) issue(prev, l);
        }
      });
      if constexpr (s == NT) read_fragment(std::integral_constant<int, TN>{}, nx);             // A0
      if constexpr (s > NT && m == 1) read_fragment(std::integral_constant<int, j>{}, nx);     // (B_j: done with)
      if constexpr (s == 2 * NT - 1) read_fragment(std::integral_constant<int, TN + 1>{}, nx); // A1
      if constexpr (ODD && s == 2 * NT - 3)            // the next pair's scales: of this tile, or the next one's first
        read_scales(LAST ? 0 : kt + 1, (sblk - (LAST || !((kt + 1) & 7) ? 1 : 2)) & 1);
      __builtin_amdgcn_sched_barrier(0);
    });
    prev = stage;
    stage = nx;
  };

  static_for<TN + TM>([&](auto f) { read_fragment(f, 0); });
  read_scales(0, 0);
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  for (;;) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) res[t][r] = 0.f;
    if constexpr (TOKEN) parked = p.As[min(tile_of<BN, OUT>(p, die_first + at).m0 + tid, p.M - 1)];
    group_step(yes, no, no, 0);
    if constexpr (TOKEN) ((__half*)sc_a)[tid] = parked;  // (read in the epilogue, many barriers later)
    for (int kt = 1; kt < KT - 1; kt += 2) {
      group_step(no, no, yes, kt);
      group_step(no, no, no, kt + 1);
    }
    group_step(no, yes, yes, KT - 1);
    constexpr std::integral_constant<int, NT - 2> t6{};
    constexpr std::integral_constant<int, NT - 1> t7{};
    fold(t6, I0, chan[2]), fold(t6, I1, chan[2]), fold(t7, I0, chan[3]), fold(t7, I1, chan[3]);

    // ---- outputs, 32 rows at a time through the slot of the stage just multiplied, which is refilled after this, and there
    // through the part that this same wave refills.  Lane: channel fr of a 32 x 32 tile, tokens 8 g + 4 fc + 0..3 in
    // register quad g.
    const Tile cur = tile_of<BN, OUT>(p, die_first + at);
    uint8_t* const ep = lds + prev * STAGE + wave * NB * kRowBlock;
    static_assert(32 * kPitch <= NB * kRowBlock, "staging tile");
    static_for<TM>([&](auto i_tag) {
      constexpr int i = decltype(i_tag)::value;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        h4 sa4 = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
        if constexpr (TOKEN) sa4 = *(const h4*)((const __half*)sc_a + wm + i * 32 + 8 * g + 4 * fc);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float f = TOKEN ? res[i * TN + j][4 * g + e] * (float)sa4[e] : res[i * TN + j][4 * g + e];
            *(_Float16*)(ep + (8 * g + 4 * fc + e) * kPitch + (j * 32 + fr) * 2) = (_Float16)round_here(f);
          }
      }
      store_rows<32, OUT>(p, cur, ep, cur.m0 + wm + i * 32, 0, lane);
      __builtin_amdgcn_sched_barrier(0);
    });
    wait_lgkmcnt0();                                   // the staged rows have been read: the slot may be refilled
    static_for<SPLIT>([&](auto l) { issue(prev, l); });
    stored = OUT != kRope && cur.m0 + BM <= p.M && cur.n0 + (OUT == kSwiglu ? BN / 2 : BN) <= cur.N;
    at += die_wgs;
    if (at >= die_count) break;
  }
  wait_vmcnt<0>();                                     // the loads past the last tile land before the ring goes away
}

template <int EPI, int OUT>
int launch(GemmArgs a, hipStream_t stream) {
  using S = Shape<EPI>;
  constexpr int BNC = OUT == kSwiglu ? S::BN / 2 : S::BN;
  a.tiles_m = (a.M + S::BM - 1) / S::BM;
  a.tiles_n = (a.N + BNC - 1) / BNC;
  for (int s = 1; s < a.n_seg; ++s) {
    a.seg_tile0[s] = a.tiles_n;
    a.tiles_n += (a.seg_N[s] + S::BN - 1) / S::BN;
  }
  a.group_m = a.tiles_m < 4 ? a.tiles_m : 4;
  auto kern = gemm_f6_large_group_kernel<EPI, OUT>;
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)kern, S::LDS, grant, "gemm_f6")) return rc;
  const long tiles = (long)a.tiles_m * a.tiles_n;
  const unsigned grid = (unsigned)(tiles < 256 ? tiles : 256);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * S::WAVES), S::LDS, stream, a);
  return check_launch("gemm_f6");
}

}  // namespace

int launch_large_group(const GemmArgs& a, bool token, Out out, hipStream_t stream) {
  switch (out) {
    case kSwiglu: return token ? launch<kTokenGroup, kSwiglu>(a, stream) : launch<kGroupScale, kSwiglu>(a, stream);
    case kRope: return token ? launch<kTokenGroup, kRope>(a, stream) : launch<kGroupScale, kRope>(a, stream);
    case kResidual: return token ? launch<kTokenGroup, kResidual>(a, stream) : launch<kGroupScale, kResidual>(a, stream);
    default: return token ? launch<kTokenGroup, kPlain>(a, stream) : launch<kGroupScale, kPlain>(a, stream);
  }
}

}  // namespace f6l
}  // namespace flh
