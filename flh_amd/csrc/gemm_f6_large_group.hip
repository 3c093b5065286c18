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
// Eight waves, two per SIMD, of 64 x 64 outputs (tile 256 x 128) or 32 x 64 (128 x 128, for launches that leave compute units
// without one of the larger tiles).  One wave issues at most one instruction every 4.4 clocks, so that four waves of 64 x
// 128, one per SIMD, spent 704 clocks of a step on its MFMAs and folds (44 per MFMA and its eight multiply-adds) and as many again
// on loads, fragment reads, scales and barriers with the matrix pipe idle; a second wave issues beside the first.  Measured
// against those four waves, us, token / group scales: 8192 x 14336 x 4096 398 -> 372 / 420 -> 397, 2048 x 28672 204 -> 188 / 215 -> 202,
// 2048 x 4096 x 14336 93 -> 89 / 105 -> 100, 1000 x 4096 x 14336 (128 tiles) - / 91 -> 79; with tiles of 128 x 128 65, 1000 x 4096 x
// 4096 31 -> 21.  The same four waves with fewer instructions (buffer loads, no clamped offsets) gave 1-3 %.
//
// What bounds it now: no unit is full.  Of the 1575 clocks of a step with token scales (2048 x 28672, outputs included) the matrix pipe is
// busy for 512 and vector instructions are issued for 728, LDS beside them for 630, a third of it bank conflicts; with group scales 768,
// 812 and 692 of 1705 (counters; four waves 1800 and 1970).  A fifth resp. a fourteenth of the clocks is neither matrix nor vector work.
// On top of that power: 1.82 GHz over 8192 x 14336 x 4096, 2.0 over half of that, 2.2 in launches of 65 us.  Everything adds to
// both: without the operand loads 294 us instead of 361 (token scales, 8192 x 14336 x 4096), from a cached slab 331, without the fragment
// reads 323, without the folds 278, the MFMAs alone 173; the outputs of a tile 40.  The 128 x 128 tile: its LDS traffic (24 fragments
// and 24 KB of loads per step of 256 matrix clocks; 490 of 1076 clocks busy).
#include "gemm_f6_large.h"

namespace flh {
namespace f6l {
namespace {

template <int EPI, int BM>
struct Shape {
  static constexpr int BN = 128, WAVES = 8, WM = BM / 4, WN = 64;   // waves: 4 x 2
  static constexpr int BLK = (BM + BN) / 32, STAGES = BM == 256 ? 4 : 6, STAGE = BLK * kRowBlock;
  // behind the ring: two blocks of eight groups per channel [2][BN][8], the same per token or one scale per token
  static constexpr int SC_B = 2 * BN * 16, SC_A = EPI == kGroupScale ? 2 * BM * 16 : BM * 2;
  static constexpr int LDS = STAGES * STAGE + SC_B + SC_A;
  static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
};

template <int EPI, int OUT, int BM>
__global__ __launch_bounds__(512, 1) void gemm_f6_large_group_kernel(const GemmArgs p) {
  using S = Shape<EPI, BM>;
  constexpr bool TOKEN = EPI == kTokenGroup, TALL = BM == 256;
  constexpr int BN = S::BN, STAGES = S::STAGES, STAGE = S::STAGE;
  constexpr int TM = S::WM / 32, TN = S::WN / 32, NT = TM * TN, ABLK = BM / 32;
  static_assert((TM == 2 || TM == 1) && TN == 2, "order of the fragment reads and folds");
  // which 32 weight rows of the tile are block b of a stage: SwiGLU and rotary epilogues need the channels c and c + 64 of the
  // tile (gate and up, the halves of a head) in one wave, whose blocks are 2 wcol and 2 wcol + 1
  constexpr bool PAIRED = OUT == kSwiglu || OUT == kRope;
  auto source_block = [](int b) { return PAIRED ? (b & 1) * 2 + (b >> 1) : b; };
  extern __shared__ __align__(1024) uint8_t lds[];    // [STAGES][STAGE], weight scales, activation scales
  uint8_t* const sc_b = lds + STAGES * STAGE;
  uint8_t* const sc_a = sc_b + S::SC_B;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lds0 = (unsigned)(size_t)lds;
  const int wrow = wave >> 1, wcol = wave & 1, wm = wrow * S::WM;
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

  // ---- operand loads.  A stage is BM / 32 blocks of 32 rows x 96 bytes of the activations and four of the weights, a block
  // three 1 KiB instructions.  128 rows: wave w requests block w.  256 rows: wave w requests block w of the activations and, of
  // weight block w % 4, the first two thirds or the last one, in turn by steps, so that any two steps are nine instructions for
  // every wave, which is what its waits count.  16-byte chunk s = 6 r + c of a block is stored in slot s ^ ((s >> 4) & 1): rows 8
  // apart, whose chunks lie in the same banks, swap neighbours, and the pattern repeats within the 64 chunks of an
  // instruction, so that one lane offset and immediates serve all of them.  Buffer loads with the slab as the buffer: rows
  // past the end of a matrix read as zero (their results are never stored).
  const unsigned lane_off = (unsigned)(lane ^ ((lane >> 4) & 1)) * 16;
  const bool first_is_a = TALL || wave < ABLK;         // what the wave's whole block is of
  const unsigned step_a = (unsigned)p.M * kBlock;
  v4i srd = buffer_of(p.A, step_a), srd_b = srd;       // slabs of the step to be requested next: of the whole block, the shared one
  unsigned off = 0, off_b = 0, step = step_a, step_b = 0;
  int kld = 0, turn = 0;                               // index of that step inside its tile; whose turn it is
  auto set_loads = [&](const Tile& t) __attribute__((always_inline)) {
    const int blk = source_block(wave & 3);
    const bool up = OUT == kSwiglu && blk >= 2;
    step_b = (unsigned)t.N * kBlock;
    srd_b = buffer_of(up ? t.B2 : t.B, step_b);
    off_b = (unsigned)(t.n0 + (OUT == kSwiglu ? (blk & 1) : blk) * 32) * kBlock + lane_off;
    if (first_is_a) {
      srd = buffer_of(p.A, step_a);
      off = (unsigned)(t.m0 + wave * 32) * kBlock + lane_off;
      step = step_a;
    } else {
      srd = srd_b, off = off_b, step = step_b;
    }
    kld = 0;
  };
  auto issue = [&](int slot_base) __attribute__((always_inline)) {
    load_block_to_lds(srd, off, lds0 + slot_base + wave * kRowBlock);
  };
  auto issue_shared = [&](int slot_base) __attribute__((always_inline)) {
    if constexpr (TALL) {
      const unsigned dst = lds0 + slot_base + (ABLK + (wave & 3)) * kRowBlock;
      if (turn ^ (wave >> 2)) load_last_third_to_lds(srd_b, off_b, dst);
      else load_two_thirds_to_lds(srd_b, off_b, dst);
    }
  };
  // the step after the one just requested; past a tile's last one the next tile's first (past the last tile: the same slab
  // again, which nobody reads).  The step is added to descriptors that start one step early: no branch in the common case.
  auto advance = [&]() __attribute__((always_inline)) {
    turn ^= 1;
    if (__builtin_expect(++kld == KT, 0)) {
      if (at + die_wgs < die_count) set_loads(tile_of<BN, OUT, BM>(p, die_first + at + die_wgs));
      else kld = KT - 1;
      buffer_advance(srd, 0ull - step);
      if (TALL) buffer_advance(srd_b, 0ull - step_b);
    }
    buffer_advance(srd, step);
    if (TALL) buffer_advance(srd_b, step_b);
  };

  // ---- scales: eight groups at a time, 16-byte pieces of the rows of scales straight to LDS ([row][8 groups]), double
  // buffered by blocks of eight steps.  A block is requested in the first step of the one before it (the next tile's
  // first block in the first step of a tile's last block); the last block of a row may start early.
  int sblk = 0;                                        // blocks requested so far
  auto sc_issue = [&](const Tile& t, int blk) __attribute__((always_inline)) {
    constexpr int PIECES = TOKEN ? 2 : 2 + BM / 64;
    const int g0 = min(8 * blk, KT - 8);
    if (wave < PIECES) {
      const int piece = wave;
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
    const unsigned* tb = (const unsigned*)(sc_b + parity * (BN * 16) + gi * 2 + (wcol * (PAIRED ? 32 : 64) + fr) * 16);
#pragma unroll
    for (int j = 0; j < TN; ++j) raw_b[j] = tb[j * (PAIRED ? 64 : 32) * 4];
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
  auto chunk_at = [&](int k) { const int c = 6 * fr + 3 * fc + k; return (c ^ ((c >> 4) & 1)) * 16; };
  const int a_base = wrow * TM * kRowBlock, b_base = (ABLK + wcol * TN) * kRowBlock;
  int ao[4] = {a_base + chunk_at(0), a_base + chunk_at(1), a_base + chunk_at(1) + 8, a_base + chunk_at(2)};
  int bo[4] = {b_base + chunk_at(0), b_base + chunk_at(1), b_base + chunk_at(1) + 8, b_base + chunk_at(2)};
  // (adjacent 8-byte reads would be merged into one of 16 bytes and taken apart with copies, if the compiler saw that
  // they are adjacent; three 16-byte reads into one tuple cost copies of the middle one, too)
  asm("" : "+v"(ao[2]), "+v"(bo[2]));
  // [set][half of the step][B0, B1, A0, A1]: tiles of 128 rows read a step's fragments into the other set than the one in use
  constexpr int SETS = TALL ? 1 : 2;
  v4i f4[SETS][2][TN + TM];
  v2i f2[SETS][2][TN + TM];
  auto read_fragment = [&](auto set_tag, auto f_tag, int slot_base) __attribute__((always_inline)) {
    constexpr int f = decltype(f_tag)::value, set = decltype(set_tag)::value % SETS;
    const int* o = f < TN ? bo : ao;
    const uint8_t* st = lds + slot_base + (f < TN ? f : f - TN) * kRowBlock;
    f4[set][0][f] = *(const v4i*)(st + o[0]);
    f2[set][0][f] = *(const v2i*)(st + o[1]);
    f2[set][1][f] = *(const v2i*)(st + o[2]);
    f4[set][1][f] = *(const v4i*)(st + o[3]);
  };
  auto operand = [&](auto set_tag, auto m_tag, int f) __attribute__((always_inline)) {
    constexpr int m = decltype(m_tag)::value, set = decltype(set_tag)::value % SETS;
    const v4i a = f4[set][m][f];
    const v2i b = f2[set][m][f];
    return m == 0 ? v8i{a[0], a[1], a[2], a[3], b[0], b[1], 0, 0} : v8i{b[0], b[1], a[0], a[1], a[2], a[3], 0, 0};
  };

  // ---- prologue
  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  int stage = 0;                                       // byte offset of a ring slot
  set_loads(tile_of<BN, OUT, BM>(p, die_first + at));
  sc_issue(tile_of<BN, OUT, BM>(p, die_first + at), 0);
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) {
    issue(s * STAGE);
    issue_shared(s * STAGE);
    advance();
  }
  issue((STAGES - 1) * STAGE);
  // load instructions of a wave in the stages that may be outstanding when one is needed: all but that and the one in use
  static_assert(!TALL || STAGES == 4, "two stages are nine instructions");
  constexpr int kBehind = TALL ? 9 : (STAGES - 3) * 3;
  wait_vmcnt<kBehind + 3>();
  __syncthreads();

  // float32 results: scalars, not a matrix-instruction tuple, on whose registers the compiler forms multiply-adds of
  // eight bytes instead of four
  float res[NT][16];
  // sums of the two pairs of tiles in flight; with one pair per step, of this step's and the one's before
  v16f sums[4], prod[TOKEN ? 1 : 4];
  constexpr int ODD_PAIR = NT == 2 ? 2 : 0;
  float chan[TN], chan_last[2];                        // (one scale per token) this step's weight scales; the last pair's of the one before
  auto fold = [&](auto t_tag, auto b_tag, auto h_tag, float sb) __attribute__((always_inline)) {
    constexpr int t = decltype(t_tag)::value, b = decltype(b_tag)::value, h = decltype(h_tag)::value;
#pragma unroll
    for (int r = 8 * h; r < 8 * h + 8; ++r) res[t][r] = __builtin_fmaf(sums[b][r], TOKEN ? sb : prod[TOKEN ? 0 : b][r], res[t][r]);
    float* q = &res[t][8 * h];                         // here, and not sunk past the branches half way through a step
    asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]), "+v"(q[4]), "+v"(q[5]), "+v"(q[6]), "+v"(q[7]));
  };
  const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // vector-memory operations that are certain to be younger than the next stage's loads in a tile's first step, besides
  // the stages behind it: the stores of the tile before, if it was a whole one
  constexpr int kStores = (OUT == kSwiglu ? 2 : 4) * TM;
  static_assert(kBehind + kStores < 64, "vmcnt range");
  bool stored = false;
  int prev = (STAGES - 1) * STAGE;
  // One step: four pairs of tiles.  The four slots of a pair issue the first MFMA of either tile, then the second (which
  // would wait for the first if it came right behind it), and the half folds of the pair before (the previous step's last
  // pair in the first).  The next step's fragments go into the registers of fragments that are done with.  ODD: the
  // second step of a pair, whose scales are the upper halves of what the first step's were read with.
  auto group_step = [&](auto first_tag, auto last_tag, auto odd_tag, int kt) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_tag)::value, LAST = decltype(last_tag)::value, ODD = decltype(odd_tag)::value;
    const int nx = stage == (STAGES - 1) * STAGE ? 0 : stage + STAGE;
    h4 sbv[TN], sav[TM];
    if constexpr (TOKEN) {
      chan_last[0] = chan[TN - 2], chan_last[1] = chan[TN - 1];
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
          if (kt + 8 < KT) sc_issue(tile_of<BN, OUT, BM>(p, die_first + at), (kt >> 3) + 1);
          else if (at + die_wgs < die_count) sc_issue(tile_of<BN, OUT, BM>(p, die_first + at + die_wgs), 0);
          else ++sblk;
        }
      }
      constexpr std::integral_constant<int, ODD> SET{};
      constexpr std::integral_constant<int, !ODD> NEXT{};
      constexpr int at_sums = t + (ODD ? ODD_PAIR : 0);
      if constexpr (m == 0)
        sums[at_sums] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(operand(SET, I0, TN + i), operand(SET, I0, j), zero, kBf6, kBf6,
                                                                       0, 0, 0, 0);
      else
        sums[at_sums] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(operand(SET, I1, TN + i), operand(SET, I1, j), sums[at_sums],
                                                                       kBf6, kBf6, 0, 0, 0, 0);
      if constexpr (!TOKEN && m == 1) prod[at_sums] = __builtin_amdgcn_mfma_f32_32x32x8f16(sav[i], sbv[j], zero, 0, 0, 0);
      constexpr std::integral_constant<int, (s & 1)> half{};
      constexpr int ft = (s < 4 ? NT : 2 * (s / 4)) - 2 + ((s >> 1) & 1);
      constexpr std::integral_constant<int, ft> FT{};
      if constexpr (s >= 4) fold(FT, FT, half, chan[ft % TN]);
      else if constexpr (!FIRST) fold(FT, std::integral_constant<int, ft + (ODD ? 0 : ODD_PAIR)>{}, half, chan_last[ft - (NT - 2)]);
      if constexpr (s == 1) issue_shared(prev);
      if constexpr (!LAST && s == NT + 1) issue(stage);
      constexpr std::integral_constant<int, TN> A0{};
      constexpr std::integral_constant<int, TN + 1> A1{};
      if constexpr (TALL) {
        if constexpr (s == NT) read_fragment(NEXT, A0, nx);
        if constexpr (s > NT && m == 1) read_fragment(NEXT, std::integral_constant<int, j>{}, nx);   // (B_j: done with)
        if constexpr (s == 2 * NT - 1) read_fragment(NEXT, A1, nx);
      } else {
        if constexpr (s == 0) read_fragment(NEXT, A0, nx);
        if constexpr (s == 1) read_fragment(NEXT, I0, nx);
        if constexpr (s == 2) read_fragment(NEXT, I1, nx);
      }
      if constexpr (ODD && s == 2 * NT - 3)            // the next pair's scales: of this tile, or the next one's first
        read_scales(LAST ? 0 : kt + 1, (sblk - (LAST || !((kt + 1) & 7) ? 1 : 2)) & 1);
      __builtin_amdgcn_sched_barrier(0);
    });
    prev = stage;
    stage = nx;
  };

  static_for<TN + TM>([&](auto f) { read_fragment(I0, f, 0); });
  read_scales(0, 0);
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  for (;;) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) res[t][r] = 0.f;
    if constexpr (TOKEN) parked = p.As[min(tile_of<BN, OUT, BM>(p, die_first + at).m0 + (tid & (BM - 1)), p.M - 1)];
    group_step(yes, no, no, 0);
    if constexpr (TOKEN) ((__half*)sc_a)[tid & (BM - 1)] = parked;  // (read in the epilogue, many barriers later)
    for (int kt = 1; kt < KT - 1; kt += 2) {
      group_step(no, no, yes, kt);
      group_step(no, no, no, kt + 1);
    }
    group_step(no, yes, yes, KT - 1);
    static_for<2>([&](auto u_tag) {                    // the last pair (KT is even: the last step is an odd one)
      constexpr int u = decltype(u_tag)::value;
      constexpr std::integral_constant<int, NT - 2 + u> FT{};
      constexpr std::integral_constant<int, NT - 2 + u + ODD_PAIR> B{};
      fold(FT, B, I0, chan[TN - 2 + u]), fold(FT, B, I1, chan[TN - 2 + u]);
    });

    // ---- outputs, 16 rows at a time through the slot of the stage just multiplied, which is refilled after this, and there
    // through the block that this same wave refills.  Lane: channel fr of a 32 x 32 tile, tokens 8 g + 4 fc + 0..3 in
    // register quad g.
    const Tile cur = tile_of<BN, OUT, BM>(p, die_first + at);
    uint8_t* const ep = lds + prev + wave * kRowBlock;
    static_assert(16 * kHalfPitch <= kRowBlock, "staging tile");
    static_for<2 * TM>([&](auto c_tag) {
      constexpr int i = decltype(c_tag)::value / 2, g0 = decltype(c_tag)::value % 2 * 2;
#pragma unroll
      for (int g = g0; g < g0 + 2; ++g) {
        h4 sa4 = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
        if constexpr (TOKEN) sa4 = *(const h4*)((const __half*)sc_a + wm + i * 32 + 8 * g + 4 * fc);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float f = TOKEN ? res[i * TN + j][4 * g + e] * (float)sa4[e] : res[i * TN + j][4 * g + e];
            *(_Float16*)(ep + (8 * (g - g0) + 4 * fc + e) * kHalfPitch + (j * 32 + fr) * 2) = (_Float16)round_here(f);
          }
      }
      store_half_rows<16, OUT>(p, cur, ep, cur.m0 + wm + i * 32 + g0 * 8, wcol, lane);
      __builtin_amdgcn_sched_barrier(0);
    });
    wait_lgkmcnt0();                                   // the staged rows have been read: the slot may be refilled
    issue(prev);
    stored = OUT != kRope && cur.m0 + BM <= p.M && cur.n0 + (OUT == kSwiglu ? BN / 2 : BN) <= cur.N;
    at += die_wgs;
    if (at >= die_count) break;
  }
  wait_vmcnt<0>();                                     // the loads past the last tile land before the ring goes away
}

template <int EPI, int OUT, int BM>
int launch(GemmArgs a, hipStream_t stream) {
  using S = Shape<EPI, BM>;
  constexpr int BNC = OUT == kSwiglu ? S::BN / 2 : S::BN;
  a.tiles_m = (a.M + BM - 1) / BM;
  a.tiles_n = (a.N + BNC - 1) / BNC;
  for (int s = 1; s < a.n_seg; ++s) {
    a.seg_tile0[s] = a.tiles_n;
    a.tiles_n += (a.seg_N[s] + S::BN - 1) / S::BN;
  }
  a.group_m = a.tiles_m < 4 ? a.tiles_m : 4;
  auto kern = gemm_f6_large_group_kernel<EPI, OUT, BM>;
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)kern, S::LDS, grant, "gemm_f6")) return rc;
  const long tiles = (long)a.tiles_m * a.tiles_n;
  const unsigned grid = (unsigned)(tiles < 256 ? tiles : 256);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * S::WAVES), S::LDS, stream, a);
  return check_launch("gemm_f6");
}

template <int OUT>
int launch(const GemmArgs& a, bool token, bool tall, hipStream_t stream) {
  if (tall) return token ? launch<kTokenGroup, OUT, 256>(a, stream) : launch<kGroupScale, OUT, 256>(a, stream);
  return token ? launch<kTokenGroup, OUT, 128>(a, stream) : launch<kGroupScale, OUT, 128>(a, stream);
}

}  // namespace

int launch_large_group(const GemmArgs& a, bool token, bool tall, Out out, hipStream_t stream) {
  switch (out) {
    case kSwiglu: return launch<kSwiglu>(a, token, tall, stream);
    case kRope: return launch<kRope>(a, token, tall, stream);
    case kResidual: return launch<kResidual>(a, token, tall, stream);
    default: return launch<kPlain>(a, token, tall, stream);
  }
}

}  // namespace f6l
}  // namespace flh
