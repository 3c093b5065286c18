// int4 GEMM on the int8 matrix instruction for launches between the small tiles (gemm_i4_stream.hip) and the per-call 6-bit
// encoding: group-scaled weights (groups of 128) with group-scaled or per-token activations, tiles of 128 x 128.
//
// Persistent workgroups of eight waves (4 x 2, 32 x 64 outputs each, two per SIMD) walk over the launch's tiles, with the
// schedule, the scale blocks and the epilogues of gemm_f6_large_group.hip; the operands are the wire format.  A stage of the
// ring is two groups (256 codes, one 128-byte line of every row), so that loads are whole lines and there is one barrier
// per two groups.  A packed dword gives two int8 operand dwords with three instructions, codes x 16; the sums are 256 times
// the integer sums, exact, and so are the float32 results (a power of two commutes with every rounding of the fold), until the
// epilogue takes the factor out: the bits of the other kernels.
//
// What bounds it: vector instructions.  Per group a wave unpacks three operands (72 shifts and masks, 3.8 clocks each with two
// waves on a SIMD), converts 32 sums and folds them, around 1400 clocks for the SIMD's two waves, of which the matrix pipe is
// busy 530.  Sums whose first operand is the bits of 1.5 x 2^23, so that a subtraction takes the conversion's place: no faster.
// us, token / group scales, the tiles this replaces -> this: 1000 x 4096 x 4096 33 -> 26 / 38 -> 27, 250 x 14336 x 4096 32 ->
// 27 / 38 -> 27, 250 x 28672 x 4096 with SwiGLU 57 -> 52 (group), 128 x 22016 34 -> 28 / 39 -> 29, q / k / v + rotary 512 x
// 6144 33 -> 28 / 39 -> 30.
#include "gemm_f6_large.h"

namespace flh {
namespace {

using namespace f6l;

constexpr int kSqTile = 128, kSqRows = 32, kSqLine = 128;            // rows of a block, bytes of a row in a stage
constexpr int kSqBlock = kSqRows * kSqLine, kSqStage = 8 * kSqBlock, kSqStages = 4;

// 4 KiB: 8 rows per instruction, to lds_base + 0, 1024, 2048, 3072
__device__ __forceinline__ void load_lines_to_lds(const v4i& d, unsigned v0, unsigned v1, unsigned v2, unsigned v3, unsigned lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %1, %5, 0 offen lds\n\t"
               "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %2, %5, 0 offen lds\n\t"
               "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %3, %5, 0 offen lds\n\t"
               "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %4, %5, 0 offen lds" ::"s"(lds_base), "v"(v0), "v"(v1), "v"(v2), "v"(v3),
               "s"(d) : "memory", "m0", "scc");
}

template <int EPI, int OUT>
__global__ __launch_bounds__(512, 1) void gemm_i4_square_kernel(const GemmArgs p) {
  constexpr bool TOKEN = EPI == kTokenGroup;
  constexpr int BN = kSqTile, BM = kSqTile, TN = 2;
  constexpr bool PAIRED = OUT == kSwiglu || OUT == kRope;   // as in gemm_f6_large_group.hip
  auto source_block = [](int b) { return PAIRED ? (b & 1) * 2 + (b >> 1) : b; };
  extern __shared__ __align__(1024) uint8_t lds[];    // [kSqStages][kSqStage], weight scales [2][BN][8], activation scales
  uint8_t* const sc_b = lds + kSqStages * kSqStage;
  uint8_t* const sc_a = sc_b + 2 * BN * 16;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lds0 = (unsigned)(size_t)lds;
  const int wrow = wave >> 1, wcol = wave & 1, wm = wrow * 32;
  const int fr = lane & 31, fc = lane >> 5;

  const unsigned total = p.tiles_m * p.tiles_n;
  const unsigned xcd = blockIdx.x % kNumXCD, slot = blockIdx.x / kNumXCD;
  const unsigned per = total / kNumXCD, rem = total % kNumXCD;
  const unsigned die_first = xcd * per + (xcd < rem ? xcd : rem), die_count = per + (xcd < rem ? 1 : 0);
  const unsigned die_wgs = (gridDim.x - xcd + kNumXCD - 1) / kNumXCD;
  unsigned at = slot;
  if (at >= die_count) return;
  const int KT = p.K / 128, ST = KT / 2;               // groups, stages

  // ---- operand loads: wave w requests block w of a stage (four of activations, four of weights).  16-byte chunk c of row r of
  // a block is stored in slot c ^ ((r >> 1) & 7): sixteen rows read at one chunk are free of bank conflicts.  Buffer loads:
  // rows past the end of a matrix read as zero (their results are never stored).
  const unsigned pitch = (unsigned)p.K / 2;
  v4i srd = buffer_of(p.A, (unsigned)p.M * pitch);
  unsigned off[4];
  int kld = 0;
  auto set_loads = [&](const Tile& t) __attribute__((always_inline)) {
    const int blk = source_block(wave & 3);
    const bool is_a = wave < 4, up = OUT == kSwiglu && blk >= 2;
    srd = buffer_of(is_a ? p.A : up ? t.B2 : t.B, (unsigned)(is_a ? p.M : t.N) * pitch);
    const unsigned first = (unsigned)(is_a ? t.m0 + wave * 32 : t.n0 + (OUT == kSwiglu ? (blk & 1) : blk) * 32);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      off[q] = (first + 8 * q + (lane >> 3)) * pitch + (unsigned)((lane & 7) ^ ((4 * q + (lane >> 4)) & 7)) * 16;
    kld = 0;
  };
  auto issue = [&](int slot_base) __attribute__((always_inline)) {
    load_lines_to_lds(srd, off[0], off[1], off[2], off[3], lds0 + slot_base + wave * kSqBlock);
  };
  auto advance = [&]() __attribute__((always_inline)) {
    if (__builtin_expect(++kld == ST, 0)) {
      if (at + die_wgs < die_count) set_loads(tile_of<BN, OUT, BM>(p, die_first + at + die_wgs));
      else kld = ST - 1;                               // past the last tile: the same lines again, which nobody reads
      buffer_advance(srd, 0ull - kSqLine);
    }
    buffer_advance(srd, kSqLine);
  };

  // ---- scales, as in gemm_f6_large_group.hip: blocks of eight groups, requested in the first stage of the block before
  int sblk = 0;
  auto sc_issue = [&](const Tile& t, int blk) __attribute__((always_inline)) {
    constexpr int PIECES = TOKEN ? 2 : 4;
    const int g0 = min(8 * blk, KT - 8);
    if (wave < PIECES) {
      const int piece = wave;
      const bool isB = piece < 2, up = OUT == kSwiglu && piece == 1;
      const int r = (isB ? piece : piece - 2) * 64 + lane;
      const int row = isB ? min(t.n0 + (up ? r - 64 : r), t.N - 1) : min(t.m0 + r, p.M - 1);
      const __half* base = isB ? (up ? t.Bs2 : t.Bs) : p.As;
      const unsigned dst = lds0 + kSqStages * kSqStage + (isB ? (sblk & 1) * (BN * 16) + piece * 1024
                                                             : 2 * BN * 16 + (sblk & 1) * (BM * 16) + (piece - 2) * 1024);
      load_to_lds16(wave_uniform(base), (unsigned)(row * KT + g0) * 2, dst);
    }
    ++sblk;
  };
  __half parked = __float2half(1.f);
  unsigned raw_b[TN], raw_a;                           // a stage's two groups
  auto read_scales = [&](int kt, int parity) __attribute__((always_inline)) {
    const int gi = kt - min(kt & ~7, KT - 8);
    const unsigned* tb = (const unsigned*)(sc_b + parity * (BN * 16) + gi * 2 + (wcol * (PAIRED ? 32 : 64) + fr) * 16);
#pragma unroll
    for (int j = 0; j < TN; ++j) raw_b[j] = tb[j * (PAIRED ? 64 : 32) * 4];
    if constexpr (!TOKEN) raw_a = *(const unsigned*)(sc_a + parity * (BM * 16) + gi * 2 + (wm + fr) * 16);
  };
  auto rank1 = [&](unsigned bits) __attribute__((always_inline)) {   // K element 0 of the lane's row / column
    const v2i d = {fc == 0 ? (int)bits : 0, 0};
    return __builtin_bit_cast(h4, d);
  };

  // ---- fragments: of group g of a stage a lane takes the chunks 4 g + 2 fc and the next one, raw; [set = group][B0, B1, A][chunk]
  int bo[4], ao[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {                        // i = 2 g + u
    const int c = ((i >> 1) * 4 + 2 * fc + (i & 1)) ^ ((fr >> 1) & 7);
    bo[i] = (4 + wcol * TN) * kSqBlock + fr * kSqLine + c * 16;
    ao[i] = wrow * kSqBlock + fr * kSqLine + c * 16;
  }
  v4i raw[2][TN + 1][2];
  auto read_raw = [&](auto g_tag, auto f_tag, int slot_base) __attribute__((always_inline)) {
    constexpr int g = decltype(g_tag)::value, f = decltype(f_tag)::value;
    const int* o = f < TN ? bo : ao;
    const uint8_t* st = lds + slot_base + (f < TN ? f : 0) * kSqBlock;
    raw[g][f][0] = *(const v4i*)(st + o[2 * g]);
    raw[g][f][1] = *(const v4i*)(st + o[2 * g + 1]);
  };
  auto nibbles = [&](auto h_tag, const v4i& w) __attribute__((always_inline)) {   // codes x 16 of the low (0) or high (1) nibbles
    v4i o;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const unsigned u = (unsigned)w[d];
      o[d] = (int)((decltype(h_tag)::value ? u : u << 4) & 0xF0F0F0F0u);
    }
    return o;
  };
  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  constexpr std::integral_constant<int, 2> I2{};

  // ---- prologue
  int stage = 0;
  set_loads(tile_of<BN, OUT, BM>(p, die_first + at));
  sc_issue(tile_of<BN, OUT, BM>(p, die_first + at), 0);
#pragma unroll
  for (int s = 0; s < kSqStages - 1; ++s) {
    issue(s * kSqStage);
    advance();
  }
  issue((kSqStages - 1) * kSqStage);
  // Where in a stage's second group the next stage's first fragments are read: at once, and the stage has to have arrived a
  // whole one ahead (group scales 94.4 -> 92.5 us at 1000 x 14336 x 4096), or behind the barrier (token scales: 91.1 -> 89.4)
  constexpr int kReadAt = TOKEN ? 4 : 0;
  // What a wave's waits count, as in gemm_f6_large_group.hip: loads come back in order, four instructions per stage (`issue`), so
  // that with kBehind outstanding everything older than the stages behind the needed one has arrived -- the scales' requests,
  // which are older still or come on top, only make a wait longer.  In a tile's first stage the kStores stores of the tile before
  // are certain to be younger as well, if every wave made them all (`stored`).
  constexpr int kBehind = (kSqStages - (kReadAt ? 2 : 3)) * 4, kStores = OUT == kSwiglu ? 2 : 4;
  wait_vmcnt<kBehind + 4>();
  __syncthreads();

  float res[TN][16];                                   // 256 times the float32 results
  v16i sums[2][TN];                                    // [group of the stage][tile]
  v16f prod[TOKEN ? 1 : TN];
  h4 a_last = {}, b_last = {};                         // the last group's scales of tile 1, whose products are made a group later
  float chan[TN], chan_last[TN];
  auto fold = [&](auto t_tag, auto b_tag, auto r_tag, float sb) __attribute__((always_inline)) {   // four values
    constexpr int t = decltype(t_tag)::value, b = decltype(b_tag)::value, r0 = decltype(r_tag)::value;
#pragma unroll
    for (int r = r0; r < r0 + 4; ++r) res[t][r] = __builtin_fmaf((float)sums[b][t][r], TOKEN ? sb : prod[TOKEN ? 0 : t][r], res[t][r]);
    float* q = &res[t][r0];                            // here, and not sunk past the branches inside a stage
    asm volatile("" : "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]));
  };
  const v16i zero_i = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  bool stored = false;
  int prev = (kSqStages - 1) * kSqStage;
  // One group: eight slots of one MFMA, which unpack the operands of a quarter of the group every other slot and fold four
  // values of the group before each.  G: which of the stage's two.
  auto group = [&](auto first_tag, auto last_tag, auto g_tag, int st) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_tag)::value, LAST = decltype(last_tag)::value;
    constexpr int G = decltype(g_tag)::value;
    const int nx = stage == (kSqStages - 1) * kSqStage ? 0 : stage + kSqStage;
    h4 sbv[TN], sav;
    if constexpr (TOKEN) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        chan_last[j] = chan[j];
        chan[j] = round_here((float)__builtin_bit_cast(_Float16, (unsigned short)(G ? raw_b[j] >> 16 : raw_b[j])));
      }
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) sbv[j] = rank1(G ? raw_b[j] >> 16 : raw_b[j] & 0xFFFFu);
      sav = rank1(G ? raw_a >> 16 : raw_a & 0xFFFFu);
    }
    v4i a_op, b_op[TN];
    static_for<8>([&](auto s_tag) {
      constexpr int s = decltype(s_tag)::value, u = s >> 2, h = (s >> 1) & 1, t = s & 1;
      if constexpr (G == 1 && s == 4) {                // the next stage is there, and nobody reads this one any more
        advance();
        if (FIRST && stored) wait_vmcnt<kBehind + kStores>();
        else wait_vmcnt<kBehind>();
        wait_lgkmcnt0();
        barrier_no_fence();
        if (!(st & 3)) {
          if (2 * st + 8 < KT) sc_issue(tile_of<BN, OUT, BM>(p, die_first + at), (st >> 2) + 1);
          else if (at + die_wgs < die_count) sc_issue(tile_of<BN, OUT, BM>(p, die_first + at + die_wgs), 0);
          else ++sblk;
        }
        if constexpr (!LAST) issue(stage);
      }
      constexpr std::integral_constant<int, h> H{};
      if constexpr (t == 0) {
        a_op = nibbles(H, raw[G][TN][u]);
#pragma unroll
        for (int j = 0; j < TN; ++j) b_op[j] = nibbles(H, raw[G][j][u]);
      }
      if constexpr (!TOKEN && s == 0) {                // the products of the group before's second tile
        if constexpr (!(FIRST && G == 0)) prod[1] = __builtin_amdgcn_mfma_f32_32x32x8f16(a_last, b_last, zero, 0, 0, 0);
      }
      sums[G][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_op, b_op[t], s < 2 ? zero_i : sums[G][t], 0, 0, 0);
      if constexpr (!(FIRST && G == 0))
        fold(std::integral_constant<int, u>{}, std::integral_constant<int, 1 - G>{}, std::integral_constant<int, 4 * (s & 3)>{},
             chan_last[u]);
      if constexpr (!TOKEN && s == 4) prod[0] = __builtin_amdgcn_mfma_f32_32x32x8f16(sav, sbv[0], zero, 0, 0, 0);
      if constexpr (G == 0) {
        if constexpr (s == 0) read_raw(I1, I2, stage);
        if constexpr (s == 1) read_raw(I1, I0, stage);
        if constexpr (s == 2) read_raw(I1, I1, stage);
      } else {
        if constexpr (s == kReadAt) read_raw(I0, I2, nx);
        if constexpr (s == kReadAt + 1) read_raw(I0, I0, nx);
        if constexpr (s == kReadAt + 2) read_raw(I0, I1, nx);
        if constexpr (s == 7) read_scales(LAST ? 0 : 2 * st + 2, (sblk - (LAST || !((2 * st + 2) & 7) ? 1 : 2)) & 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (!TOKEN) a_last = sav, b_last = sbv[1];
    if constexpr (G == 1) prev = stage, stage = nx;
  };

  read_raw(I0, I0, 0), read_raw(I0, I1, 0), read_raw(I0, I2, 0);
  read_scales(0, 0);
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  for (;;) {
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) res[t][r] = 0.f;
    if constexpr (TOKEN) parked = p.As[min(tile_of<BN, OUT, BM>(p, die_first + at).m0 + (tid & (BM - 1)), p.M - 1)];
    group(yes, no, I0, 0);
    group(yes, no, I1, 0);
    if constexpr (TOKEN) ((__half*)sc_a)[tid & (BM - 1)] = parked;   // (read in the epilogue, many barriers later)
    for (int st = 1; st < ST - 1; ++st) {
      group(no, no, I0, st);
      group(no, no, I1, st);
    }
    group(no, yes, I0, ST - 1);
    group(no, yes, I1, ST - 1);
    if constexpr (!TOKEN) prod[1] = __builtin_amdgcn_mfma_f32_32x32x8f16(a_last, b_last, zero, 0, 0, 0);
    static_for<8>([&](auto s_tag) {
      constexpr int s = decltype(s_tag)::value;
      fold(std::integral_constant<int, (s >> 2)>{}, I1, std::integral_constant<int, 4 * (s & 3)>{}, chan[s >> 2]);
    });

    // ---- outputs, 16 rows at a time through the block of the stage just multiplied that this same wave refills.  Lane: channel
    // fr of a 32 x 32 tile, tokens 8 g + 4 fc + 0..3 in register quad g.
    const Tile cur = tile_of<BN, OUT, BM>(p, die_first + at);
    uint8_t* const ep = lds + prev + wave * kSqBlock;
    static_assert(16 * kHalfPitch <= kSqBlock, "staging tile");
    static_for<2>([&](auto c_tag) {
      constexpr int g0 = decltype(c_tag)::value * 2;
#pragma unroll
      for (int g = g0; g < g0 + 2; ++g) {
        h4 sa4 = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
        if constexpr (TOKEN) sa4 = *(const h4*)((const __half*)sc_a + wm + 8 * g + 4 * fc);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float f = res[j][4 * g + e] * (TOKEN ? (float)sa4[e] * (1.f / 256.f) : 1.f / 256.f);
            *(_Float16*)(ep + (8 * (g - g0) + 4 * fc + e) * kHalfPitch + (j * 32 + fr) * 2) = (_Float16)round_here(f);
          }
      }
      store_half_rows<16, OUT>(p, cur, ep, cur.m0 + wm + g0 * 8, wcol, lane);
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

template <int EPI, int OUT>
int launch_square(GemmArgs a, hipStream_t stream) {
  constexpr int BNC = OUT == kSwiglu ? kSqTile / 2 : kSqTile;
  constexpr size_t LDS = kSqStages * kSqStage + 2 * kSqTile * 16 + (EPI == kGroupScale ? 2 * kSqTile * 16 : kSqTile * 2);
  a.tiles_m = (a.M + kSqTile - 1) / kSqTile;
  a.tiles_n = (a.N + BNC - 1) / BNC;
  for (int s = 1; s < a.n_seg; ++s) {
    a.seg_tile0[s] = a.tiles_n;
    a.tiles_n += (a.seg_N[s] + kSqTile - 1) / kSqTile;
  }
  a.group_m = a.tiles_m < 4 ? a.tiles_m : 4;
  auto kern = gemm_i4_square_kernel<EPI, OUT>;
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)kern, LDS, grant, "gemm")) return rc;
  const long tiles = (long)a.tiles_m * a.tiles_n;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles < 256 ? tiles : 256)), dim3(512), LDS, stream, a);
  return check_launch("gemm");
}

template <int OUT>
int launch_square(const GemmArgs& a, hipStream_t stream) {
  return a.a_cols == 1 ? launch_square<kTokenGroup, OUT>(a, stream) : launch_square<kGroupScale, OUT>(a, stream);
}

}  // namespace

// What the kernel takes: group-scaled weights in groups of 128, an even number of groups of which a last block of eight leaves the
// next tile's scales time to arrive, scale rows of whole dwords, output rows of whole 16-byte stores.
bool gemm_square_takes(const GemmArgs& a) {
  const int kt = a.K >> 7;
  if (a.K % 256 || kt < 8 || (kt % 8 && kt % 8 < 6) || a.b_cols != kt || (a.a_cols != 1 && a.a_cols != kt) || a.N % 8) return false;
  auto off4 = [](const void* q) { return ((uintptr_t)q & 3) != 0; };
  if (off4(a.As) || off4(a.Bs) || off4(a.Bs2)) return false;
  long n = a.N;
  for (int s = 1; s < a.n_seg; ++s) {
    if (a.seg_N[s] % 8 || off4(a.seg_Bs[s])) return false;
    n += a.seg_N[s];
  }
  return (uint64_t)(a.M > n ? a.M : n) * kt < (1ull << 31);
}

int gemm_square_dispatch(const GemmArgs& a, SquareOut out, hipStream_t stream) {
  switch (out) {
    case kSquareSwiglu: return launch_square<kSwiglu>(a, stream);
    case kSquareRope: return launch_square<kRope>(a, stream);
    default: return a.R ? launch_square<kResidual>(a, stream) : launch_square<kPlain>(a, stream);
  }
}

}  // namespace flh
