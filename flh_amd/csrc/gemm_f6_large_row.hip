// One scale per row and channel: the large-tile kernel of gemm_f6_large.h.
#include "gemm_f6_large.h"

namespace flh {
namespace f6l {
namespace {

template <int WM>
struct Shape {
  static constexpr int WN = 128, BM = 256, WAVES_N = WM == 128 ? 2 : 1, BN = WN * WAVES_N;
  static constexpr int BLK = (BM + BN) / 32, STAGES = WM == 128 ? 3 : 4, STAGE = BLK * kRowBlock;
  static constexpr int NI = BLK * 3 / 4;              // load instructions per wave and stage
  static constexpr int SC_B = BN * 2, SC_A = BM * 2;  // behind the ring: the tile's scales
  static constexpr int LDS = STAGES * STAGE + SC_B + SC_A;
  static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
};

// A value of an accumulator where it is used and not before: left to itself, the compiler fetches most of the 256
// accumulation registers of a 128 x 128 wave tile ahead of the branches of the epilogue, and spills.  The compiler does not see
// that the instruction reads a matrix result and inserts no wait states for it: at least 18 cycles have to lie between the last
// MFMA into a register and this read.  They do: the first value read is of acc[0][0], 15 MFMAs (of 8 passes or more) and the scale
// product's MFMAs after its last one, and the last MFMA, into acc[3][0], is followed by three quarters of the epilogue.
template <bool IN_AGPR>
__device__ __forceinline__ float accumulator(float v) {
  if constexpr (IN_AGPR) {
    float r;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(r) : "a"(v));
    return r;
  } else {
    return v;
  }
}

template <int WM, int OUT>
__global__ __launch_bounds__(256, 1) void gemm_f6_large_kernel(const GemmArgs p) {
  using S = Shape<WM>;
  constexpr int BM = S::BM, BN = S::BN, WN = S::WN, STAGES = S::STAGES, STAGE = S::STAGE, NI = S::NI;
  constexpr int TM = WM / 32, TN = WN / 32, ABLK = BM / 32;
  constexpr int NF = TM + TN;
  extern __shared__ __align__(1024) uint8_t lds[];    // [STAGES][STAGE], weight scales, activation scales
  uint8_t* const sc_b = lds + STAGES * STAGE;
  uint8_t* const sc_a = sc_b + S::SC_B;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned lds0 = (unsigned)(size_t)lds;
  const int wcol = wave % S::WAVES_N;
  const int wm = (wave / S::WAVES_N) * WM, wn = wcol * WN;
  const int fr = lane & 31, fc = lane >> 5;

  // tiles of this workgroup: every die (workgroup i runs on die i % 8) owns a contiguous range of the launch's tiles and
  // its workgroups take them in turn, so that at any time a die works on neighbouring tiles
  const unsigned total = p.tiles_m * p.tiles_n;
  const unsigned xcd = blockIdx.x % kNumXCD, slot = blockIdx.x / kNumXCD;
  const unsigned per = total / kNumXCD, rem = total % kNumXCD;
  const unsigned die_first = xcd * per + (xcd < rem ? xcd : rem), die_count = per + (xcd < rem ? 1 : 0);
  const unsigned die_wgs = (gridDim.x - xcd + kNumXCD - 1) / kNumXCD;
  unsigned at = slot;                                  // tile of the range being multiplied
  if (at >= die_count) return;
  const int KT = p.K / 128;

  // ---- operand loads.  A wave requests NB row blocks of 32 rows per stage, a third of one (1 KiB) per instruction; lane ->
  // 16-byte chunk as in the ring of gemm_f6.hip (chunk c of row r in slot 6 r + (c ^ ((r >> 3) & 1)): sixteen rows read
  // at one chunk are free of bank conflicts).  A block is a wave-uniform pointer plus one of three lane offsets; past
  // the last row of a matrix the offset is held inside it (those rows' results are never stored).
  constexpr int NB = NI / 3;
  unsigned loff[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int s = q * 64 + lane, r = s / 6;
    loff[q] = (unsigned)r * kBlock + ((s % 6) ^ ((r >> 3) & 1)) * 16;
  }
  const uint8_t* lp[NB];                               // block b's slab of the step to be requested next
  unsigned lim[NB];                                    // last 16-byte chunk inside the matrix, from there
  unsigned b_step = 0;
  int kld = 0;                                         // index of that step inside its tile
  auto set_loads = [&](const Tile& t) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int blk = wave * NB + b, wb = blk - ABLK;
      const bool isA = blk < ABLK, up = OUT == kSwiglu && (wb & 3) >= 2;
      // SwiGLU: a wave column's 128 weight rows are 64 gate rows and the same 64 up rows
      const int first = isA ? t.m0 + blk * 32 : t.n0 + (OUT == kSwiglu ? (wb >> 2) * 64 + (wb & 1) * 32 : wb * 32);
      const int all = isA ? p.M : t.N, rows = all - first;   // rows of the matrix, and from the block's first on
      lp[b] = wave_uniform((isA ? p.A : up ? t.B2 : t.B) + (rows > 0 ? (size_t)first * kBlock : 0));
      lim[b] = (unsigned)min(rows > 0 ? rows : all, 32) * kBlock - 16;
    }
    b_step = (unsigned)t.N * kBlock;
    kld = 0;
  };
  // (the step is added to a pointer that starts one step early, so that the common case has no branch of its own)
  auto step_of = [&](int b) { return wave * NB + b < ABLK ? (unsigned)p.M * kBlock : b_step; };
  auto issue = [&](int stage, auto i_tag) __attribute__((always_inline)) {
    constexpr int b = decltype(i_tag)::value / 3, q = decltype(i_tag)::value % 3;
    load_to_lds16(lp[b], min(loff[q], lim[b]), lds0 + stage * STAGE + (wave * NB + b) * kRowBlock + q * 1024);
  };
  // the step after the one just requested; past a tile's last one the next tile's first (past the last tile: the same
  // slab again, which nobody reads -- the number of outstanding loads stays what the waits below count on)
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

  // ---- fragments: 24 bytes per lane and MFMA, as 16 + 8 (first 64 codes of a step) and 8 + 16 (second) bytes
  const int sw = (fr >> 3) & 1;
  const int c0 = ((3 * fc) ^ sw) * 16, c1 = ((3 * fc + 1) ^ sw) * 16, c2 = ((3 * fc + 2) ^ sw) * 16;
  const int a_base = (wm / 32) * kRowBlock + fr * kBlock, b_base = (ABLK + wn / 32) * kRowBlock + fr * kBlock;
  const int ao[4] = {a_base + c0, a_base + c1, a_base + c1 + 8, a_base + c2};
  const int bo[4] = {b_base + c0, b_base + c1, b_base + c1 + 8, b_base + c2};
  v4i f4[2][NF];
  v2i f2[2][NF];
  // piece r of the 2 NF reads of half m: fragments in the order in which the MFMAs below need them first
  auto read_piece = [&](auto m_tag, auto r_tag, int stage) __attribute__((always_inline)) {
    constexpr int m = decltype(m_tag)::value, r = decltype(r_tag)::value, o = r / 2;
    constexpr int f = o == 0 ? 0 : o <= TN ? TM + o - 1 : o - TN;   // A0, B0 .. B(TN-1), A1 ..
    const uint8_t* st = lds + stage * STAGE + (f < TM ? f : f - TM) * kRowBlock;
    const int* off = f < TM ? ao : bo;
    if constexpr (r % 2 == 0) f4[m][f] = *(const v4i*)(st + off[m == 0 ? 0 : 3]);
    else f2[m][f] = *(const v2i*)(st + off[m == 0 ? 1 : 2]);
  };
  auto operand = [&](int m, int f) __attribute__((always_inline)) {
    const v4i a = f4[m][f];
    const v2i b = f2[m][f];
    return m == 0 ? v8i{a[0], a[1], a[2], a[3], b[0], b[1], 0, 0} : v8i{b[0], b[1], a[0], a[1], a[2], a[3], 0, 0};
  };
  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};

  v16f acc[TM][TN];

  // ---- scales
  // One per row and channel: read in a tile's first step, parked in LDS after it.
  constexpr int PARK = (BM + BN + 255) / 256;
  __half parked[PARK];
  auto park_load = [&]() __attribute__((always_inline)) {
    const Tile cur = tile_of<BN, OUT>(p, die_first + at);
#pragma unroll
    for (int i = 0; i < PARK; ++i) {
      const int e = tid + i * 256;
      if (e < BM) {
        parked[i] = p.As[min(cur.m0 + e, p.M - 1)];
      } else if (e < BM + BN) {
        const int r = e - BM, b = r >> 5;
        const int n = cur.n0 + (OUT == kSwiglu ? (b >> 2) * 64 + (b & 1) * 32 + (r & 31) : r);
        parked[i] = (OUT == kSwiglu && (b & 3) >= 2 ? cur.Bs2 : cur.Bs)[min(n, cur.N - 1)];
      }
    }
  };
  auto park_store = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PARK; ++i) {
      const int e = tid + i * 256;
      if (e < BM) ((__half*)sc_a)[e] = parked[i];
      else if (e < BM + BN) ((__half*)sc_b)[e - BM] = parked[i];
    }
  };

  // ---- prologue
  constexpr int SPLIT = NI / 2;                        // loads of a stage issued in the second half of a step, the rest follow
  int stage = 0;
  set_loads(tile_of<BN, OUT>(p, die_first + at));
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) {
    static_for<NI>([&](auto i) { issue(s, i); });
    advance();
  }
  static_for<SPLIT>([&](auto i) { issue(STAGES - 1, i); });
  wait_vmcnt<(STAGES - 2) * NI + SPLIT>();
  __syncthreads();
  constexpr int NM = TM * TN;                          // MFMAs of half a step
  // Outstanding vector-memory operations a wave may have when it needs its part of the next stage: the stages behind
  // that one, and in the first step of a tile also the stores of the tile before (kStores of them are certain).
  constexpr int kBehind = (STAGES - 2) * NI, kStores = TM * (OUT == kSwiglu ? 4 : 8);
  bool stored = false;                                 // a whole tile's stores went out right before this tile

  const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int prev = STAGES - 1;                               // slot of the stage before `stage`
  // one step of K; FIRST: a tile's first (its sums start at zero), LAST: its last (the slot is refilled after the outputs)
  auto k_step = [&](auto first_tag, auto last_tag, int kt) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_tag)::value, LAST = decltype(last_tag)::value;
    const int nx = stage + 1 == STAGES ? 0 : stage + 1;
    // Between two MFMAs (32 clocks of the matrix pipe each) go a fragment read or two and now and then a load: issued in
    // bunches they would take longer than the MFMA in front of them.
    // first half: multiplies the first 64 codes, reads the second 64
    static_for<NM>([&](auto n_tag) {
      constexpr int n = decltype(n_tag)::value, i = n / TN, j = i & 1 ? TN - 1 - n % TN : n % TN;
      static_for<2 * NF>([&](auto r) {
        if constexpr (decltype(r)::value * NM / (2 * NF) == n) read_piece(I1, r, stage);
      });
      static_for<NI - SPLIT>([&](auto l) {
        constexpr int li = SPLIT + decltype(l)::value;
        if constexpr (decltype(l)::value * NM / (NI - SPLIT) == n) issue(prev, std::integral_constant<int, li>{});
      });
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(operand(0, TM + j), operand(0, i),
                                                                 FIRST ? zero : acc[i][j], kBf6, kBf6, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    advance();
    // every wave's part of the next stage has landed, and nobody reads this one any more
    if (FIRST && stored) wait_vmcnt<kBehind + kStores>();
    else wait_vmcnt<kBehind>();
    wait_lgkmcnt0();
    barrier_no_fence();
    // second half: multiplies the second 64 codes, reads the next step's first 64, refills this stage's slot
    static_for<NM>([&](auto n_tag) {
      constexpr int n = decltype(n_tag)::value, i = n / TN, j = i & 1 ? TN - 1 - n % TN : n % TN;
      static_for<2 * NF>([&](auto r) {
        if constexpr (decltype(r)::value * NM / (2 * NF) == n) read_piece(I0, r, nx);
      });
      static_for<SPLIT>([&](auto l) {
        if constexpr (!LAST && decltype(l)::value * NM / SPLIT == n) issue(stage, l);
      });
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(operand(1, TM + j), operand(1, i), acc[i][j], kBf6, kBf6,
                                                                 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    prev = stage;
    stage = nx;
  };
  static_for<2 * NF>([&](auto r) { read_piece(I0, r, 0); });
  for (;;) {
    park_load();
    k_step(std::true_type{}, std::false_type{}, 0);
    park_store();                                      // (read in the epilogue, many barriers later)
    for (int kt = 1; kt < KT - 1; ++kt) k_step(std::false_type{}, std::false_type{}, kt);
    k_step(std::false_type{}, std::true_type{}, KT - 1);

    // ---- outputs.  Lane: token fr of a 32 x 32 tile, channels 8 g + 4 fc + 0..3 in register quad g.
    // The scale products a * b of a 32 x 32 tile are an outer product: one fp16 MFMA with a single non-zero K element
    // gives all of them in the accumulators' own layout, exact in float32, instead of a conversion and a multiplication
    // per output on the vector ALU.
    const __half* la = (const __half*)sc_a + wm;
    const __half* lb = (const __half*)sc_b + wn;
    auto rank1 = [&](const __half* at_lds) __attribute__((always_inline)) {   // K element 0 of the lane's row / column
      const _Float16 v = *(const _Float16*)at_lds;
      return h4{fc == 0 ? v : (_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
    };
    h4 sb[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) sb[j] = rank1(lb + j * 32 + fr);
    auto product = [&](h4 sa, int j) __attribute__((always_inline)) {
      return __builtin_amdgcn_mfma_f32_32x32x8f16(sb[j], sa, zero, 0, 0, 0);
    };
    auto value = [&](int i, int j, int g, const v16f& ab) __attribute__((always_inline)) {
      h4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e)   // float(sum) * (a * b), rounded once to float32, then to fp16
        v[e] = (_Float16)round_here(accumulator<WM == 128>(acc[i][j][4 * g + e]) * ab[4 * g + e]);
      return v;
    };
    // One 32-row block at a time, the fp16 results go through LDS, so that whole 256-byte row segments are stored: into
    // the slot of the stage just multiplied, which is refilled after this, and there into the part that this same wave
    // refills -- no other wave is involved.
    const Tile cur = tile_of<BN, OUT>(p, die_first + at);
    uint8_t* const ep = lds + prev * STAGE + wave * NB * kRowBlock;
    {
      static_for<TM>([&](auto i_tag) {
        constexpr int i = decltype(i_tag)::value;
        const h4 sa = rank1(la + i * 32 + fr);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const v16f ab = product(sa, j);
#pragma unroll
          for (int g = 0; g < 4; ++g) *(h4*)(ep + fr * kPitch + (j * 32 + 8 * g + 4 * fc) * 2) = value(i, j, g, ab);
        }
        store_rows<32, OUT>(p, cur, ep, cur.m0 + wm + i * 32, wcol, lane);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    wait_lgkmcnt0();                                   // the staged rows have been read: the slot may be refilled
    static_for<SPLIT>([&](auto l) { issue(prev, l); });
    stored = OUT != kRope && cur.m0 + BM <= p.M && cur.n0 + (OUT == kSwiglu ? BN / 2 : BN) <= cur.N;
    at += die_wgs;
    if (at >= die_count) break;
  }
  wait_vmcnt<0>();                                     // the loads past the last tile land before the ring goes away
}

template <int WM, int OUT>
int launch_large(GemmArgs a, hipStream_t stream) {
  using S = Shape<WM>;
  constexpr int BNC = OUT == kSwiglu ? S::BN / 2 : S::BN;
  a.tiles_m = (a.M + S::BM - 1) / S::BM;
  a.tiles_n = (a.N + BNC - 1) / BNC;
  for (int s = 1; s < a.n_seg; ++s) {
    a.seg_tile0[s] = a.tiles_n;
    a.tiles_n += (a.seg_N[s] + S::BN - 1) / S::BN;
  }
  a.group_m = a.tiles_m < 4 ? a.tiles_m : 4;
  auto kern = gemm_f6_large_kernel<WM, OUT>;
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)kern, S::LDS, grant, "gemm_f6")) return rc;
  const long tiles = (long)a.tiles_m * a.tiles_n;
  const unsigned grid = (unsigned)(tiles < 256 ? tiles : 256);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), S::LDS, stream, a);
  return check_launch("gemm_f6");
}

}  // namespace

int launch_large_row(const GemmArgs& a, bool wide, Out out, hipStream_t stream) {
  switch (out) {
    case kSwiglu: return wide ? launch_large<128, kSwiglu>(a, stream) : launch_large<64, kSwiglu>(a, stream);
    case kRope: return wide ? launch_large<128, kRope>(a, stream) : launch_large<64, kRope>(a, stream);
    case kResidual: return wide ? launch_large<128, kResidual>(a, stream) : launch_large<64, kResidual>(a, stream);
    default: return wide ? launch_large<128, kPlain>(a, stream) : launch_large<64, kPlain>(a, stream);
  }
}

}  // namespace f6l
}  // namespace flh
