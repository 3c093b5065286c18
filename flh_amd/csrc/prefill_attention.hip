// Causal attention of a block of new tokens over a key / value cache (prefill), fp16 with float32 softmax and
// accumulation, heads of 128 channels, grouped queries: what the reference's attention module hands to flash-attn
// after the rotary embedding and the cache update (flh/quantized_model/modeling_llama.py:426-460).  Inputs in the
// layouts the q / k / v GEMM of this library writes: queries token-major [B, T, Hq, 128], keys / values in cache slots
// [B, Hkv, max_len, 128]; query t of the block sees the slots 0 .. past + t.  Output token-major [B, T, Hq * 128], the
// layout the quantiser of o_proj reads.
//
// One workgroup = 4 waves = 128 consecutive queries of one head, 32 per wave; keys in blocks of 64, K and V tiles
// double-buffered in LDS by direct-to-LDS loads (row-major, 16-byte chunks XOR-swizzled by the row; the V tile has a
// swizzle of its own for the transpose loads).  Both products run
// on v_mfma_f32_32x32x16_f16 in transposed form, so that a lane owns one query throughout:
//
//   S^T[key, query] = sum_d K[key, d] Q[query, d]         A = K tile rows from LDS, B = the wave's queries (registers)
//   O^T[d, query]  += sum_key V[key, d] P[query, key]     A = V^T fragments, B = P^T as it sits in the S^T accumulators
//
// The S^T accumulator of lane (query n, half h) holds keys 8 g + 4 h + e (g, e in 0..3) of a 32-key tile, which as B
// operand of the second product means contraction slot 8 h + 4 g' + e <-> key 16 s + 8 g' + 4 h + e for step s; the V^T
// fragment is read to match with the LDS transpose load of this part (ds_read_b64_tr_b16: within 16 lanes, lane i
// receives element i % 4 of the 8-byte rows addressed by lanes i / 4 + 4 j, j = 0..3), i.e. four consecutive keys for
// the lane's channel straight from the row-major tile.  Online softmax in base 2 per lane; only the running maximum is
// exchanged between the two lanes of a query per key block.
//
// Sixteen fragments of four registers serve both products: while the scores' MFMAs use up the step's K, V is read into the
// registers they leave, and the next step's K while the second product uses up V; the second half of the exponentials sits
// between MFMAs too.  A wave waits for LDS only at the step's one barrier.
// What bounds it: power on long launches (8192 tokens of 32 heads: 1.8 GHz, where the form that read fragments right before
// use ran at 2.0, and took 15 % more clocks per step; MFMAs alone take 364 us at 1.8 GHz, the fragment reads add 59, the loads 57, the
// exponentials 36), clocks on short ones.  us before -> now: 1 x 8192 tokens 602 -> 597, 1 x 4096 of 8 key / value heads 181 -> 171,
// 1 x 2048 54 -> 49.4, 2 x 1500 behind 100 82 -> 76, 1 x 1000 behind 531 36.7 -> 31.8, 1 x 513 15.3 -> 13.5, 8 x 512 37.5 -> 36.5.
// Not taken: a running maximum that may lag behind by 8 powers of two, 3-6 % faster (fewer rescaled steps) but with the largest
// probabilities rounded instead of 1 (largest error at 1000 behind 531 9.7e-5 -> 1.6e-4); raised wave priority around the MFMAs: nothing.
#include <atomic>

#include "lane_ops.h"

namespace flh {

namespace {

constexpr int kHeadDim = 128;
constexpr int kQueriesPerBlock = 128;                  // 32 per wave
constexpr int kKeysPerStep = 64;
constexpr int kTileBytes = kKeysPerStep * kHeadDim * 2;   // one K or V tile in LDS (16 KiB)
constexpr int kOutPitch = kHeadDim * 2 + 16;           // bytes per query row of the output staging tile

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s4 lds_s4;

// byte offset inside a tile of the 16-byte chunk `c` (8 channels) of key row `r`
__device__ __forceinline__ int chunk_at(int r, int c) { return r * (kHeadDim * 2) + ((c ^ (r & 15)) << 4); }
// the same for a V tile, whose swizzle serves the transpose loads: one of them reads 64 bytes (four chunks) of each of
// four consecutive rows, which must fall into four different quarters of the 256-byte bank line
__device__ __forceinline__ int v_swizzle(int r) { return (r & 3) << 2; }
__device__ __forceinline__ int v_chunk_at(int r, int c) { return r * (kHeadDim * 2) + ((c ^ v_swizzle(r)) << 4); }

// 1 KiB: lane i's 16 bytes at voff go to lds_base + 16 i
__device__ __forceinline__ void load_rows_to_lds(const v4i& d, unsigned voff, unsigned lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds_base), "v"(voff), "s"(d) : "memory", "m0");
}
// the same four times, 1 KiB further in memory and in LDS each
__device__ __forceinline__ void load_four_rows_to_lds(const v4i& d, unsigned voff, unsigned lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen offset:1024 lds\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen offset:2048 lds\n\t"
               "buffer_load_dwordx4 %1, %2, 0 offen offset:3072 lds" ::"s"(lds_base), "v"(voff), "s"(d) : "memory", "m0");
}

__global__ __launch_bounds__(256, 2) void prefill_attention_kernel(const __half* __restrict__ q,
                                                                   const __half* __restrict__ k_cache,
                                                                   const __half* __restrict__ v_cache,
                                                                   __half* __restrict__ out, int T, int Hq, int Hkv,
                                                                   int past, int max_len, float scale_log2) {
  extern __shared__ __align__(1024) uint8_t lds[];     // K[2], V[2] tiles; the output staging tile afterwards
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // workgroup -> (sequence, head, query block): every die takes a contiguous range of (sequence, head) pairs, so the
  // keys / values of a head (of a group of heads that share them) are fetched into one L2 only; within a head the long
  // blocks (late queries) come first
  const int n_blocks = (T + kQueriesPerBlock - 1) / kQueriesPerBlock;
  const unsigned L = xcd_contiguous(blockIdx.x, gridDim.x);
  const int head = (int)((L / n_blocks) % Hq), b = (int)(L / ((unsigned)n_blocks * Hq));
  // a die's 32 compute units take its workgroups in order, two each: every other row of 32 workgroups walks its heads'
  // blocks in the opposite direction, so that a compute unit's two residents are a long and a short block
  // (heads of 32 blocks or more fill whole rows: they keep the long blocks first)
  const bool ascending = n_blocks < 32 && (((L / n_blocks) / (32 / n_blocks)) & 1);
  const int qb = ascending ? (int)(L % n_blocks) : n_blocks - 1 - (int)(L % n_blocks);
  const int hkv = head / (Hq / Hkv);
  const int q_first = qb * kQueriesPerBlock + wave * 32;
  const int my_q = min(q_first + n, T - 1);            // rows past the end repeat the last query; never stored

  // this lane's query as B operand: channels 16 s + 8 h .. + 7
  h8 qf[8];
  {
    const __half* qrow = q + ((size_t)((size_t)b * T + my_q) * Hq + head) * kHeadDim;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *(const h8*)(qrow + 16 * s + 8 * h);
  }

  const int total_keys = past + T;
  const int block_keys = min(past + (qb + 1) * kQueriesPerBlock, total_keys);   // slots any query of the block sees
  const int n_steps = (block_keys + kKeysPerStep - 1) / kKeysPerStep;
  // steps with a key that some query of this wave sees, and whether the last of them has one in its second tile of 32
  const int wave_limit = past + min(q_first + 31, T - 1);
  const int live_steps = __builtin_amdgcn_readfirstlane(q_first < T ? wave_limit / kKeysPerStep + 1 : 0);
  const bool half_step = __builtin_amdgcn_readfirstlane(wave_limit % kKeysPerStep < 32);
  const size_t cache = ((size_t)b * Hkv + hkv) * (size_t)max_len * kHeadDim;
  const unsigned lds0 = (unsigned)(size_t)lds;

  // one load instruction moves four key rows (1 KiB); a wave issues four for K and four for V per step.  The descriptors
  // cover what is left of a step's 64 rows: rows past the end arrive as zeros
  unsigned k_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = (wave * 4 + i) * 4 + (lane >> 4);
    k_off[i] = (unsigned)(r * kHeadDim + ((lane & 15) ^ (r & 15)) * 8) * 2;
  }
  const unsigned v_off = (unsigned)((wave * 16 + (lane >> 4)) * kHeadDim + ((lane & 15) ^ v_swizzle(lane >> 4)) * 8) * 2;
  const uint8_t *k_next = (const uint8_t*)(k_cache + cache), *v_next = (const uint8_t*)(v_cache + cache);   // the steps requested next
  int k_left = total_keys, v_left = total_keys;        // keys from there on
  auto rows_left = [](int keys) { return (unsigned)__builtin_amdgcn_readfirstlane(max(0, min(keys, kKeysPerStep)) * (kHeadDim * 2)); };
  auto issue_k = [&](int buf) {
    const v4i d = buffer_of(k_next, rows_left(k_left));
#pragma unroll
    for (int i = 0; i < 4; ++i) load_rows_to_lds(d, k_off[i], lds0 + buf * kTileBytes + (wave * 4 + i) * 1024);
    k_next += kTileBytes, k_left -= kKeysPerStep;
  };
  auto issue_v = [&](int buf) {
    load_four_rows_to_lds(buffer_of(v_next, rows_left(v_left)), v_off, lds0 + (2 + buf) * kTileBytes + wave * 4096);
    v_next += kTileBytes, v_left -= kKeysPerStep;
  };

  v16f o[4];                                           // O^T: [channel tile], lane = query, register r = channel 8 (r/4) + 4 h + r % 4
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;                // running maximum (scaled, base 2) and this lane's share of the sum
  const int q_limit = past + my_q;                     // last visible slot of this lane's query

  // K fragment 2 s + kt of a step: rows 32 kt + n, channels 16 s + 8 h .. + 7 (chunk 2 s + h; s enters the swizzled address by XOR)
  const int k_at = chunk_at(n, h);
  // per-lane offsets of the V^T transpose loads: lane i of a group of 16 addresses the 8-byte piece (i % 4) of the
  // 32-byte run of channels the group's sixteen lanes will own, in key row i / 4 of the four keys of one load
  const int grp = lane >> 4, gi = lane & 15;
  const int tr_key = gi >> 2;                          // + key0 of the load
  const int tr_half = (gi & 1) << 3;                   // byte inside the 16-byte chunk
  const int tr_chunk0 = ((grp & 1) << 1) + ((gi & 3) >> 1);   // + 4 dt: chunk of 8 channels inside the row
  // the lane's part of a transpose-load address for channel tile dt (the key rows of a load add a constant to it)
  int tr_off[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) tr_off[dt] = v_chunk_at(4 * (grp >> 1) + tr_key, 4 * dt + tr_chunk0) + tr_half;

  h8 f[16];                                            // the fragments of one operand: K's during the scores, V's afterwards
  auto read_k = [&](auto j_, int buf, int at) {
    constexpr int j = decltype(j_)::value;
    f[j] = *(const h8*)(lds + buf * kTileBytes + (at ^ ((j >> 1) << 5)) + (j & 1) * (32 * kHeadDim * 2));
  };
  // V fragment 4 (2 kt + ks) + dt: this half-wave's slots 8 h .. 8 h + 7 are keys 32 kt + 16 ks + 4 h + {0..3} and + 8 + {0..3}
  // (rows 32 kt + 16 ks and + 8 on: multiples of four, which the V swizzle does not see)
  auto read_v = [&](auto j_, int buf) {
    constexpr int j = decltype(j_)::value;
    const uint8_t* at = lds + (2 + buf) * kTileBytes + tr_off[j & 3] + (j >> 2) * (16 * kHeadDim * 2);
    const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)at);
    const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(at + 8 * (kHeadDim * 2)));
    f[j] = __builtin_bit_cast(h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // Step `step` with K and V of it in the buffers of parity P
  auto run = [&](auto p_, int step) {
    constexpr int P = decltype(p_)::value;
    wait_vmcnt<0>();
    __syncthreads();   // V of this step and K of the next are complete; everybody has read the buffers refilled here
    issue_k(P);
    issue_v(P ^ 1);
    if (step >= live_steps) return;
    // ---- S^T = K Q^T for two tiles of 32 keys; every fragment's registers take one of V's
    v16f st[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 16; ++r) st[kt][r] = 0.f;
    __builtin_amdgcn_sched_barrier(0);
    static_for<16>([&](auto j_) {
      constexpr int j = decltype(j_)::value;
      st[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[j], qf[j >> 1], st[j & 1], 0, 0, 0);
      read_v(j_, P);
      __builtin_amdgcn_sched_barrier(0);
    });
    // ---- causal mask, online softmax in base 2 on scale_log2 * s (register r of tile kt: key = 64 step + 32 kt +
    // 8 (r/4) + 4 h + r % 4)
    const int key0 = step * kKeysPerStep + 4 * h;
    if (step * kKeysPerStep + kKeysPerStep - 1 > past + q_first) {   // (a branch of its own: most steps carry no mask arithmetic at all;
      asm volatile("" ::: "memory");                   //  the empty statement keeps the compiler from predicating it)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (key0 + 32 * kt + 8 * (r >> 2) + (r & 3) > q_limit) st[kt][r] = -INFINITY;
    }
    __builtin_amdgcn_sched_barrier(0);
    float mx[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      mx[c] = fmaxf(st[c >> 1][8 * (c & 1)], st[c >> 1][8 * (c & 1) + 1]);
#pragma unroll
      for (int r = 2; r < 8; ++r) mx[c] = fmaxf(mx[c], st[c >> 1][8 * (c & 1) + r]);
    }
    float top = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]));
    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_int(top), __float_as_int(top), false, false);
    top = fmaxf(__int_as_float(halves[0]), __int_as_float(halves[1])) * scale_log2;   // (the scale is positive: the maximum commutes with it)
    const float m_new = fmaxf(m_run, top);             // finite from the first step on: slot 0 is visible to every query
    // rescale what has been accumulated -- unless no lane's maximum moved (the common case after the first steps)
    if (__builtin_amdgcn_ballot_w64(m_new != m_run) != 0) {
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      m_run = m_new;
    }
    float sum = 0.f;
    h8 pb[2][2];                                       // P^T as B operand: [tile][step of 16 slots]
    auto two = [&](auto kt_, auto i_) {                // probabilities 2 i and 2 i + 1 of a tile
      constexpr int kt = decltype(kt_)::value, i = decltype(i_)::value;
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[kt][2 * i], scale_log2, -m_run));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[kt][2 * i + 1], scale_log2, -m_run));
      sum += p0, sum += p1;
      pb[kt][i >> 2][(2 * i) & 7] = (_Float16)p0, pb[kt][i >> 2][(2 * i + 1) & 7] = (_Float16)p1;
    };
    static_for<8>([&](auto i_) { two(std::integral_constant<int, 0>{}, i_); });
    __builtin_amdgcn_sched_barrier(0);
    // ---- O^T += V^T P^T, a tile's MFMAs between the next tile's exponentials; every fragment's registers take one of the next step's K
    int k_now = k_at;
    asm("" : "+v"(k_now));                             // (eight addresses kept across the steps are registers there are not)
    const bool half = half_step && step + 1 == live_steps;
    static_for<8>([&](auto j_) {
      constexpr int j = decltype(j_)::value;
      o[j & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[j], pb[0][j >> 2], o[j & 3], 0, 0, 0);
      read_k(j_, P ^ 1, k_now);
      two(std::integral_constant<int, 1>{}, j_);
      __builtin_amdgcn_sched_barrier(0);
    });
    l_run += sum;
    if (half) return;                                  // (the wave's last step, whose second tile it does not see)
    static_for<8>([&](auto j_) {
      constexpr int j = decltype(j_)::value + 8;
      o[j & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[j], pb[1][(j >> 2) & 1], o[j & 3], 0, 0, 0);
      read_k(std::integral_constant<int, j>{}, P ^ 1, k_now);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  issue_k(0);
  issue_v(0);
  issue_k(1);
  wait_vmcnt<8>();                                     // K of step 0
  barrier_no_fence();
  static_for<16>([&](auto j_) { read_k(j_, 0, k_at); });
  for (int step = 0; step < n_steps; step += 2) {
    run(std::integral_constant<int, 0>{}, step);
    if (step + 1 < n_steps) run(std::integral_constant<int, 1>{}, step + 1);
  }
  wait_vmcnt<0>();                                     // (zeros requested past the last step must not land in the staging tiles)

  // ---- normalise, transpose through LDS, store whole rows
  const float l_all = l_run + lane_xor_f<32>(l_run);
  const float inv = 1.0f / l_all;
  __syncthreads();                                     // every wave is done with the tiles
  uint8_t* stage = lds + wave * (32 * kOutPitch);
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      h4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (_Float16)(o[dt][4 * g + e] * inv);
      *(h4*)(stage + n * kOutPitch + (32 * dt + 8 * g + 4 * h) * 2) = v;
    }
  // (the staging tile is private to the wave: a wave-level wait is enough)
  __builtin_amdgcn_s_waitcnt(0xc07f);                  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int row = it * 4 + (lane >> 4), c = lane & 15;
    const int tq = q_first + row;
    const v4i v = *(const v4i*)(stage + row * kOutPitch + c * 16);
    if (tq < T) *(v4i*)(out + ((size_t)((size_t)b * T + tq) * Hq + head) * kHeadDim + c * 8) = v;
  }
}

}  // namespace

}  // namespace flh

using namespace flh;

extern "C" int flh_prefill_attention_f16(const flh_half* q, const flh_half* k_cache, const flh_half* v_cache, flh_half* out,
                                         uint32_t B, uint32_t T, uint32_t Hq, uint32_t Hkv, uint32_t head_dim, uint32_t past,
                                         uint32_t max_len, float scale, void* stream) {
  if (!q || !k_cache || !v_cache || !out) return fail(FLH_EINVAL, "prefill_attention: null pointer");
  if (misaligned16(q, k_cache, v_cache, out)) return fail(FLH_EINVAL, "prefill_attention: tensors must be 16-byte aligned");
  if (head_dim != kHeadDim) return fail(FLH_EINVAL, "prefill_attention: head_dim (%u) must be 128", head_dim);
  if (Hq == 0 || Hkv == 0 || Hq % Hkv) return fail(FLH_EINVAL, "prefill_attention: %u query heads do not divide into %u key / value heads", Hq, Hkv);
  if ((uint64_t)past + T > max_len) return fail(FLH_EINVAL, "prefill_attention: past (%u) + T (%u) exceeds the cache length %u", past, T, max_len);
  if (B == 0 || T == 0) return FLH_OK;
  if ((uint64_t)B * Hq * ((T + kQueriesPerBlock - 1) / kQueriesPerBlock) > 0x7FFFFFFFull || (uint64_t)B * T * Hq * kHeadDim > (1ull << 40) || (uint64_t)B * Hkv * max_len * kHeadDim > (1ull << 40) ||
      (uint64_t)past + T > (1u << 30))
    return fail(FLH_EINVAL, "prefill_attention: problem too large");
  if (!(scale > 0.f)) return fail(FLH_EINVAL, "prefill_attention: the scale must be positive");
  const size_t smem = 4 * (size_t)kTileBytes;          // 64 KiB: two workgroups per compute unit
  static_assert(4 * 32 * kOutPitch <= 4 * kTileBytes, "the output staging tiles reuse the K / V buffers");
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)prefill_attention_kernel, smem, grant, "prefill_attention")) return rc;
  const unsigned blocks = (T + kQueriesPerBlock - 1) / kQueriesPerBlock;
  hipLaunchKernelGGL(prefill_attention_kernel, dim3(blocks * Hq * B), dim3(256), smem, (hipStream_t)stream, (const __half*)q,
                     (const __half*)k_cache, (const __half*)v_cache, (__half*)out, (int)T, (int)Hq, (int)Hkv, (int)past,
                     (int)max_len, scale * 1.4426950408889634f);
  return check_launch("prefill_attention");
}
