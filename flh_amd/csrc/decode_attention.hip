// Attention of ONE new token per sequence over a preallocated fp16 key / value cache (the decode step), with grouped
// queries: out[b, h] = softmax(q[b, h] . K[b, h / rep]^T * scale) V[b, h / rep] over the first kv_len cache slots.
//
// Stands where the reference calls the flash-attn package (flh/quantized_model/modeling_llama.py:449-460,
// _flash_attention_forward on the cached keys / values); the stock fused attention kernels are built for long query
// blocks and take ~80 us for this shape, the same arithmetic as separate tensor operations ~30 us in five launches.
// Here the cached positions are split into chunks, one workgroup per (sequence, key / value head, chunk): scores and
// probabilities in float32, a partial (maximum, sum, weighted values) per chunk goes to a scratch buffer, and a second
// small kernel combines the chunks' partials -- two launches, every key and value read once, all query heads of a
// key / value head served by the same read.
#include <atomic>

#include "group_codes.h"
#include "lane_ops.h"

namespace flh {
namespace {

constexpr int kAttnThreads = 256;

// partial of one (sequence, kv head, chunk): REP heads x (D weighted values, maximum, sum) as float
template <int D>
constexpr int partial_floats(int rep) { return rep * (D + 2); }

// One value of the rotary embedding with the roundings of the tensor expression x * cos + rotate_half(x) * sin evaluated
// op by op in fp16 (the same as the stand-alone kernel, rope_cache.hip): `first_half` says whether x sits in the first
// half of the head vector (its partner xp then enters negated).
__device__ __forceinline__ _Float16 rope_value(_Float16 x, _Float16 xp, _Float16 c, _Float16 s, bool first_half) {
  const _Float16 a = (_Float16)round_here((float)x * (float)c);
  const _Float16 r = (_Float16)round_here((first_half ? -1.f : 1.f) * (float)xp * (float)s);
  return (_Float16)round_here((float)a + (float)r);
}

// ROPE: the step's new token comes in un-rotated -- q, and k_new / v_new [B, Hkv, D] -- together with the cos / sin row of
// its position and the cache slot `positions[0]` it takes (the same for every sequence).  The queries are rotated while
// they are loaded; the workgroup whose chunk holds the slot rotates the new key, uses it and the new value in place of
// what the cache holds there, and writes both into the cache.  One launch less in front of attention, and the same
// bytes in the cache as the stand-alone rotary / cache kernel writes -- also for a slot in kv_len .. max_len - 1, which
// attention does not read: the first workgroup of every (sequence, key / value head) writes it there, as the
// stand-alone kernel would.
//
// Values pass the caches by (16 x 32 / 8 heads x 4096 64.2 -> 62.6 us, 12 x 32 / 8 x 2048 31.3 -> 30.5).  With one query per
// key the keys do as well, and both are requested before anything else.  us with the combine launch, replayed over caches that
// together don't fit the last-level one, otherwise -> so, sequences x heads / key-value heads x positions: 5 x 32 / 32 x 777
// 18.7 -> 17.3, 8 x 32 / 32 x 2048 54.6 -> 49.6, 16 x 32 / 32 x 777 44.8 -> 42.1;  grouped queries the same up to two chunks
// per compute unit (4 x 32 / 8 x 1024 10.3 -> 10.5) and slower beyond (16 x 32 / 8 x 777 17.3 -> 18.7, 8 x 32 / 4 x 3000 21.2
// -> 24.2).  Inside a decode step there is less in it: 5 x 32 / 32 x 777 14.7 -> 14.4 for the kernel.
template <int D, int REP, int CHUNK, bool ROPE>
__global__ __launch_bounds__(kAttnThreads) void decode_attention_partial_kernel(
    const __half* __restrict__ q, __half* k_cache, __half* v_cache, float* __restrict__ partials, uint32_t Hkv,
    uint32_t kv_len, uint32_t max_len, uint32_t splits, float scale, const __half* __restrict__ k_new,
    const __half* __restrict__ v_new, const __half* __restrict__ cos, const __half* __restrict__ sin,
    const long long* __restrict__ positions) {
  static_assert(D == 128 || D == 64, "head dimension");
  static_assert(CHUNK == 64, "one key per lane in the softmax step");
  constexpr bool AHEAD = REP == 1;
  static_assert(REP <= 16, "the heads of a key / value head are the columns of one matrix tile");
  constexpr int KS = D / 32;                           // matrix steps over the channels
  constexpr int RPW = CHUNK / (kAttnThreads / 64);     // keys / value rows per wave: 16
  __shared__ __align__(16) _Float16 qs[REP * D];       // the query heads
  __shared__ float sc[REP][CHUNK];                     // scores, then probabilities
  // the new token's rotated key, later the waves' weighted values
  __shared__ __align__(16) float red[kAttnThreads / 64][REP * D];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // One or two queries per key: the chunks of one place in all the caches next to each other, whose strides are often a power
  // of two; more (more work per chunk, fewer caches): the chunks of a cache.  us, chunks of a cache -> of one place: 8 x 32 /
  // 32 x 2048 52.5 -> 46.1, 16 x 32 / 32 x 2048 101 -> 91, 8 x 32 / 32 x 1024 29.4 -> 26.2, 5 x 32 / 32 x 777 16.8 -> 16.8;
  // two queries per key go either way: 12 x 32 / 16 x 1024 27.6 -> 26.7, 8 x 32 / 16 x 2048 33.9 -> 32.9, 4 x 32 / 16 x 2048
  // 21.7 -> 22.3, 2 x 32 / 16 x 2048 14.4 -> 16.1;  four: 4 x 32 / 8 x 2048 14.7 -> 17.2
  const uint32_t caches = gridDim.x / splits;
  const uint32_t split = REP <= 2 ? blockIdx.x / caches : blockIdx.x % splits;
  const uint32_t bh = REP <= 2 ? blockIdx.x % caches : blockIdx.x / splits;   // b * Hkv + kvh
  const uint32_t t0 = split * CHUNK;
  const uint32_t n_live = kv_len > t0 ? min((uint32_t)CHUNK, kv_len - t0) : 0u;
  const uint32_t last = n_live ? n_live - 1 : 0;       // rows past the live range read the last live one again (any valid address)

  // Scores on the matrix cores: wave w owns the keys 16 w .. 16 w + 15 as the rows of a 16 x 16 tile whose columns are
  // the query heads; a lane holds eight consecutive channels (block `kb` of the step's 32) of key row `krow`.
  // Values: wave w takes rows 16 w .. 16 w + 15 of the chunk, a lane one channel pair (one channel for D = 64) of each.
  const int krow = lane & 15, kb = lane >> 4;
  typedef std::conditional_t<D == 128, unsigned, unsigned short> raw_t;
  h8 ka[KS];
  raw_t vr[RPW];
  __half* const vbase = v_cache + ((size_t)bh * max_len + t0) * D;
  auto request = [&]() __attribute__((always_inline)) {
    const __half* kr = k_cache + ((size_t)bh * max_len + t0 + min((uint32_t)(wave * RPW + krow), last)) * D + kb * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const v4i* src = (const v4i*)(kr + ks * 32);
      ka[ks] = __builtin_bit_cast(h8, AHEAD ? __builtin_nontemporal_load(src) : *src);
    }
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const raw_t* src = (const raw_t*)(vbase + (size_t)min((uint32_t)(wave * RPW + i), last) * D) + lane;
      vr[i] = __builtin_nontemporal_load(src);
    }
    if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (AHEAD) request();
  uint32_t slot = 0xFFFFFFFFu;                         // cache slot of the new token (ROPE), if it is inside kv_len
  if constexpr (ROPE) {
    const long long pos = positions[0];
    if (pos >= 0 && pos < (long long)kv_len) slot = (uint32_t)pos;
    if (pos >= (long long)kv_len && pos < (long long)max_len && split == 0 && wave == 0) {
      // a slot attention does not read: written, not used
      const _Float16 *kn = (const _Float16*)k_new + (size_t)bh * D, *vn = (const _Float16*)v_new + (size_t)bh * D;
      const _Float16 *cf = (const _Float16*)cos, *sf = (const _Float16*)sin;
      _Float16* kd = (_Float16*)k_cache + ((size_t)bh * max_len + (size_t)pos) * D;
      _Float16* vd = (_Float16*)v_cache + ((size_t)bh * max_len + (size_t)pos) * D;
      for (int c = lane; c < D; c += 64) {
        kd[c] = rope_value(kn[c], kn[c ^ (D / 2)], cf[c], sf[c], c < D / 2);
        vd[c] = vn[c];
      }
    }
  }
  const _Float16* qf = (const _Float16*)q + (size_t)bh * REP * D;   // q [B, Hq, D]: the REP heads of this kv head are adjacent
  for (int i = tid; i < REP * D; i += kAttnThreads) {
    if constexpr (ROPE) {
      const _Float16 *cf = (const _Float16*)cos, *sf = (const _Float16*)sin;
      const int d = i % D;
      qs[i] = rope_value(qf[i], qf[i ^ (D / 2)], cf[d], sf[d], d < D / 2);
    } else {
      qs[i] = qf[i];
    }
  }
  // The new token's chunk: its key is rotated like the queries, by all threads through LDS (in its lanes' registers, next to the
  // requested keys and values, it took 70 registers and with them the eighth wave of a SIMD, most of all where a launch just fits
  // one round of eight: 16 x 32 / 4 heads x 2048 28.1 -> 24.4 us, 8 x 32 / 8 x 2048 23.3 -> 20.8, 16 x 32 / 8 x 2048 37.5 -> 33.9).
  _Float16* const new_key = (_Float16*)red[0];
  const bool fresh_chunk = ROPE && slot - t0 < (uint32_t)CHUNK;
  if (fresh_chunk) {
    const _Float16 *kn = (const _Float16*)k_new + (size_t)bh * D, *cf = (const _Float16*)cos, *sf = (const _Float16*)sin;
    for (int c = tid; c < D; c += kAttnThreads) new_key[c] = rope_value(kn[c], kn[c ^ (D / 2)], cf[c], sf[c], c < D / 2);
  }
  if constexpr (!AHEAD) request();
  __syncthreads();                                     // the queries, and the new key, are in LDS
  if (fresh_chunk && (slot - t0) / RPW == (uint32_t)wave) {
    // the new token's wave: key and value take the place of what the cache held, here and there
    const uint32_t r = (slot - t0) % RPW;
    if ((uint32_t)krow == r) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        ka[ks] = *(const h8*)(new_key + ks * 32 + kb * 8);
        *(h8*)(k_cache + ((size_t)bh * max_len + slot) * D + ks * 32 + kb * 8) = ka[ks];
      }
    }
    const raw_t fresh = ((const raw_t*)(v_new + (size_t)bh * D))[lane];
    ((raw_t*)(vbase + (size_t)(slot - t0) * D))[lane] = fresh;
#pragma unroll
    for (int i = 0; i < RPW; ++i)
      if ((uint32_t)i == r) vr[i] = fresh;
  }
  {
    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      h8 qb = {0, 0, 0, 0, 0, 0, 0, 0};
      if (krow < REP) qb = *(const h8*)(qs + krow * D + ks * 32 + kb * 8);   // column `krow` of the tile: head krow
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[ks], qb, acc, 0, 0, 0);
    }
    // acc[i]: key 16 w + 4 kb + i, head krow
    if (krow < REP) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t key = wave * RPW + 4 * kb + i;
        sc[krow][key] = t0 + key < kv_len ? acc[i] * scale : -INFINITY;
      }
    }
  }
  __syncthreads();

  // softmax pieces of this chunk, head h by wave h (REP > 4: two heads per wave)
  float* out = partials + ((size_t)bh * splits + split) * partial_floats<D>(REP);
  for (int h = wave; h < REP; h += kAttnThreads / 64) {
    const float s = sc[h][lane];
    const float m = wave_max(s);
    const float p = m == -INFINITY ? 0.f : __expf(s - m);      // a chunk wholly past kv_len: nothing
    const float l = wave_sum(p);
    sc[h][lane] = p;
    if (lane == 0) {
      out[h * (D + 2) + D] = m;
      out[h * (D + 2) + D + 1] = l;
    }
  }
  __syncthreads();
  // weighted values: every wave its own rows for all heads, then the four waves' sums in a fixed order (rows past the live
  // range as zeros: their probability is zero, but 0 x NaN is not)
  float vv0[RPW], vv1[D == 128 ? RPW : 1];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const bool have = (uint32_t)(wave * RPW + i) < n_live;
    if constexpr (D == 128) {
      const h2 v = __builtin_bit_cast(h2, vr[i]);
      vv0[i] = have ? (float)v[0] : 0.f;
      vv1[i] = have ? (float)v[1] : 0.f;
    } else {
      vv0[i] = have ? (float)__builtin_bit_cast(_Float16, vr[i]) : 0.f;
    }
  }
#pragma unroll
  for (int h = 0; h < REP; ++h) {
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int i = 0; i < RPW; ++i) {                    // probabilities past kv_len are zero, their values were not loaded
      const float p = sc[h][wave * RPW + i];
      a0 = __builtin_fmaf(p, vv0[i], a0);
      if constexpr (D == 128) a1 = __builtin_fmaf(p, vv1[i], a1);
    }
    if constexpr (D == 128) *(v2f*)(&red[wave][h * D + 2 * lane]) = v2f{a0, a1};
    else red[wave][h * D + lane] = a0;
  }
  __syncthreads();
  for (int i = tid; i < REP * D; i += kAttnThreads)
    out[(i / D) * (D + 2) + i % D] = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
}

// one workgroup of four waves per (sequence, query head): the chunks' partials -> fp16 output.  Every wave reads all
// maxima and sums (lane s: chunk s, 64 chunks per pass; two wave reductions) and accumulates the weighted values of
// every fourth chunk with the chunk's weight read from its lane; the four waves' sums meet in LDS.
// QUANT (heads of 128 channels): the head is a group of the quantiser that follows, so its codes and scale leave instead, the
// bytes of the group quantiser on the fp16 output: a launch of 4.6 us less in a decode step's layer.
template <int D, bool QUANT = false>
__global__ __launch_bounds__(256) void decode_attention_combine_kernel(const float* __restrict__ partials,
                                                                       __half* __restrict__ out, uint32_t rep,
                                                                       uint32_t splits, uint8_t* __restrict__ codes,
                                                                       __half* __restrict__ scales) {
  static_assert(!QUANT || D == 128, "a head is a group");
  __shared__ float acc[4][2][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t bhq = blockIdx.x;                     // b * Hq + hq
  const uint32_t bh = bhq / rep, h = bhq % rep;
  const float* base = partials + (size_t)bh * splits * (rep * (D + 2)) + h * (D + 2);
  const size_t stride = (size_t)rep * (D + 2);
  float m = -INFINITY;
  for (uint32_t s0 = 0; s0 < splits; s0 += 64)
    if (s0 + lane < splits) m = __builtin_fmaxf(m, base[(s0 + lane) * stride + D]);
  m = wave_max(m);
  float l = 0.f, a0 = 0.f, a1 = 0.f;
  for (uint32_t s0 = 0; s0 < splits; s0 += 64) {
    float w = 0.f;
    if (s0 + lane < splits) {
      const float ms = base[(s0 + lane) * stride + D];
      w = ms == -INFINITY ? 0.f : __expf(ms - m);
      l = __builtin_fmaf(w, base[(s0 + lane) * stride + D + 1], l);
    }
    const uint32_t n = min(64u, splits - s0);
#pragma unroll 4
    for (uint32_t i = wave; i < n; i += 4) {
      const float wi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), (int)i));
      if constexpr (D == 128) {
        const v2f v = *(const v2f*)(base + (s0 + i) * stride + 2 * lane);
        a0 = __builtin_fmaf(wi, v[0], a0);
        a1 = __builtin_fmaf(wi, v[1], a1);
      } else {
        a0 = __builtin_fmaf(wi, base[(s0 + i) * stride + lane], a0);
      }
    }
  }
  l = wave_sum(l);
  acc[wave][0][lane] = a0;
  acc[wave][1][lane] = a1;
  __syncthreads();
  if (wave != 0) return;
  a0 = (acc[0][0][lane] + acc[1][0][lane]) + (acc[2][0][lane] + acc[3][0][lane]);
  a1 = (acc[0][1][lane] + acc[1][1][lane]) + (acc[2][1][lane] + acc[3][1][lane]);
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  if constexpr (D == 128) {
    const h2 r = {(_Float16)(a0 * inv), (_Float16)(a1 * inv)};
    if constexpr (QUANT) {
      const unsigned y = __builtin_bit_cast(unsigned, r);
      const h2 mag = __builtin_bit_cast(h2, y & 0x7FFF7FFFu);
      float m = __builtin_fmaxf((float)mag[0], (float)mag[1]);
      m = __builtin_fmaxf(m, lane_xor_f<16>(m));
      m = __builtin_fmaxf(m, lane_xor_f<32>(m));
      const GroupScale s = group_scale<16>(m);             // (and over the sixteen lanes of a row)
      // four adjacent lanes hold the eight values of a dword of codes
      const unsigned y0 = dpp_i<0x00>(y), y1 = dpp_i<0x55>(y), y2 = dpp_i<0xAA>(y), y3 = dpp_i<0xFF>(y);
      const h2 hb = {(_Float16)65504.0f, (_Float16)65504.0f};
      const unsigned w = s.careful ? nibbles8<true>(y0, y1, y2, y3, s.r, hb) : nibbles8<false>(y0, y1, y2, y3, s.r, hb);
      if ((lane & 3) == 0) *(unsigned*)(codes + (size_t)bhq * (D / 2) + lane) = w;
      if (lane == 0) scales[bhq] = __builtin_bit_cast(__half, s.s);
    } else {
      *(h2*)(out + (size_t)bhq * D + 2 * lane) = r;
    }
  } else {
    out[(size_t)bhq * D + lane] = __float2half(a0 * inv);
  }
}

constexpr int kChunk = 64;

// where the result goes: fp16, or (heads of 128) int4 codes and a scale per head
struct AttentionOut {
  __half* out;
  uint8_t* codes;
  __half* scales;
};

// the new token's inputs of the variant with the rotary embedding and the cache write inside (all null without it)
struct NewToken {
  const __half *k, *v, *cos, *sin;
  const long long* positions;
};

template <int D, int REP>
int launch_attention(const __half* q, __half* k, __half* v, const AttentionOut& out, float* partials, uint32_t B, uint32_t Hkv,
                     uint32_t kv_len, uint32_t max_len, float scale, const NewToken& nt, hipStream_t stream) {
  const uint32_t splits = (kv_len + kChunk - 1) / kChunk;
  const dim3 grid(B * Hkv * splits), block(kAttnThreads);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, block, 0, stream, q, k, v, partials, Hkv, kv_len, max_len, splits, scale, nt.k, nt.v, nt.cos, nt.sin,
                       nt.positions);
  };
  if (nt.k) go(decode_attention_partial_kernel<D, REP, kChunk, true>);
  else go(decode_attention_partial_kernel<D, REP, kChunk, false>);
  if (int rc = check_launch("decode_attention (partials)")) return rc;
  auto combine = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(B * Hkv * REP), dim3(256), 0, stream, partials, out.out, (uint32_t)REP, splits, out.codes, out.scales);
  };
  if constexpr (D == 128)
    if (out.codes) {
      combine(decode_attention_combine_kernel<D, true>);
      return check_launch("decode_attention (combine)");
    }
  combine(decode_attention_combine_kernel<D>);
  return check_launch("decode_attention (combine)");
}

}  // namespace
}  // namespace flh

using namespace flh;

extern "C" size_t flh_decode_attention_workspace_bytes(uint32_t B, uint32_t Hq, uint32_t head_dim, uint32_t kv_len) {
  const size_t splits = ((size_t)kv_len + kChunk - 1) / kChunk;
  return (size_t)B * Hq * splits * (head_dim + 2) * sizeof(float);
}

namespace {
int decode_attention_checked(const flh_half* q, flh_half* k_cache, flh_half* v_cache, const AttentionOut& out, uint32_t B, uint32_t Hq,
                             uint32_t Hkv, uint32_t head_dim, uint32_t kv_len, uint32_t max_len, float scale,
                             void* workspace, size_t workspace_bytes, const NewToken& nt, void* stream) {
  if (!q || !k_cache || !v_cache || !(out.out || (out.codes && out.scales))) return fail(FLH_EINVAL, "decode_attention: null pointer");
  if (misaligned16(q, k_cache, v_cache, out.out, out.codes)) return fail(FLH_EINVAL, "decode_attention: tensors must be 16-byte aligned");
  if (head_dim != 128 && head_dim != 64) return fail(FLH_EINVAL, "decode_attention: head_dim (%u) must be 64 or 128", head_dim);
  if (Hkv == 0 || Hq % Hkv) return fail(FLH_EINVAL, "decode_attention: %u query heads do not divide over %u key / value heads", Hq, Hkv);
  const uint32_t rep = Hq / Hkv;
  if (rep != 1 && rep != 2 && rep != 4 && rep != 8)
    return fail(FLH_EINVAL, "decode_attention: %u query heads per key / value head (1, 2, 4 or 8 supported)", rep);
  if (kv_len == 0 || kv_len > max_len) return fail(FLH_EINVAL, "decode_attention: kv_len (%u) must be in 1 .. max_len (%u)", kv_len, max_len);
  if (B == 0) return FLH_OK;
  const size_t need = flh_decode_attention_workspace_bytes(B, Hq, head_dim, kv_len);
  if (!workspace || ((uintptr_t)workspace & 15)) return fail(FLH_EINVAL, "decode_attention: a 16-byte aligned workspace is required");
  if (workspace_bytes < need)
    return fail(FLH_EINVAL, "decode_attention: the workspace has %zu bytes, this call needs %zu", workspace_bytes, need);
  if ((uint64_t)B * Hkv * ((kv_len + kChunk - 1) / kChunk) > 0x7FFFFFFFull) return fail(FLH_EINVAL, "decode_attention: too many chunks");
  const __half* qh = (const __half*)q;
  __half *kh = (__half*)k_cache, *vh = (__half*)v_cache;
  float* ws = (float*)workspace;
  hipStream_t st = (hipStream_t)stream;
#define FLH_ATTN(D, R) return launch_attention<D, R>(qh, kh, vh, out, ws, B, Hkv, kv_len, max_len, scale, nt, st)
  if (head_dim == 128) {
    switch (rep) {
      case 1: FLH_ATTN(128, 1);
      case 2: FLH_ATTN(128, 2);
      case 4: FLH_ATTN(128, 4);
      default: FLH_ATTN(128, 8);
    }
  }
  switch (rep) {
    case 1: FLH_ATTN(64, 1);
    case 2: FLH_ATTN(64, 2);
    case 4: FLH_ATTN(64, 4);
    default: FLH_ATTN(64, 8);
  }
#undef FLH_ATTN
}
}  // namespace

extern "C" int flh_decode_attention_f16(const flh_half* q, const flh_half* k_cache, const flh_half* v_cache, flh_half* out,
                                        uint32_t B, uint32_t Hq, uint32_t Hkv, uint32_t head_dim, uint32_t kv_len,
                                        uint32_t max_len, float scale, void* workspace, size_t workspace_bytes,
                                        void* stream) {
  // (without a new token the kernel only reads the caches)
  return decode_attention_checked(q, (flh_half*)k_cache, (flh_half*)v_cache, AttentionOut{(__half*)out, nullptr, nullptr}, B, Hq, Hkv, head_dim, kv_len, max_len, scale,
                                  workspace, workspace_bytes, NewToken{nullptr, nullptr, nullptr, nullptr, nullptr}, stream);
}

namespace {
int decode_attention_rope_checked(const flh_half* q, const flh_half* k_new, const flh_half* v_new, const flh_half* cos, const flh_half* sin,
                                  const int64_t* positions, flh_half* k_cache, flh_half* v_cache, const AttentionOut& out, uint32_t B,
                                  uint32_t Hq, uint32_t Hkv, uint32_t head_dim, uint32_t kv_len, uint32_t max_len, float scale,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  if (!k_new || !v_new || !cos || !sin || !positions) return fail(FLH_EINVAL, "decode_attention (rotary): null pointer");
  if (misaligned16(k_new, v_new, cos, sin)) return fail(FLH_EINVAL, "decode_attention (rotary): tensors must be 16-byte aligned");
  return decode_attention_checked(q, k_cache, v_cache, out, B, Hq, Hkv, head_dim, kv_len, max_len, scale, workspace, workspace_bytes,
                                  NewToken{(const __half*)k_new, (const __half*)v_new, (const __half*)cos, (const __half*)sin,
                                           (const long long*)positions}, stream);
}
}  // namespace

extern "C" int flh_decode_attention_rope_f16(const flh_half* q, const flh_half* k_new, const flh_half* v_new,
                                             const flh_half* cos, const flh_half* sin, const int64_t* positions,
                                             flh_half* k_cache, flh_half* v_cache, flh_half* out, uint32_t B, uint32_t Hq,
                                             uint32_t Hkv, uint32_t head_dim, uint32_t kv_len, uint32_t max_len, float scale,
                                             void* workspace, size_t workspace_bytes, void* stream) {
  return decode_attention_rope_checked(q, k_new, v_new, cos, sin, positions, k_cache, v_cache, AttentionOut{(__half*)out, nullptr, nullptr},
                                       B, Hq, Hkv, head_dim, kv_len, max_len, scale, workspace, workspace_bytes, stream);
}

extern "C" int flh_decode_attention_rope_group_quant_i4(const flh_half* q, const flh_half* k_new, const flh_half* v_new,
                                                        const flh_half* cos, const flh_half* sin, const int64_t* positions,
                                                        flh_half* k_cache, flh_half* v_cache, uint8_t* q_packed, flh_half* scales,
                                                        uint32_t B, uint32_t Hq, uint32_t Hkv, uint32_t head_dim, uint32_t kv_len,
                                                        uint32_t max_len, float scale, void* workspace, size_t workspace_bytes,
                                                        void* stream) {
  if (head_dim != 128) return fail(FLH_EINVAL, "decode_attention (quantised): head_dim (%u) must be 128, the group of the quantiser", head_dim);
  return decode_attention_rope_checked(q, k_new, v_new, cos, sin, positions, k_cache, v_cache,
                                       AttentionOut{nullptr, q_packed, (__half*)scales}, B, Hq, Hkv, head_dim, kv_len, max_len, scale,
                                       workspace, workspace_bytes, stream);
}

// ---- the same for callers that cannot allocate ---------------------------------------------------------------------
// The partials live in a static device array of a fixed size instead of a caller's workspace.  Every device the library
// runs on holds its own copy of the array until the process ends; the address of the current device's copy is looked
// up once per device.  Calls on one device share that array: calls that overlap in time (different streams) race.
constexpr size_t kScratchBytes = 16u << 20;            // 16 MiB: e.g. 31 sequences x 32 query heads x 2048 positions, d = 128
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
std::atomic<void*> g_scratch_ptr[kMaxDevices];         // per device: where that device's copy of `scratch` lives

int scratch_of_current_device(void** out) {
  int dev = 0;
  if (int rc = current_device(&dev, "decode_attention")) return rc;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));   // of the current device
    if (e != hipSuccess || !ptr)
      return fail(FLH_ELAUNCH, "decode_attention: cannot locate the static scratch array: %s", hipGetErrorString(e));
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return FLH_OK;
}
}  // namespace

extern "C" size_t flh_decode_attention_static_scratch_bytes(void) { return kScratchBytes; }

extern "C" int flh_decode_attention_f16_static(const flh_half* q, const flh_half* k_cache, const flh_half* v_cache,
                                               flh_half* out, uint32_t B, uint32_t Hq, uint32_t Hkv, uint32_t head_dim,
                                               uint32_t kv_len, uint32_t max_len, float scale, void* stream) {
  const size_t need = flh_decode_attention_workspace_bytes(B, Hq, head_dim, kv_len);
  if (need > kScratchBytes)
    return fail(FLH_EINVAL, "decode_attention (static scratch): this call needs %zu bytes of scratch, the static array has "
                "%zu; use flh_decode_attention_f16 with a workspace", need, kScratchBytes);
  void* ptr = nullptr;
  if (int e = scratch_of_current_device(&ptr)) return e;
  // every chunk's partial is written before the combine kernel reads it: nothing has to start at zero
  return flh_decode_attention_f16(q, k_cache, v_cache, out, B, Hq, Hkv, head_dim, kv_len, max_len, scale, ptr,
                                  kScratchBytes, stream);
}
