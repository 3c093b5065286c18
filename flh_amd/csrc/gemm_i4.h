// Shared declarations of the int4 GEMM translation units.
#pragma once
#include <atomic>

#include "common.h"

namespace flh {

// kTokenGroup: group-scaled weights with one activation scale per token, applied after the groups
enum Epilogue { kRowScale = 0, kGroupScale = 1, kInt32 = 2, kTokenGroup = 3 };

constexpr int kMaxGemmSegments = 4;

// tile / K-split override of the shape heuristics (0 = automatic), set by flh_gemm_set_tuning
extern std::atomic<int> g_tune_tile, g_tune_ks;

struct GemmArgs {
  const uint8_t* A;     // [M, K/2] packed activations
  const uint8_t* B;     // [N, K/2] packed weights
  const __half* As;     // [M, a_cols]
  const __half* Bs;     // [N, b_cols]
  void* D;              // [M, N] fp16 (int32 for kInt32)
  int M, N, K;          // K in codes
  int a_cols, b_cols;   // scale columns (1 or K/group)
  int tiles_m, tiles_n, group_m;
  // Further weight matrices that share A (q / k / v, gate / up): segment s > 0 starts at output-column tile
  // seg_tile0[s] of the launch and has its own B, scales, output and N; segment 0 is B / Bs / D / N above.
  int n_seg;            // 0 or 1: a single weight matrix
  int seg_tile0[kMaxGemmSegments];
  int seg_N[kMaxGemmSegments];
  const uint8_t* seg_B[kMaxGemmSegments];
  const __half* seg_Bs[kMaxGemmSegments];
  void* seg_D[kMaxGemmSegments];
  // SwiGLU launches (gate = B / Bs, up = B2 / Bs2, N = channels of each, D [M, N] = fp16(fp16(silu(gate)) * up))
  const uint8_t* B2;
  const __half* Bs2;
  // q / k / v launches with the rotary embedding and the cache write in the epilogue (three segments q, k, v of heads of
  // 128 channels; row m = b * rope_T + t): q -> D [M, N] rotated; k -> seg_D[1] = key cache [B, rope_hkv, rope_max_len,
  // 128] at slot rope_pos[t], rotated; v -> seg_D[2] = value cache, as it is.  cos / sin [rope_T, 128].
  const __half* rope_cos;
  const __half* rope_sin;
  const long long* rope_pos;
  int rope_T, rope_max_len, rope_hkv;
  // residual (single weight matrix, fp16 output): D = fp16(R + fp16(the launch's result)), R [M, N]; may be D itself
  const __half* R;
};

// fp16(fp16(x cos) + fp16(rotate_half(x) sin)) of one channel pair (c, c + 64), as rope_cache.hip rounds it
__device__ __forceinline__ void rope_pair(_Float16& x1, _Float16& x2, _Float16 c1, _Float16 c2, _Float16 s1, _Float16 s2) {
  const _Float16 a1 = (_Float16)round_here((float)x1 * (float)c1), r1 = (_Float16)round_here(-1.f * (float)x2 * (float)s1);
  const _Float16 a2 = (_Float16)round_here((float)x2 * (float)c2), r2 = (_Float16)round_here(1.f * (float)x1 * (float)s2);
  x1 = (_Float16)round_here((float)a1 + (float)r1);
  x2 = (_Float16)round_here((float)a2 + (float)r2);
}

// product of element H (0 / 1) of two fp16 pairs, exact in float32
template <int H>
__device__ __forceinline__ float mul_halves(unsigned a, unsigned b) {
  float d;
  if constexpr (H == 0) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,1,0]" : "=v"(d) : "v"(a), "v"(b));
  else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(d) : "v"(a), "v"(b));
  return d;
}
// fma(v, element H of the fp16 pair s, acc)
template <int H>
__device__ __forceinline__ float fma_half(float v, unsigned s, float acc) {
  float d;
  if constexpr (H == 0) asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,1,0]" : "=v"(d) : "v"(v), "v"(s), "v"(acc));
  else asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(d) : "v"(v), "v"(s), "v"(acc));
  return d;
}

// Small-M (decode) kernels: weight-streaming, split over K inside a workgroup.
constexpr int kDecodeMaxM = 64;
bool gemm_dot_supports(const GemmArgs& a, int epi, int group);        // up to four tokens
int gemm_dot_dispatch(const GemmArgs& a, int epi, hipStream_t stream);
bool gemm_lines_supports(const GemmArgs& a, int epi);      // (within gemm_decode_dispatch)
bool gemm_lines_over_stream(const GemmArgs& a, int epi);
bool gemm_decode_supports(const GemmArgs& a, int epi, int group);
int gemm_decode_dispatch(const GemmArgs& a, int epi, hipStream_t stream);

// Between decoding and prefill: small tiles over the whole of K (gemm_i4_stream.hip).
bool gemm_stream_supports(const GemmArgs& a, int epi, int group);
int gemm_stream_dispatch(const GemmArgs& a, int epi, hipStream_t stream);
bool gemm_stream_rope_supports(const GemmArgs& a, int epi);
int gemm_stream_rope_dispatch(const GemmArgs& a, hipStream_t stream);

// 128 x 128 tiles of eight waves for group-scaled weights (gemm_i4_square.hip).
enum SquareOut { kSquarePlain = 0, kSquareSwiglu = 1, kSquareRope = 2 };
bool gemm_square_takes(const GemmArgs& a);
int gemm_square_dispatch(const GemmArgs& a, SquareOut out, hipStream_t stream);

}  // namespace flh
