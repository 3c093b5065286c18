// fp16 linear for a handful of rows: y[m][n] = fp16(sum_k x[m][k] w[n][k]), float32 accumulation on the matrix cores -- the
// language-model head of a decode step (flh/quantized_model/modeling_llama.py:693), whose weights are the largest single read
// of a step.
//
// What bounds it: HBM.  A workgroup of four waves owns 64 output channels for the whole of K; 128 inputs of each (256 bytes,
// two whole cache lines) per stage go straight to LDS, three stages ahead, two workgroups to a compute unit: 96 KB in flight
// on each.  The weights are read once and marked non-temporal (a plain read of 1 GB runs at 6.4 TB/s here, a non-temporal one
// at 7.2); the tokens, shared by all, come from L2.  Every workgroup starts at its own place of K (and wraps around): rows are
// a power of two apart, and workgroups that walk along them together meet in a few memory channels.
// us, weights from HBM, against the vendor's product: 128256 x 4096, 1 / 16 rows 157 / 155 (6.8 TB/s) against 186 (in step
// from the start of K: 184), 32000 x 4096 43 / 41 against 56.
#include "gemm_i4.h"

namespace flh {
namespace {

typedef __attribute__((address_space(3))) uint8_t lds_byte;
typedef _Float16 h4 __attribute__((ext_vector_type(4)));

constexpr int kStages = 4, kRows = 64, kTokens = 16;   // channels per workgroup, tokens per tile
constexpr int kLineBytes = 256;                        // of a row per stage: 128 values
constexpr int kStage = (kRows + kTokens) * kLineBytes;
constexpr int kLoads = 5;                              // 1 KiB load instructions per wave and stage: 16 channels, 4 tokens

__global__ __launch_bounds__(256, 2) void linear_f16_kernel(const __half* __restrict__ x, const __half* __restrict__ w,
                                                            __half* __restrict__ y, int M, int N, int K) {
  extern __shared__ __align__(16) uint8_t lds[];
  lds_byte* ring = (lds_byte*)lds;
  const int lane = threadIdx.x & 63, r = lane & 15, c = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * kRows, stages = K >> 7;
  // a load instruction brings 256 bytes of four rows, chunk i of row q to slot i ^ (q % 16)
  const uint8_t* src[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = i < 4 ? wave * 16 + i * 4 + c : wave * 4 + c;
    src[i] = (const uint8_t*)(i < 4 ? w + (size_t)min(n0 + row, N - 1) * K : x + (size_t)min(row, M - 1) * K) +
             ((lane & 15) ^ (row & 15)) * 16;
  }
  const unsigned base = (unsigned)(uintptr_t)ring;
  // workgroups start at different places of K: rows are a power of two apart, at one place they would meet in a few channels
  const int turn = (int)((blockIdx.x / kNumXCD * 5 + blockIdx.x) % (unsigned)stages);
  auto request = [&](int s, int slot) {
    s = s + turn < stages ? s + turn : s + turn - stages;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const unsigned at = base + slot + (i < 4 ? wave * 16 + i * 4 : kRows + wave * 4) * kLineBytes;
      const void* q = src[i] + (size_t)s * kLineBytes;
      if (i < 4) load_to_lds16_nt(q, at);
      else load_to_lds16(q, at);
    }
  };
  int chunk[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) chunk[g] = r * kLineBytes + ((g * 4 + c) ^ r) * 16;

#pragma unroll
  for (int s = 0; s < kStages - 1; ++s)
    if (s < stages) request(s, s * kStage);
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  for (int s = 0; s < stages; ++s) {
    // stage s is there for every wave, and every wave has read stage s - 1: its slot takes stage s + 3
    if (s + kStages - 2 < stages) wait_vmcnt<(kStages - 2) * kLoads>();
    else wait_vmcnt<0>();
    wait_lgkmcnt0();
    barrier_no_fence();
    if (s + kStages - 1 < stages) request(s + kStages - 1, slot == 0 ? (kStages - 1) * kStage : slot - kStage);
    const lds_byte* st = ring + slot;
    h8 a[4], b[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      a[g] = *(const __attribute__((address_space(3))) h8*)(st + chunk[g] + wave * 16 * kLineBytes);
      b[g] = *(const __attribute__((address_space(3))) h8*)(st + chunk[g] + kRows * kLineBytes);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[g], b[g], acc, 0, 0, 0);
    slot = slot == (kStages - 1) * kStage ? 0 : slot + kStage;
  }
  // lane: token r, channels 4 c + e
  const int n = n0 + wave * 16 + 4 * c;
  if (r >= M || n >= N) return;
  __half* dst = y + (size_t)r * N + n;
  const h4 v = {(_Float16)acc[0], (_Float16)acc[1], (_Float16)acc[2], (_Float16)acc[3]};
  if (N % 4 == 0) {
    *(h4*)dst = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) ((_Float16*)dst)[e] = v[e];
  }
}

}  // namespace
}  // namespace flh

using namespace flh;

extern "C" int flh_linear_f16(const flh_half* x, const flh_half* w, flh_half* y, uint32_t M, uint32_t N, uint32_t K, void* stream) {
  if (!x || !w || !y) return fail(FLH_EINVAL, "linear_f16: null pointer");
  if (misaligned16(x, w, y)) return fail(FLH_EINVAL, "linear_f16: tensors must be 16-byte aligned");
  if (M > (uint32_t)kTokens) return fail(FLH_EINVAL, "linear_f16: at most %d rows (%u given)", kTokens, M);
  if (K == 0 || K % 128 || K > (1u << 20)) return fail(FLH_EINVAL, "linear_f16: K (%u) must be a positive multiple of 128", K);
  if (N > (1u << 30)) return fail(FLH_EINVAL, "linear_f16: N too large");
  if (M == 0 || N == 0) return FLH_OK;
  static LdsGrant grant;
  if (int rc = reserve_lds((const void*)linear_f16_kernel, (size_t)kStages * kStage, grant, "linear_f16")) return rc;
  hipLaunchKernelGGL(linear_f16_kernel, dim3((N + kRows - 1) / kRows), dim3(256), (size_t)kStages * kStage, (hipStream_t)stream,
                     (const __half*)x, (const __half*)w, (__half*)y, (int)M, (int)N, (int)K);
  return check_launch("linear_f16");
}
