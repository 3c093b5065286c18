// Packed int4 codes -> the operand format of the 6-bit matrix instruction (gemm_f6.hip): a launch of its own, or workgroups behind those of
// the quantiser whose codes meet the encoded weights (fwht_quant.hip).
#pragma once
#include "f6_codes.h"
#include "gemm_i4.h"

namespace flh {
namespace {

// Bound by memory: 0.5 byte in and 0.75 byte out per code.  A workgroup takes 32 rows x 4 blocks: a lane encodes two
// 16-byte chunks of nibbles (each one 24-byte piece), sixteen lanes read 256 contiguous bytes of a row, and the pieces meet
// in LDS, from where every slab's 32 x 96 bytes leave as one contiguous run.
// 28672 x 4096 codes: 26.5 us (5.5 TB/s), 36.5 with 48-byte stores straight from the lanes; 4096 x 4096: 6.4 against 7.1.
// The matrices of one GEMM launch share one launch here as well.
constexpr int kEncodeRows = 32, kEncodeBlocks = 4, kEncodeLds = kEncodeBlocks * kEncodeRows * kF6BlockBytes;
struct EncodeArgs {   // up to four matrices of one K: 32-row blocks [block0[i], block0[i + 1]) of the launch
  const uint8_t* src[kMaxGemmSegments];
  uint8_t* dst[kMaxGemmSegments];
  size_t rows[kMaxGemmSegments];
  unsigned block0[kMaxGemmSegments];
  int count, blocks_per_row;
};
// lds: kEncodeLds bytes, 16-byte aligned (of the caller, which may have another use for them in other workgroups)
__device__ __forceinline__ void encode_f6_block(const EncodeArgs& p, unsigned block_x, unsigned block_y, uint8_t* lds) {
  uint8_t(*tile)[kEncodeRows * kF6BlockBytes] = (uint8_t(*)[kEncodeRows * kF6BlockBytes])lds;
  const uint8_t* src = p.src[0];
  uint8_t* dst = p.dst[0];
  size_t rows = p.rows[0];
  unsigned first = 0;
  for (int i = 1; i < p.count; ++i)
    if (block_x >= p.block0[i]) src = p.src[i], dst = p.dst[i], rows = p.rows[i], first = p.block0[i];
  const int blocks_per_row = p.blocks_per_row;
  const int t = threadIdx.x, c = t & 15, blk = c >> 2, q = c & 3;   // chunk q of a block: wave half q & 1, MFMA q >> 1
  const size_t row0 = (size_t)(block_x - first) * kEncodeRows;
  const int kt0 = block_y * kEncodeBlocks;
  const int n_rows = (int)(rows - row0 < (size_t)kEncodeRows ? rows - row0 : (size_t)kEncodeRows);
  const int n_blocks = min(blocks_per_row - kt0, kEncodeBlocks);
  v4i w[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = min((t >> 4) + 16 * i, n_rows - 1);
    w[i] = *(const v4i*)(src + ((row0 + r) * blocks_per_row + kt0 + min(blk, n_blocks - 1)) * 64 + 16 * q);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const unsigned long long q0 = bf6_of_nibbles((unsigned)w[i][0]), q1 = bf6_of_nibbles((unsigned)w[i][1]),
                             q2 = bf6_of_nibbles((unsigned)w[i][2]), q3 = bf6_of_nibbles((unsigned)w[i][3]);
    unsigned long long* o = (unsigned long long*)(&tile[blk][((t >> 4) + 16 * i) * kF6BlockBytes + 48 * (q & 1) + 24 * (q >> 1)]);
    o[0] = q0 | (q1 << 48);
    o[1] = (q1 >> 16) | (q2 << 32);
    o[2] = (q2 >> 32) | (q3 << 16);
  }
  __syncthreads();
  constexpr int kChunks = kEncodeRows * kF6BlockBytes / 16;           // 16-byte chunks of a slab's run: 192
#pragma unroll
  for (int i = 0; i < kEncodeBlocks * kChunks / 256; ++i) {
    const int e = t + 256 * i, b = e / kChunks, x = e % kChunks;
    if (b < n_blocks && x * 16 < n_rows * kF6BlockBytes)
      *(v4i*)(dst + ((size_t)(kt0 + b) * rows + row0) * kF6BlockBytes + x * 16) = *(const v4i*)(&tile[b][x * 16]);
  }
}

struct EncodeLaunch {
  EncodeArgs args;
  unsigned x, y;                                   // workgroups; x = 0: nothing to do
};
inline int encode_launch(int count, const uint8_t* const* packed_i4, uint8_t* const* encoded, const size_t* rows, size_t K, EncodeLaunch& l) {
  l = EncodeLaunch{};
  if (count < 1 || count > kMaxGemmSegments) return fail(FLH_EINVAL, "encode_f6: count = %d, must be 1 .. %d", count, kMaxGemmSegments);
  if (!packed_i4 || !encoded || !rows) return fail(FLH_EINVAL, "encode_f6: null array");
  if (K == 0 || K % 128) return fail(FLH_EINVAL, "encode_f6: K (%zu) must be a positive multiple of 128", K);
  EncodeArgs& a = l.args;
  a.blocks_per_row = (int)(K / 128);
  uint64_t blocks = 0;
  for (int i = 0; i < count; ++i) {
    if (rows[i] == 0) continue;
    if (!packed_i4[i] || !encoded[i]) return fail(FLH_EINVAL, "encode_f6: null pointer");
    if (misaligned16(packed_i4[i], encoded[i])) return fail(FLH_EINVAL, "encode_f6: packed_i4 and encoded must be 16-byte aligned");
    if ((rows[i] + kEncodeRows - 1) / kEncodeRows > 0x7FFFFFFFull) return fail(FLH_EINVAL, "encode_f6: matrix too large");
    a.src[a.count] = packed_i4[i], a.dst[a.count] = encoded[i], a.rows[a.count] = rows[i], a.block0[a.count] = (unsigned)blocks;
    blocks += (rows[i] + kEncodeRows - 1) / kEncodeRows;
    ++a.count;
  }
  const uint64_t slabs = (K / 128 + kEncodeBlocks - 1) / kEncodeBlocks;
  if (blocks > 0x7FFFFFFFull || slabs > 65535) return fail(FLH_EINVAL, "encode_f6: matrix too large");
  l.x = (unsigned)blocks, l.y = (unsigned)slabs;
  return FLH_OK;
}

}  // namespace
}  // namespace flh
