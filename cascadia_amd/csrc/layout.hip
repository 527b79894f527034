// layout.hip -- the MFMA-tiled device layout of an INT4 matrix.
//
// The crate's row-major layout (format.rs:3-17) makes one wave instruction of
// the decode GEMM touch 16 rows x 64 bytes, 2 KB apart, and a row's next 64
// bytes arrive much later -- poor DRAM page locality.  The tiled layout stores
// each (16-row tile T, 128-column k-block kb) as one contiguous 1 KB block in
// MFMA lane order, so every wave streams sequentially:
//
//   packed_tiled[(T*KB + kb)*1024 + 16*l .. +16]
//       = swz(packed[16*T + (l & 15)][kb*64 + 16*(l >> 4) .. +16])  (l = lane 0..63)
//   scale_tiled[(T*NG + g)*16 + r] = scale[16*T + r][g]             (u16)
//
// with KB = ceil(K/128), NG = K/G, rows past N and bytes past K/2 zero.
// swz re-orders the 8 nibbles of each dword: the crate's byte b holds columns
// 2b (low) and 2b+1 (high); the tiled byte b holds columns b (low) and b+4
// (high), so that the MFMA decode (two masks, one shift, four byte permutes)
// yields the dword's 8 columns in natural order and the activations need no
// re-ordering.  The nibble codes and scale bits are moved, never changed: a
// kernel that takes both layouts computes bit-identical results from either
// (grouped.hip, few.hip and the one-token GEMV take the tiled one only).
//
// Groups of fewer than 128 columns (G not a multiple of 128): every 32-column
// MFMA step must cover whole groups, so its lanes' dwords must be the block's
// columns 32 s .. 32 s + 31.  Those blocks are stored with the dwords
// transposed across the four 16-lane rows -- dword s of lane row c is dword c
// of lane row s above:
//
//   packed_tiled[(T*KB + kb)*1024 + 16*l + 4*s .. +4]
//       = swz(packed[16*T + (l & 15)][kb*64 + 16*s + 4*(l >> 4) .. +4])
//
// -- so the kernels load a step's fragment as stored (the transpose, four
// lane permutes per fragment, was otherwise paid in every k-loop).
#include "int4_common.hpp"
#include "layout.hpp"

namespace cai4 {

void tiled_sizes(int N, int K, int G, size_t *packed_bytes, size_t *scale_bytes) {
  const size_t tiles = (size_t)(N + 15) / 16, kb = (size_t)(K + 127) / 128;
  *packed_bytes = tiles * kb * 1024;
  *scale_bytes = tiles * (size_t)(K / G) * 16 * 2;
}

// Nibbles n0 .. n7 of d -> bytes n0 | n4, n1 | n5, n2 | n6, n3 | n7.
CAI4_DEV uint32_t swizzle_dword(uint32_t d) {
  uint32_t lo = d & 0xFFFFu, hi = d >> 16;
  lo = (lo | (lo << 8)) & 0x00FF00FFu;
  hi = (hi | (hi << 8)) & 0x00FF00FFu;
  lo = (lo | (lo << 4)) & 0x0F0F0F0Fu;
  hi = (hi | (hi << 4)) & 0x0F0F0F0Fu;
  return lo | (hi << 4);
}

// Bound: HBM, each byte read and written once.  A wave takes kTileBlocks
// k-blocks of one tile: lane (r, c) reads row r's 16-byte parts c of each, all
// in flight (a row's kTileBlocks * 64 bytes are contiguous), and writes the
// blocks in lane order; where the layout transposes, the lanes' dwords trade
// places in registers.  Reading each dword of the transposed form from memory
// (four 4-byte loads a lane, 16 bytes apart) took 22 us for 7168 x 8192, and the
// scales' launch 7; this one launch 15.  The blocks past the code blocks move
// the scales, through LDS: [16 rows][64 groups] read along the rows, written
// along the tile.
constexpr int kTileBlocks = 4, kTileGroups = 64;

__global__ __launch_bounds__(256) void tile_kernel(const uint8_t *__restrict__ packed,
                                                   const uint16_t *__restrict__ scales, int N,
                                                   int K, int NG, int xposed,
                                                   unsigned code_blocks,
                                                   uint8_t *__restrict__ out,
                                                   uint16_t *__restrict__ out_s) {
  if (blockIdx.x < code_blocks) {
    const size_t kbt = (size_t)(K + 127) / 128, per = (kbt + kTileBlocks - 1) / kTileBlocks;
    const size_t wave = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const size_t T = wave / per, kb0 = (wave - T * per) * kTileBlocks;
    if (T >= (size_t)(N + 15) / 16) return;
    const int lane = threadIdx.x & 63;
    const size_t r = 16 * T + (lane & 15), row_bytes = (size_t)K / 2;
    u32x4_t w[kTileBlocks];
#pragma unroll
    for (int i = 0; i < kTileBlocks; ++i) {
      // row_bytes is a multiple of 16: a part is wholly inside the row or past it
      const size_t part = (kb0 + i) * 64 + 16 * (lane >> 4);
      w[i] = u32x4_t{0u, 0u, 0u, 0u};
      if (r < (size_t)N && part < row_bytes)
        w[i] = *reinterpret_cast<const u32x4_t *>(packed + r * row_bytes + part);
    }
#pragma unroll
    for (int i = 0; i < kTileBlocks; ++i) {
      if (kb0 + i >= kbt) break;  // uniform in the wave
      const u32x4_t v = xposed ? xpose_rows(w[i]) : w[i];
      reinterpret_cast<u32x4_t *>(out)[(T * kbt + kb0 + i) * 64 + lane] =
          u32x4_t{swizzle_dword(v.x), swizzle_dword(v.y), swizzle_dword(v.z), swizzle_dword(v.w)};
    }
    return;
  }
  __shared__ uint16_t t[kTileGroups][18];
  const size_t blk = blockIdx.x - code_blocks, nb = (size_t)(NG + kTileGroups - 1) / kTileGroups;
  const size_t T = blk / nb;
  const int g0 = (int)(blk - T * nb) * kTileGroups;
  const int ng = NG - g0 < kTileGroups ? NG - g0 : kTileGroups;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int g = threadIdx.x & 63, r = (threadIdx.x >> 6) + 4 * i;
    if (g < ng)
      t[g][r] = 16 * T + r < (size_t)N ? scales[(16 * T + r) * NG + g0 + g] : (uint16_t)0;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < ng * 16; i += 256)
    out_s[(T * NG + g0) * 16 + i] = t[i >> 4][i & 15];
}

hipError_t tile_weights(const uint8_t *packed, const uint8_t *scale_bits, int N, int K, int G,
                        uint8_t *packed_tiled, uint8_t *scale_tiled, hipStream_t st) {
  const size_t tiles = (size_t)(N + 15) / 16, kbt = (size_t)(K + 127) / 128;
  const int NG = K / G;
  const size_t code = (tiles * ((kbt + kTileBlocks - 1) / kTileBlocks) + 3) / 4;
  const size_t sc = tiles * (size_t)((NG + kTileGroups - 1) / kTileGroups);
  if (code + sc > 0x7FFFFFFFu) return hipErrorInvalidValue;
  hipLaunchKernelGGL(tile_kernel, dim3((unsigned)(code + sc)), dim3(256), 0, st, packed,
                     reinterpret_cast<const uint16_t *>(scale_bits), N, K, NG,
                     tiled_xposed(G) ? 1 : 0, (unsigned)code, packed_tiled,
                     reinterpret_cast<uint16_t *>(scale_tiled));
  return hipGetLastError();
}

}  // namespace cai4
