// quant.hip -- load-time INT4 quantiser on the GPU: bf16 weights [N, K] ->
// packed nibbles [N, K/2] + bf16 group scales [N, K/G], as the crate's
// quantize_int4_group (crates/cascadia-int4-gemm/src/shell_int4.rs:148-212,
// fixed G = 32 there; any G that is a multiple of 32 dividing K here).
//
// Per group: max|w| (NaNs never win the comparison), scale = max / 7 (1e-10
// for an all-zero group), stored as bf16 by the crate's rounding
// (shell_int4.rs:214-220: bits + 0x7FFF + lsb, no NaN branch); then
// q = clamp(round(w * (1 / scale_bf16)), -8, 7) with round half away from
// zero, and nibble q + 8 (column 2i low, 2i+1 high).  The divisions are
// IEEE-rounded and the product is not fused with anything, so the bytes match
// the crate bit for bit.  A NaN weight becomes q = 0 (Rust's `as i32` of NaN),
// nibble 8.
//
// Bound: HBM (2 bytes read and half a byte written per weight) beside about 10
// VALU instructions per weight.  Groups of a power of two columns up to 512: a
// lane takes 16 bytes (eight columns), G / 8 neighbouring lanes share a group
// and add up its max by lane swaps, so a wave's loads and stores are
// contiguous and the weights are read once; four chunks per lane are in flight.
// One thread per group, reading its chunks twice and 64 bytes apart from its
// neighbour's, took 54 us for 7168 x 8192 at G 32, this form 32 us.  Other
// group sizes (96, 160, ...) keep the thread per group.
#include <math.h>

#include "int4_common.hpp"
#include "quant.hpp"

namespace cai4 {

namespace {

// The scale bits of a group from its max|w| (shell_int4.rs:171-178, 214-220).
CAI4_DEV uint32_t scale_bits_of(float mx) {
  const float scale = mx == 0.0f ? 1.0e-10f : __fdiv_rn(mx, 7.0f);
  const uint32_t b = fbits(scale);
  return (b + 0x7FFFu + ((b >> 16) & 1u)) >> 16;
}

// Eight bf16 weights -> eight nibbles, column c in bits 4 c.  round() half away
// from zero as trunc(t + copysign(0.5 - 2^-25, t)): t + 0.5 itself would round
// 0.5 - 2^-25 up to 1.  The conversion truncates, saturates and takes NaN to 0.
CAI4_DEV uint32_t quantize8(u32x4_t v, float inv) {
  // the product rounds before the sum: no contraction.  (__fmul_rn / __fadd_rn
  // are plain operators defined outside this scope, which it would still fuse)
#pragma clang fp contract(off)
  uint32_t out = 0x88888888u;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t bits = (j & 1) ? v[j >> 1] & 0xFFFF0000u : v[j >> 1] << 16;
    const float t = bitsf(bits) * inv;
    const float r = t + __builtin_copysignf(bitsf(0x3EFFFFFFu), t);
    int q;
#ifdef __HIP_DEVICE_COMPILE__
    asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(r));
#else
    q = (int)r;
#endif
    q = q < -8 ? -8 : q > 7 ? 7 : q;
    out += (uint32_t)q << (4 * j);  // (q + 8) << 4 j, the eights in out's start value
  }
  return out;
}

CAI4_DEV float max_abs8(u32x4_t v) {
  float mx = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    // shell_int4.rs:167-170 (a NaN never compares greater)
    mx = fmaxf(mx, fabsf(bitsf(v[e] << 16)));
    mx = fmaxf(mx, fabsf(bitsf(v[e] & 0xFFFF0000u)));
  }
  return mx;
}

// L = G / 8 lanes per group (a power of two, 4 .. 64).
constexpr int kQuantChunks = 4;  // 16-byte chunks per lane

template <int L>
__global__ __launch_bounds__(256) void quantize_lanes_kernel(const uint16_t *w, size_t chunks,
                                                             uint8_t *packed, uint16_t *scales) {
  constexpr int C = kQuantChunks;
  const int lane = threadIdx.x & 63;
  const size_t c0 = ((size_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 * C) + lane;
  u32x4_t v[C];
#pragma unroll
  for (int i = 0; i < C; ++i) {
    const size_t c = c0 + 64 * i;  // (a clamped read past the end: its lanes store nothing)
    v[i] = *reinterpret_cast<const u32x4_t *>(w + 8 * (c < chunks ? c : chunks - 1));
  }
#pragma unroll
  for (int i = 0; i < C; ++i) {
    const size_t c = c0 + 64 * i;
    float mx = max_abs8(v[i]);
#pragma unroll
    for (int d = 1; d < L; d *= 2) mx = fmaxf(mx, __shfl_xor(mx, d));
    const uint32_t sb = scale_bits_of(mx);
    const uint32_t out = quantize8(v[i], __fdiv_rn(1.0f, bf16_to_f32(sb)));
    // whole groups are inside or past the end: chunks is a multiple of L
    if (c < chunks) {
      if ((lane & (L - 1)) == 0) scales[c / L] = (uint16_t)sb;
      reinterpret_cast<uint32_t *>(packed)[c] = out;
    }
  }
}

__global__ __launch_bounds__(256) void quantize_group_kernel(const uint16_t *w, int N, int K,
                                                             int G, uint8_t *packed,
                                                             uint16_t *scales) {
  const int ng = K / G;
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (long)N * ng) return;
  const uint16_t *src = w + gid * G;
  float mx = 0.0f;
  for (int c = 0; c < G; c += 8)
    mx = fmaxf(mx, max_abs8(*reinterpret_cast<const u32x4_t *>(src + c)));
  const uint32_t sb = scale_bits_of(mx);
  scales[gid] = (uint16_t)sb;
  const float inv = __fdiv_rn(1.0f, bf16_to_f32(sb));
  uint32_t *dst = reinterpret_cast<uint32_t *>(packed + gid * G / 2);
  for (int c = 0; c < G; c += 8)
    dst[c / 8] = quantize8(*reinterpret_cast<const u32x4_t *>(src + c), inv);
}

}  // namespace

hipError_t quantize_group(const uint16_t *w_bf16, int N, int K, int G, uint8_t *packed,
                          uint16_t *scale_bits, hipStream_t st) {
  const long groups = (long)N * (K / G);
  if (groups == 0) return hipSuccess;
  const size_t chunks = (size_t)N * K / 8, per = 256 * kQuantChunks;
  const dim3 grid((unsigned)((chunks + per - 1) / per)), block(256);
#define CAI4_QL(L)                                                                             \
  hipLaunchKernelGGL(quantize_lanes_kernel<L>, grid, block, 0, st, w_bf16, chunks, packed, \
                     scale_bits);                                                             \
  return hipGetLastError()
  switch ((chunks + per - 1) / per <= 0x7FFFFFFFu ? G : 0) {
    case 32: CAI4_QL(4);
    case 64: CAI4_QL(8);
    case 128: CAI4_QL(16);
    case 256: CAI4_QL(32);
    case 512: CAI4_QL(64);
    default: break;
  }
#undef CAI4_QL
  hipLaunchKernelGGL(quantize_group_kernel, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0,
                     st, w_bf16, N, K, G, packed, scale_bits);
  return hipGetLastError();
}

}  // namespace cai4
