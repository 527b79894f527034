// few.hip -- INT4 weight-only GEMM for up to 32 token rows over MFMA-tiled
// weights (gfx950): the two GEMMs of a decode batch's FFN.
//
// y[t, r] = sum_g s[r, g] * sum_{c in g} (nibble[r, c] - 8) * x[t, c], the sum of
// dequant_gemm_int4_multi_auto (kernel_avx512_multi.rs:66-245) and, with the
// SwiGLU epilogue, of expert_forward's gate/up (kernel.rs:75-136).
//
// Bound: HBM (each weight byte once).  The skinny kernel stages its rows'
// whole k-range in LDS before it streams (16 rows of 4,096 columns: 128 KB, one
// workgroup per CU, two k-blocks of weights per wave in flight meanwhile).
// Here activations and weights arrive together: a stage holds two k-blocks of
// the workgroup's eight weight tiles and of its rows, global -> LDS by buffer
// loads with an LDS destination, as many stages ahead as LDS holds (2 to 4: 32-64
// KB of weights in flight per CU from the first microsecond on), one barrier per
// stage.  Eight waves: four by columns (two tiles each: a gate and an up tile
// with SwiGLU), two by k-block of the stage, added through LDS at the end.
// K is cut into slices until the workgroups fill the CUs; the reduce kernels of
// grouped.hip add the slices in order.  Measured on a 4096 x 14336 FFN, G 128
// (88 MB): 16 rows 36.0 -> 33.7 us (gate/up 18.5 -> 17.5, 3.4 TB/s of weights;
// down 14.6 -> 12.6, 2.3 TB/s, half its LDS traffic two planes of activations),
// 32 rows 62.5 -> 42.7; G 32: 16 rows 47.4 -> 35.0.  Walking the k-blocks from
// a different one per workgroup changed nothing.
//
// Arithmetic as the skinny kernel's: 16x16x32 MFMAs over bf16 128 + nibble, the
// zero point as MFMAs against a constant -136, the scale in f32 per group.  Two
// planes accumulate apart (hi, lo) and are added once at the end: the large
// partials of hi round no more often than one plane's.
#include "few.hpp"
#include "int4_common.hpp"
#include "lds_dma.hpp"

namespace cai4 {

namespace {

// MT: 16-row M-tiles; PL: activation planes; GPK: groups per k-block.
template <int MT, int PL, int GPK>
struct Few {
  static constexpr int W = 8, NT16 = 8;  // waves, weight tiles per workgroup
  static constexpr int A = 0, B = MT * PL * 8192, S = B + NT16 * 2048, BYTES = S + W * 256;
  static constexpr int AL = MT * PL;     // 1 KB activation loads per wave and stage
  static constexpr int LOADS = AL + 2 + 1;
  static constexpr int PIECES = 2 * GPK;  // 256-byte pieces of scales: [2 k-blocks][8 tiles][GPK][16]
  static constexpr int ST = 155 * 1024 / BYTES;  // stages: 3 .. 5
  static_assert(ST >= 3 && ST <= 5 && (ST - 2) * LOADS <= 63 && PIECES <= W, "stage");
};

template <int N>
CAI4_DEV void few_wait(int ahead) {  // uniform: stages that may still be in flight (ST - 2 at most)
  if (ahead == 3)
    dma_wait_barrier<3 * N>();
  else if (ahead == 2)
    dma_wait_barrier<2 * N>();
  else if (ahead == 1)
    dma_wait_barrier<N>();
  else
    dma_wait_barrier<0>();
}

template <int MT, int PL, int GPK, bool SW, int SDT>
__global__ __launch_bounds__(512, 2) void few_kernel(GgArgs a) {
  using P = Few<MT, PL, GPK>;
  __shared__ __attribute__((aligned(256))) uint8_t st[P::ST * P::BYTES];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave & 3, wk = wave >> 2;
  const int KB = a.K >> 7, NG = a.K / a.G, KPG = GPK > 1 ? 1 : a.G >> 7;
  const int ntiles = (a.N + 15) >> 4;
  // SwiGLU: LDS tiles 0-3 gate, 4-7 up of the same four 16-column tiles
  constexpr int TM = SW ? P::NT16 / 2 : P::NT16;
  // consecutive workgroups (one per XCD in turn) take the slices in turn: an XCD
  // then reads few slices of the activations
  const int nsl = (KB + a.kper - 1) / a.kper;
  const int tile = blockIdx.x / nsl, slice = blockIdx.x - tile * nsl;
  const int T0 = tile * TM;
  const int tv = __builtin_amdgcn_readfirstlane(ntiles - T0 > TM ? TM : ntiles - T0);
  const size_t wo = (size_t)T0 * KB * 1024, so = (size_t)T0 * NG * 32;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_void *)st);
  const int kb0 = slice * a.kper, KE = min(KB, kb0 + a.kper), nst = (KE - kb0 + 1) / 2;

  // ---- this wave's loads: tile `wave` of both k-blocks, AL blocks of rows, a
  // piece of the scales (a k-block past KE reads KE - 1 again: in range, unused)
  const bool up = SW && wave >= 4;
  const rsrc_t wr = rsrc_scalar((up ? a.w1 : a.w0) + wo, (size_t)tv * KB * 1024);
  const uint32_t vb = (uint32_t)((wave - (up ? 4 : 0)) * KB) * 1024 + 16 * lane;
  const rsrc_t xr0 = rsrc_scalar(a.x, (size_t)a.M * a.K * 2);
  const rsrc_t xr1 = rsrc_scalar(PL == 2 ? a.x2 : a.x, PL == 2 ? (size_t)a.M * a.K * 2 : 0);
  // block b = (k-block half, plane, four rows): 4 MT PL blocks per half
  uint32_t va[P::AL];
#pragma unroll
  for (int l = 0; l < P::AL; ++l) {
    const int b = (wave * P::AL + l) % (4 * MT * PL), rb = b % (4 * MT);
    const int row = 4 * rb + (lane >> 4), q = lr ^ (row & 15);
    va[l] = row < a.M ? (uint32_t)(row * a.K + 8 * q) * 2 : kDmaOOB;
  }
  // piece m: k-block half m / GPK, tiles (m % GPK) * 8 / GPK ..., 8 GPK lanes a tile
  const int m = wave < P::PIECES ? wave : wave % P::PIECES;
  const int mh = m / GPK, mt0 = (m % GPK) * (8 / GPK);
  const bool mu = SW && mt0 >= 4;  // (GPK 1: one piece spans both matrices, below)
  const int ltile = mt0 + lane / (8 * GPK), lj = lane % (8 * GPK);
  const rsrc_t sr0 = rsrc_scalar((mu ? a.s1 : a.s0) + so, (size_t)tv * NG * 32);
  const uint32_t vs = (uint32_t)((ltile - (mu ? 4 : 0)) * NG * 32 + 4 * lj);
  // SwiGLU with one piece per k-block: lanes 0-31 gate's tiles, 32-63 up's, so
  // waves 0 / 1 load gate's half and waves 2 / 3 up's
  constexpr bool kSplit = SW && GPK == 1;
  const rsrc_t srx = kSplit ? rsrc_scalar(((wave & 2) ? a.s1 : a.s0) + so, (size_t)tv * NG * 32) : sr0;
  auto issue = [&](int buf, int t) {
    const uint32_t L = lds0 + buf * P::BYTES;
    const int k0 = kb0 + 2 * t, k1 = min(k0 + 1, KE - 1);
    lds_dma<16>(wr, L + P::B + wave * 2048, vb, (uint32_t)k0 * 1024);
    lds_dma<16>(wr, L + P::B + wave * 2048 + 1024, vb, (uint32_t)k1 * 1024);
#pragma unroll
    for (int l = 0; l < P::AL; ++l) {
      const int blk = wave * P::AL + l, half = blk / (4 * MT * PL), b = blk % (4 * MT * PL);
      lds_dma<16>(PL == 2 && b >= 4 * MT ? xr1 : xr0, L + P::A + blk * 1024, va[l],
                  (uint32_t)(half ? k1 : k0) * 256);
    }
    if constexpr (kSplit) {
      // waves 0-3: k-block half wave & 1, matrix (wave & 2): 32 lanes each; waves
      // 4-7 the same into the spare pieces
      const int kb = (wave & 1) ? k1 : k0;
      if (lane < 32)
        lds_dma<4>(srx, L + P::S + (wave >> 2) * 1024 + (wave & 1) * 256 + ((wave & 2) ? 128 : 0),
                   (uint32_t)((lane >> 3) * NG * 32 + 4 * (lane & 7)), (uint32_t)(kb / KPG) * 32);
    } else {
      const int kb = mh ? k1 : k0;
      lds_dma<4>(sr0, L + P::S + wave * 256, vs, (uint32_t)(GPK > 1 ? kb * GPK : kb / KPG) * 32);
    }
  };
#pragma unroll
  for (int t = 0; t < P::ST - 1; ++t)
    if (t < nst) issue(t, t);

  // ---- LDS read offsets within a stage: this wave's k-block half wk ----
  // A row 16 i + lr, step s: chunk (GPK 1: 4 lg + s; else 4 s + lg) ^ lr
  const uint32_t ax = lds0 + P::A + wk * (MT * PL * 4096) + lr * 256 +
                      16 * ((GPK == 1 ? 4 * lg : lg) ^ lr);
  // tiles of this wave: 2 wn, 2 wn + 1; SwiGLU: wn of gate, wn of up
  constexpr int JT = SW ? 4 : 1;
  const int t0 = SW ? wn : 2 * wn;
  const uint32_t bx = lds0 + P::B + t0 * 2048 + wk * 1024 + 16 * lane;
  const uint32_t sx = lds0 + P::S + wk * GPK * 256 + t0 * 32 * GPK + 2 * lr;

  f32x4_t acc[PL][MT][2];
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[p][i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  u32x4_t B136 = {0xC308C308u, 0xC308C308u, 0xC308C308u, 0xC308C308u};  // bf16 -136 x 8
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+v"(B136));  // one register copy for the loop
#endif
  int buf = 0;
#pragma unroll 1
  for (int t = 0; t < nst; ++t) {
    few_wait<P::LOADS>(min(P::ST - 2, nst - 1 - t));
    // every wave is past stage t - 1: its buffer takes stage t + ST - 1
    if (t + P::ST - 1 < nst) issue(buf == 0 ? P::ST - 1 : buf - 1, t + P::ST - 1);
    if (kb0 + 2 * t + wk < KE) {
      const uint32_t base = buf * P::BYTES;
      u32x4_t b[2], af[PL][MT][4];
      float sc[2][GPK];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = lds_at<u32x4_t>(base + bx, j * JT * 2048);
#pragma unroll
      for (int p = 0; p < PL; ++p)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int s = 0; s < 4; ++s)
            af[p][i][s] = lds_at<u32x4_t>((base + ax) ^ (16 * (GPK == 1 ? s : 4 * s)),
                                          (p * MT + i) * 4096);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < GPK; ++g)
          sc[j][g] = scale_to_f32<SDT>(
              (uint32_t)lds_at<uint16_t>(base + sx, j * JT * 32 * GPK + g * 32));
      constexpr int SPG = 4 / GPK;
#pragma unroll
      for (int g = 0; g < GPK; ++g) {
        u32x4_t d[2][SPG];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int s = 0; s < SPG; ++s) d[j][s] = decode8(b[j][g * SPG + s]);
#pragma unroll
        for (int p = 0; p < PL; ++p)
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            f32x4_t corr = zero4;
#pragma unroll
            for (int s = 0; s < SPG; ++s) corr = mfma_bf16(af[p][i][g * SPG + s], B136, corr);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              f32x4_t q = corr;
#pragma unroll
              for (int s = 0; s < SPG; ++s) q = mfma_bf16(af[p][i][g * SPG + s], d[j][s], q);
              acc[p][i][j] += sc[j][g] * q;
            }
          }
      }
    }
    buf = buf == P::ST - 1 ? 0 : buf + 1;
  }

  // ---- hi + lo, then the two k-block halves through LDS ----
  f32x4_t y[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      y[i][j] = acc[0][i][j];
      if (PL == 2) y[i][j] += acc[PL - 1][i][j];
    }
  __syncthreads();
  f32x4_t *red = reinterpret_cast<f32x4_t *>(st);
  if (wk == 1) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) red[((wn * MT + i) * 2 + j) * 64 + lane] = y[i][j];
  }
  __syncthreads();
  if (wk == 1) return;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) y[i][j] += red[((wn * MT + i) * 2 + j) * 64 + lane];

  // ---- epilogue: D lane l holds column lr and rows 4 lg + v ----
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int t = 16 * i + 4 * lg + v;
      if (t >= a.M) continue;
      if constexpr (SW) {
        const int n = (T0 + wn) * 16 + lr;
        if (n >= a.N) continue;
        if (a.part) {
          float *o = a.part + ((size_t)slice * a.M + t) * 2 * a.N + n;
          o[0] = y[i][0][v];
          o[a.N] = y[i][1][v];
        } else {
          const float h = silu_f32(y[i][0][v]) * y[i][1][v];
          const size_t o = (size_t)t * a.ldy + n;
          const uint32_t hb = split_hi(h);
          static_cast<uint16_t *>(a.y)[o] = (uint16_t)hb;
          static_cast<uint16_t *>(a.y2)[o] = (uint16_t)split_lo(h, hb);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = (T0 + 2 * wn + j) * 16 + lr;
          if (n >= a.N) continue;
          if (a.part)
            a.part[((size_t)slice * a.M + t) * a.N + n] = y[i][j][v];
          else
            static_cast<uint16_t *>(a.y)[(size_t)t * a.ldy + n] = (uint16_t)f32_to_bf16_rne(y[i][j][v]);
        }
      }
    }
}

struct FewPlan {
  int nsl, kper;
};

// Slices of K: as many as fill the CUs once, each of at least four k-blocks (an
// even number: a stage holds two).
FewPlan few_plan(int N, int K, bool sw, int num_cus) {
  const int KB = K / 128, tiles = (N + (sw ? 63 : 127)) / (sw ? 64 : 128);
  int s = num_cus / tiles;
  if (s > KB / 4) s = KB / 4;
  if (s > 64) s = 64;
  if (s < 1 || N % 4) s = 1;  // (the partials' rows are N apart here)
  int kper = (KB + s - 1) / s;
  kper += kper & 1;
  return FewPlan{(KB + kper - 1) / kper, kper};
}

template <int MT, int PL, bool SW>
hipError_t few_launch(const GgArgs &a, int nsl, hipStream_t st) {
  const dim3 grid((a.N + (SW ? 63 : 127)) / (SW ? 64 : 128) * nsl), block(512);
#define CAI4_FEW(GPK)                                                                        \
  do {                                                                                       \
    if (a.sdt)                                                                               \
      hipLaunchKernelGGL((few_kernel<MT, PL, GPK, SW, SCALE_F16>), grid, block, 0, st, a);  \
    else                                                                                     \
      hipLaunchKernelGGL((few_kernel<MT, PL, GPK, SW, SCALE_BF16>), grid, block, 0, st, a); \
  } while (0)
  switch (a.G == 32 ? 4 : a.G == 64 ? 2 : 1) {
    case 4: CAI4_FEW(4); break;
    case 2: CAI4_FEW(2); break;
    default: CAI4_FEW(1);
  }
#undef CAI4_FEW
  return hipGetLastError();
}

}  // namespace

bool few_supported(int M, int N, int K, int G, int tiled) {
  return M >= 1 && M <= kFewMaxRows && N >= 16 && gg_supported(K, G, tiled);
}

size_t few_workspace(int M, int N, int K, bool sw, int num_cus) {
  const FewPlan p = few_plan(N, K, sw, num_cus);
  return p.nsl > 1 ? (size_t)p.nsl * M * (sw ? 2 * (size_t)N : N) * 4 : 0;
}

hipError_t few_gemm(GgArgs a, void *ws, int num_cus, hipStream_t st) {
  const bool sw = a.epi == GG_SWIGLU_HILO;
  if (a.M < 1 || a.M > kFewMaxRows || sw == (a.hilo != 0) || (!sw && a.epi != GG_BF16))
    return hipErrorInvalidValue;
  const FewPlan p = few_plan(a.N, a.K, sw, num_cus);
  a.kper = p.kper;
  a.part = p.nsl > 1 ? static_cast<float *>(ws) : nullptr;
  hipError_t e;
  if (sw)
    e = a.M <= 16 ? few_launch<1, 1, true>(a, p.nsl, st) : few_launch<2, 1, true>(a, p.nsl, st);
  else
    e = a.M <= 16 ? few_launch<1, 2, false>(a, p.nsl, st) : few_launch<2, 2, false>(a, p.nsl, st);
  if (e != hipSuccess || p.nsl == 1) return e;
  return gg_reduce_slices(a, p.nsl, st);
}

}  // namespace cai4
