// grouped.hip -- INT4 weight-only GEMM on MFMA tiles of up to 128 rows, for
// one matrix (dense prefill) or for the row groups of many experts in one
// launch (a MoE layer whose experts receive many tokens each).
//
// The crate runs these as per-token GEMVs (kernel_avx512_multi.rs:240-244;
// the runner's per-(token, expert) loop, runner.rs:2079-2108); every output
// element is the same sum, y = sum_g s_g * sum_{c in g} (nibble - 8) x_c, with
// exact products and f32 accumulation.
//
// Arithmetic: weights enter v_mfma_f32_32x32x16_bf16 as the exact bf16 value
// 128 + nibble (or 16 + nibble: gg_small_offset); each group's partial starts
// from the seed -136 (-24) * sum(x) over the group's columns (computed once per
// row and group by gg_prep) and is scaled in f32 when the group ends, acc +=
// s * p.  A k-block of 128 columns is
// four sub-steps of 32: a sub-step is dword s of every weight fragment.  Groups
// of 32 or 64 columns end with a sub-step: the tiled layout stores those
// matrices' fragments with their four dwords transposed across the lane rows
// (layout.hip), so that dword s holds columns 32 s .. 32 s + 31.
//
// Two-plane activations (PL = 2): the A operand is hi + lo (two bf16 planes
// whose sum carries an f32 value to 2^-16: the SwiGLU intermediate, or an f32
// input); both planes run with the same decoded weights.
//
// SwiGLU: each wave has 32 gate and the same 32 up columns, and the epilogue
// writes hi / lo of silu(g) * u and, for the down projection, their seeds.
//
// Grouped mode: workgroup row y takes chunk y of a table written by the MoE
// grouping -- (expert, first grouped row, rows) -- and reads expert e's
// matrices at + e * estride.  A tile's rows past its count read zeros and are
// not stored; a wave whose rows are all past it only loads and waits.
//
// Bound: matrix-core and VALU issue.  Measured on the card: a 32x32x16 MFMA
// takes 32 cycles of its SIMD's matrix core and, with two waves, about 10 of
// the issue slots the VALU also needs (two 16x16x32 ones take 15), a VALU
// instruction 4; so V VALU instructions per MFMA cost max(32, 10 + 4 V).  V is
// the nibble decode (7 per fragment, shared by the NT MFMAs that use it: 3.5)
// and the scaled adds (16 per MFMA and group: 2 at G 128, 8 at G 32), nothing
// else: load offsets step in scalar registers, LDS offsets are immediates.  On
// data like the weights' the power limit holds the clock at 1.9-2.1 GHz.
//
// Schedule: one slot per MFMA (a scheduling barrier ends it) holding that
// MFMA's share of everything else -- half a fragment's decode, an LDS read for
// the next sub-step, a stage load, eight scaled adds of the group before -- so
// that a wave keeps the matrix core fed by itself and its VALU work runs in
// the MFMAs' shadow.  Written as decode / MFMA / add blocks, the two waves of
// a SIMD, held together by the stage barriers, ran the same phase at once.
//
// Pipeline: three LDS stages of one k-block; activations, weight tiles, scales
// and seeds go global -> LDS by buffer loads with an LDS destination.  The
// barrier that publishes stage k + 1 stands before the last sub-step of k, when
// no wave reads stage k any more: its buffer takes the loads of k + 3, and the
// first fragments of k + 1 are read while the last MFMAs of k run.
//
// Measured (M 2048, N 14336, K 4096, G 128): 264 -> 230 us against the
// 16x16x32 kernel with block phases (3600 -> 2900 cycles per k-block; the tile
// through LDS in 16-byte stores, 14.5k cycles of 2-byte stores before); 1024
// tokens over 384 experts, G 32: 2.39 -> 1.98 ms a layer (with the other changes
// to its tiles' rules).
#include "grouped.hpp"
#include "int4_common.hpp"
#include "lds_dma.hpp"

namespace cai4 {

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

CAI4_DEV f32x16_t mfma32_bf16(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Workgroup geometry (WM x WN waves of 32 MT rows x 64 columns, PL activation
// planes, GPK scale groups per 128-column k-block) and the LDS of one stage:
// activations [PL][BM][256 B] (16-byte chunk c of row r at slot c ^ (r & 15)),
// weight tiles [NT16][1 KB], then 256-byte pieces of scales [NT16][GPK][16] u16
// and seeds [GPK][BM] f32, MPW pieces per wave (the last ones spare: every
// wave issues the same number of loads, the stage waits count them).
template <int MT, int WM, int WN, int GPK, int PL, bool SW>
struct Gg {
  static constexpr int W = WM * WN;
  static constexpr int RM = 32 * MT, BM = RM * WM, BN = 64 * WN;
  static constexpr int NT16 = BN / 16;                 // weight tiles per stage
  static constexpr int OUTC = SW ? BN / 2 : BN;        // output columns per workgroup
  static constexpr int SLD = NT16 * GPK / 8, XLD = GPK * BM / 64;  // 256-byte pieces
  static constexpr int MPW = (SLD + XLD + W - 1) / W;
  static constexpr int A = 0, B = PL * BM * 256, S = B + NT16 * 1024, X = S + SLD * 256,
                       BYTES = S + MPW * W * 256;
  static constexpr int AL = PL * BM / (4 * W);         // 1 KB activation loads per wave
  static constexpr int BL = NT16 / W;                  // weight tiles per wave
  static constexpr int LOADS = AL + BL + MPW;
  static constexpr int NT = MT * PL;                   // A fragments per 16-column step
  static constexpr int SLOTS = 4 * NT;                 // MFMAs per 32-column sub-step
  static_assert(AL >= 1 && BL >= 1 && SLD >= 1 && XLD >= 1, "workgroup shape");
  static_assert(NT == 1 || NT == 2, "fragments per step");
  static_assert(!SW || (W % 2 == 0 && SLD % 2 == 0), "SwiGLU shape");
  static_assert(3 * BYTES <= 160 * 1024, "LDS");
};

// Keeps these values' computation in its slot: the instruction selector orders
// arithmetic freely between scheduling barriers unless something there uses it.
CAI4_DEV void gg_pin(float &a, float &b, float &c, float &d, float &e, float &f, float &g,
                     float &h) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f), "+v"(g), "+v"(h));
#endif
}

// The weights' encoding: bf16 128 + n (0x43 over the nibble), offset 136 with
// the zero point; or 16 + n (0x41 over 0x80 | n << 3), offset 24, one
// instruction more per half fragment.  A group's partial starts at -offset *
// sum(x) and comes down to sum((n - 8) x), so its f32 roundings grow with the
// offset and the group, and two planes share one partial, where the skinny
// kernel adds them up apart.  Two planes in groups of 64 columns and more take
// the small one.  Error against 64 bits with the large / the small offset / in
// the skinny kernel:
//   FFN 4096 x 14336 f32, 130 rows  G 64 8.7e-6 / 4.2e-6 / 8.2e-6 (133 / 139 us)
//                                   G 128 9.9e-6 / 4.4e-6 / 9.1e-6
//                                   G 32 7.5e-6 / 4.1e-6 / 8.2e-6
//   GEMM 7168 x 8192 f32, 333 rows  G 64 3.3e-6 / 2.5e-6 / 4.9e-6 (90 / 93 us)
//                                   G 32 3.0e-6 / 2.5e-6 / 4.9e-6 (100 / 105 us)
// (rows of mean 1 instead of 0: G 64 1.8e-6 / 5.3e-7 / 9.3e-7, G 32 1.2e-6 /
// 4.7e-7 / 9.3e-7 of a result ten times as large.)
constexpr bool gg_small_offset(int GPK, int PL) { return GPK <= 2 && PL == 2; }
constexpr float gg_seed_factor(int GPK, int PL) { return gg_small_offset(GPK, PL) ? -24.f : -136.f; }

// Bytes of the low (0) or high (1) nibbles of w, encoded.
template <bool SMALL>
CAI4_DEV uint32_t gg_nibbles(uint32_t w, int hi) {
  if constexpr (SMALL)
    return ((hi ? w >> 1 : w << 3) & 0x78787878u) | 0x80808080u;
  else
    return (hi ? w >> 4 : w) & 0x0F0F0F0Fu;
}
template <bool SMALL>
CAI4_DEV u32x4_t gg_decode8(uint32_t w) {
  const uint32_t C = SMALL ? 0x41414141u : 0x43434343u;
  const uint32_t t = gg_nibbles<SMALL>(w, 0), u = gg_nibbles<SMALL>(w, 1);
  return u32x4_t{__builtin_amdgcn_perm(C, t, 0x04010400u), __builtin_amdgcn_perm(C, t, 0x04030402u),
                 __builtin_amdgcn_perm(C, u, 0x04010400u), __builtin_amdgcn_perm(C, u, 0x04030402u)};
}

struct GgTrue { static constexpr bool value = true; };
struct GgFalse { static constexpr bool value = false; };

// Sum over groups of L consecutive lanes (L = 4, 8, 16 within a DPP row):
// quad sums, then a half-row mirror (lane i <- 7 - i of its 8 lanes: the other
// quad of the same half), then a row mirror (the other half).
template <int L>
CAI4_DEV float lane_group_sum(float t) {
  t += dpp_f32<0xB1>(t);                          // quad_perm 1,0,3,2
  t += dpp_f32<0x4E>(t);                          // quad_perm 2,3,0,1
  if constexpr (L >= 8) t += dpp_f32<0x141>(t);   // row_half_mirror
  if constexpr (L >= 16) t += dpp_f32<0x140>(t);  // row_mirror
  return t;
}

// A [BM][OUTC] u16 tile from LDS (row pitch `pitch` bytes) to rows row0.. of
// dst [., ldy], columns col0..: 16 bytes per thread where dst allows it.
template <int OUTC>
CAI4_DEV void gg_store_tile(const uint8_t *lds, int pitch, uint16_t *dst, size_t row0, int mrows,
                            int col0, int N, int ldy, int tid, int nth) {
  const bool wide = (ldy & 7) == 0 && ((uintptr_t)dst & 15) == 0;
  for (int c = tid; c < mrows * (OUTC / 8); c += nth) {
    const int row = c / (OUTC / 8), col = 8 * (c - row * (OUTC / 8));
    const u32x4_t v = *reinterpret_cast<const u32x4_t *>(lds + row * pitch + col * 2);
    const int n = col0 + col;
    if (n >= N) continue;
    uint16_t *p = dst + (row0 + row) * (size_t)ldy + n;
    if (wide && n + 8 <= N) {
      *reinterpret_cast<u32x4_t *>(p) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < N) p[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// SDT: the scale dtype (a.sdt) as a constant.
template <int MT, int WM, int WN, int GPK, int PL, bool SW, int SDT>
__global__ __launch_bounds__(64 * WM * WN, 2) void gg_kernel(GgArgs a) {
  using P = Gg<MT, WM, WN, GPK, PL, SW>;
  __shared__ __attribute__((aligned(256))) uint8_t st[3 * P::BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int h = lane >> 5, l15 = lane & 15, l31 = lane & 31, t16 = (lane >> 4) & 1;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % WM, wn = wave / WM;
  // this workgroup's rows
  int e = 0, row0, mrows;
  if (a.tiles) {
    const int sub = blockIdx.y % a.tile_split;
    const SkinnyChunk c = a.tiles[blockIdx.y / a.tile_split];
    const int cnt = c.count - sub * P::BM;
    if (cnt <= 0) return;  // uniform: an empty table entry, or past its rows
    e = c.expert;
    row0 = c.row0 + sub * P::BM;
    mrows = cnt < P::BM ? cnt : P::BM;
  } else {
    row0 = blockIdx.y * P::BM;
    mrows = a.M - row0 < P::BM ? a.M - row0 : P::BM;
  }
  e = __builtin_amdgcn_readfirstlane(e);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  mrows = __builtin_amdgcn_readfirstlane(mrows);
  const int KB = a.K >> 7, NG = a.K / a.G, KPG = GPK > 1 ? 1 : a.G >> 7;
  const int ntiles = (a.N + 15) >> 4;
  const int T0 = blockIdx.x * (P::OUTC / 16);
  constexpr int TM = SW ? P::NT16 / 2 : P::NT16;  // tiles per matrix per workgroup
  const int tv = __builtin_amdgcn_readfirstlane(ntiles - T0 > TM ? TM : ntiles - T0);
  const size_t eo = (size_t)e * a.estride;
  const size_t wo = eo + (size_t)T0 * KB * 1024, so = eo + (size_t)T0 * NG * 32;
  const size_t wbytes = (size_t)tv * KB * 1024, sbytes = (size_t)tv * NG * 32;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const lds_void *)st);

  // ---- this wave's loads of a stage: descriptors and per-lane offsets ----
  const bool up = SW && wave >= P::W / 2;  // SwiGLU: the upper waves load up's tiles
  const rsrc_t wr = rsrc_scalar((up ? a.w1 : a.w0) + wo, wbytes);
  rsrc_t xr0 = rsrc(a.x + (size_t)row0 * a.K, (size_t)mrows * a.K * 2);
  const rsrc_t xr1 = rsrc(PL == 2 ? a.x2 + (size_t)row0 * a.K : a.x,
                          PL == 2 ? (size_t)mrows * a.K * 2 : 0);
  const bool ind = PL == 1 && a.row_map != nullptr;  // rows through a row map
  if (ind) xr0 = rsrc(a.x, (size_t)a.x_rows * a.K * 2);
  uint32_t va[P::AL], vb[P::BL], vm[P::MPW];
#pragma unroll
  for (int l = 0; l < P::AL; ++l) {
    const int blk = wave * P::AL + l, rb = blk % (P::BM / 4);
    const int row = 4 * rb + (lane >> 4), q = l15 ^ (row & 15);
    if (ind)
      va[l] = row < mrows ? (uint32_t)(((size_t)a.row_map[row0 + row] * a.K + 8 * q) * 2) : kDmaOOB;
    else
      va[l] = row < mrows ? (uint32_t)(row * a.K + 8 * q) * 2 : kDmaOOB;
  }
#pragma unroll
  for (int l = 0; l < P::BL; ++l) {
    const int tile = wave * P::BL + l - (up ? P::NT16 / 2 : 0);
    vb[l] = (uint32_t)(tile * KB) * 1024 + 16 * lane;
  }
  // pieces m = wave, wave + W, ...: scales (8 / GPK tiles' 32 GPK bytes), seeds, spare
  rsrc_t mr[P::MPW];
  bool mx[P::MPW];
#pragma unroll
  for (int k = 0; k < P::MPW; ++k) {
    const int m = wave + k * P::W, mm = m < P::SLD + P::XLD ? m : m - P::SLD - P::XLD;
    mx[k] = mm >= P::SLD;
    const bool u = SW && mm >= P::SLD / 2;
    const void *mb = (u ? a.s1 : a.s0) + so;
    size_t ms = sbytes;
    if (!mx[k]) {
      const int lane_tile = mm * (8 / GPK) + lane / (8 * GPK), j = lane % (8 * GPK);
      vm[k] = (uint32_t)((lane_tile - (u ? P::NT16 / 2 : 0)) * NG * 32 + 4 * j);
    } else {
      const int idx = (mm - P::SLD) * 64 + lane, g = idx / P::BM, r = idx - g * P::BM;
      mb = ind ? a.seeds : a.seeds + row0;
      ms = ((size_t)KB * GPK * a.rows_pad - (ind ? 0 : row0)) * 4;
      vm[k] = r < mrows ? (uint32_t)(((size_t)g * a.rows_pad + (ind ? a.row_map[row0 + r] : r)) * 4)
                        : kDmaOOB;
    }
    mr[k] = rsrc_scalar(mb, ms);
  }
  // load l of this wave for k-block kb (scale group row g = first group of kb)
  auto issue1 = [&](int l, int buf, int kb, int g) {
    const uint32_t L = lds0 + buf * P::BYTES;
    if (l < P::AL) {
      const int blk = wave * P::AL + l;
      lds_dma<16>(PL == 2 && blk >= P::BM / 4 ? xr1 : xr0, L + P::A + blk * 1024, va[l < P::AL ? l : 0],
                 (uint32_t)kb * 256);
    } else if (l < P::AL + P::BL) {
      const int t = l - P::AL;
      lds_dma<16>(wr, L + P::B + (wave * P::BL + t) * 1024, vb[t < P::BL ? t : 0],
                 (uint32_t)kb * 1024);
    } else {
      const int k = l - P::AL - P::BL < P::MPW ? l - P::AL - P::BL : 0;
      lds_dma<4>(mr[k], L + P::S + (wave + k * P::W) * 256, vm[k],
                mx[k] ? (uint32_t)(kb * GPK * a.rows_pad) * 4 : (uint32_t)g * 32);
    }
  };
  const int kb0 = blockIdx.z * a.kper, KE = min(KB, kb0 + a.kper);
#pragma unroll
  for (int s = 0; s < 3; ++s)
    if (kb0 + s < KE) {
#pragma unroll
      for (int l = 0; l < P::LOADS; ++l)
        issue1(l, s, kb0 + s, GPK > 1 ? (kb0 + s) * GPK : (kb0 + s) / KPG);
    }

  // ---- LDS read offsets within a stage ----
  // A row 32 i + l31; the fragment of sub-step s, step q: chunk (GPK 1: 4 (2 q + h)
  // + s; else 4 s + 2 q + h) ^ (row & 15); rows and stages are 256-byte aligned,
  // so the constant part of the chunk is one XOR of the address
  const uint32_t ax = lds0 + P::A + (uint32_t)(wm * P::RM + l31) * 256 +
                      16 * ((GPK == 1 ? 4 * h : h) ^ l15);
  // B: tile (4 wn + 2 j + t16; SwiGLU: 2 wn + t16 of gate, of up), chunk 2 q + h, row l15
  constexpr int JT = SW ? P::NT16 / 2 : 2;  // tiles between j = 0 and j = 1
  const int bt = (SW ? 2 : 4) * wn + t16;
  const uint32_t bx = lds0 + P::B + (uint32_t)bt * 1024 + h * 256 + l15 * 16;
  const uint32_t sx = lds0 + P::S + (uint32_t)bt * 32 * GPK + l15 * 2;
  const uint32_t xx = lds0 + P::X + (uint32_t)(wm * P::RM + 4 * h) * 4;

  float acc[MT][2][16];
  // With one M-tile there are registers for two sets of partials: groups that
  // end with a sub-step (GPK 2, 4) alternate, so that a group's adds spread
  // over the next one's slots
  constexpr int PB = MT == 1 && GPK > 1 ? 2 : 1;
  f32x16_t p[PB][MT][2], seed[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = p[0][i][j][v] = p[PB - 1][i][j][v] = 0.f;
  u32x4_t af[2][P::NT][2], b[2][2], d[PL == 2 ? 4 : 2];
  constexpr bool SMALL = gg_small_offset(GPK, PL);
  constexpr uint32_t C = SMALL ? 0x41414141u : 0x43434343u;
  uint32_t dx = 0, dy = 0;
  uint32_t su[2], sn[2];            // scale bits of the group in flight, of the next
  float sc[2] = {0.f, 0.f};         // scales of the group being added
  uint32_t base = 0, nbase = 0;  // byte offsets of this k-block's stage and the next
  auto read_a1 = [&](uint32_t from, int s, int buf, int r) {  // fragment r = q NT + t
    const int q = r / P::NT, t = r % P::NT;
    const uint32_t at = (ax + from) ^ (16 * (GPK == 1 ? 8 * q + s : 4 * s + 2 * q));
    af[buf][t][q] = lds_at<u32x4_t>(at, t * (PL == 2 ? P::BM * 256 : 32 * 256));
  };
  auto read_b1 = [&](uint32_t from, int f) {  // fragment f = 2 q + j
    b[f & 1][f >> 1] = lds_at<u32x4_t>(from + bx, (f & 1) * JT * 1024 + (f >> 1) * 512);
  };
  auto read_seed1 = [&](uint32_t from, int g, int r) {  // rows 32 (r / 4) + 8 (r % 4) ..
    const f32x4_t t = lds_at<f32x4_t>(from + xx, g * P::BM * 4 + (32 * (r >> 2) + 8 * (r & 3)) * 4);
#pragma unroll
    for (int v = 0; v < 4; ++v) seed[r >> 2][4 * (r & 3) + v] = t[v];
  };
  auto read_scale = [&](uint32_t from, int g, int j) -> uint32_t {
    return lds_at<uint16_t>(from + sx, j * JT * 32 * GPK + g * 32);
  };
  // eight scaled adds: acc += s * p, half `c & 1` of tile (i, j)
  auto add8 = [&](int c, int pb = 0) {
    const int i = MT == 2 ? (c >> 1) & 1 : 0, j = MT == 2 ? c >> 2 : c >> 1;
#pragma unroll
    for (int v = 0; v < 8; ++v) acc[i][j][8 * (c & 1) + v] += sc[j] * p[pb][i][j][8 * (c & 1) + v];
    float *o = &acc[i][j][8 * (c & 1)];
    gg_pin(o[0], o[1], o[2], o[3], o[4], o[5], o[6], o[7]);
  };

  if (kb0 + 2 < KE)
    dma_wait_barrier<2 * P::LOADS>();
  else if (kb0 + 1 < KE)
    dma_wait_barrier<P::LOADS>();
  else
    dma_wait_barrier<0>();
  int cur = 0;

  if (wm * P::RM < mrows) {
#pragma unroll
    for (int r = 0; r < 2 * P::NT; ++r) read_a1(0, 0, 0, r);
#pragma unroll
    for (int f = 0; f < 4; ++f) read_b1(0, f);
#pragma unroll
    for (int r = 0; r < 4 * MT; ++r) read_seed1(0, 0, r);
    sn[0] = read_scale(0, 0, 0);
    sn[1] = read_scale(0, 0, 1);
    // fragments decoded before the first slot: one ahead of their use (PL 2: two)
    d[0] = gg_decode8<SMALL>(b[0][0][0]);
    if (PL == 2) d[1] = gg_decode8<SMALL>(b[1][0][0]);

    // One k-block.  Slot n of a sub-step issues one MFMA and the work beside
    // it: half a weight fragment's decode (one or two fragments ahead), an LDS
    // read for the next sub-step, a stage load, eight of the last group's
    // scaled adds.  A scheduling barrier ends every slot.
    auto kblock = [&](auto dma_tag, int kb, int g3) {
      constexpr bool DMA = decltype(dma_tag)::value;
      base = cur * P::BYTES;
      const int nxt = cur == 2 ? 0 : cur + 1;
      nbase = nxt * P::BYTES;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        constexpr int SPG = 4 / GPK;  // sub-steps per group
        const bool first = s % SPG == 0, last = s % SPG == SPG - 1;
        const int g = s / SPG, pb = PB == 2 ? g & 1 : 0;
#pragma unroll
        for (int n = 0; n < P::SLOTS; ++n) {
          constexpr int NT = P::NT, SL = P::SLOTS;
          const int q = n / (2 * NT);
          const int t = MT == 2 ? n & 1 : PL == 2 ? (n >> 1) & 1 : 0;
          const int j = MT == 2 ? (n >> 1) & 1 : n & 1;
          const int i = MT == 2 ? t : 0;
          if (s == 3 && n == 0) {
            if (DMA)
              dma_wait_barrier<P::LOADS>();
            else if (kb + 1 < KE)
              dma_wait_barrier<0>();
          }
          // LDS reads: the next sub-step's activations, the group's scales, the
          // next group's seeds, the next k-block's weights once their last
          // dword is decoded
          const uint32_t from = s == 3 ? nbase : base;
          if ((n & 1) == 0) read_a1(from, (s + 1) & 3, (s + 1) & 1, n / 2);
          if (first && n == 0) su[0] = sn[0], su[1] = sn[1];
          if (last && n >= SL / 2) {
            if (n < SL / 2 + 2)
              sn[n - SL / 2] = read_scale(from, GPK > 1 ? (g + 1) % GPK : 0, n - SL / 2);
            constexpr int RS = 4 * MT / (SL / 2);  // seed reads per slot: 2 (MT 1, PL 2: 1)
#pragma unroll
            for (int r = 0; r < RS; ++r)
              read_seed1(from, GPK > 1 ? (g + 1) % GPK : 0, (n - SL / 2) * RS + r);
          }
          if (s == 3) {
#pragma unroll
            for (int f = 0; f < 4; ++f)
              if (n == (NT == 1 ? f : PL == 2 ? (f < 3 ? f : 4) : 2 * f)) read_b1(nbase, f);
          }
          // the adds that must precede this slot's MFMA (it overwrites their p)
          if (MT == 2) {
            if (first && n == 0) add8(3), add8(4);
            if (first && n == 1) add8(5);
            if (first && n == 2) add8(6), add8(7);
            if (last && n == 6) {
              sc[0] = scale_to_f32<SDT>(su[0]);
              add8(0);
            }
            if (last && n == 7) {
              add8(1), add8(2);
            }
          } else {
            if (PB == 2) {
              if (first && n >= SL / 8 && n < SL / 8 + 4) add8(n - SL / 8, pb ^ 1);
            } else {
              if (first && n == 0) add8(0), add8(1);
              if (first && n == 1) add8(2), add8(3);
            }
          }
          p[pb][i][j] = mfma32_bf16(af[s & 1][t][q], d[PL == 2 ? 2 * q + j : (2 * q + j) & 1],
                                    first && q == 0 && (PL == 1 || t == 0) ? seed[i] : p[pb][i][j]);
#ifdef __HIP_DEVICE_COMPILE__
          // the seeds stay live past their last use: that MFMA must not take
          // their registers for its result (64 copies per k-block if it does)
          if (first && n == (MT == 2 ? 3 : 1)) {
            asm volatile("" ::"v"(seed[0]));
            if (MT == 2) asm volatile("" ::"v"(seed[MT - 1]));
          }
#endif
          // the scales replace the last group's once its adds are done
          if (last && n == SL - 1) {
            if (MT == 1) sc[0] = scale_to_f32<SDT>(su[0]);
            sc[1] = scale_to_f32<SDT>(su[1]);
          }
          // decode: half a fragment per slot (MT 1 with one plane: a whole one)
          const int f = (NT == 1 ? n + 1 : PL == 2 ? (n >> 1) + 2 : (n >> 1) + 1);
          const int fs = (s + (f >> 2)) & 3, fj = f & 1, fq = (f >> 1) & 1;
          const uint32_t w = b[fj][fq][fs];
          u32x4_t &o = d[PL == 2 ? f & 3 : f & 1];
          if (NT == 1) {
            o = gg_decode8<SMALL>(w);
          } else if ((n & 1) == 0) {
            const uint32_t lo = gg_nibbles<SMALL>(w, 0);
            dx = __builtin_amdgcn_perm(C, lo, 0x04010400u);
            dy = __builtin_amdgcn_perm(C, lo, 0x04030402u);
          } else {
            const uint32_t hi = gg_nibbles<SMALL>(w, 1);
            o.x = dx;
            o.y = dy;
            o.z = __builtin_amdgcn_perm(C, hi, 0x04010400u);
            o.w = __builtin_amdgcn_perm(C, hi, 0x04030402u);
          }
          if (DMA && s == 3) {
#pragma unroll
            for (int l = 0; l < P::LOADS; ++l)
              if (l * SL / P::LOADS == n) issue1(l, cur, kb + 3, g3);
          }
          __builtin_amdgcn_sched_barrier(0);
          asm volatile("" ::: "memory");
        }
      }
      cur = nxt;
    };
    int kb = kb0;
    int g3 = GPK > 1 ? (kb0 + 3) * GPK : (kb0 + 3) / KPG, gr = GPK > 1 ? 0 : (kb0 + 3) % KPG;
#pragma unroll 1
    for (; kb + 3 < KE; ++kb) {
      kblock(GgTrue{}, kb, g3);
      if (GPK > 1) {
        g3 += GPK;
      } else if (++gr == KPG) {
        gr = 0;
        ++g3;
      }
    }
#pragma unroll 1
    for (; kb < KE; ++kb) kblock(GgFalse{}, kb, 0);
#pragma unroll
    for (int c = MT == 2 ? 3 : 0; c < 4 * MT; ++c) add8(c, PB - 1);
  } else {
    // no live rows in this wave's tiles: its loads and barriers only
    int g3 = GPK > 1 ? (kb0 + 3) * GPK : (kb0 + 3) / KPG, gr = GPK > 1 ? 0 : (kb0 + 3) % KPG;
#pragma unroll 1
    for (int kb = kb0; kb + 1 < KE; ++kb) {
      if (kb + 3 < KE) {
        dma_wait_barrier<P::LOADS>();
#pragma unroll
        for (int l = 0; l < P::LOADS; ++l) issue1(l, cur, kb + 3, g3);
        if (GPK > 1) {
          g3 += GPK;
        } else if (++gr == KPG) {
          gr = 0;
          ++g3;
        }
      } else {
        dma_wait_barrier<0>();
      }
      cur = cur == 2 ? 0 : cur + 1;
    }
  }

  // ---- epilogue: D lane l holds column l31 and rows 8 (v / 4) + 4 h + v % 4 ----
  const bool live = wm * P::RM < mrows;
  if constexpr (SW) {
    if (a.part) {  // a slice of K: gate and up partials, columns n and N + n
      float *part = a.part + (size_t)blockIdx.z * a.M * 2 * a.N;
      const int n = T0 * 16 + 32 * wn + l31;
      if (live && n < a.N) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int m = wm * P::RM + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
            if (m >= mrows) continue;
            float *o = part + (size_t)(row0 + m) * 2 * a.N + n;
            o[0] = acc[i][0][v];
            o[a.N] = acc[i][1][v];
          }
      }
      return;
    }
    // hi / lo of silu(g) * u, through LDS so that the planes are stored 16 bytes a lane
    constexpr int pitch = P::OUTC * 2 + 16;
    uint8_t *lo_t = st + P::BM * pitch;
    __syncthreads();  // every wave is past its last read of the stages
    if (live) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = wm * P::RM + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
          const float y = silu_f32(acc[i][0][v]) * acc[i][1][v];
          const uint32_t hb = split_hi(y);
          const uint32_t o = m * pitch + (32 * wn + l31) * 2;
          *reinterpret_cast<uint16_t *>(st + o) = (uint16_t)hb;
          *reinterpret_cast<uint16_t *>(lo_t + o) = (uint16_t)split_lo(y, hb);
        }
    }
    __syncthreads();
    gg_store_tile<P::OUTC>(st, pitch, reinterpret_cast<uint16_t *>(a.y), row0, mrows, T0 * 16, a.N,
                           a.ldy, tid, 64 * P::W);
    gg_store_tile<P::OUTC>(lo_t, pitch, reinterpret_cast<uint16_t *>(a.y2), row0, mrows, T0 * 16,
                           a.N, a.ldy, tid, 64 * P::W);
    if (a.seeds_out) {
      // the seeds of the planes just written, for the GEMM that reads them as A
      // (in place of a pass over them): 16 consecutive lanes hold a row's 128
      // columns, 16 / GPK of them a group
      constexpr int L = 16 / GPK;
      for (int c = tid; c < P::BM * 16; c += 64 * P::W) {
        const int m = c >> 4, col = 8 * (c & 15), n = T0 * 16 + col;
        const uint32_t o = m * pitch + col * 2;
        float t = sum8_bf16(*reinterpret_cast<const u32x4_t *>(st + o)) +
                  sum8_bf16(*reinterpret_cast<const u32x4_t *>(lo_t + o));
        t = lane_group_sum<L>(t);
        if ((c & (L - 1)) == 0 && m < mrows && n < a.N)
          a.seeds_out[(size_t)(n / (8 * L)) * a.seeds_rp + row0 + m] = gg_seed_factor(GPK, 2) * t;
      }
    }
  } else if (a.part || a.epi == GG_F32) {
    const size_t ld = a.part ? gg_part_ld(a.N) : a.ldy;
    float *y = a.part ? a.part + (size_t)blockIdx.z * a.M * ld : reinterpret_cast<float *>(a.y);
    if (live) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = wm * P::RM + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
          const int n = T0 * 16 + 64 * wn + l31;
          if (m >= mrows) continue;
          float *o = y + (size_t)(row0 + m) * ld + n;
          if (n < a.N) o[0] = acc[i][0][v];
          if (n + 32 < a.N) o[32] = acc[i][1][v];
        }
    }
  } else {
    constexpr int pitch = P::BN * 2 + 16;
    __syncthreads();
    if (live) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = wm * P::RM + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
          uint8_t *o = st + m * pitch + (64 * wn + l31) * 2;
          *reinterpret_cast<uint16_t *>(o) = (uint16_t)f32_to_bf16_rne(acc[i][0][v]);
          *reinterpret_cast<uint16_t *>(o + 64) = (uint16_t)f32_to_bf16_rne(acc[i][1][v]);
        }
    }
    __syncthreads();
    gg_store_tile<P::OUTC>(st, pitch, reinterpret_cast<uint16_t *>(a.y), row0, mrows, T0 * 16, a.N,
                           a.ldy, tid, 64 * P::W);
  }
}

// The sum of the nsl slices' partials at part + i (slices `stride` apart), in
// slice order; W slices' loads are issued before their adds (clamped: all in
// range) and pinned there.
template <int W>
CAI4_DEV f32x4_t sum_slices_by(const float *part, size_t stride, size_t i, int nsl) {
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
  for (int z0 = 0; z0 < nsl; z0 += W) {
    f32x4_t v[W];
#pragma unroll
    for (int z = 0; z < W; ++z)
      v[z] = *reinterpret_cast<const f32x4_t *>(part + (size_t)min(z0 + z, nsl - 1) * stride + i);
#pragma unroll
    for (int z = 0; z < W; ++z) asm volatile("" : "+v"(v[z]));
#pragma unroll
    for (int z = 0; z < W; ++z)
      if (z0 + z < nsl) s = z0 + z ? s + v[z] : v[z];
  }
  return s;
}
// Loads past the last slice repeat it, so few slices take the narrow form.  Back
// to back (us, four / eight wide, bf16 out): 3 slices of 333 x 4096 2.9 / 3.5, 4 of
// 200 x 7168 2.9 / 3.6, 4 of 512 x 4096 4.1 / 4.8, 2 of 1024 x 4096 6.3 / 7.3; up to
// 100 x 4096 both at the launch floor (2.4); eight slices 2.40 / 2.44 (16 x 4096),
// 11.8 / 12.6 (512 x 4096): there the order of the loads matters little.
CAI4_DEV f32x4_t sum_slices(const float *part, size_t stride, size_t i, int nsl) {
  return nsl <= 4 ? sum_slices_by<4>(part, stride, i, nsl) : sum_slices_by<8>(part, stride, i, nsl);
}

// y = sum over the K slices' partials, in slice order; bf16 (RNE) or f32.  The
// partials' rows are gg_part_ld(N) apart: a thread's four columns are aligned
// and in one row whatever N is (those past N are read and not used).
__global__ __launch_bounds__(256) void gg_reduce_kernel(const float *part, void *y, int M, int N,
                                                        int ldy, int nsl, int out_f32) {
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  const uint32_t ld = gg_part_ld(N);
  const size_t n = (size_t)M * ld;
  if (i >= n) return;  // n is a multiple of 4
  const f32x4_t s = sum_slices(part, n, i, nsl);
  const size_t r = n >> 32 ? i / ld : (uint32_t)i / ld;
  const int c = (int)(i - r * ld);
  const bool four = c + 4 <= N;
  const size_t o = r * ldy + c;
  if (out_f32) {
    float *yf = reinterpret_cast<float *>(y) + o;
    if (four && ((uintptr_t)yf & 15) == 0) {
      *reinterpret_cast<f32x4_t *>(yf) = s;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < N) yf[e] = s[e];
    }
  } else {
    uint16_t *yb = reinterpret_cast<uint16_t *>(y) + o;
    u32x2_t b;
    b.x = f32_to_bf16_rne(s.x) | (f32_to_bf16_rne(s.y) << 16);
    b.y = f32_to_bf16_rne(s.z) | (f32_to_bf16_rne(s.w) << 16);
    if (four && ((uintptr_t)yb & 7) == 0) {
      *reinterpret_cast<u32x2_t *>(yb) = b;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < N) yb[e] = (uint16_t)(b[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// The SwiGLU of gate / up partials [nsl][M][gate N | up N], in slice order: the
// hi / lo planes of silu(g) * u ([M, ldy]) and, with seeds, their seeds per
// group of 8 L columns (N a multiple of 8 L): what the tile kernel's epilogue
// writes when K is not split.  A thread per eight columns.
template <int L>
__global__ __launch_bounds__(256) void gg_swiglu_reduce_kernel(const float *part, uint16_t *hi,
                                                               uint16_t *lo, float *seeds, int M,
                                                               int N, int ldy, int nsl,
                                                               int seeds_rp) {
  const int per = N / 8;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)M * per) return;  // whole groups of L lanes: per is a multiple of L
  const size_t r = t / per;
  const int c = 8 * (int)(t - r * per);
  const size_t stride = (size_t)M * 2 * N, i = r * 2 * N + c;
  float g[8], u[8];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const f32x4_t a = sum_slices(part, stride, i + 4 * q, nsl);
    const f32x4_t b = sum_slices(part, stride, i + N + 4 * q, nsl);
#pragma unroll
    for (int v = 0; v < 4; ++v) g[4 * q + v] = a[v], u[4 * q + v] = b[v];
  }
  u32x4_t h, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t hb[2], lb[2];
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const float y = silu_f32(g[2 * e + v]) * u[2 * e + v];
      hb[v] = split_hi(y);
      lb[v] = split_lo(y, hb[v]);
    }
    h[e] = hb[0] | (hb[1] << 16);
    l[e] = lb[0] | (lb[1] << 16);
  }
  const size_t o = r * ldy + c;
  *reinterpret_cast<u32x4_t *>(hi + o) = h;
  *reinterpret_cast<u32x4_t *>(lo + o) = l;
  if (seeds) {
    const float sum = lane_group_sum<L>(sum8_bf16(h) + sum8_bf16(l));
    if ((t & (L - 1)) == 0)
      seeds[(size_t)(c / (8 * L)) * seeds_rp + r] = gg_seed_factor(16 / L, 2) * sum;
  }
}

// ---------------------------------------------------------------------------
// gg_prep: seeds (and converted activations), one wave per row
// ---------------------------------------------------------------------------

// One wave per row and kGgPrepPasses passes of 512 columns (blockIdx.y: which),
// every load issued before the first sum: the pass is latency-bound, so it is
// spread over as many waves as the rows and columns give.
constexpr int kGgPrepPasses = 2;

template <int L>
__global__ __launch_bounds__(256) void gg_prep_kernel(int mode, const void *src, const void *src2,
                                                      uint16_t *out, uint16_t *out2, float *seeds,
                                                      int rows, int rows_pad, int K) {
  constexpr int P = kGgPrepPasses;
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;  // whole waves; no barriers here
  const int gw = 8 * L;   // columns per seed group
  const size_t srow = (size_t)r;
  const int c0 = blockIdx.y * P * 512 + 8 * lane;
  u32x4_t v[P], w[P];  // 8 columns a pass: bf16 hi (and lo), or two halves of f32
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int c = c0 + 512 * q;
    v[q] = w[q] = u32x4_t{0u, 0u, 0u, 0u};
    if (c >= K) continue;
    if (mode <= 1) {
      v[q] = *reinterpret_cast<const u32x4_t *>(static_cast<const uint16_t *>(src) + srow * K + c);
      if (mode == 1)
        w[q] = *reinterpret_cast<const u32x4_t *>(static_cast<const uint16_t *>(src2) + srow * K + c);
    } else {
      const float *f = static_cast<const float *>(src) + srow * K + c;
      v[q] = *reinterpret_cast<const u32x4_t *>(f);
      w[q] = *reinterpret_cast<const u32x4_t *>(f + 4);
    }
  }
#pragma unroll
  for (int q = 0; q < P; ++q) {
    const int c = c0 + 512 * q;
    float t;
    if (mode <= 1) {
      t = sum8_bf16(v[q]);
      if (mode == 1) t += sum8_bf16(w[q]);
    } else if (mode == 2) {
      u32x4_t o;
      o.x = f32_to_bf16_rne(bitsf(v[q].x)) | (f32_to_bf16_rne(bitsf(v[q].y)) << 16);
      o.y = f32_to_bf16_rne(bitsf(v[q].z)) | (f32_to_bf16_rne(bitsf(v[q].w)) << 16);
      o.z = f32_to_bf16_rne(bitsf(w[q].x)) | (f32_to_bf16_rne(bitsf(w[q].y)) << 16);
      o.w = f32_to_bf16_rne(bitsf(w[q].z)) | (f32_to_bf16_rne(bitsf(w[q].w)) << 16);
      if (c < K) *reinterpret_cast<u32x4_t *>(out + (size_t)r * K + c) = o;
      t = sum8_bf16(o);
    } else {
      u32x4_t hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0 = bitsf(e < 2 ? v[q][2 * e] : w[q][2 * e - 4]);
        const float x1 = bitsf(e < 2 ? v[q][2 * e + 1] : w[q][2 * e - 3]);
        const uint32_t h0 = split_hi(x0), h1 = split_hi(x1);
        hi[e] = h0 | (h1 << 16);
        lo[e] = split_lo(x0, h0) | (split_lo(x1, h1) << 16);
      }
      if (c < K) {
        *reinterpret_cast<u32x4_t *>(out + (size_t)r * K + c) = hi;
        *reinterpret_cast<u32x4_t *>(out2 + (size_t)r * K + c) = lo;
      }
      t = sum8_bf16(hi) + sum8_bf16(lo);
    }
    t = lane_group_sum<L>(t);
    if ((lane & (L - 1)) == 0 && c < K)
      seeds[(size_t)(c / gw) * rows_pad + r] =
          (mode & 1 ? gg_seed_factor(16 / L, 2) : gg_seed_factor(16 / L, 1)) * t;
  }
}

template <int MT, int WM, int WN, int GPK, int PL, bool SW>
hipError_t gg_launch(const GgArgs &a, int rows_y, int nsl, hipStream_t st) {
  using P = Gg<MT, WM, WN, GPK, PL, SW>;
  const dim3 grid((a.N + P::OUTC - 1) / P::OUTC, rows_y ? rows_y : (a.M + P::BM - 1) / P::BM, nsl);
  if (a.sdt)
    hipLaunchKernelGGL((gg_kernel<MT, WM, WN, GPK, PL, SW, SCALE_F16>), grid, dim3(64 * P::W), 0, st,
                       a);
  else
    hipLaunchKernelGGL((gg_kernel<MT, WM, WN, GPK, PL, SW, SCALE_BF16>), grid, dim3(64 * P::W), 0,
                       st, a);
  return hipGetLastError();
}

// rows_y: workgroup rows (0: as many as a.M takes); nsl: slices of K.
template <int MT, int WM, int WN, int PL, bool SW>
hipError_t gg_launch_g(const GgArgs &a, int rows_y, int nsl, hipStream_t st) {
  switch (a.G == 32 ? 4 : a.G == 64 ? 2 : 1) {
    case 4: return gg_launch<MT, WM, WN, 4, PL, SW>(a, rows_y, nsl, st);
    case 2: return gg_launch<MT, WM, WN, 2, PL, SW>(a, rows_y, nsl, st);
    default: return gg_launch<MT, WM, WN, 1, PL, SW>(a, rows_y, nsl, st);
  }
}

// How a dense GEMM runs: the tile and the slices of K.
struct GgPlan {
  bool small;  // one-plane, not SwiGLU: 64 x 128 tiles (4 waves, two workgroups per CU)
  int nsl, kper;
};

// The plan with the least estimated time, from times measured on the card: a
// k-block of a 128 x 256 (64 x 256 with two planes, 64 x 128) tile, a tile's
// prologue and epilogue, and the reduce launch with its partials written and
// read.  Slices of at least four k-blocks (the pipeline's depth), at most
// eight.  max_slices 1: no partials (a workspace that cannot grow).
// A small tile alone on its CU takes 0.6 of the time per k-block of two, and a
// split of two planes 1.5 us more than its reduce: without the two, short K was
// split to its loss (163 x 10703 x 1536, G 32: 26.5 us in three slices of large
// tiles, 21.0 in one of small ones; 384 x 2431 x 1152 of f32 rows 24.8 / 22.7).
// Over 92 shapes of 64-2048 bf16 rows with every plan measured, the one chosen
// is 2.4 % behind the best on average; of 33-500 f32 rows, 36 shapes, 1.1 %.
GgPlan gg_plan(int M, int N, int K, int G, bool two, bool sw, int num_cus, int max_slices) {
  const int KB = K / 128, ncol = sw ? 2 * N : N;
  const double tkb128 = G == 32 ? 2.4 : G == 64 ? 1.9 : 1.5;
  const double tkb64x2 = G == 32 ? 1.6 : 1.4, tkb_small = G == 32 ? 1.8 : 1.25;
  constexpr double kTile = 6.0, kTileSmall = 4.5, kAlone = 0.6, kBytesPerUs = 1.2e7;
  const double reduce = two && !sw ? 4.5 : 3.0;
  GgPlan best{false, 1, KB};
  double best_t = -1.0;
  for (int small = 0; small < (two || sw ? 1 : 2); ++small) {
    const int bm = small || two ? 64 : 128, bn = small ? 128 : sw ? 128 : 256;
    const long tiles = (long)((N + bn - 1) / bn) * ((M + bm - 1) / bm);
    const long slots = small ? 2L * num_cus : num_cus;
    for (int s = 1; s <= max_slices && s <= 8; ++s) {
      if (s > 1 && KB / s < 4) break;
      const int kper = (KB + s - 1) / s, nsl = (KB + kper - 1) / kper;
      const long rounds = (tiles * nsl + slots - 1) / slots;
      const double tkb = !small ? (two ? tkb64x2 : tkb128)
                         : tiles * nsl <= num_cus ? kAlone * tkb_small : tkb_small;
      double t = rounds * (kper * tkb + (small ? kTileSmall : kTile));
      if (nsl > 1) t += reduce + (double)nsl * M * ncol * 8.0 / kBytesPerUs;
      if (best_t < 0 || t < best_t) {
        best_t = t;
        best = GgPlan{small != 0, nsl, kper};
      }
    }
  }
  return best;
}

}  // namespace

bool gg_supported(int K, int G, int tiled) {
  return tiled && K % 128 == 0 && (G == 32 || G == 64 || G % 128 == 0) && K % G == 0;
}

int gg_rows_pad(int rows) { return (rows + 127) / 128 * 128; }

hipError_t gg_prep(int mode, const void *src, const void *src2, uint16_t *out, uint16_t *out2,
                   float *seeds, int rows, int rows_pad, int K, int G, hipStream_t st) {
  if (rows <= 0) return hipSuccess;
  const dim3 grid((rows + 3) / 4, (K + 512 * kGgPrepPasses - 1) / (512 * kGgPrepPasses)), block(256);
  const int gw = gg_group_width(G);
  if (gw == 32)
    hipLaunchKernelGGL(gg_prep_kernel<4>, grid, block, 0, st, mode, src, src2, out, out2, seeds,
                       rows, rows_pad, K);
  else if (gw == 64)
    hipLaunchKernelGGL(gg_prep_kernel<8>, grid, block, 0, st, mode, src, src2, out, out2, seeds,
                       rows, rows_pad, K);
  else
    hipLaunchKernelGGL(gg_prep_kernel<16>, grid, block, 0, st, mode, src, src2, out, out2, seeds,
                       rows, rows_pad, K);
  return hipGetLastError();
}

namespace {
size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }
}  // namespace

hipError_t gg_reduce_slices(const GgArgs &a, int nsl, hipStream_t st) {
  const bool sw = a.epi == GG_SWIGLU_HILO;
  if (sw) {
    const size_t n = (size_t)a.M * (a.N / 8);
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    uint16_t *hi = static_cast<uint16_t *>(a.y), *lo = static_cast<uint16_t *>(a.y2);
    switch (gg_group_width(a.G)) {
      case 32:
        hipLaunchKernelGGL(gg_swiglu_reduce_kernel<4>, grid, block, 0, st, a.part, hi, lo,
                           a.seeds_out, a.M, a.N, a.ldy, nsl, a.seeds_rp);
        break;
      case 64:
        hipLaunchKernelGGL(gg_swiglu_reduce_kernel<8>, grid, block, 0, st, a.part, hi, lo,
                           a.seeds_out, a.M, a.N, a.ldy, nsl, a.seeds_rp);
        break;
      default:
        hipLaunchKernelGGL(gg_swiglu_reduce_kernel<16>, grid, block, 0, st, a.part, hi, lo,
                           a.seeds_out, a.M, a.N, a.ldy, nsl, a.seeds_rp);
    }
    return hipGetLastError();
  }
  const size_t n = (size_t)a.M * gg_part_ld(a.N);
  // small outputs: one wave per workgroup, so that every CU has one (16 x 4096 is
  // 64 workgroups of 256).  Back to back the two sizes are within 1 % up to 100 x
  // 4096, 4 % at 1024 x 7168 either way: the line is not sharp.
  const unsigned bs = n / 4 >= 1u << 17 ? 256 : 64;
  hipLaunchKernelGGL(gg_reduce_kernel, dim3((unsigned)((n / 4 + bs - 1) / bs)), dim3(bs), 0, st,
                     a.part, a.y, a.M, a.N, a.ldy, nsl, a.epi == GG_F32 ? 1 : 0);
  return hipGetLastError();
}

size_t gg_dense_workspace(int M, int N, int K, int G, int amode, int epi, int num_cus,
                          bool have_seeds, int max_slices, int rows) {
  const bool sw = epi == GG_SWIGLU_HILO;
  if (!rows) rows = M;
  size_t b = have_seeds ? 0 : al256((size_t)(K / gg_group_width(G)) * gg_rows_pad(rows) * 4);
  if (amode == GG_A_F32) b += 2 * al256((size_t)rows * K * 2);  // the A planes
  const GgPlan p = gg_plan(M, N, K, G, amode != GG_A_BF16, sw, num_cus, max_slices);
  return b + (p.nsl > 1 ? (size_t)p.nsl * rows * (sw ? 2 * (size_t)N : gg_part_ld(N)) * 4 : 0);
}

hipError_t gg_dense(GgArgs a, int amode, void *ws, int num_cus, hipStream_t st, int max_slices) {
  a.row_map = nullptr;
  a.tiles = nullptr;
  a.tile_split = 1;
  a.hilo = amode != GG_A_BF16;
  const bool sw = a.epi == GG_SWIGLU_HILO;
  if (a.seeds_out && !sw) return hipErrorInvalidValue;
  uint8_t *w = static_cast<uint8_t *>(ws);
  if (!a.seeds) {
    a.rows_pad = gg_rows_pad(a.M);
    float *seeds = reinterpret_cast<float *>(w);
    a.seeds = seeds;
    w += al256((size_t)(a.K / gg_group_width(a.G)) * a.rows_pad * 4);
    hipError_t e;
    if (amode == GG_A_F32) {
      uint16_t *hi = reinterpret_cast<uint16_t *>(w);
      w += al256((size_t)a.M * a.K * 2);
      uint16_t *lo = reinterpret_cast<uint16_t *>(w);
      w += al256((size_t)a.M * a.K * 2);
      e = gg_prep(3, a.x, nullptr, hi, lo, seeds, a.M, a.rows_pad, a.K, a.G, st);
      a.x = hi;
      a.x2 = lo;
    } else {
      e = gg_prep(a.hilo ? 1 : 0, a.x, a.x2, nullptr, nullptr, seeds, a.M, a.rows_pad, a.K, a.G,
                  st);
    }
    if (e != hipSuccess) return e;
  } else if (amode == GG_A_F32) {
    return hipErrorInvalidValue;  // the planes are made here, their seeds with them
  }
  const GgPlan p = gg_plan(a.M, a.N, a.K, a.G, a.hilo, sw, num_cus, max_slices);
  a.kper = p.kper;
  a.part = p.nsl > 1 ? reinterpret_cast<float *>(w) : nullptr;
  hipError_t e;
  if (a.hilo)
    e = sw ? gg_launch_g<1, 2, 4, 2, true>(a, 0, p.nsl, st)
           : gg_launch_g<1, 2, 4, 2, false>(a, 0, p.nsl, st);
  else if (sw)
    e = gg_launch_g<2, 2, 4, 1, true>(a, 0, p.nsl, st);
  else if (p.small)
    e = gg_launch_g<1, 2, 2, 1, false>(a, 0, p.nsl, st);
  else
    e = gg_launch_g<2, 2, 4, 1, false>(a, 0, p.nsl, st);
  if (e != hipSuccess || p.nsl == 1) return e;
  return gg_reduce_slices(a, p.nsl, st);
}

hipError_t gg_grouped(const GgArgs &a0, int max_tiles, hipStream_t st) {
  GgArgs a = a0;
  a.kper = a.K / 128;
  a.part = nullptr;
  if (max_tiles <= 0) return hipSuccess;
  const bool sw = a.epi == GG_SWIGLU_HILO;
  if (a.seeds_out && (!sw || a.seeds_rp <= 0)) return hipErrorInvalidValue;
  // rows through a row map: one bf16 plane, x rows addressable in 31 bits
  if (a.row_map && (a.hilo || a.x_rows <= 0 || (size_t)a.x_rows * a.K * 2 > 0x7FFFFFFFu))
    return hipErrorInvalidValue;
  if (a.hilo) {  // 64-row tiles: two per table entry
    a.tile_split = kGgChunkRows / 64;
    if (sw) return gg_launch_g<1, 2, 4, 2, true>(a, max_tiles * a.tile_split, 1, st);
    return gg_launch_g<1, 2, 4, 2, false>(a, max_tiles * a.tile_split, 1, st);
  }
  a.tile_split = kGgChunkRows / 128;
  if (sw) return gg_launch_g<2, 2, 4, 1, true>(a, max_tiles * a.tile_split, 1, st);
  return gg_launch_g<2, 2, 4, 1, false>(a, max_tiles * a.tile_split, 1, st);
}

}  // namespace cai4
