// few.hpp -- INT4 weight-only GEMM for a few token rows (up to 32) over
// MFMA-tiled weights: the two GEMMs of a decode batch's FFN.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "grouped.hpp"

namespace cai4 {

constexpr int kFewMaxRows = 32;

// Whether the kernel takes this shape: 1 .. 32 rows, MFMA-tiled weights, K a
// multiple of 128, G 32, 64 or a multiple of 128.
bool few_supported(int M, int N, int K, int G, int tiled);

// Bytes of the f32 partials of the slices of K (0: K is not split) for M rows of
// N output columns, or (sw) of N gate and N up columns.
size_t few_workspace(int M, int N, int K, bool sw, int num_cus);

// The SwiGLU planes of a gate / up pair (a.epi GG_SWIGLU_HILO, a.x bf16 [M, K]),
// or bf16 y = x W^T of two planes (a.hilo: a.x, a.x2); M <= 32; a.part is set
// from ws.
hipError_t few_gemm(GgArgs a, void *ws, int num_cus, hipStream_t st);

}  // namespace cai4
