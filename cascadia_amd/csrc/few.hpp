// few.hpp -- INT4 weight-only GEMM for a few token rows (2 .. 32) over
// MFMA-tiled weights: a decode batch's FFN and projections.
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

// f32 partials of the slices of K (0: K is not split).  ncol: output columns (N).
size_t few_workspace(int M, int N, int K, bool sw, int num_cus, int max_slices = 64);

// y = x W^T (a.x bf16 [M, K], or with a.hilo two planes a.x, a.x2), or the
// SwiGLU planes of a gate / up pair (a.epi), M <= 32; a.part is set from ws.
hipError_t few_gemm(GgArgs a, void *ws, int num_cus, hipStream_t st, int max_slices = 64);

}  // namespace cai4
