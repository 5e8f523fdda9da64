// The 4-wave kernel of 256 x 256 tiles (gemm_quad.hip).
#pragma once
#include "gemm_common.h"

namespace evgpt {

// What it takes: at least two K-tiles in every split, byte offsets of a tile's rows within 31 bits, and an output it stores in whole
// 16-byte chunks (bf16, plain or gated; fp32 sums as they are) or fp32 slabs.
bool gemm_quad_serves(const GemmParams& p);
// Whether it is ahead of the 8-wave kernel there; tiles: of the output, times the splits
bool gemm_quad_ahead(const GemmParams& p, int tiles);
void launch_gemm_quad(const GemmParams& p, int grid, hipStream_t st);

}  // namespace evgpt
