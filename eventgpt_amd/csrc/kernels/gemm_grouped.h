// Grouped products of a few rows a group (gemm_grouped.hip).
#pragma once
#include "gemm_common.h"

namespace evgpt {

// Where it serves and is ahead; rows: in all groups
bool gemm_grouped_few_serves(const GemmParams& p, int rows);
void launch_gemm_grouped_few(const GemmParams& p, int rows, hipStream_t st);

}  // namespace evgpt
