// Products of one round of workgroups on a deep ring (gemm_ring.hip).
#pragma once
#include "gemm_common.h"

namespace evgpt {

enum RingTile { RING_NONE = 0, RING_64x64, RING_128x64, RING_64x128, RING_64x192, RING_128x128 };
// The tile it takes the product on, where it is ahead of the tiles of gemm.hip; K-contiguous operands, splits as set in `p`.  w8: the other
// choice is the 64 x 128 tile of eight waves.
RingTile gemm_ring_tile(const GemmParams& p, bool w8);
void launch_gemm_ring(const GemmParams& p, RingTile tile, hipStream_t st);

}  // namespace evgpt
