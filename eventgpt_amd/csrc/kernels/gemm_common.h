// What the GEMM kernels share: their parameters, the walk over the tiles of an output, counted waits.
#pragma once
#include "common.h"
#include "../evgpt_kernels.h"

namespace evgpt {

constexpr int BK = 64;

typedef const void __attribute__((address_space(1)))* gptr_t;
typedef void __attribute__((address_space(3)))* lptr_t;

struct GemmParams {
  const bf16_t* A;     // [M][lda]
  const bf16_t* W;     // [N][ldw]
  bf16_t* C;           // [M][ldc]
  const bf16_t* bias;  // [N] or null
  const bf16_t* res;   // [M][ldc] or null (may alias C)
  float* Cf;           // optional fp32 output [M][ldc] (C may be null)
  int M, N, K, lda, ldw, ldc, act;
  // optional row-argmax partials: [M][n_part] (value, index), n_part = tiles_n * WGN,
  // taken on the fp32 accumulators so C is never written.
  float* amax_val;
  int* amax_idx;
  // split-K: blockIdx = tile * splitk + ks; each split covers k_per_split (a
  // multiple of 64) of K and stores its raw fp32 tile to partial[ks][M][N]; a
  // second launch sums the slabs and applies the epilogue.
  int splitk, k_per_split;
  float* partial;
  int raw_partial;     // store the fp32 slab even when splitk == 1 (a fused consumer sums it)
  // K-strided operands only: k-rows that exist in memory.  A padded contraction (K rounded up
  // to 64) re-reads the last real row for k >= k_rows; the other operand holds zeros there.
  int ka_rows, kw_rows;
  // Gated-linear-unit mode (K-contiguous operands, no K split): W is [gate rows | up rows], each
  // glu_half rows; the output has glu_half (= N) columns  silu(x·gate_n) * (x·up_n).  A block stages,
  // for every wave column, half of its tile rows from the gate region and the matching half from the
  // up region, so a lane holds both factors of its output columns and the intermediate [M, 2I]
  // tensor is never written.
  int glu_half;
  int glu_act;         // GluAct of that mode
  // K-contiguous operands only: the columns a row really has when that is not a multiple of 64
  // (0: K itself).  K is then the contraction rounded up to 64, and the last K-tile's chunks past
  // k_cols -- which in memory are the start of the next row -- are staged as zeros.
  int k_cols;
  // RoPE + cache-append epilogue of a q | k | v projection (ROPE instance of the 128 x 128 tile, head_dim
  // 128 so that a column tile is one head): rotated q rows go to rope_q [M][Hq * 128], rotated k and
  // plain v rows into the cache slices rope_k / rope_v [Hkv][l_max][128] at position pos0[0] + row.
  bf16_t* rope_q; bf16_t* rope_k; bf16_t* rope_v;
  const float* rope_cos; const float* rope_sin;     // [l_max][64]
  const int* rope_pos0;
  int rope_hq, rope_hkv, rope_lmax;
  int rope_head0;      // the head of the output's first column (the last heads of a projection are a launch of their own)
  // row tiles per group of the tile walk (0: whole columns); set by the launchers
  int group_m;
  int rows_epilogue;   // 8-wave kernel: bf16 output stored as whole lines through LDS (set by launch_256)
  // 4-wave kernel with split K: workgroup index = split * tiles + tile instead of tile * splits + split
  int split_major;
  // Grouped product (GRP instances of the 4-wave kernel): the rows are sorted into grp_count groups (group e: rows
  // grp_start[e] .. grp_start[e + 1]), each with its own weights W + e * grp_wstride; row i is row grp_perm[i] / grp_top of
  // A (grp_perm null: row i) and goes to row i of C.
  const int* grp_start; const int* grp_perm;
  int grp_count, grp_top;
  long long grp_wstride;
};

// What a kernel needs for its first loads, as arguments of their own ahead of the other parameters: with kernel argument preload
// (build.py) they are in scalar registers when a wave starts; a structure is fetched.  Vision tower, one frame, 1867 us without preload, 1830
// with it where arguments were scalars already (norms, slab sums), 1800 with these.  cols_: the gated half, or -- instances with a short last K-tile, which
// no gated product takes -- the rows' true columns.
#define EVGPT_GEMM_ARGS                                                                                                              \
  const bf16_t *a_, const bf16_t *w_, int m_, int n_, int k_, int lda_, int ldw_, int splitk_, int k_per_split_, int cols_, GemmParams p
#define EVGPT_GEMM_TAKE \
  p.A = a_, p.W = w_, p.M = m_, p.N = n_, p.K = k_, p.lda = lda_, p.ldw = ldw_, p.splitk = splitk_, p.k_per_split = k_per_split_, p.glu_half = cols_
#define EVGPT_GEMM_PASS_COLS(p, cols) (p).A, (p).W, (p).M, (p).N, (p).K, (p).lda, (p).ldw, (p).splitk, (p).k_per_split, cols, p
#define EVGPT_GEMM_PASS(p) EVGPT_GEMM_PASS_COLS(p, (p).glu_half)

// wait until at most `n` of this wave's direct-to-LDS loads are still in flight
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N <= 24, "vmcnt literal");
  if constexpr (N == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else if constexpr (N == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
  else if constexpr (N == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
  else if constexpr (N == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else if constexpr (N == 5) asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
  else if constexpr (N == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  else if constexpr (N == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  else if constexpr (N == 9) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
  else if constexpr (N == 10) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
  else if constexpr (N == 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  else if constexpr (N == 15) asm volatile("s_waitcnt vmcnt(15)" ::: "memory");
  else if constexpr (N == 16) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  else if constexpr (N == 18) asm volatile("s_waitcnt vmcnt(18)" ::: "memory");
  else if constexpr (N == 24) asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
  else static_assert(N == 0, "add the literal");
}

// 16 bytes per lane from `src + voff` (range-checked against `bytes`: past it, zeros) straight
// into LDS at `lds + 16 * lane`.  Kept out of the kernel template: the descriptor type exists
// only in the device pass, and a template body the host pass cannot instantiate loses its
// launch stub.
__device__ __forceinline__ void buffer_to_lds16(const unsigned char* src, int bytes, unsigned char* lds, int voff) {
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(src), 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)lds, 16, voff, 0, 0, 0);
}

// Tile index -> (row tile, column tile).  Consecutive tiles walk down a group of about `group_m` row tiles, then
// move one column tile over, group after group (group_m <= 0 or few row tiles: whole columns).  The workgroups
// of an XCD that run side by side then cover a near-square patch of the output and share its operand panels
// in their L2 -- about 8 + 4 panels for 32 tiles instead of 32 + 1 when a tall output is walked column by
// column.  The groups are balanced (27 row tiles at group_m = 8: 7, 7, 7, 6).  Only from 3 group_m row tiles on:
// every group streams the whole weight matrix again, which a tall, compute-bound product takes from the
// die-level cache, while a few hundred rows are bound by exactly that stream (636-token prefill with groups of
// five 64-row tiles: 11.55 -> 11.89 ms; 8192^3 on the 8-wave kernel 1182 -> 1441 TFLOP/s, 4643 x 12288 x 4096 on
// 128 x 128 tiles 929 -> 1070, 19 row tiles of 256: no change either way).
__device__ __forceinline__ void tile_walk(int tile, int tiles_m, int tiles_n, int group_m, int& tm, int& tn) {
  if (group_m > 0 && tiles_m >= 3 * group_m) {
    const int ngroups = (tiles_m + group_m - 1) / group_m;
    const int gsize = (tiles_m + ngroups - 1) / ngroups;
    const int per_group = gsize * tiles_n;
    const int g = tile / per_group, within = tile % per_group;
    const int first = g * gsize;
    const int rows = min(gsize, tiles_m - first);
    tm = first + within % rows;
    tn = within / rows;
  } else {
    tm = tile % tiles_m;
    tn = tile / tiles_m;
  }
}

}  // namespace evgpt
