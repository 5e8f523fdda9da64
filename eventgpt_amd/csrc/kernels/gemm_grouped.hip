// Grouped products (experts) of a few rows a group: a stream of the weights, as gemm_fewrow_kernel is for one matrix.
//
// A decode step of 32 rows gives each of 8 experts about 8 rows, and what counts is how fast the experts' matrices arrive.  The
// 32 x 128 tile of the general kernel fetches 128 bytes of a weight row per K-tile and makes 352 workgroups of the gate / up product and
// 128 of the down product.  Here a tile is 32 output columns: 32 gate and 32 up rows, or 32 rows whose K is divided between
// two pairs of waves (704 and 512 workgroups), in K-tiles of 128, 256 contiguous bytes of a weight row each; rows that a group
// does not have are neither fetched nor, past the first 16, multiplied.
//
// us, general tile -> this, weights from memory, 8 experts of 4096 x 5504 (two a row, 8 to 64 rows): gate / up 139 -> 128 (721 MB: 5.6 TB/s),
// down 92 -> 75; of 2048 x 2816 42.7 -> 40.0 and 23.0 -> 18.1.  Two stages: gate / up 155, down 94 where three take 132 and 75; four: down level.
#include <type_traits>

#include "gemm_common.h"

namespace evgpt {

namespace {

constexpr int TK = 128, AM = 32, TN = 32, STAGES = 3, RUN = 16;

// ONE: all rows are one group (a dense gated product of a decode step); its gate and up sums are not rounded on the way
template <bool GLU, bool ONE>
__global__ __launch_bounds__(256) void gemm_grouped_few_kernel(EVGPT_GEMM_ARGS) {
  EVGPT_GEMM_TAKE;
  constexpr int W_ROWS = GLU ? 2 * TN : TN, WI = W_ROWS / 16;      // staging instructions per wave: 4 rows x 256 bytes each
  constexpr int A_BYTES = AM * TK * 2, STAGE = A_BYTES + W_ROWS * TK * 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles_n = p.N / TN;
  // The XCDs take turns in runs of sixteen tiles: the grid is for the most tiles there can be, and cut into eight ranges it left the last XCDs
  // those that there are not (no more rows than experts: 0.66 of the general tile's time at the mean, in ranges 0.93; gated 0.69 and 0.98).
  // Ranges of the tiles there are lie a power of two apart for many shapes and meet in the same channels (0.67, more rows than experts
  // level), single tiles read 4096 k slower than runs do (0.85 against 0.79).
  const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
  int tile = ((turn / RUN) * 8 + xcd) * RUN + turn % RUN;
  int e = 0, first = 0, all = p.M;
  if constexpr (ONE) {
    if (tile >= (p.M + AM - 1) / AM * tiles_n) return;
  } else {
    e = group_of_tile(p.grp_start, p.grp_count, AM, tiles_n, tile);
    if (e < 0) return;
    first = p.grp_start[e], all = p.grp_start[e + 1] - first;
  }
  const int tiles_m = (all + AM - 1) / AM;
  const int m0 = tile % tiles_m * AM, n0 = tile / tiles_m * TN, rows = min(all - m0, AM);
  const int nk = p.K / TK;

  const int r4 = lane >> 4, slot = lane & 15;
  auto run = [&](auto ai_c) {
    constexpr int AI = decltype(ai_c)::value, G = WI + AI;         // 16-row blocks of x; staging instructions per wave and K-tile
    int voff_a[AI], voff_w[WI];
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const int row = (wid * AI + i) * 4 + r4, at = first + m0 + min(row, rows - 1);
      const int src = !ONE && p.grp_perm ? p.grp_perm[at] / p.grp_top : at;
      voff_a[i] = row < rows ? (src * p.lda + ((slot ^ (row & 15)) * 8)) * 2 : 0x7fffff00;     // (past the range: zeros)
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int row = (wid * WI + i) * 4 + r4;
      voff_w[i] = ((n0 + (row & (TN - 1)) + (row / TN) * p.glu_half) * p.ldw + ((slot ^ (row & 15)) * 8)) * 2;
    }
    const unsigned char* A = reinterpret_cast<const unsigned char*>(p.A);
    const unsigned char* W = reinterpret_cast<const unsigned char*>(p.W + (ONE ? 0 : e * p.grp_wstride));
    const int bytes_a = 2 * p.M * p.lda, bytes_w = 2 * (GLU ? 2 * p.glu_half : p.N) * p.ldw;
    auto stage_w = [&](int buf, int kt) {
#pragma unroll
      for (int i = 0; i < WI; ++i)
        buffer_to_lds16(W + kt * (2 * TK), bytes_w - kt * (2 * TK), smem + buf * STAGE + A_BYTES + (wid * WI + i) * 1024, voff_w[i]);
    };
    auto stage_a = [&](int buf, int kt) {
#pragma unroll
      for (int i = 0; i < AI; ++i)
        buffer_to_lds16(A + kt * (2 * TK), bytes_a - kt * (2 * TK), smem + buf * STAGE + (wid * AI + i) * 1024, voff_a[i]);
    };
    f32x4_t acc[AI];
#pragma unroll
    for (int i = 0; i < AI; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int frow = lane & 15, fq = lane >> 4, col = wid & 1, half = wid >> 1;
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
      if (s < nk) {
        stage_w(s, s);
        stage_a(s, s);
      }
    int cur = 0;
    for (int kt = 0; kt < nk; ++kt) {
      const int ahead = min(STAGES - 2, nk - 1 - kt);              // younger K-tiles that may still be on their way
      if (ahead <= 0) wait_vm<0>();
      else if (ahead == 1) wait_vm<G>();
      else wait_vm<2 * G>();
      __builtin_amdgcn_s_barrier();
      if (kt + STAGES - 1 < nk) {
        int nb = cur + STAGES - 1;
        if (nb >= STAGES) nb -= STAGES;
        stage_w(nb, kt + STAGES - 1);
        stage_a(nb, kt + STAGES - 1);
      }
      const unsigned char* a_img = smem + cur * STAGE + frow * 256;
      const unsigned char* w_img = smem + cur * STAGE + A_BYTES + ((GLU ? half * TN : 0) + col * 16 + frow) * 256;
#pragma unroll
      for (int k = 0; k < (GLU ? 4 : 2); ++k) {
        const int ks = GLU ? k : half * 2 + k, off = ((ks * 4 + fq) ^ frow) * 16;
        const bf16x8_t wf = *reinterpret_cast<const bf16x8_t*>(w_img + off);
#pragma unroll
        for (int i = 0; i < AI; ++i) {
          const bf16x8_t af = *reinterpret_cast<const bf16x8_t*>(a_img + i * 4096 + off);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, af, acc[i], 0, 0, 0);
        }
      }
      cur = cur + 1 == STAGES ? 0 : cur + 1;
    }
    // the second pair of waves (up rows, or the other half of K) hands its sums to the first
    __syncthreads();
    f32x4_t* pass = reinterpret_cast<f32x4_t*>(smem);
    if (half) {
#pragma unroll
      for (int i = 0; i < AI; ++i) pass[(col * AI + i) * 64 + lane] = acc[i];
    }
    __syncthreads();
    if (half) return;
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const f32x4_t o = pass[(col * AI + i) * 64 + lane];
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        v[r] = !GLU ? acc[i][r] + o[r] : ONE ? glu_gate(acc[i][r], p.glu_act) * o[r]
                                             : glu_gate(bf16_to_f32(f32_to_bf16(acc[i][r])), p.glu_act) * bf16_to_f32(f32_to_bf16(o[r]));
      if (i * 16 + frow < rows) {
        const u32x2_t w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        *reinterpret_cast<u32x2_t*>(p.C + static_cast<size_t>(first + m0 + i * 16 + frow) * p.ldc + n0 + col * 16 + fq * 4) = w;
      }
    }
  };
  if (rows <= 16) run(std::integral_constant<int, 1>{});
  else run(std::integral_constant<int, 2>{});
}

template <bool GLU, bool ONE>
void launch(const GemmParams& p, int grid, hipStream_t st) {
  constexpr int smem = STAGES * (AM + (GLU ? 2 * TN : TN)) * TK * 2;
  static const bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_grouped_few_kernel<GLU, ONE>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, smem) == hipSuccess;
  (void)attr;
  hipLaunchKernelGGL((gemm_grouped_few_kernel<GLU, ONE>), dim3(grid), dim3(256), smem, st, EVGPT_GEMM_PASS(p));
}

}  // namespace

// Up to 16 rows an average group: 24 (96 rows, two experts each) down 25.4 vs 30.6 us.  Time over the general tile's at the mean of 11 600
// products of 2 to 32 experts, 512 to 5 504 k, 512 to 9 000 columns, rows dealt at random, weights from memory: 0.78 and gated 0.84, 2 % of
// them behind by more than 2.5 %.  Not the gated ones of 257 to 384 workgroups (groups x columns / 32: over a round of one a CU, most CUs with one)
// and more rows than groups, 0.94 at the mean and a fifth of them behind; up to 256 are at 0.80, up to 512 at 0.84.
bool gemm_grouped_few_serves(const GemmParams& p, int rows) {
  if (p.K % TK || p.N % TN || p.ldc % 4 || rows > 16 * p.grp_count) return false;
  const int most = p.grp_count * (p.N / TN);
  return !p.glu_half || rows <= p.grp_count || most <= 256 || most > 384;
}

void launch_gemm_grouped_few(const GemmParams& p, int rows, hipStream_t st) {
  const int most = (rows / AM + p.grp_count) * (p.N / TN);        // at least as many as there can be
  const int grid = (most + 8 * RUN - 1) / (8 * RUN) * (8 * RUN);  // every XCD's whole turns
  if (p.glu_half) launch<true, false>(p, grid, st);
  else launch<false, false>(p, grid, st);
}

// A dense gated product of a decode step, against the slabs of gemm_fewrow_kernel and the launch that sums and gates them; the error against 64
// bits is the same.  What it saves is the slabs; what it gives up is K divided over more workgroups than there are tiles, and whole rounds.
// Time with it / without, weights from memory, 5 / 16 / 32 rows:
//  * K below 2048, 4 to 1024 tiles: 0.5 to 0.99 (1920 and 64 tiles 1.03 at 32 rows)
//  * K 2048, tiles 48 / 64 / 72 / 88 / 128 / 176 / 256: 1.17 1.17 1.20 / 1.11 1.07 1.14 / 0.97 0.94 0.94 / 0.98 0.94 0.93 / 0.92 0.89 0.92 / 0.79 0.78
//    0.80 / 0.86 0.84 0.78 (2 x 5632 columns 13.9 -> 10.9 us, 14.2 -> 11.1, 14.9 -> 12.0)
//  * K 2560 to 4608 below 136 tiles: 0.9 to 1.6; 144: 0.88 to 0.99, 176: 0.90 to 0.98, 256: 0.78 to 0.98.  K 5120: 144 between 0.94 and 1.11 from run to
//    run, 176 0.89 0.89 0.93, 256 0.85 0.84 0.80
//  * a round and a part, 257 / 288 / 320 / 352 / 400 tiles: K 2048 1.01 1.03 1.02 / 1.01 1.02 1.02 / 0.96 0.92 0.95 / 0.93 0.90 0.87 / 0.93 0.87 0.85; 4096
//    1.14 1.14 1.12 / 1.18 1.18 1.18 / 1.08 1.02 1.06 / 1.04 0.98 0.98 / 0.96 0.93 0.91; 5120 1.10 1.09 1.12 / 1.12 1.10 1.14 / 1.09 1.07 1.08 / 1.05 1.00
//    0.99 / 0.94 0.92 0.89; 512: 0.87 to 1.02, 0.80 to 0.96, 0.73 to 0.86
//  * more rounds, 576 / 640 / 768 / 1024 tiles: K 2048 1.10 1.00 0.92 / 1.05 0.93 0.84 / 1.04 0.92 0.80 / 0.97 0.95 0.91; 4096 1.15 1.03 0.99 / 1.02 0.91 0.85 /
//    0.97 0.84 0.80 / 0.97 0.94 0.94
//  * K 6144: 1.0 to 1.3 below 400 tiles; 8192: 0.9 to 1.2
bool gemm_few_glu_serves(int rows, int I, int K) {
  if (rows > AM || K <= 0 || K % TK || I % TN) return false;
  const int tiles = I / TN;
  if (K < 2048) return true;
  if (K > 5120) return false;
  if (tiles <= 256) return tiles >= (K < 2304 ? 72 : 160);
  if (tiles <= 512) return tiles >= (K < 2304 ? 320 : 400);
  return rows > 8 && tiles >= 640;
}
void launch_gemm_few_glu(const bf16_t* A, const bf16_t* W, bf16_t* C, int rows, int I, int K, int glu_act, hipStream_t st) {
  GemmParams p{};
  p.A = A, p.W = W, p.C = C, p.M = rows, p.N = I, p.K = p.lda = p.ldw = K, p.ldc = I, p.splitk = 1, p.k_per_split = K;
  p.glu_half = I, p.glu_act = glu_act;
  launch<true, true>(p, (I / TN + 8 * RUN - 1) / (8 * RUN) * (8 * RUN), st);
}

}  // namespace evgpt
