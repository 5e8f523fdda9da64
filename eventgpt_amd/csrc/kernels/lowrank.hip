// Rank-r projection of a low-rank adapter: C [M, R] = alpha * A [M, K] · W [R, K]^T with R <= 16.
//
// The output is 16 columns wide and the contraction is the model width, so a tiled GEMM spends its
// time on a 64- or 128-column W tile that is mostly padding and on a split-K reduction pass.  Here a
// block owns 16 rows of A and its 16 waves share the contraction: wave w takes the 32-column K-steps
// w, w + 16, ..., loads the A and W fragments of a step straight from memory in the MFMA operand
// layout (row = lane % 16, eight consecutive k at 8 * (lane / 16)), and the 16 partial 16 x 16
// accumulators are summed through LDS.  A [836, 4096] input is 53 blocks of 1024 threads with every
// load of a wave in flight at once; W (128 KB at r = 16) stays in L2.
//
// A may be a column block of a wider matrix (row stride lda), and the adapter's input dropout can be
// applied while A is loaded (DROP): element (m, k) is zeroed unless its bit of lowrank_keep8(seed,
// chunk (m K + k) / 8) is set -- the 1 / (1 - p) factor rides on alpha -- so the dropped copy of the
// layer input is never written.  The backward's kernels recompute the same mask from the seed while they load x (weight
// gradient of A) and store the input gradient.
#include "common.h"
#include "../evgpt_kernels.h"

namespace evgpt {

constexpr int LR_WAVES = 16;

// keep bits of the 8 elements of 16-byte chunk `chunk`: two 64-bit mixes, one 16-bit field per element
__device__ __forceinline__ unsigned int lowrank_keep8(unsigned long long seed, unsigned long long chunk,
                                                      unsigned int thresh16) {
  unsigned int bits = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    unsigned long long z = seed + (2 * chunk + h) * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
#pragma unroll
    for (int f = 0; f < 4; ++f)
      bits |= (static_cast<unsigned int>(z >> (16 * f)) & 0xffffu) >= thresh16 ? 1u << (4 * h + f) : 0u;
  }
  return bits;
}
// zero the dropped elements of a chunk (element e: low / high half of word e / 2)
__device__ __forceinline__ u32x4_t lowrank_apply8(u32x4_t v, unsigned int keep) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned int m = ((keep >> (2 * j)) & 1u ? 0x0000ffffu : 0u) | ((keep >> (2 * j + 1)) & 1u ? 0xffff0000u : 0u);
    v[j] &= m;
  }
  return v;
}
static unsigned int lowrank_thresh16(float p) {
  if (p <= 0.f) return 0u;
  const double t = static_cast<double>(p) * 65536.0;
  return t >= 65535.0 ? 65535u : static_cast<unsigned int>(t);
}

// NA adapters that read the same A (q, k and v of a grouped projection): A is loaded once, each has its own W, C and mask.
template <int NA, bool DROP>
__global__ __launch_bounds__(LR_WAVES * 64) void lowrank_out_kernel(const bf16_t* __restrict__ A, LowrankSet set, int M, int R, int K,
                                                                   long long lda, float alpha, unsigned int thresh16) {
  __shared__ float red[LR_WAVES][256];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 15, fq = lane >> 4;
  const int m = blockIdx.x * 16 + frow;
  const bool a_ok = m < M, w_ok = frow < R;
  const bf16_t* a_row = A + static_cast<size_t>(a_ok ? m : 0) * lda;
  const u32x4_t z4 = {0u, 0u, 0u, 0u};
  const bf16x8_t zero = __builtin_bit_cast(bf16x8_t, z4);
  f32x4_t acc[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int UN = 8;   // K = 4096: the eight steps of a wave are issued together
  // the loop bound is the same for all lanes of a wave (an MFMA needs every lane's operands, so no lane
  // may leave early); a lane whose chunk of the last step lies past K contributes zeros
  for (int kb = wid * 32; kb < K; kb += UN * LR_WAVES * 32) {
    bf16x8_t af[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int k = kb + u * LR_WAVES * 32 + fq * 8;      // K is a multiple of 8: a chunk is inside or outside as a whole
      af[u] = (k < K && a_ok) ? *reinterpret_cast<const bf16x8_t*>(a_row + k) : zero;
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const bf16_t* w_row = set.b[i] + static_cast<size_t>(w_ok ? frow : 0) * K;
      bf16x8_t wf[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int k = kb + u * LR_WAVES * 32 + fq * 8;
        wf[u] = (k < K && w_ok) ? *reinterpret_cast<const bf16x8_t*>(w_row + k) : zero;
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        bf16x8_t x = af[u];
        if constexpr (DROP) {
          const int k = kb + u * LR_WAVES * 32 + fq * 8;
          const unsigned long long chunk = (static_cast<unsigned long long>(a_ok ? m : 0) * K + (k < K ? k : 0)) >> 3;
          x = __builtin_bit_cast(bf16x8_t, lowrank_apply8(__builtin_bit_cast(u32x4_t, x),
                                                          lowrank_keep8(set.seed[i], chunk, thresh16)));
        }
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], x, acc[i], 0, 0, 0);
      }
    }
  }
  // acc[e] = sum over this wave's steps of  W[r = 4 * fq + e] · A[m = frow]
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    if (i) __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wid][lane * 4 + e] = acc[i][e];
    __syncthreads();
    if (t < 256) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < LR_WAVES; ++w) s += red[w][t];
      const int ln = t >> 2, e = t & 3;
      const int r = 4 * (ln >> 4) + e, mm = blockIdx.x * 16 + (ln & 15);
      if (mm < M && r < R) set.out[i][static_cast<size_t>(mm) * R + r] = f32_to_bf16(s * alpha);
    }
  }
}

void launch_lowrank_out(const bf16_t* A, const LowrankSet& set, int M, int R, int K, long long lda, float alpha, float drop_p,
                        hipStream_t st) {
  if (M <= 0) return;
  const unsigned int t16 = lowrank_thresh16(drop_p);
  const float s = t16 ? alpha / (1.f - drop_p) : alpha;
  const dim3 grid((M + 15) / 16), block(LR_WAVES * 64);
#define LR_OUT(NA)                                                                                                      \
  if (t16) hipLaunchKernelGGL((lowrank_out_kernel<NA, true>), grid, block, 0, st, A, set, M, R, K, lda, s, t16);        \
  else hipLaunchKernelGGL((lowrank_out_kernel<NA, false>), grid, block, 0, st, A, set, M, R, K, lda, s, 0u)
  if (set.n == 1) { LR_OUT(1); }
  else if (set.n == 2) { LR_OUT(2); }
  else { LR_OUT(3); }
#undef LR_OUT
}

// Y [M, N] += sum over the adapters of  m_i (.) (T_i [M, R] · B_i^T),  B_i [N, R] (or [R, N]: TRANS), R = 8 or 16, in place.
//
// Bound by memory: Y is read and written once and nothing else is large.  As a GEMM with a residual epilogue the product
// ran one K-tile of 64 for a contraction of 16 behind a three-stage ring and one pass over Y per adapter: 6 688 x 4 096
// 89 us (110 MB: 1.2 TB/s).  Here a wave takes 64 rows x 64 columns: the Y loads are issued first, T and B fragments come
// from L2, and the columns are dealt to the MFMA rows so that a lane ends up with 8 consecutive ones (two MFMAs, rows
// 4 q + e -> columns 8 q + e and 8 q + 4 + e): every access to Y is 16 bytes.  Same shape: 27 us (4.1 TB/s), 40 us
// for three adapters in one pass.
template <int NA, bool TRANS, bool DROP>
__global__ __launch_bounds__(256) void lowrank_add_kernel(LowrankSet set, bf16_t* __restrict__ Y, int M, int N, int R, long long ldy,
                                                          unsigned int thresh16) {
  const int lane = threadIdx.x & 63, frow = lane & 15, fq = lane >> 4;
  const int c0 = blockIdx.x * 256 + (threadIdx.x >> 6) * 64, m0 = (blockIdx.z * 65535 + blockIdx.y) * 64;
  if (c0 >= N || m0 >= M) return;
  const u32x4_t z4 = {0u, 0u, 0u, 0u};
  const bool k_ok = fq * 8 < R;
  u32x4_t y[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int m = m0 + i * 16 + frow, c = c0 + g * 32 + fq * 8;
      y[i][g] = m < M && c < N ? load16(Y + m * ldy + c) : z4;
    }
  f32x4_t acc[4][2][2];
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    bf16x8_t tf[4], bfr[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + i * 16 + frow;
      tf[i] = __builtin_bit_cast(bf16x8_t, k_ok && m < M ? load16(set.t[a] + static_cast<size_t>(m) * R + fq * 8) : z4);
    }
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = c0 + g * 32 + 8 * (frow >> 2) + 4 * h + (frow & 3);
        u32x4_t v = z4;
        if (k_ok && n < N) {
          if constexpr (TRANS) {
            const bf16_t* b = set.b[a] + static_cast<size_t>(fq) * 8 * N + n;
#pragma unroll
            for (int j = 0; j < 4; ++j)
              v[j] = b[static_cast<size_t>(2 * j) * N] | static_cast<unsigned int>(b[static_cast<size_t>(2 * j + 1) * N]) << 16;
          } else {
            v = load16(set.b[a] + static_cast<size_t>(n) * R + fq * 8);
          }
        }
        bfr[g][h] = __builtin_bit_cast(bf16x8_t, v);
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
        if constexpr (DROP) {
          const int m = m0 + i * 16 + frow, c = c0 + g * 32 + fq * 8;
          const unsigned int keep = lowrank_keep8(set.seed[a], (static_cast<unsigned long long>(m < M ? m : 0) * N + (c < N ? c : 0)) >> 3,
                                                  thresh16);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const f32x4_t p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[g][h], tf[i], zero, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float v = (keep >> (4 * h + e)) & 1u ? p[e] : 0.f;
              acc[i][g][h][e] = a == 0 ? v : acc[i][g][h][e] + v;
            }
          }
        } else {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            acc[i][g][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[g][h], tf[i], a == 0 ? zero : acc[i][g][h], 0, 0, 0);
        }
      }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int m = m0 + i * 16 + frow, c = c0 + g * 32 + fq * 8;
      if (m >= M || c >= N) continue;
      u32x4_t v;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = pack_bf16x2(bf16lo(y[i][g][j]) + acc[i][g][j >> 1][(j & 1) * 2], bf16hi(y[i][g][j]) + acc[i][g][j >> 1][(j & 1) * 2 + 1]);
      *reinterpret_cast<u32x4_t*>(Y + m * ldy + c) = v;
    }
}

void launch_lowrank_add(const LowrankSet& set, bf16_t* Y, int M, int N, int R, long long ldy, bool trans, float drop_p, hipStream_t st) {
  if (M <= 0) return;
  const unsigned int t16 = lowrank_thresh16(drop_p);
  const int rows = (M + 63) / 64;                 // blocks of 64 rows, over two dimensions of the grid
  const dim3 grid((N + 255) / 256, rows < 65535 ? rows : 65535, (rows + 65534) / 65535), block(256);
#define LR_ADD(NA, TR, DR) hipLaunchKernelGGL((lowrank_add_kernel<NA, TR, DR>), grid, block, 0, st, set, Y, M, N, R, ldy, t16)
#define LR_ADD_N(TR, DR)                          \
  if (set.n == 1) LR_ADD(1, TR, DR);              \
  else if (set.n == 2) LR_ADD(2, TR, DR);         \
  else LR_ADD(3, TR, DR)
  if (!trans) { LR_ADD(1, false, false); }        // (the forward adds one adapter to its own columns, unmasked)
  else if (t16) { LR_ADD_N(true, true); }
  else { LR_ADD_N(true, false); }
#undef LR_ADD_N
#undef LR_ADD
}

// D_i [R, C] = T_i [M, R]^T · (m_i (.) G [M, C]) for adapters that share G: both weight gradients of an adapter (the output is
// written [R, C] for A, [C, R] for B), R = 8 or 16.
//
// Bound by reading G once.  The contraction runs over rows, so the MFMA wants eight rows of one column in a lane: a lane
// loads 16 bytes of eight rows (its 8 x 8 patch; 16 lanes are 256 contiguous bytes of a row) and turns the patch by 32
// v_perm, column j of every lane's patch then being the operand of the j-th MFMA -- no trip of G through LDS.  T, a
// thousandth of G, is turned through LDS once per block.  Rows are split over blocks into fp32 slabs [R, C] (about 512
// blocks), which lowrank_wgrad_sum_kernel adds.  As a K-strided GEMM with a 16-wide tile side: 79 us at M = 6 688,
// C = 4 096 (55 MB); here 14.6 and 5.0 for the slabs' sum, 21.6 for three adapters in one pass.  Up to LW_ROWS rows are one
// slab, which the block writes as the result: one launch and no partials, as the GEMM had there (launch-bound).
constexpr int LW_ROWS = 256;     // rows of T staged at a time

template <int NA, bool DROP>
__global__ __launch_bounds__(256) void lowrank_wgrad_kernel(const bf16_t* __restrict__ G, LowrankSet set, float* __restrict__ part, int M,
                                                            int C, int R, long long ldg, int rows_per_block, unsigned int thresh16,
                                                            int transposed) {
  __shared__ __attribute__((aligned(16))) bf16_t tt[NA][16][LW_ROWS + 8];
  const int tid = threadIdx.x, lane = tid & 63, frow = lane & 15, fq = lane >> 4;
  const int c = (blockIdx.x * 4 + (tid >> 6)) * 128 + frow * 8;
  const bool c_ok = c < C;
  const u32x4_t z4 = {0u, 0u, 0u, 0u};
  const int row0 = blockIdx.y * rows_per_block, row1 = min(M, row0 + rows_per_block);
  f32x4_t acc[NA][8];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[a][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int base = row0; base < row1; base += LW_ROWS) {
    __syncthreads();
    const int tm = base + tid;
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4_t v = tm < row1 && h * 8 < R ? load16(set.t[a] + static_cast<size_t>(tm) * R + h * 8) : z4;
#pragma unroll
        for (int e = 0; e < 8; ++e) tt[a][h * 8 + e][tid] = static_cast<bf16_t>(v[e >> 1] >> (16 * (e & 1)));
      }
    __syncthreads();
    const int steps = (min(row1 - base, LW_ROWS) + 31) / 32;
#pragma unroll 2
    for (int s = 0; s < steps; ++s) {
      u32x4_t v[8];
      const int m = base + s * 32 + fq * 8;
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = c_ok && m + r < row1 ? load16(G + (m + r) * ldg + c) : z4;
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        const bf16x8_t tf = *reinterpret_cast<const bf16x8_t*>(&tt[a][frow][s * 32 + fq * 8]);
        u32x4_t x[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          x[r] = v[r];
          if constexpr (DROP) {
            const unsigned long long chunk = (static_cast<unsigned long long>(m + r < M ? m + r : 0) * C + (c_ok ? c : 0)) >> 3;
            x[r] = lowrank_apply8(x[r], lowrank_keep8(set.seed[a], chunk, thresh16));
          }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          u32x4_t f;                       // column j of the patch: rows 2 i and 2 i + 1 in word i
#pragma unroll
          for (int i = 0; i < 4; ++i)
            f[i] = __builtin_amdgcn_perm(x[2 * i + 1][j >> 1], x[2 * i][j >> 1], j & 1 ? 0x07060302u : 0x05040100u);
          acc[a][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tf, __builtin_bit_cast(bf16x8_t, f), acc[a][j], 0, 0, 0);
        }
      }
    }
  }
  // acc[a][j][e]: rank 4 fq + e, column c + j
  if (!c_ok) return;
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 4 * fq + e;
      if (r >= R) continue;
      if (gridDim.y == 1) {                      // one slab: there is nothing to add
#pragma unroll
        for (int j = 0; j < 8; ++j)
          set.out[a][transposed ? static_cast<size_t>(c + j) * R + r : static_cast<size_t>(r) * C + c + j] = f32_to_bf16(acc[a][j][e]);
        continue;
      }
      float* dst = part + ((static_cast<size_t>(blockIdx.y) * NA + a) * R + r) * C + c;
      *reinterpret_cast<f32x4_t*>(dst) = f32x4_t{acc[a][0][e], acc[a][1][e], acc[a][2][e], acc[a][3][e]};
      *reinterpret_cast<f32x4_t*>(dst + 4) = f32x4_t{acc[a][4][e], acc[a][5][e], acc[a][6][e], acc[a][7][e]};
    }
}

// sums the slabs; thread: four consecutive columns of one rank
__global__ __launch_bounds__(256) void lowrank_wgrad_sum_kernel(const float* __restrict__ part, LowrankSet set, int slabs, int C, int R,
                                                                int transposed) {
  const int i = blockIdx.x * 256 + threadIdx.x, per = R * C / 4;
  if (i >= set.n * per) return;
  const size_t stride = static_cast<size_t>(set.n) * R * C;
  const float* src = part + static_cast<size_t>(i) * 4;
  f32x4_t s = *reinterpret_cast<const f32x4_t*>(src);
#pragma unroll 8
  for (int z = 1; z < slabs; ++z) s += *reinterpret_cast<const f32x4_t*>(src + z * stride);
  const int a = i / per, r = (i % per) * 4 / C, c = (i % per) * 4 % C;
  bf16_t* out = set.out[a];
#pragma unroll
  for (int e = 0; e < 4; ++e) out[transposed ? static_cast<size_t>(c + e) * R + r : static_cast<size_t>(r) * C + c + e] = f32_to_bf16(s[e]);
}

// slabs of the split: about 512 blocks of 4 x 128 columns, no slab under LW_ROWS rows
int lowrank_wgrad_slabs(int M, int C) {
  const int cols = (C + 511) / 512, most = (M + LW_ROWS - 1) / LW_ROWS;
  const int want = (512 + cols - 1) / cols;
  return want < most ? want : (most < 1 ? 1 : most);
}

void launch_lowrank_wgrad(const bf16_t* G, const LowrankSet& set, float* part, int M, int C, int R, long long ldg, bool transposed,
                          float drop_p, hipStream_t st) {
  const unsigned int t16 = lowrank_thresh16(drop_p);
  const int slabs = lowrank_wgrad_slabs(M, C), rows = ((M + slabs - 1) / slabs + 31) / 32 * 32;
  const dim3 grid((C + 511) / 512, slabs), block(256);
#define LR_WG(NA)                                                                                                                \
  if (t16) hipLaunchKernelGGL((lowrank_wgrad_kernel<NA, true>), grid, block, 0, st, G, set, part, M, C, R, ldg, rows, t16, transposed);      \
  else hipLaunchKernelGGL((lowrank_wgrad_kernel<NA, false>), grid, block, 0, st, G, set, part, M, C, R, ldg, rows, 0u, transposed)
  if (set.n == 1) { LR_WG(1); }
  else if (set.n == 2) { LR_WG(2); }
  else { LR_WG(3); }
#undef LR_WG
  if (slabs > 1)
    hipLaunchKernelGGL(lowrank_wgrad_sum_kernel, dim3((set.n * R * C / 4 + 255) / 256), block, 0, st, part, set, slabs, C, R, transposed);
}

// y = m (.) x over contiguous [rows][K] tensors, m the keep mask of lowrank_keep8 (no 1 / (1 - p) factor), for checking the
// kernels that apply it on the way
__global__ __launch_bounds__(256) void lowrank_mask_kernel(const bf16_t* __restrict__ x, bf16_t* __restrict__ y, long long n8,
                                                           unsigned int thresh16, unsigned long long seed) {
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n8; i += gridDim.x * 256ll)
    *reinterpret_cast<u32x4_t*>(y + i * 8) = lowrank_apply8(load16(x + i * 8), lowrank_keep8(seed, static_cast<unsigned long long>(i), thresh16));
}
void launch_lowrank_mask(const bf16_t* x, bf16_t* y, long long n, float drop_p, unsigned long long seed, hipStream_t st) {
  if (n <= 0) return;
  long long b = (n / 8 + 255) / 256;
  const unsigned blocks = static_cast<unsigned>(b > 8192 ? 8192 : (b < 1 ? 1 : b));
  hipLaunchKernelGGL(lowrank_mask_kernel, dim3(blocks), dim3(256), 0, st, x, y, n / 8, lowrank_thresh16(drop_p), seed);
}

}  // namespace evgpt
