// The epilogue that the GEMM kernels share.
#pragma once
#include "gemm_common.h"

namespace evgpt {

// Epilogue shared by the GEMM kernels: lane holds C[m][n .. n+3] of each 16x16 tile (m = row
// lane & 15, n = 4 * (lane >> 4)); wave (wr, wc) owns the WM x WN sub-tile at (wr*WM, wc*WN).
// ACT: the activation as a constant (-1: p.act, a choice among all of them unrolled for every element).
template <int TM, int TN, int WM, int WN, int WGN, int ACT = -1>
__device__ __forceinline__ void gemm_epilogue(const GemmParams& p, f32x4_t (&acc)[TM][TN], int m0, int n0, int wr,
                                              int wc, int tn, int tiles_n, int ksplit, int lane) {
  const int frow = lane & 15, fq = lane >> 4;
  if constexpr (TN % 2 == 0) {
    if (p.glu_half) {
      // tile columns j < TN/2 are gate, j + TN/2 the matching up columns; both factors are rounded to
      // bf16 first (what a separate activation kernel would read back)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = m0 + wr * WM + i * 16 + frow;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < TN / 2; ++j) {
          const int n = n0 + wc * (WN / 2) + j * 16 + fq * 4;
          if (n >= p.N) continue;
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = glu_gate(bf16_to_f32(f32_to_bf16(acc[i][j][r])), p.glu_act) * bf16_to_f32(f32_to_bf16(acc[i][j + TN / 2][r]));
          const size_t o = static_cast<size_t>(m) * p.ldc + n;
          if (n + 3 < p.N && (p.ldc & 3) == 0) {
            u32x2_t w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            *reinterpret_cast<u32x2_t*>(p.C + o) = w;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) if (n + r < p.N) p.C[o + r] = f32_to_bf16(v[r]);
          }
        }
      }
      return;
    }
  }
  if (p.splitk > 1 || p.raw_partial) {
    float* slab = p.partial + static_cast<size_t>(ksplit) * p.M * p.N;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + wr * WM + i * 16 + frow;
      if (m >= p.M) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wc * WN + j * 16 + fq * 4;
        float* dst = slab + static_cast<size_t>(m) * p.N + n;
        if (n + 3 < p.N && (p.N & 3) == 0) {
          *reinterpret_cast<f32x4_t*>(dst) = acc[i][j];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) if (n + r < p.N) dst[r] = acc[i][j][r];
        }
      }
    }
    return;
  }
  // A bf16 output in whole quads of columns (ACT < 0: without an activation): the bias is read once, a row's residual together.  (The general
  // way below asks for bias, activation, residual and edges at every quad and waits for each load of its own.  us, so / now, with a bias, a
  // residual, both: 577 x 4096 x 1024 13.0 / 11.2, 16.0 / 12.7, 18.1 / 12.7; 836 x 4096 x 4096 36.7 / 34.5, 40.9 / 36.3, 44.1 / 36.3; 40 x 4096 x
  // 1024 7.7 / 7.2, 8.0 / 7.3, 8.5 / 7.4.  Without either it was as fast.)
  if (p.C && !p.Cf && !p.amax_val && (ACT >= 0 || p.act == ACT_NONE) && ((p.N | p.ldc) & 3) == 0 &&
      ((reinterpret_cast<uintptr_t>(p.C) | reinterpret_cast<uintptr_t>(p.bias) | reinterpret_cast<uintptr_t>(p.res)) & 7) == 0) {
    const int n = n0 + wc * WN + fq * 4;
    u32x2_t bw[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bw[j] = u32x2_t{0, 0};
    if (p.bias)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        if (n + j * 16 < p.N) bw[j] = *reinterpret_cast<const u32x2_t*>(p.bias + n + j * 16);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + wr * WM + i * 16 + frow;
      if (m >= p.M) continue;
      const size_t o = static_cast<size_t>(m) * p.ldc + n;
      u32x2_t rw[TN];
      if (p.res)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          if (n + j * 16 < p.N) rw[j] = *reinterpret_cast<const u32x2_t*>(p.res + o + j * 16);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (n + j * 16 >= p.N) continue;
        float v[4] = {acc[i][j][0] + bf16lo(bw[j][0]), acc[i][j][1] + bf16hi(bw[j][0]), acc[i][j][2] + bf16lo(bw[j][1]), acc[i][j][3] + bf16hi(bw[j][1])};
        if constexpr (ACT > 0) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = apply_act(v[r], ACT);
        }
        u32x2_t w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        if (p.res)
          w = u32x2_t{pack_bf16x2(bf16lo(w[0]) + bf16lo(rw[j][0]), bf16hi(w[0]) + bf16hi(rw[j][0])),
                      pack_bf16x2(bf16lo(w[1]) + bf16lo(rw[j][1]), bf16hi(w[1]) + bf16hi(rw[j][1]))};
        *reinterpret_cast<u32x2_t*>(p.C + o + j * 16) = w;
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + wr * WM + i * 16 + frow;
    if (p.amax_val) {
      // row max over this wave's WN columns: in-lane over j and r, then across the
      // 4 lanes (fq) that share the row
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = n0 + wc * WN + j * 16 + fq * 4 + r;
          float v = acc[i][j][r];
          if (p.bias && n < p.N) v += bf16_to_f32(p.bias[n]);
          if (n < p.N && (v > bv || (v == bv && n < bi))) { bv = v; bi = n; }
        }
#pragma unroll
      for (int off = 16; off < 64; off <<= 1) {
        const float ov = __shfl_xor(bv, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
      }
      if (fq == 0 && m < p.M) {
        const int n_part = tiles_n * WGN;
        p.amax_val[static_cast<size_t>(m) * n_part + tn * WGN + wc] = bv;
        p.amax_idx[static_cast<size_t>(m) * n_part + tn * WGN + wc] = bi;
      }
    }
    if (m >= p.M || (!p.C && !p.Cf)) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wc * WN + j * 16 + fq * 4;
      if (n >= p.N) continue;
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      const size_t o = static_cast<size_t>(m) * p.ldc + n;
      const bool full = (n + 3 < p.N) && ((p.ldc & 3) == 0);
      if (p.bias) {
#pragma unroll
        for (int r = 0; r < 4; ++r) if (n + r < p.N) v[r] += bf16_to_f32(p.bias[n + r]);
      }
      if (ACT < 0 ? p.act != ACT_NONE : ACT != ACT_NONE) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = apply_act(v[r], ACT < 0 ? p.act : ACT);
      }
      if (p.res) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < p.N) v[r] = bf16_to_f32(f32_to_bf16(v[r])) + bf16_to_f32(p.res[o + r]);
      }
      if (p.Cf) {
        if (full) {
          *reinterpret_cast<f32x4_t*>(p.Cf + o) = f32x4_t{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) if (n + r < p.N) p.Cf[o + r] = v[r];
        }
      }
      if (p.C) {
        if (full) {
          u32x2_t w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
          *reinterpret_cast<u32x2_t*>(p.C + o) = w;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) if (n + r < p.N) p.C[o + r] = f32_to_bf16(v[r]);
        }
      }
    }
  }
}

}  // namespace evgpt
