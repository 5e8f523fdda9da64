// Flash-attention backward for the training paths (causal head_dim 128 of the decoder,
// non-causal head_dim 64 of the vision tower): dQ, dK, dV from Q, K, V, dO and the forward's
// per-row log-sum-exp, without ever materialising the score matrix.
//
// P is recomputed tile by tile:  P = exp2(S * scale*log2e - LSE),  dS = P * (dP - delta) * scale
// with dP = dO V^T and delta = rowsum(dO * O).  Two kernels, each the forward kernel's
// structure (attn_prefill.hip) with the roles of the operands rearranged, so that every
// product is an MFMA whose transposed operand comes from ds_read_b64_tr_b16 on the same
// swizzled LDS image and whose "probability" operand never leaves the registers:
//
//   * dq kernel -- one block per 64 query rows of a (batch, head); K and V tiles stream
//     through LDS.  S^T = K Q^T and dP^T = V dO^T put the query on the lane, so LSE / delta
//     are per-lane scalars and dS^T (bf16) is directly the B operand of
//     dQ^T[d][q] += K^T[d][key] dS^T[key][q]  (K^T by transposed reads of the K tile).
//   * dkv kernel -- one block per 64 keys of a (batch, kv head); Q and dO tiles stream
//     through LDS.  S = Q K^T and dP = dO V^T put the KEY on the lane (K / V fragments of the
//     wave's 16 keys stay in registers), P and dS are the B operands of
//     dV^T[d][key] += dO^T[d][q] P[q][key]   and   dK^T[d][key] += Q^T[d][q] dS[q][key].
//     dK and dV are owned by the block: no atomics, bitwise reproducible.  Grouped KV heads
//     loop over the query heads of the group.
//
// Streamed tiles go straight into LDS, one on its way while another is multiplied, behind one barrier a tile.  Bound by the chain of a
// tile (operands out of LDS, products, exponentials, transposed operands, products) and by LDS reads of about twice the matrix time,
// which the waves of other blocks fill: so small tiles, and registers for three waves a SIMD (without that bound two: 406 us of the 342
// below).  Both kernels and delta, tiles of 64 rows through registers behind two barriers / this, us: eight sequences of 836, 32 heads
// of 128 500 / 342 (0.33 PFLOP/s of 5 products); two of 700 120 / 75; one of 2 048 394 / 179; two of 500, 8 key heads 132 / 108; eight of
// 577, 16 heads of 64, no mask 102 / 81.  Tiles of 64 rows of 128 values (64 KB, two blocks a CU) 393 where 32 take 331, of 32 rows of 64 values 80
// where 64 take 75; two column tiles a wave, half the reads, 429 (256 registers); priority for the products: level.
//
// Recomputing S and dP in both kernels costs 7 products instead of 5; in exchange dQ needs
// no cross-block float atomics (which run at a sixth of the store rate on this chip) and no
// ordered hand-off.  At the sequence lengths trained here (<= 2K tokens) attention is a few
// percent of a step.
#include "common.h"
#include "attn_common.h"
#include "../evgpt_kernels.h"

namespace evgpt {

struct AttnBwdParams {
  const bf16_t* q; const bf16_t* k; const bf16_t* v; const bf16_t* d_o;
  const float* lse; const float* delta;
  bf16_t* dq; bf16_t* dk; bf16_t* dv;
  int Sq, Sk, Hq, Hkv, q_offset;
  float scale, scale_log2e;
};

// delta[b][h][q] = sum_d dO[b][q][h][d] * O[b][q][h][d]
template <int D>
__global__ __launch_bounds__(256) void attn_delta_kernel(const bf16_t* __restrict__ o,
                                                         const bf16_t* __restrict__ d_o,
                                                         float* __restrict__ delta, long long rows, int Sq,
                                                         int Hq) {
  constexpr int LPR = D / 8;                 // lanes per row
  const long long r = (blockIdx.x * 256ll + threadIdx.x) / LPR;   // row = (b, q, h)
  const int dl = threadIdx.x % LPR;
  float s = 0.f;
  if (r < rows) {
    const u32x4_t a = load16(o + r * D + dl * 8), g = load16(d_o + r * D + dl * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) s += bf16lo(a[i]) * bf16lo(g[i]) + bf16hi(a[i]) * bf16hi(g[i]);
  }
  s = group_sum<LPR>(s);
  if (r < rows && dl == 0) {
    const long long h = r % Hq, bq = r / Hq, qq = bq % Sq, b = bq / Sq;
    delta[(b * Hq + h) * Sq + qq] = s;
  }
}

// rows of a streamed tile: two stages of two tiles are 32 KB for either D, so that three to six blocks of a CU work beside each other
template <int D> constexpr int bwd_tile() { return 4096 / D; }

// A tile [bwd_tile][D] of rows row0.. of a [S, H, D] tensor's head goes straight into the swizzled LDS image, 1 KB an instruction
// and wave; rows past the end come back as zeros from the descriptor's range check.
__device__ __forceinline__ void bwd_to_lds16(const unsigned char* src, int bytes, unsigned char* lds, int voff) {
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(src), 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (void __attribute__((address_space(3)))*)lds, 16, voff, 0, 0, 0);
}
template <int D>
__device__ __forceinline__ void bwd_stage(const bf16_t* head, long long row_stride, int row0, int n_rows, unsigned char* lds, int wid, int lane) {
  constexpr int CPR = D / 8, NIW = bwd_tile<D>() * D * 2 / 1024 / 4;
  const long long left = 2 * ((static_cast<long long>(n_rows) - 1 - row0) * row_stride + D);
  const int bytes = static_cast<int>(left < 0 ? 0 : (left > 0x7fffffff ? 0x7fffffff : left));
  const unsigned char* src = reinterpret_cast<const unsigned char*>(head + row0 * row_stride);
#pragma unroll
  for (int j = 0; j < NIW; ++j) {
    const int idx = (wid * NIW + j) * 64 + lane, row = idx / CPR, ch = (idx % CPR) ^ swz<D>(row);
    bwd_to_lds16(src, bytes, lds + (wid * NIW + j) * 1024, static_cast<int>((row * row_stride + ch * 8) * 2));
  }
}

// st[n] = rows 32 s + 16 n .. of the LDS tile (A operand, ds_read_b128) times the register fragments; the k-step outermost, so that
// independent products follow each other
template <int D>
__device__ __forceinline__ void mma_rows(f32x4_t (&st)[2], const unsigned char* lds, const bf16x8_t (&bfrag)[D / 32], int s, int fr, int g) {
  st[0] = st[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks)
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const bf16x8_t af = *reinterpret_cast<const bf16x8_t*>(lds + tile_off<D>(s * 32 + n * 16 + fr, ks * 4 + g));
      st[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfrag[ks], st[n], 0, 0, 0);
    }
}

// acc[dt] += T^T[d][x] * Pb[x][lane column]: T is rows 32 s .. of an LDS tile read transposed, pk the packed bf16 weights of this
// lane's column for these 32 x-rows (the forward kernel's P layout)
template <int D>
__device__ __forceinline__ void mma_tr(f32x4_t (&acc)[D / 16], const unsigned char* lds, const unsigned int (&pk)[2][2], int s, int fr, int g) {
  typedef __attribute__((ext_vector_type(8))) short s16x8_t;
  const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, u32x4_t{pk[0][0], pk[0][1], pk[1][0], pk[1][1]});
  const int q4 = fr >> 2, p4 = fr & 3;
  const int r0 = s * 32 + g * 4 + q4, r1 = r0 + 16;
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) {
    const int ch = dt * 2 + (p4 >> 1);
    const s16x4_t lo = read_tr16((lds_s16x4_t*)(lds + tile_off<D>(r0, ch) + 8 * (p4 & 1)));
    const s16x4_t hi = read_tr16((lds_s16x4_t*)(lds + tile_off<D>(r1, ch) + 8 * (p4 & 1)));
    const s16x8_t vv = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vv), pf, acc[dt], 0, 0, 0);
  }
}

// ------------------------------------------------------------------------ dQ
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 3) void attn_bwd_dq_kernel(AttnBwdParams p) {
  constexpr int TR = bwd_tile<D>(), TILE_BYTES = TR * D * 2, KS = D / 32, DT = D / 16;
  __shared__ __attribute__((aligned(16))) unsigned char lds[4 * TILE_BYTES];      // [2][K | V]
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, g = lane >> 4;
  const int b = blockIdx.z, h = blockIdx.x, hk = h / (p.Hq / p.Hkv);
  const int qb0 = (CAUSAL ? gridDim.y - 1 - blockIdx.y : blockIdx.y) * 64, qw0 = qb0 + wid * 16, qi = qw0 + fr, qi_c = min(qi, p.Sq - 1);
  const long long q_row = static_cast<long long>(p.Hq) * D, k_row = static_cast<long long>(p.Hkv) * D;
  const bf16_t* qp = p.q + (static_cast<long long>(b) * p.Sq + qi_c) * q_row + h * D;
  const bf16_t* dop = p.d_o + (static_cast<long long>(b) * p.Sq + qi_c) * q_row + h * D;
  bf16x8_t qf[KS], dof[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = *reinterpret_cast<const bf16x8_t*>(qp + ks * 32 + g * 8);
    dof[ks] = *reinterpret_cast<const bf16x8_t*>(dop + ks * 32 + g * 8);
  }
  const long long stat = (static_cast<long long>(b) * p.Hq + h) * p.Sq + qi_c;
  const float lse = p.lse[stat], dlt = p.delta[stat];
  const bf16_t* kbase = p.k + static_cast<long long>(b) * p.Sk * k_row + hk * D;
  const bf16_t* vbase = p.v + static_cast<long long>(b) * p.Sk * k_row + hk * D;
  int k_end = p.Sk;
  if (CAUSAL) k_end = min(p.Sk, min(qb0 + 63, p.Sq - 1) + p.q_offset + 1);
  const int ntiles = (k_end + TR - 1) / TR;
  const int q_last = min(qw0 + 15, p.Sq - 1);

  f32x4_t acc[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto stage = [&](int buf, int t) {
    unsigned char* d = lds + buf * 2 * TILE_BYTES;
    bwd_stage<D>(kbase, k_row, t * TR, p.Sk, d, wid, lane);
    bwd_stage<D>(vbase, k_row, t * TR, p.Sk, d + TILE_BYTES, wid, lane);
  };
  if (ntiles > 0) stage(0, 0);
  for (int t = 0; t < ntiles; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                        // the tile is there, and every wave is done with the one before it
    if (t + 1 < ntiles) stage((t + 1) & 1, t + 1);
    if (qw0 >= p.Sq || (CAUSAL && t * TR > q_last + p.q_offset)) continue;      // nothing of the tile is visible
    const unsigned char* k_lds = lds + (t & 1) * 2 * TILE_BYTES;
    const unsigned char* v_lds = k_lds + TILE_BYTES;
    const int lim = CAUSAL ? min(p.Sk - 1, qi + p.q_offset) : p.Sk - 1;
    const bool edge = !CAUSAL || t * TR + TR > p.Sk || t * TR + TR - 1 > qw0 + p.q_offset;
#pragma unroll
    for (int s = 0; s < TR / 32; ++s) {
      f32x4_t st[2], dp[2];
      mma_rows<D>(st, k_lds, qf, s, fr, g);      // S^T[key][q]
      mma_rows<D>(dp, v_lds, dof, s, fr, g);     // dP^T[key][q]
      const int key0 = t * TR + s * 32 + g * 4;
      unsigned int pk[2][2];
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        float ds[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = key0 + n * 16 + r;
          const float pr = !edge || key <= lim ? __builtin_amdgcn_exp2f(st[n][r] * p.scale_log2e - lse) : 0.f;
          ds[r] = pr * (dp[n][r] - dlt) * p.scale;
        }
        pk[n][0] = pack_bf16x2(ds[0], ds[1]);
        pk[n][1] = pack_bf16x2(ds[2], ds[3]);
      }
      mma_tr<D>(acc, k_lds, pk, s, fr, g);       // dQ^T[d][q] += K^T dS^T
    }
  }
  if (qi >= p.Sq) return;
  bf16_t* dqp = p.dq + (static_cast<long long>(b) * p.Sq + qi) * q_row + h * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const u32x2_t w = {pack_bf16x2(acc[dt][0], acc[dt][1]), pack_bf16x2(acc[dt][2], acc[dt][3])};
    *reinterpret_cast<u32x2_t*>(dqp + dt * 16 + g * 4) = w;
  }
}

// ------------------------------------------------------------------- dK, dV
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 3) void attn_bwd_dkv_kernel(AttnBwdParams p) {
  constexpr int TR = bwd_tile<D>(), TILE_BYTES = TR * D * 2, KS = D / 32, DT = D / 16;
  __shared__ __attribute__((aligned(16))) unsigned char lds[4 * TILE_BYTES];      // [2][Q | dO]
  __shared__ __attribute__((aligned(16))) float stats[2][2][TR];                  // [2][log-sum-exp | delta]
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, g = lane >> 4;
  const int b = blockIdx.z, hk = blockIdx.x, rep = p.Hq / p.Hkv;
  const int kb0 = blockIdx.y * 64, kw0 = kb0 + wid * 16, ki = kw0 + fr, ki_c = min(ki, p.Sk - 1);
  const long long q_row = static_cast<long long>(p.Hq) * D, k_row = static_cast<long long>(p.Hkv) * D;
  const bf16_t* kp = p.k + (static_cast<long long>(b) * p.Sk + ki_c) * k_row + hk * D;
  const bf16_t* vp = p.v + (static_cast<long long>(b) * p.Sk + ki_c) * k_row + hk * D;
  bf16x8_t kf[KS], vf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    kf[ks] = *reinterpret_cast<const bf16x8_t*>(kp + ks * 32 + g * 8);
    vf[ks] = *reinterpret_cast<const bf16x8_t*>(vp + ks * 32 + g * 8);
  }
  // first query tile that can see this key block: q + q_offset >= kb0
  int t_begin = 0;
  if (CAUSAL) t_begin = max(0, kb0 - p.q_offset) / TR;
  const int per = max(0, (p.Sq + TR - 1) / TR - t_begin), steps = rep * per;      // tiles of a query head, and of all of them

  f32x4_t dk[DT], dv[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) { dk[i] = f32x4_t{0.f, 0.f, 0.f, 0.f}; dv[i] = f32x4_t{0.f, 0.f, 0.f, 0.f}; }
  float stat = 0.f;                                     // of the tile on its way; wave 0: log-sum-exp, wave 1: delta
  int next_h = hk * rep, next_t = t_begin;
  auto stage = [&](int buf) {
    unsigned char* d = lds + buf * 2 * TILE_BYTES;
    const long long head = static_cast<long long>(b) * p.Sq * q_row + next_h * D;
    bwd_stage<D>(p.q + head, q_row, next_t * TR, p.Sq, d, wid, lane);
    bwd_stage<D>(p.d_o + head, q_row, next_t * TR, p.Sq, d + TILE_BYTES, wid, lane);
    if (wid < 2 && lane < TR)
      stat = (wid ? p.delta : p.lse)[(static_cast<long long>(b) * p.Hq + next_h) * p.Sq + min(next_t * TR + lane, p.Sq - 1)];
    if (++next_t == t_begin + per) { next_t = t_begin; ++next_h; }
  };
  if (steps > 0) stage(0);
  int t = t_begin;
  for (int i = 0; i < steps; ++i, t = t + 1 == t_begin + per ? t_begin : t + 1) {
    const int buf = i & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (wid < 2 && lane < TR) stats[buf][wid][lane] = stat;
    __syncthreads();                        // the tile is there, and every wave is done with the one before it
    if (i + 1 < steps) stage(buf ^ 1);
    if (kw0 >= p.Sk || (CAUSAL && kw0 > min(t * TR + TR, p.Sq) - 1 + p.q_offset)) continue;      // no query of the tile sees these keys
    const unsigned char* q_lds = lds + buf * 2 * TILE_BYTES;
    const unsigned char* do_lds = q_lds + TILE_BYTES;
    const bool edge = !CAUSAL || t * TR + TR > p.Sq || kw0 + 16 > p.Sk || kw0 + 15 > t * TR + p.q_offset;
#pragma unroll
    for (int s = 0; s < TR / 32; ++s) {
      f32x4_t st[2], dp[2];
      mma_rows<D>(st, q_lds, kf, s, fr, g);      // S[q][key]: key on the lane
      mma_rows<D>(dp, do_lds, vf, s, fr, g);     // dP[q][key]
      unsigned int pp[2][2], pd[2][2];
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const int q0 = s * 32 + n * 16 + g * 4;
        const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(&stats[buf][0][q0]);
        const f32x4_t d4 = *reinterpret_cast<const f32x4_t*>(&stats[buf][1][q0]);
        float pr[4], ds[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int qq = t * TR + q0 + r;
          const bool vis = !edge || (qq < p.Sq && ki < p.Sk && (!CAUSAL || ki <= qq + p.q_offset));
          pr[r] = vis ? __builtin_amdgcn_exp2f(st[n][r] * p.scale_log2e - l4[r]) : 0.f;
          ds[r] = pr[r] * (dp[n][r] - d4[r]) * p.scale;
        }
        pp[n][0] = pack_bf16x2(pr[0], pr[1]); pp[n][1] = pack_bf16x2(pr[2], pr[3]);
        pd[n][0] = pack_bf16x2(ds[0], ds[1]); pd[n][1] = pack_bf16x2(ds[2], ds[3]);
      }
      mma_tr<D>(dv, do_lds, pp, s, fr, g);       // dV^T[d][key] += dO^T P
      mma_tr<D>(dk, q_lds, pd, s, fr, g);        // dK^T[d][key] += Q^T dS
    }
  }
  if (ki >= p.Sk) return;
  const long long at = (static_cast<long long>(b) * p.Sk + ki) * k_row + hk * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const u32x2_t wk = {pack_bf16x2(dk[dt][0], dk[dt][1]), pack_bf16x2(dk[dt][2], dk[dt][3])};
    const u32x2_t wv = {pack_bf16x2(dv[dt][0], dv[dt][1]), pack_bf16x2(dv[dt][2], dv[dt][3])};
    *reinterpret_cast<u32x2_t*>(p.dk + at + dt * 16 + g * 4) = wk;
    *reinterpret_cast<u32x2_t*>(p.dv + at + dt * 16 + g * 4) = wv;
  }
}

template <int D>
static void launch_bwd_d(const AttnBwdParams& p, const bf16_t* o, float* delta, int B, int causal, hipStream_t st) {
  const long long rows = static_cast<long long>(B) * p.Sq * p.Hq;
  const long long threads = rows * (D / 8);
  hipLaunchKernelGGL(attn_delta_kernel<D>, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, st,
                     o, p.d_o, delta, rows, p.Sq, p.Hq);
  // a head's blocks follow each other at a distance of the heads (one XCD and its L2 where the heads are a multiple of eight), those
  // with the most tiles ahead
  const dim3 gq(p.Hq, (p.Sq + 63) / 64, B), gk(p.Hkv, (p.Sk + 63) / 64, B), blk(256);
  if (causal) {
    hipLaunchKernelGGL((attn_bwd_dq_kernel<D, true>), gq, blk, 0, st, p);
    hipLaunchKernelGGL((attn_bwd_dkv_kernel<D, true>), gk, blk, 0, st, p);
  } else {
    hipLaunchKernelGGL((attn_bwd_dq_kernel<D, false>), gq, blk, 0, st, p);
    hipLaunchKernelGGL((attn_bwd_dkv_kernel<D, false>), gk, blk, 0, st, p);
  }
}

void launch_attn_bwd(const bf16_t* q, const bf16_t* k, const bf16_t* v, const bf16_t* o, const bf16_t* d_o,
                     const float* lse, float* delta, bf16_t* dq, bf16_t* dk, bf16_t* dv, int B, int Sq,
                     int Sk, int Hq, int Hkv, int D, int causal, int q_offset, float scale, hipStream_t st) {
  AttnBwdParams p;
  p.q = q; p.k = k; p.v = v; p.d_o = d_o; p.lse = lse; p.delta = delta; p.dq = dq; p.dk = dk; p.dv = dv;
  p.Sq = Sq; p.Sk = Sk; p.Hq = Hq; p.Hkv = Hkv; p.q_offset = q_offset;
  p.scale = scale; p.scale_log2e = scale * 1.4426950408889634f;
  if (D == 128) launch_bwd_d<128>(p, o, delta, B, causal, st);
  else launch_bwd_d<64>(p, o, delta, B, causal, st);
}

}  // namespace evgpt
