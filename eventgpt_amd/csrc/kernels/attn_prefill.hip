// Fused (flash-style) attention for many query rows: LLM prefill (causal,
// head_dim 128), speculative-verify batches (causal with an offset into a long
// cache) and the ViT encoder (non-causal, head_dim 64, 577 tokens).
//
// One block = 4 or 8 waves = 64 or 128 query rows of one (batch, head); each wave owns 16
// rows.  K/V tiles of 64 keys go straight into LDS, the next one while a tile is
// multiplied.  The score tile is computed TRANSPOSED,
//     S^T[key][q] = K · Q^T        (K rows = MFMA A operand, Q^T = B operand)
// so that the query index lives on the lane (lane & 15) and a lane's 16
// accumulator values are 16 different keys of ONE query.  Consequences:
//   * softmax row statistics are in-lane reductions + 2 lane swaps (maxima) or shuffles (sums);
//   * the exponentiated tile, converted to bf16, already *is* the B operand of
//     the second product  O^T[d][q] = V^T · P^T  — no LDS round trip for P
//     (the contraction index is permuted consistently on both operands);
//   * V^T fragments come from the row-major V tile with the hardware
//     transposing read ds_read_b64_tr_b16, so V is staged exactly like K;
//   * rescaling O by exp(m_old - m_new) is a per-lane scalar multiply.
// LDS images are XOR-swizzled at 16-byte-chunk granularity so both the row
// reads (ds_read_b128) and the transposed reads spread over the banks.
#include <type_traits>

#include "common.h"
#include "attn_common.h"
#include "../evgpt_kernels.h"

namespace evgpt {

// what rounding the pair to bf16 left out
__device__ __forceinline__ unsigned int bf16_rest(float a, float b, unsigned int packed) {
  return pack_bf16x2(a - bf16lo(packed), b - bf16hi(packed));
}

// The largest of a lane's sixteen scores, then of the four lanes (16 apart) that hold the query's other keys.  v_maximum3 takes
// three scores as an MFMA leaves them (fmaxf quiets its operands first, two instructions more a pair); the lanes trade rows of
// 16 and 32 in registers, where a shuffle waits for the LDS four times a key tile.
__device__ __forceinline__ float maximum3(float a, float b, float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}
__device__ __forceinline__ float score_max(const f32x4_t (&st)[4]) {
  float a = maximum3(st[0][0], st[0][1], st[0][2]), b = maximum3(st[0][3], st[1][0], st[1][1]);
  a = maximum3(a, st[1][2], st[1][3]);
  b = maximum3(b, st[2][0], st[2][1]);
  a = maximum3(a, st[2][2], st[2][3]);
  b = maximum3(b, st[3][0], st[3][1]);
  a = maximum3(a, st[3][2], st[3][3]);
  a = __builtin_elementwise_maximum(a, b);
  return max_of_quads(a);
}
__device__ __forceinline__ float score_max(const f32x4_t (&st)[2]) {
  float a = maximum3(st[0][0], st[0][1], st[0][2]);
  const float b = maximum3(st[0][3], st[1][0], st[1][1]);
  a = maximum3(a, st[1][2], st[1][3]);
  return max_of_quads(__builtin_elementwise_maximum(a, b));
}
struct AttnParams {
  const bf16_t* q; const bf16_t* k; const bf16_t* v; bf16_t* o;
  long long q_sb, q_ss, q_sh;   // element strides: batch, sequence, head
  long long k_sb, k_ss, k_sh;
  long long v_sb, v_ss, v_sh;
  long long o_sb, o_ss, o_sh;
  const int* kv_len;            // optional device-side key count per batch
  int Sq, Sk, Hq, Hkv;
  int q_offset;                 // absolute position of query row 0 minus key 0 (causal)
  int q_offset_from_len;        // if set: q_offset = kv_len[b] - Sq
  float scale_log2e;            // positive: the softmax takes maxima of raw scores; see set_scale
  unsigned int q_and, q_xor;    // applied to the words of Q
  // split-KV mode (few query rows against a long cache): block x = key split
  float* part_o;                // [B][Hq][nsplit][Sq][D] unnormalised fp32
  float* part_ml;               // [B][Hq][nsplit][Sq][2] (running max in log2 units, sum)
  int nsplit;
  float* lse;                   // optional [B][Hq][Sq]: log2 of the row's softmax denominator in the
                                // scaled-log2 domain (max + log2(sum)); the backward recomputes P from it
  const bf16_t* gate;           // optional [B * Sq][gate_ld]: head h's output is multiplied by sigmoid of column h
  int gate_ld;
  const int* items;             // ITEMS: [blocks][4] first query row, rows (<= 64), key row of the chunk, position in it
};
// softmax(s Q K^T) with any s, by a positive scale: a negative s flips the signs of Q, zero clears Q (all scores are then equal)
static void set_scale(AttnParams& p, float scale) {
  p.q_and = scale == 0.f ? 0u : 0xffffffffu;
  p.q_xor = scale < 0.f ? 0x80008000u : 0u;
  p.scale_log2e = (scale == 0.f ? 1.f : (scale < 0.f ? -scale : scale)) * 1.4426950408889634f;
}
__device__ __forceinline__ bf16x8_t load_q(const AttnParams& p, const bf16_t* src) {
  u32x4_t v = load16(src);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (v[i] & p.q_and) ^ p.q_xor;
  return __builtin_bit_cast(bf16x8_t, v);
}
__device__ __forceinline__ float head_gate(const AttnParams& p, long long row, int h) {
  return 1.f / (1.f + __expf(-bf16_to_f32(p.gate[row * p.gate_ld + h])));
}

__device__ __forceinline__ void attn_buffer_to_lds16(const unsigned char* src, int bytes, unsigned char* lds, int voff) {
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(src), 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (void __attribute__((address_space(3)))*)lds, 16, voff, 0, 0, 0);
}

// GROUPS = 2: the block is two such groups of 4 waves over the SAME 64 query rows; group 0 takes the
// even key tiles of the block's range and group 1 the odd ones, each through its own K / V tile
// buffers, and group 1's running (max, sum, O) is merged into group 0's at the end through LDS.  A
// few hundred query rows of a few heads are fewer blocks than CUs, each a serial chain over its key
// tiles; two groups halve the chain and double the waves (used for the ViT, see launch_attn_prefill).
// WAVES = 8: 128 query rows share the tiles, so that a CU has twice the waves in the same LDS.
// Bound by the chain of a tile (scores, maxima, exponentials, weights times values) and by LDS reads of twice the matrix time, which
// other waves fill.  Tiles through registers behind two barriers / straight into LDS behind one, us: 636 causal rows, 32 heads of 128
// 22.8 / 17.8; 300 10.6 / 8.3; 1 024 39.3 / 28.4; 100 rows over 300 keys, 8 key heads 10.8 / 8.0; one frame of 577 tokens, 16 heads of
// 64 9.2 / 8.3, two 15.9 / 13.5; ITEMS, eight prompts of 342 to 685, 32 heads 77 / 67.  With D = 128 tiles of 32 keys, five blocks a CU instead
// of two, 23 where these take 18, in 170 registers instead of 150 20; ITEMS of 200 and fewer rows 2 to 10 % ahead with them, longer
// ones as much behind.
// WP: the softmax weights enter the second product as two bf16 parts (16 mantissa bits) instead of one.
// ITEMS: block x takes the query rows, keys and position of an entry of `items`, so runs of any lengths and sequences share
// a launch.  Eight prompts of 342 to 682 tokens, 32 heads of 128: one launch a prompt 170 us a layer, one for all 80; 32 prompts of
// 200, 16 heads: 52 (148 with the 64-column blocks of attn_chunk.hip).
template <int D, bool CAUSAL, bool SPLIT = false, int GROUPS = 1, bool WP = false, bool ITEMS = false, int WAVES = 4>
__global__ __launch_bounds__(64 * WAVES * GROUPS, WAVES == 8 || GROUPS == 2 ? 4 : 2) void attn_prefill_kernel(AttnParams p) {
  constexpr int TR = D == 128 && GROUPS == 2 ? 32 : 64;       // keys of a tile
  constexpr int CPR = D / 8;                  // 16-byte chunks per row
  constexpr int TILE_BYTES = TR * D * 2;
  constexpr int NIW = TILE_BYTES / 1024 / WAVES;  // 1 KB staging instructions per wave and tile
  constexpr int KS = D / 32;                  // k-steps of the QK^T product
  constexpr int DT = D / 16;                  // 16-wide output column tiles
  constexpr int NT = TR / 16;                 // 16-key sub-tiles
  static_assert(GROUPS == 1 || GROUPS == 2, "one or two groups of four waves");
  static_assert(GROUPS == 1 || (DT * 4 + 2) * 256 * 4 <= GROUPS * 4 * TILE_BYTES, "merge buffer fits the tile buffers");
  __shared__ __attribute__((aligned(16))) unsigned char lds[GROUPS * 4 * TILE_BYTES];
  const int grp = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * WAVES));
  unsigned char* ring = lds + grp * 4 * TILE_BYTES;       // [2][K | V]

  const int tid = threadIdx.x % (64 * WAVES), lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);   // within the group
  const int fr = lane & 15, g = lane >> 4;
  const int b = blockIdx.z, h = blockIdx.y;
  const int hk = h / (p.Hq / p.Hkv);
  // a device-side key count can never address past the buffer capacity p.Sk
  int Sk = p.kv_len ? p.kv_len[b] : p.Sk;
  Sk = Sk > p.Sk ? p.Sk : (Sk < 0 ? 0 : Sk);
  int q_off = p.q_offset_from_len ? (Sk - p.Sq) : p.q_offset;
  long long row0 = static_cast<long long>(b) * p.Sq;      // the block's rows in the gate
  if constexpr (ITEMS) {                       // (p is this thread's copy)
    const int* it = p.items + (gridDim.x - 1 - blockIdx.x) * 4;      // a sequence's last rows see the most keys: first
    row0 = it[0];
    q_off = it[3];
    p.Sq = min(it[1], 64);
    Sk = q_off + p.Sq;
    p.q += row0 * p.q_ss; p.o += row0 * p.o_ss;
    p.k += static_cast<long long>(it[2]) * p.k_ss; p.v += static_cast<long long>(it[2]) * p.v_ss;
  }
  const int qb0 = SPLIT || ITEMS ? 0 : (CAUSAL && WAVES == 8 ? gridDim.x - 1 - blockIdx.x : blockIdx.x) * (16 * WAVES);  // first query row of the block
  const int qi = qb0 + wid * 16 + fr;        // this lane's query row
  const int qi_c = qi < p.Sq ? qi : p.Sq - 1;

  // Q^T fragments straight from global: Q[qi][ks*32 + 8g .. +8]
  bf16x8_t qf[KS];
  {
    const bf16_t* qp = p.q + b * p.q_sb + static_cast<long long>(qi_c) * p.q_ss + h * p.q_sh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = load_q(p, qp + ks * 32 + g * 8);
  }

  const unsigned char* kbase = reinterpret_cast<const unsigned char*>(p.k + b * p.k_sb + hk * p.k_sh);
  const unsigned char* vbase = reinterpret_cast<const unsigned char*>(p.v + b * p.v_sb + hk * p.v_sh);

  // keys this block needs: all of them, or up to its last query's diagonal
  int k_end = Sk;
  if (CAUSAL) {
    const int last_q = min(qb0 + 16 * WAVES - 1, p.Sq - 1);
    k_end = min(Sk, last_q + q_off + 1);
  }
  int ntiles = (k_end + TR - 1) / TR;
  int t_begin = 0;
  if (SPLIT) {
    const int per = (ntiles + p.nsplit - 1) / p.nsplit;
    t_begin = min(static_cast<int>(blockIdx.x) * per, ntiles);
    ntiles = min(t_begin + per, ntiles);
  }
  // waves whose 16 query rows are all padding only help staging the tiles
  const bool wave_active = qb0 + wid * 16 < p.Sq;

  const int q_hi = min(qb0 + wid * 16 + 15, p.Sq - 1);       // last query row of this wave

  // Tiles go straight into LDS (the swizzle applied to the source; rows past the last key are zeros from the descriptor's range
  // check), the next one while a tile is multiplied, one barrier a tile.
  const long long k_bytes = Sk > 0 ? 2ll * ((Sk - 1) * p.k_ss + D) : 0;
  const long long v_bytes = Sk > 0 ? 2ll * ((Sk - 1) * p.v_ss + D) : 0;
  int voff_k[NIW], voff_v[NIW];
#pragma unroll
  for (int j = 0; j < NIW; ++j) {
    const int idx = (wid * NIW + j) * 64 + lane, row = idx / CPR, ch = (idx % CPR) ^ swz<D>(row);
    voff_k[j] = static_cast<int>((row * p.k_ss + ch * 8) * 2);
    voff_v[j] = static_cast<int>((row * p.v_ss + ch * 8) * 2);
  }
  auto range = [](long long left) { return static_cast<int>(left < 0 ? 0 : (left > 0x7fffffff ? 0x7fffffff : left)); };
  auto stage = [&](int buf, int t) {
    unsigned char* kd = ring + buf * 2 * TILE_BYTES + wid * NIW * 1024;
    const long long ka = 2ll * t * TR * p.k_ss, va = 2ll * t * TR * p.v_ss;
#pragma unroll
    for (int j = 0; j < NIW; ++j) attn_buffer_to_lds16(kbase + ka, range(k_bytes - ka), kd + j * 1024, voff_k[j]);
#pragma unroll
    for (int j = 0; j < NIW; ++j) attn_buffer_to_lds16(vbase + va, range(v_bytes - va), kd + TILE_BYTES + j * 1024, voff_v[j]);
  };

  f32x4_t o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  auto compute = [&](int buf, int t) {
    const unsigned char* k_lds = ring + buf * 2 * TILE_BYTES;
    const unsigned char* v_lds = k_lds + TILE_BYTES;
    // ---- S^T tile: sub-tiles of 16 keys
    f32x4_t st[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) st[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)      // k-step outermost: independent accumulators in turn
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(
            k_lds + tile_off<D>(n * 16 + fr, ks * 4 + g));
        st[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], st[n], 0, 0, 0);
      }

    // ---- online softmax on the RAW scores (lane = one query; 16 keys in registers).  The scale
    // is positive, so the maximum commutes with it and exp2(s * scale - m * scale) is one fma and
    // one v_exp_f32 per score; keys are masked only in tiles that cross the diagonal or the end
    // of the keys; the accumulators (AGPRs) are rescaled only when some row's maximum moved.
    const int key0 = t * TR + g * 4;
    const int last_key = t * TR + TR - 1;
    if (last_key > Sk - 1 || (CAUSAL && last_key > qb0 + wid * 16 + q_off)) {
      const int lim = CAUSAL ? min(Sk - 1, qi + q_off) : Sk - 1;  // last visible key
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (key0 + n * 16 + r > lim) st[n][r] = -INFINITY;
    }
    const float mt = score_max(st);
    const float mn = fmaxf(m, mt);
    const float msafe = mn == -INFINITY ? 0.f : mn;
    if (__builtin_amdgcn_ballot_w64(mn != m) != 0) {
      const float alpha = __builtin_amdgcn_exp2f((m - msafe) * p.scale_log2e);  // m = -inf -> 0
      l *= alpha;
#pragma unroll
      for (int i = 0; i < DT; ++i) o[i] *= alpha;
      m = mn;
    }
    const float ms = msafe * p.scale_log2e;
    float psum = 0.f;
    unsigned int pk[NT][2], pl[NT][2];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      float e[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) { e[r] = __builtin_amdgcn_exp2f(fmaf(st[n][r], p.scale_log2e, -ms)); psum += e[r]; }
      pk[n][0] = pack_bf16x2(e[0], e[1]);
      pk[n][1] = pack_bf16x2(e[2], e[3]);
      if constexpr (WP) {
        pl[n][0] = bf16_rest(e[0], e[1], pk[n][0]);
        pl[n][1] = bf16_rest(e[2], e[3], pk[n][1]);
      }
    }
    l += psum;

    // ---- O^T += V^T · P^T, two k-steps of 32 keys; slot (g, j) <-> key
    //      32s + 4g + j (j < 4) or 32s + 16 + 4g + (j - 4)
#pragma unroll
    for (int s = 0; s < TR / 32; ++s) {
      u32x4_t pw = {pk[2 * s][0], pk[2 * s][1], pk[2 * s + 1][0], pk[2 * s + 1][1]};
      const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, pw);
      bf16x8_t pf_lo = pf;
      if constexpr (WP) {
        const u32x4_t lw = {pl[2 * s][0], pl[2 * s][1], pl[2 * s + 1][0], pl[2 * s + 1][1]};
        pf_lo = __builtin_bit_cast(bf16x8_t, lw);
      }
      const int q4 = fr >> 2, p4 = fr & 3;
      const int r0 = s * 32 + g * 4 + q4, r1 = r0 + 16;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int ch = dt * 2 + (p4 >> 1);
        const s16x4_t lo = read_tr16((lds_s16x4_t*)(v_lds + tile_off<D>(r0, ch) + 8 * (p4 & 1)));
        const s16x4_t hi = read_tr16((lds_s16x4_t*)(v_lds + tile_off<D>(r1, ch) + 8 * (p4 & 1)));
        typedef __attribute__((ext_vector_type(8))) short s16x8_t;
        const s16x8_t vv = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        if constexpr (WP)
          o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vv), pf_lo, o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vv), pf,
                                                        o[dt], 0, 0, 0);
      }
    }
  };

  // this group's tiles: first, first + GROUPS, ...; the trip count is group 0's (block-uniform:
  // the loop contains barriers), a group past its last tile only keeps step
  const int first = t_begin + grp;
  const int n_mine = first < ntiles ? (ntiles - first + GROUPS - 1) / GROUPS : 0;
  const int n_iter = t_begin < ntiles ? (ntiles - t_begin + GROUPS - 1) / GROUPS : 0;
  if (0 < n_mine) stage(0, first);
  for (int k = 0; k < n_iter; ++k) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                             // the tile is there, and every wave is done with the one before it
    if (k + 1 < n_mine) stage((k + 1) & 1, first + GROUPS * (k + 1));
    const int t = first + GROUPS * k;
    if (wave_active && k < n_mine && !(CAUSAL && t * TR > q_hi + q_off)) compute(k & 1, t);      // (else nothing of it is visible)
  }

  // ---- finalise: l is a per-lane partial over this lane's key slots
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if constexpr (GROUPS == 2) {
    // group 1 hands its state over in lane-private columns of the (now idle) tile buffers; lane
    // (wave, lane) of group 0 holds the same query row and output columns as its counterpart
    __syncthreads();
    float* xch = reinterpret_cast<float*>(lds);
    const int col = tid;   // wave * 64 + lane within the group
    if (grp == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) xch[(dt * 4 + r) * 256 + col] = o[dt][r];
      xch[(DT * 4) * 256 + col] = m;
      xch[(DT * 4 + 1) * 256 + col] = l;
    }
    __syncthreads();
    if (grp == 1) return;
    const float m1 = xch[(DT * 4) * 256 + col], l1 = xch[(DT * 4 + 1) * 256 + col];
    const float mn = fmaxf(m, m1);
    const float msafe = mn == -INFINITY ? 0.f : mn;
    const float a0 = __builtin_amdgcn_exp2f((m - msafe) * p.scale_log2e);    // -inf -> 0
    const float a1 = __builtin_amdgcn_exp2f((m1 - msafe) * p.scale_log2e);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[dt][r] = o[dt][r] * a0 + xch[(dt * 4 + r) * 256 + col] * a1;
    l = l * a0 + l1 * a1;
    m = mn;
  }
  if (SPLIT) {
    if (qi < p.Sq) {
      const long long slot = ((static_cast<long long>(b) * p.Hq + h) * p.nsplit + blockIdx.x) * p.Sq + qi;
      float* po = p.part_o + slot * D;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        *reinterpret_cast<f32x4_t*>(po + dt * 16 + g * 4) = o[dt];
      if (g == 0) { p.part_ml[slot * 2] = m * p.scale_log2e; p.part_ml[slot * 2 + 1] = l; }   // m is kept unscaled
    }
    return;
  }
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (p.gate && qi < p.Sq) inv *= head_gate(p, row0 + qi, h);
  if (p.lse && g == 0 && qi < p.Sq)
    p.lse[(static_cast<long long>(b) * p.Hq + h) * p.Sq + qi] = l > 0.f ? m * p.scale_log2e + log2f(l) : INFINITY;
  if (qi < p.Sq) {
    bf16_t* op = p.o + b * p.o_sb + static_cast<long long>(qi) * p.o_ss + h * p.o_sh;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      u32x2_t w = {pack_bf16x2(o[dt][0] * inv, o[dt][1] * inv),
                   pack_bf16x2(o[dt][2] * inv, o[dt][3] * inv)};
      *reinterpret_cast<u32x2_t*>(op + dt * 16 + g * 4) = w;
    }
  }
}

// Same computation for long query ranges: one block = 256 query rows, each wave owns TWO 16-row
// query tiles, so every K fragment (ds_read_b128) and every V^T fragment (two transposing reads)
// feeds two MFMAs instead of one -- with 16 rows per wave the kernel above reads 32 KB of LDS
// per wave and key tile for 32 MFMAs and is bound by the LDS pipe.  K / V tiles are staged
// straight into LDS (buffer_load ... lds, swizzle applied to the per-lane source offset; keys past
// the end come back as zeros from the descriptor's range check) into a ring of AW_STAGES tiles:
// loads are in flight while other tiles are computed, and no staging registers are held.
constexpr int AW_STAGES = 4;   // K / V tiles in the LDS ring: three are read between two barriers, one is on its way

// QT: 16-row query tiles per wave (2: every K / V fragment feeds two MFMAs); 256 query rows per block
constexpr int AW_WAVES = 8, QT = 2;
template <int D, bool CAUSAL, bool WP = false>
__global__ __launch_bounds__(AW_WAVES * 64) void attn_prefill_wide_kernel(AttnParams p) {
  constexpr int CPR = D / 8;
  constexpr int TILE_BYTES = TK * D * 2;
  constexpr int NIW = TILE_BYTES / 1024 / AW_WAVES;   // 1 KB staging instructions per wave and tile
  constexpr int KS = D / 32;
  constexpr int DT = D / 16;
  constexpr int BR = AW_WAVES * 16 * QT;              // query rows per block
  static_assert(NIW >= 1, "a tile is at least one staging instruction per wave");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // [stage][K | V]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, g = lane >> 4;
  // grid = (heads, query blocks, batch): consecutive blocks are the same query block of different
  // heads, so under causal masking the whole grid starts in order of decreasing work
  const int b = blockIdx.z, h = blockIdx.x;
  const int hk = h / (p.Hq / p.Hkv);
  int Sk = p.kv_len ? p.kv_len[b] : p.Sk;
  Sk = Sk > p.Sk ? p.Sk : (Sk < 0 ? 0 : Sk);
  const int q_off = p.q_offset_from_len ? (Sk - p.Sq) : p.q_offset;
  // causal: the blocks with the most keys start first
  const int qb0 = (CAUSAL ? gridDim.y - 1 - blockIdx.y : blockIdx.y) * BR;
  const int qw0 = qb0 + wid * 16 * QT;       // first query row of this wave

  bf16x8_t qf[QT][KS];
  int qi[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    qi[qt] = qw0 + qt * 16 + fr;
    const int qc = qi[qt] < p.Sq ? qi[qt] : p.Sq - 1;
    const bf16_t* qp = p.q + b * p.q_sb + static_cast<long long>(qc) * p.q_ss + h * p.q_sh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[qt][ks] = load_q(p, qp + ks * 32 + g * 8);
  }

  const unsigned char* kbase = reinterpret_cast<const unsigned char*>(p.k + b * p.k_sb + hk * p.k_sh);
  const unsigned char* vbase = reinterpret_cast<const unsigned char*>(p.v + b * p.v_sb + hk * p.v_sh);
  const long long k_bytes = Sk > 0 ? 2ll * ((Sk - 1) * p.k_ss + D) : 0;
  const long long v_bytes = Sk > 0 ? 2ll * ((Sk - 1) * p.v_ss + D) : 0;
  int voff_k[NIW], voff_v[NIW];
#pragma unroll
  for (int j = 0; j < NIW; ++j) {
    const int idx = (wid * NIW + j) * 64 + lane;
    const int row = idx / CPR, ch = (idx % CPR) ^ swz<D>(row);
    voff_k[j] = static_cast<int>((row * p.k_ss + ch * 8) * 2);
    voff_v[j] = static_cast<int>((row * p.v_ss + ch * 8) * 2);
  }
  auto stage = [&](int buf, int t) {
    unsigned char* kd = lds + buf * 2 * TILE_BYTES + wid * NIW * 1024;
    const long long ka = 2ll * t * TK * p.k_ss, va = 2ll * t * TK * p.v_ss;
    const int kl = static_cast<int>(k_bytes > ka ? k_bytes - ka : 0), vl = static_cast<int>(v_bytes > va ? v_bytes - va : 0);
#pragma unroll
    for (int j = 0; j < NIW; ++j) attn_buffer_to_lds16(kbase + ka, kl, kd + j * 1024, voff_k[j]);
#pragma unroll
    for (int j = 0; j < NIW; ++j) attn_buffer_to_lds16(vbase + va, vl, kd + TILE_BYTES + j * 1024, voff_v[j]);
  };

  int k_end = Sk;
  if (CAUSAL) k_end = min(Sk, min(qb0 + BR - 1, p.Sq - 1) + q_off + 1);
  const int ntiles = (k_end + TK - 1) / TK;
  const bool wave_active = qw0 < p.Sq;
  const int q_hi = min(qw0 + 16 * QT - 1, p.Sq - 1);   // last query row of this wave

  f32x4_t o[QT][DT];
  float m[QT], l[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m[qt] = -INFINITY; l[qt] = 0.f;
#pragma unroll
    for (int i = 0; i < DT; ++i) o[qt][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // The loop is software-pipelined into two phases per key tile,
  //   S: softmax of tile t (VALU)            M: P·V of tile t, then K·Q^T of tile t+1 (MFMA)
  // and the two halves of the block (waves 0-3 / 4-7, one of each per SIMD) meet at ONE barrier per tile, which the first
  // half passes after M and the second after S: while one half is in its MFMA phase the other is in its
  // softmax, so the SIMD's matrix and vector pipes work at the same time instead of taking turns.
  f32x4_t st[QT][4];
  unsigned int pk[QT][4][2], pl[QT][WP ? 4 : 1][2];
  auto qk = [&](const unsigned char* k_lds) {
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) st[qt][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // k-step outermost: eight independent accumulators between two MFMAs on the same one
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(k_lds + tile_off<D>(n * 16 + fr, ks * 4 + g));
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
          st[qt][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qt][ks], st[qt][n], 0, 0, 0);
      }
  };
  auto softmax = [&](int t) {
    // Online softmax on the RAW scores (the scale is positive, so the maximum commutes with it):
    // exp2(s * scale - m * scale) is one fma and one v_exp_f32 per score.  The softmax, not the
    // MFMA, bounds this kernel (16 scores per lane and query tile, 4 cycles per VALU instruction),
    // so everything avoidable is avoided: keys are masked only in tiles that cross the diagonal
    // or the end of the keys, and the accumulators are rescaled only when some row's maximum
    // moved (they live in AGPRs; a rescale moves all of them through VGPRs).
    const int key0 = t * TK + g * 4;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int q_lo = qw0 + qt * 16;                     // first query row of the tile (wave-uniform)
      const int last_key = t * TK + TK - 1;
      const bool need_mask = last_key > Sk - 1 || (CAUSAL && last_key > q_lo + q_off);
      if (need_mask) {
        const int lim = CAUSAL ? min(Sk - 1, qi[qt] + q_off) : Sk - 1;
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (key0 + n * 16 + r > lim) st[qt][n][r] = -INFINITY;
      }
      const float mt = score_max(st[qt]);
      const float mn = fmaxf(m[qt], mt);
      const float msafe = mn == -INFINITY ? 0.f : mn;
      if (__builtin_amdgcn_ballot_w64(mn != m[qt]) != 0) {   // some row's maximum moved
        const float alpha = __builtin_amdgcn_exp2f((m[qt] - msafe) * p.scale_log2e);   // m = -inf -> 0
        l[qt] *= alpha;
#pragma unroll
        for (int i = 0; i < DT; ++i) o[qt][i] *= alpha;
        m[qt] = mn;
      }
      const float ms = msafe * p.scale_log2e;
      float psum = 0.f;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) { e[r] = __builtin_amdgcn_exp2f(fmaf(st[qt][n][r], p.scale_log2e, -ms)); psum += e[r]; }
        pk[qt][n][0] = pack_bf16x2(e[0], e[1]);
        pk[qt][n][1] = pack_bf16x2(e[2], e[3]);
        if constexpr (WP) {
          pl[qt][n][0] = bf16_rest(e[0], e[1], pk[qt][n][0]);
          pl[qt][n][1] = bf16_rest(e[2], e[3], pk[qt][n][1]);
        }
      }
      l[qt] += psum;
    }
  };
  auto pv = [&](const unsigned char* v_lds) {
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      bf16x8_t pf[QT], pf_lo[QT];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        if constexpr (WP) {
          const u32x4_t lw = {pl[qt][2 * s2][0], pl[qt][2 * s2][1], pl[qt][2 * s2 + 1][0], pl[qt][2 * s2 + 1][1]};
          pf_lo[qt] = __builtin_bit_cast(bf16x8_t, lw);
        }
        u32x4_t pw = {pk[qt][2 * s2][0], pk[qt][2 * s2][1], pk[qt][2 * s2 + 1][0], pk[qt][2 * s2 + 1][1]};
        pf[qt] = __builtin_bit_cast(bf16x8_t, pw);
      }
      const int q4 = fr >> 2, p4 = fr & 3;
      const int r0 = s2 * 32 + g * 4 + q4, r1 = r0 + 16;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int ch = dt * 2 + (p4 >> 1);
        const s16x4_t lo = read_tr16((lds_s16x4_t*)(v_lds + tile_off<D>(r0, ch) + 8 * (p4 & 1)));
        const s16x4_t hi = read_tr16((lds_s16x4_t*)(v_lds + tile_off<D>(r1, ch) + 8 * (p4 & 1)));
        typedef __attribute__((ext_vector_type(8))) short s16x8_t;
        const s16x8_t vv = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          if constexpr (WP)
            o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vv), pf_lo[qt], o[qt][dt], 0, 0, 0);
          o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vv), pf[qt], o[qt][dt], 0, 0, 0);
        }
      }
    }
  };
  auto fence = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // Ring of AW_STAGES tiles.  Between barriers k and k + 1 the early half is in S and M of tile k, the late half in M of tile
  // k - 1 and S of tile k: tiles k - 1 to k + 1 are read, tile k + 2 is requested into the fourth stage, whose content, tile k - 2,
  // was last read before barrier k (every wave waits for its LDS reads there).  A tile has landed one barrier after its request:
  // every wave waits for its own part.  Tiles past the last one are requested too: zero fills of a stage nobody reads.
  // (With a second barrier a tile, which closed S for one half and M for the other, 4643 tokens of 32 heads took 2 to 3 % longer, eight
  // sequences of 836 6 %: a wave that had a new maximum held up all of them.  One call after another they take 201 and 99 us, were 233 and
  // 116; inside a prompt 231.)
  auto landed = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    fence();
  };
  const bool late = wid >= AW_WAVES / 2;
  stage(0, 0);
  stage(1, 1);
  landed();
  stage(2, 2);
  const int n_mine = !wave_active ? 0 : CAUSAL ? min(ntiles, (q_hi + q_off + TK) / TK) : ntiles;
  if (n_mine > 0) qk(lds);
  for (int t = 0; t < ntiles; ++t) {
    if (t < n_mine) softmax(t);
    if (late) {
      landed();
      stage((t + 3) % AW_STAGES, t + 3);
    }
    const unsigned char* v_lds = lds + (t % AW_STAGES) * 2 * TILE_BYTES + TILE_BYTES;
    const unsigned char* k_lds = lds + ((t + 1) % AW_STAGES) * 2 * TILE_BYTES;
    __builtin_amdgcn_s_setprio(1);
    if (!WP && t + 1 < n_mine) {
      // one block of code: sixteen LDS reads ahead of the products, of which a V read feeds one and a K read two
      __builtin_amdgcn_sched_barrier(0);
      pv(v_lds);
      qk(k_lds);
      __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);
#pragma unroll
      for (int i = 0; i < DT * QT - 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
#pragma unroll
      for (int i = 0; i < KS * 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 16, 0);
      __builtin_amdgcn_sched_barrier(0);
    } else {                           // (both parts of the weights leave no registers to read ahead into)
      if (t < n_mine) pv(v_lds);
      if (WP && t + 1 < n_mine) qk(k_lds);
    }
    __builtin_amdgcn_s_setprio(0);
    if (!late) {
      landed();
      stage((t + 3) % AW_STAGES, t + 3);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // zero fills land before the LDS is handed on

#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    float lt = l[qt];
    lt += __shfl_xor(lt, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
    float inv = lt > 0.f ? 1.f / lt : 0.f;
    if (qi[qt] >= p.Sq) continue;
    if (p.gate) inv *= head_gate(p, static_cast<long long>(b) * p.Sq + qi[qt], h);
    if (p.lse && g == 0)
      p.lse[(static_cast<long long>(b) * p.Hq + h) * p.Sq + qi[qt]] = lt > 0.f ? m[qt] * p.scale_log2e + log2f(lt) : INFINITY;
    bf16_t* op = p.o + b * p.o_sb + static_cast<long long>(qi[qt]) * p.o_ss + h * p.o_sh;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      u32x2_t w = {pack_bf16x2(o[qt][dt][0] * inv, o[qt][dt][1] * inv),
                   pack_bf16x2(o[qt][dt][2] * inv, o[qt][dt][3] * inv)};
      *reinterpret_cast<u32x2_t*>(op + dt * 16 + g * 4) = w;
    }
  }
}

// Merge the key splits of one query row: thread d owns output column d.
template <int D>
__global__ __launch_bounds__(D) void attn_split_combine_kernel(AttnParams p) {
  const int qi = blockIdx.x, h = blockIdx.y, b = blockIdx.z, d = threadIdx.x;
  const long long base = (static_cast<long long>(b) * p.Hq + h) * p.nsplit;
  // Every load is issued before the first use and none sits behind a branch: the
  // kernel is a handful of L2 round trips and they must overlap.  Splits past
  // nsplit re-read split 0 and are masked afterwards.
  constexpr int MAXS = 16;
  float ms[MAXS], ls[MAXS], os[MAXS];
#pragma unroll
  for (int s = 0; s < MAXS; ++s) {
    const long long slot = (base + (s < p.nsplit ? s : 0)) * p.Sq + qi;
    ms[s] = p.part_ml[slot * 2];
    ls[s] = p.part_ml[slot * 2 + 1];
    os[s] = p.part_o[slot * D + d];
  }
  float mx = -INFINITY;
#pragma unroll
  for (int s = 0; s < MAXS; ++s) {
    ms[s] = s < p.nsplit ? ms[s] : -INFINITY;
    mx = fmaxf(mx, ms[s]);
  }
  float acc = 0.f, l = 0.f;
#pragma unroll
  for (int s = 0; s < MAXS; ++s) {
    const float w = (ms[s] == -INFINITY) ? 0.f : exp2f(ms[s] - mx);
    l += w * ls[s];
    acc += w * os[s];
  }
  bf16_t* op = p.o + b * p.o_sb + static_cast<long long>(qi) * p.o_ss + h * p.o_sh;
  op[d] = f32_to_bf16(l > 0.f ? acc / l : 0.f);
}

void launch_attn_items(const bf16_t* q, const bf16_t* k, const bf16_t* v, bf16_t* o, const int* items, int n_items, int Hq, int Hkv,
                       int D, long long kld, float scale, const bf16_t* gate, int gate_ld, hipStream_t st) {
  AttnParams p{};
  p.q = q; p.k = k; p.v = v; p.o = o;
  p.q_ss = p.o_ss = static_cast<long long>(Hq) * D;
  p.k_ss = p.v_ss = kld;
  p.q_sh = p.k_sh = p.v_sh = p.o_sh = D;
  p.Hq = Hq; p.Hkv = Hkv; p.items = items; p.gate = gate; p.gate_ld = gate_ld;
  set_scale(p, scale);
  const dim3 grid(n_items, Hq), block(256);
  if (D == 128) hipLaunchKernelGGL((attn_prefill_kernel<128, true, false, 1, true, true>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((attn_prefill_kernel<64, true, false, 1, true, true>), grid, block, 0, st, p);
}

static int g_attn_groups = 0;  // key-tile groups per 64-row block: 0 = by shape, 1 / 2 = forced (tests, tuning)
void attn_force_groups(int g) { g_attn_groups = g; }
static int g_attn_wide = 1;   // the ring-staged blocks: 0 never, 1 by shape, 2 whenever the strides allow; 3: 128-row blocks of one tile a wave (tests, tuning)
void attn_enable_wide(int mode) { g_attn_wide = mode; }

void launch_attn_prefill(const bf16_t* q, const bf16_t* k, const bf16_t* v, bf16_t* o,
                         const long long* strides /*12: q,k,v,o x (b,s,h)*/, const int* kv_len,
                         int B, int Sq, int Sk, int Hq, int Hkv, int D, int causal, int q_offset,
                         int q_offset_from_len, float scale, hipStream_t st, float* part_o,
                         float* part_ml, int nsplit, float* lse, bool wide_p, const bf16_t* gate, int gate_ld) {
  AttnParams p;
  p.gate = gate; p.gate_ld = gate_ld;
  p.part_o = part_o; p.part_ml = part_ml; p.nsplit = nsplit; p.lse = lse;
  p.q = q; p.k = k; p.v = v; p.o = o;
  p.q_sb = strides[0]; p.q_ss = strides[1]; p.q_sh = strides[2];
  p.k_sb = strides[3]; p.k_ss = strides[4]; p.k_sh = strides[5];
  p.v_sb = strides[6]; p.v_ss = strides[7]; p.v_sh = strides[8];
  p.o_sb = strides[9]; p.o_ss = strides[10]; p.o_sh = strides[11];
  p.kv_len = kv_len; p.Sq = Sq; p.Sk = Sk; p.Hq = Hq; p.Hkv = Hkv;
  p.q_offset = q_offset; p.q_offset_from_len = q_offset_from_len;
  set_scale(p, scale);
  if (nsplit > 0) {
    // few query rows (Sq <= 64), causal, long cache: split the keys over blocks
    dim3 sgrid(nsplit, Hq, B), cgrid(Sq, Hq, B);
    if (D == 128) {
      hipLaunchKernelGGL((attn_prefill_kernel<128, true, true>), sgrid, dim3(256), 0, st, p);
      hipLaunchKernelGGL((attn_split_combine_kernel<128>), cgrid, dim3(128), 0, st, p);
    } else {
      hipLaunchKernelGGL((attn_prefill_kernel<64, true, true>), sgrid, dim3(256), 0, st, p);
      hipLaunchKernelGGL((attn_split_combine_kernel<64>), cgrid, dim3(64), 0, st, p);
    }
    return;
  }
  dim3 block(256);
  // Three block shapes: 64 rows (four waves), 128 rows (eight), and the ring-staged 256 rows of two tiles a wave, whose K / V must allow
  // 16-byte row chunks.  us of 64 / 128 / 256 rows, causal heads of 128 unless noted; with D = 128 there are 512, 512 and 256 blocks at a time:
  //  * 256 rows where they are one round, nearly full: 2 x 836, 32 heads 40 / 32 / 32; 1850 64 / 61 / 59; 4096, 16 heads 152 / 129 / 118;
  //    4 x 836, 16 heads of 64, no mask 31 / 27 / 25; and their rows are, without a mask more than half of them (8 x 100, 32 heads of 128 8.5 / 7.5 / 9.5,
  //    8 x 128 of 64 5.8 / 6.2 / 7.0; 8 x 200 27.5 / 20.1 / 19.4 and 16.2 / 11.7 / 11.7; 8 x 280, 16 heads 23.5 / 20.5 / 19.5; 5 x 577, 16 heads of 64 23 / 20 / 20), with
  //    one seven tenths and more than a block of them (8 x 20, 32 heads 4.2 / 4.8 / 6.1; 8 x 100 7.7 / 7.5 / 9.8; 8 x 200 23 / 16 / 19, of 64 12.6 / 9.7 / 11.2;
  //    8 x 256 25 / 19 / 21; 4 x 260 17.5 / 15.3 / 17.1; 4 x 384 25 / 20 / 18.5; 5 x 520, 16 heads 25 / 22 / 24; 5 x 600 30 / 25 / 25)
  //  * 64 rows up to 640 blocks of them: 636, 32 heads 18 / 20 / 23; 1200 35 / 39 / 40; 2048, 16 heads 43 / 64 / 65; 4096, 8 heads 82 / 95 /
  //    118.  Heads of 64 without a mask to 1056: 4 x 577, 16 heads 18 / 20 / 20; 4 x 1200 45 / 46 / 61
  //  * beyond, 128 rows where they are one round (1400, 32 heads 45 / 43 / 44; 3 x 577 33 / 26 / 32; 1500, 2 x 16 heads 53 / 44 / 51) or
  //    256 pad a tenth more rows (8 x 577 78 / 58 / 66; 8 x 836 116 / 93 / 99; 16 heads, 8 x 1200, which they don't, 96 / 88 / 88; 32
  //    184 / 164 / 155), and for heads of 64 without a mask (40 x 577, 16 heads 123 / 107 / 135; 8 x 1600 133 / 129 / 151)
  //  * 256 rows for the rest: 3000, 32 heads 129 / 139 / 93; 4643 265 / 256 / 203
  const bool strides_ok = strides[4] % 8 == 0 && strides[7] % 8 == 0 && strides[4] * 2ll * Sk < (1ll << 31) &&
                          strides[7] * 2ll * Sk < (1ll << 31);
  const long long heads = static_cast<long long>(Hq) * B, n64 = (Sq + 63) / 64 * heads, n128 = (Sq + 127) / 128 * heads,
                  n256 = (Sq + 255) / 256 * heads;
  const bool vit = D == 64 && !causal;
  const long long padded = (Sq + 255) / 256 * 256;
  const bool filled = causal ? Sq > 256 && Sq * 10ll >= padded * 7 : Sq * 2ll > padded;
  int rows = 64;
  if (g_attn_wide == 2 || (g_attn_wide == 1 && n256 > 224 && n256 <= 256 && filled)) rows = 256;
  else if (g_attn_wide == 3) rows = 128;
  else if (n64 > (vit ? 1056 : 640))
    rows = vit || (n128 <= 512 && Sq <= 1792) || n256 * 20 >= n128 * 11 || g_attn_wide == 0 ? 128 : 256;
  if (rows == 256 && !strides_ok) rows = 128;
  if (rows == 256) {
    auto go = [&](auto d, auto masked, auto parts) {
      constexpr auto kern = &attn_prefill_wide_kernel<decltype(d)::value, decltype(masked)::value, decltype(parts)::value>;
      constexpr int smem = AW_STAGES * 2 * TK * decltype(d)::value * 2;
      static const bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem) == hipSuccess;
      (void)attr;
      hipLaunchKernelGGL(kern, dim3(Hq, (Sq + 255) / 256, B), dim3(AW_WAVES * 64), smem, st, p);
    };
    using T = std::true_type;
    using F = std::false_type;
    if (D == 128) {
      const std::integral_constant<int, 128> d;
      if (wide_p && causal) go(d, T{}, T{});
      else if (causal) go(d, T{}, F{});
      else go(d, F{}, F{});
    } else {
      const std::integral_constant<int, 64> d;
      if (wide_p && causal) go(d, T{}, T{});
      else if (causal) go(d, T{}, F{});
      else go(d, F{}, F{});
    }
    return;
  }
  if (rows == 128) {
    const dim3 grid128((Sq + 127) / 128, Hq, B), block8(512);
    if (wide_p && causal) {
      if (D == 128) hipLaunchKernelGGL((attn_prefill_kernel<128, true, false, 1, true, false, 8>), grid128, block8, 0, st, p);
      else hipLaunchKernelGGL((attn_prefill_kernel<64, true, false, 1, true, false, 8>), grid128, block8, 0, st, p);
    } else if (D == 128) {
      if (causal) hipLaunchKernelGGL((attn_prefill_kernel<128, true, false, 1, false, false, 8>), grid128, block8, 0, st, p);
      else hipLaunchKernelGGL((attn_prefill_kernel<128, false, false, 1, false, false, 8>), grid128, block8, 0, st, p);
    } else {
      if (causal) hipLaunchKernelGGL((attn_prefill_kernel<64, true, false, 1, false, false, 8>), grid128, block8, 0, st, p);
      else hipLaunchKernelGGL((attn_prefill_kernel<64, false, false, 1, false, false, 8>), grid128, block8, 0, st, p);
    }
    return;
  }
  dim3 grid((Sq + 63) / 64, Hq, B);
  if (wide_p && causal) {
    if (D == 128) hipLaunchKernelGGL((attn_prefill_kernel<128, true, false, 1, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((attn_prefill_kernel<64, true, false, 1, true>), grid, block, 0, st, p);
    return;
  }
  // Two key-tile groups per block for the ViT's shape class -- head_dim 64, non-causal, so few blocks that much of the chip idles
  // (577 tokens x 16 heads: 160).  us, one group / two: 160 blocks 9.3 / 8.3, 224 7.6 / 7.5, 256 14.0 / 12.6, 320 13.8 / 13.5, 384 9.6 / 10.5, 480
  // 13.8 / 15.1.  Causal head_dim-128 blocks do not gain (636 tokens x 32 heads: 23.9 -> 25.1, 836: 30.4 -> 33.7 when tiles went through
  // registers): the diagonal splits unevenly (benchmarks/bench_attn_groups.py).
  const bool two = g_attn_groups == 2 || (g_attn_groups == 0 && vit && n64 <= 320 && Sk >= 4 * TK);
  if (two) {
    dim3 block2(512);
    if (D == 128) {
      if (causal) hipLaunchKernelGGL((attn_prefill_kernel<128, true, false, 2>), grid, block2, 0, st, p);
      else hipLaunchKernelGGL((attn_prefill_kernel<128, false, false, 2>), grid, block2, 0, st, p);
    } else {
      if (causal) hipLaunchKernelGGL((attn_prefill_kernel<64, true, false, 2>), grid, block2, 0, st, p);
      else hipLaunchKernelGGL((attn_prefill_kernel<64, false, false, 2>), grid, block2, 0, st, p);
    }
    return;
  }
  if (D == 128) {
    if (causal) hipLaunchKernelGGL((attn_prefill_kernel<128, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((attn_prefill_kernel<128, false>), grid, block, 0, st, p);
  } else {
    if (causal) hipLaunchKernelGGL((attn_prefill_kernel<64, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((attn_prefill_kernel<64, false>), grid, block, 0, st, p);
  }
}

}  // namespace evgpt
