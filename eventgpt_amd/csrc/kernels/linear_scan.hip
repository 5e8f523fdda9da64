// Linear recurrences with one scalar decay per head and token (Mamba-2's state-space duality, the matrix
// memory of xLSTM):
//     S_t = exp(a_t) S_(t-1) + b_t v_t k_t^T,      y_t = S_t q_t          (S is [V][N], value-major)
//
// Prefill runs in chunks of 128 tokens (64 with fp32 storage), three launches, all chunks of all sequences at once where the
// recurrence allows it.  With F_t = sum of a over the chunk up to t:
//   1. scan_chunk_state: what a chunk adds to the state,  dS = sum_s exp(F_L - F_s) b_s v_s k_s^T;
//   2. scan_chunk_pass: the walk over a sequence's chunks, elementwise:  S <- exp(F_L) S + dS; every
//      chunk's slot of dS ends up holding the state at the chunk's START;
//   3. scan_chunk_out: y_t = exp(F_t) S_start q_t + sum_{s <= t} exp(F_t - F_s) b_s (q_t . k_s) v_s.
// The products run on MFMA.  Whatever belongs to the recurrence -- states, decays, weighted scores --
// stays fp32: decay sums and maxima are kept in double (differences of long sums are taken), and fp32 MFMA
// operands go in as two bf16 parts (`WideFrag`).
//
// With a running maximum (log_in given; b = exp(log_in)) the stored state is S exp(-m), with
// m_t = max(a_t + m_(t-1), log_in_t), and a normaliser n_t (the same recurrence on k alone) divides the
// output: y_t = S_t q_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6).  m is a max-plus scan, so it chunks too:
// m_t = F_t + max(m_start, max_{s <= t}(log_in_s - F_s)).
//
// n and m are stored twice, indexed by the parity of the position they are read at, so that a decode step
// (decode_step.hip) can write the next ones while other blocks still read the old ones.
#include <algorithm>

#include "elem.h"
#include "../layered_kernels.h"

namespace evgpt {

// inclusive sum over the wave, in double
__device__ __forceinline__ double wave_scan_add(double v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const double o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}
__device__ __forceinline__ double wave_scan_max(double v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const double o = __shfl_up(v, d, 64);
    if (lane >= d) v = fmax(v, o);
  }
  return v;
}

// Rows [row0, row0 + len) x 64 columns from col (nc of them exist) of a T matrix, zeros past them, as MFMA operands whose contraction
// runs down the rows.  bf16: rows as they are, 16 bytes a store, read with the transposing read (chunks swizzled so that the eight rows of a
// half-wave's read lie on different banks); one element a store into a transposed tile took a third of the kernels' instructions.
template <typename T, int SL> struct Columns;
template <int SL> struct Columns<bf16_t, SL> {
  static constexpr int LOADS = SL * 8 / 256;
  unsigned char bytes[SL * 128];
  struct Regs { u32x4_t v[LOADS]; };
  static __device__ __forceinline__ int at(int row, int chunk) {
    return row * 128 + ((chunk ^ ((((row >> 1) & 1) | (((row >> 3) & 1) << 1)) << 1)) << 4);
  }
  static __device__ __forceinline__ Regs request(const bf16_t* __restrict__ p, long long ld, long long row0, int len, int col, int nc) {
    Regs r;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int idx = threadIdx.x + i * 256, row = idx >> 3, c = (idx & 7) * 8;
      r.v[i] = row < len && c < nc ? load16(p + (row0 + row) * ld + col + c) : u32x4_t{0, 0, 0, 0};
    }
    return r;
  }
  __device__ __forceinline__ void put(const Regs& r) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int idx = threadIdx.x + i * 256;
      *reinterpret_cast<u32x4_t*>(bytes + at(idx >> 3, idx & 7)) = r.v[i];
    }
  }
  // columns c0 + (lane & 15), rows 32 kb + 8 (lane >> 4) .. + 7
  __device__ __forceinline__ Frag<bf16_t> frag(int c0, int kb) const {
    typedef __attribute__((ext_vector_type(8))) short s16x8_t;
    const int lane = threadIdx.x & 63, fr = lane & 15, g = lane >> 4, row = kb * 32 + g * 8 + (fr >> 2), chunk = (c0 >> 3) + ((fr & 3) >> 1);
    const s16x4_t a = read_tr16((lds_s16x4_t*)(bytes + at(row, chunk) + 8 * (fr & 1)));
    const s16x4_t b = read_tr16((lds_s16x4_t*)(bytes + at(row + 4, chunk) + 8 * (fr & 1)));
    const s16x8_t v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return {__builtin_bit_cast(bf16x8_t, v)};
  }
  __device__ __forceinline__ f32x4_t four(int row, int c) const {            // c % 4 == 0
    return load4(reinterpret_cast<const bf16_t*>(bytes + at(row, c >> 3) + (c & 4) * 2));
  }
  __device__ __forceinline__ float one(int row, int c) const {
    return bf16_to_f32(*reinterpret_cast<const bf16_t*>(bytes + at(row, c >> 3) + (c & 7) * 2));
  }
};
template <int SL> struct Columns<float, SL> {
  static constexpr int LOADS = SL / 32, TS = SL + 8;
  float t[64 * TS];                       // [column][row]
  struct Regs { f32x4_t v[LOADS][2]; };
  static __device__ __forceinline__ Regs request(const float* __restrict__ p, long long ld, long long row0, int len, int col, int nc) {
    Regs r;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int idx = threadIdx.x + i * 256, s = idx % SL, c8 = (idx / SL) * 8;
      const bool in = s < len && c8 < nc;
      const float* g = p + (row0 + s) * ld + col + c8;
      r.v[i][0] = in ? load4(g) : f32x4_t{0.f, 0.f, 0.f, 0.f};
      r.v[i][1] = in ? load4(g + 4) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    return r;
  }
  __device__ __forceinline__ void put(const Regs& r) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int idx = threadIdx.x + i * 256, s = idx % SL, c8 = (idx / SL) * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) t[(c8 + j) * TS + s] = r.v[i][j >> 2][j & 3];
    }
  }
  __device__ __forceinline__ Frag<float> frag(int c0, int kb) const {
    const int lane = threadIdx.x & 63;
    return load_frag(t + (c0 + (lane & 15)) * TS + kb * 32 + (lane >> 4) * 8);
  }
  __device__ __forceinline__ f32x4_t four(int row, int c) const {
    return f32x4_t{t[c * TS + row], t[(c + 1) * TS + row], t[(c + 2) * TS + row], t[(c + 3) * TS + row]};
  }
  __device__ __forceinline__ float one(int row, int c) const { return t[c * TS + row]; }
};
__device__ __forceinline__ void unpack(const Frag<bf16_t>& f, float (&x)[8]) {
  const u32x4_t w = __builtin_bit_cast(u32x4_t, f.v);
#pragma unroll
  for (int i = 0; i < 4; ++i) { x[2 * i] = bf16lo(w[i]); x[2 * i + 1] = bf16hi(w[i]); }
}
__device__ __forceinline__ void unpack(const Frag<float>& f, float (&x)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = f.v[i];
}

// exp of an exponent put together in double: v_exp_f32 on its float in units of log2 (0 below 2^-126)
__device__ __forceinline__ float exp_of(double v) { return __builtin_amdgcn_exp2f(static_cast<float>(v * 1.4426950408889634074)); }

// One wave: decay sums F of a chunk's tokens (lane l: tokens l NH .. l NH + NH - 1), and with STAB the running maxima
// of log_in - F.
template <int NH, bool STAB>
__device__ __forceinline__ void chunk_gates(const ScanArgs& a, int row0, int len, int h, double (&F)[NH], float (&li)[NH],
                                            double (&top)[NH]) {
  const int lane = threadIdx.x & 63;
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    const int t = lane * NH + i;
    const long long gi = static_cast<long long>(row0 + t) * a.H + h;
    sum += t < len ? static_cast<double>(a.log_decay[gi]) : 0.0;
    F[i] = sum;
    if constexpr (STAB) li[i] = t < len ? a.log_in[gi] : -INFINITY;
    else li[i] = t < len ? a.scale_in[gi] : 0.f;
  }
  const double upto = __shfl_up(wave_scan_add(sum), 1, 64), before = lane > 0 ? upto : 0.0;     // (less `sum`, a long one would take it away)
#pragma unroll
  for (int i = 0; i < NH; ++i) F[i] += before;
  if constexpr (STAB) {
    double m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NH; ++i) {
      m = fmax(m, static_cast<double>(li[i]) - F[i]);
      top[i] = m;
    }
    const double up = __shfl_up(wave_scan_max(m), 1, 64);
    if (lane > 0)
#pragma unroll
      for (int i = 0; i < NH; ++i) top[i] = fmax(top[i], up);
  }
}

// A block's 64 value rows of a head and chunk.  The blocks of one head and chunk read the same queries and keys: one XCD takes them.  Heads of
// one block go by the grid: neighbours' value rows then meet in memory while the eight XCDs read them (head 64 wide: 103 us, by XCD 113).
struct ScanTile {
  int v0, h, chunk;
  __device__ __forceinline__ explicit ScanTile(int heads) : v0(0), h(blockIdx.y), chunk(blockIdx.z) {
    const int nx = gridDim.x;
    if (nx == 1) return;
    const int id = xcd_remap(blockIdx.x + nx * (blockIdx.y + heads * blockIdx.z), nx * heads * gridDim.z);
    v0 = id % nx * 64;
    h = id / nx % heads;
    chunk = id / nx / heads;
  }
};

// Block: 64 value rows of one head and chunk, all of N in runs of 64.
template <typename T, bool STAB, int SL>
__global__ __launch_bounds__(256) void scan_chunk_state_kernel(ScanArgs a, ScanChunks c) {
  constexpr int NH = SL / 64;
  using Tile = Columns<T, SL>;
  __shared__ __attribute__((aligned(16))) Tile kt, vt;
  __shared__ __attribute__((aligned(16))) float wgt[SL];
  __shared__ float dn_s[4][64];
  const ScanTile tile(a.H);
  const int v0 = tile.v0, h = tile.h, ci = tile.chunk;
  const int row0 = c.chunks[ci * 4], len = min(c.chunks[ci * 4 + 1], SL);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, fr = lane & 15, g = lane >> 4;
  const int nv = min(64, a.V - v0), k_col = (h / a.per_group) * a.N;
  const auto vr = Tile::request(static_cast<const T*>(a.v), a.ldv, row0, len, h * a.V + v0, nv);
  auto kr = Tile::request(static_cast<const T*>(a.k), a.ldk, row0, len, k_col, min(64, a.N));
  if (wid == 0) {
    double F[NH], m[NH];
    float li[NH];
    chunk_gates<NH, STAB>(a, row0, len, h, F, li, m);
    const double FL = __shfl(F[NH - 1], 63, 64);
    double top = 0.0;
    if constexpr (STAB) top = FL + __shfl(m[NH - 1], 63, 64);     // the largest FL - F + log_in
#pragma unroll
    for (int i = 0; i < NH; ++i) {
      const float e = static_cast<float>(FL - F[i] + (STAB ? static_cast<double>(li[i]) - top : 0.0));
      wgt[lane * NH + i] = lane * NH + i < len ? expf(e) * (STAB ? 1.f : li[i]) : 0.f;
    }
    if (v0 == 0 && lane == 0) {
      const long long o = static_cast<long long>(ci) * a.H + h;
      c.am[o] = top;
      c.fl[o] = FL;
    }
  }
  vt.put(vr);
  kt.put(kr);
  __syncthreads();
  WideFrag<T> vf[SL / 32];          // a wave owns 16 value rows, weighted
#pragma unroll
  for (int ks = 0; ks < SL / 32; ++ks) {
    float x[8], w[8];
    unpack(vt.frag(wid * 16, ks), x);
    load8(wgt + ks * 32 + g * 8, w);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] *= w[j];
    vf[ks] = wide_frag<T>(x);
  }
  float* dS = c.dS + ((static_cast<long long>(ci) * a.H + h) * a.V + v0) * a.N;
  for (int n0 = 0; n0 < a.N; n0 += 64) {
    const int nn = min(64, a.N - n0);
    if (n0 + 64 < a.N) kr = Tile::request(static_cast<const T*>(a.k), a.ldk, row0, len, k_col + n0 + 64, min(64, a.N - n0 - 64));
    f32x4_t acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < SL / 32; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = mma(kt.frag(i * 16, ks), vf[ks], acc[i]);
    // D[n][v]: a lane holds four consecutive n of value row fr
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int v = wid * 16 + fr, n = i * 16 + g * 4;
      if (v < nv && n < nn) *reinterpret_cast<f32x4_t*>(dS + static_cast<long long>(v) * a.N + n0 + n) = acc[i];
    }
    if constexpr (STAB) {
      if (v0 == 0) {                  // (block-uniform) a wave per quarter of the tokens
        float s = 0.f;
#pragma unroll 8
        for (int t = 0; t < SL / 4; ++t) s += wgt[wid * (SL / 4) + t] * kt.one(wid * (SL / 4) + t, lane);
        dn_s[wid][lane] = s;
        __syncthreads();
        if (tid < nn)
          c.dn[(static_cast<long long>(ci) * a.H + h) * a.N + n0 + tid] = dn_s[0][tid] + dn_s[1][tid] + dn_s[2][tid] + dn_s[3][tid];
      }
    }
    if (n0 + 64 < a.N) {
      __syncthreads();
      kt.put(kr);
      __syncthreads();
    }
  }
}

// One thread per four state elements (the block after the last: the normaliser), over a sequence's chunks.
template <bool STAB>
__global__ __launch_bounds__(256) void scan_chunk_pass_kernel(ScanArgs a, ScanChunks c) {
  const int* sq = c.seqs + blockIdx.z * 4;
  const int c0 = sq[0], nc = sq[1];
  const long long slot = sq[2];
  const bool fresh = (sq[3] & 1) != 0;
  const long long nm_in = (static_cast<long long>(sq[3] >> 1 & 1) * a.slots + slot) * a.H;    // [2][slots][H]
  const long long nm_out = (static_cast<long long>(sq[3] >> 2 & 1) * a.slots + slot) * a.H;
  const int h = blockIdx.y;
  const long long per = static_cast<long long>(a.V) * a.N;
  const bool norm = STAB && blockIdx.x == gridDim.x - 1;
  const long long size = norm ? a.N : per;
  const long long e0 = norm ? threadIdx.x * 4ll : (static_cast<long long>(blockIdx.x) * 256 + threadIdx.x) * 4;
  const float m_in = STAB && !fresh ? a.m[nm_in + h] : 0.f;
  const float* from = norm ? a.n + (nm_in + h) * a.N : a.S + (slot * a.H + h) * per;
  float* to = norm ? a.n + (nm_out + h) * a.N : a.S + (slot * a.H + h) * per;
  float* dbase = norm ? c.dn : c.dS;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  for (long long e = e0; e < size; e += norm ? 1024 : size) {
    f32x4_t s = fresh ? f32x4_t{0.f, 0.f, 0.f, 0.f} : load4(from + e);
    float m = m_in;
    constexpr int PF = 4;            // chunk slots in flight
    f32x4_t nxt[PF];
#pragma unroll
    for (int k = 0; k < PF; ++k)
      if (k < nc) nxt[k] = load4(dbase + (static_cast<long long>(c0 + k) * a.H + h) * size + e);
    for (int k0 = 0; k0 < nc; k0 += PF) {
#pragma unroll
      for (int k = 0; k < PF; ++k) {
        if (k0 + k >= nc) break;
        const long long o = static_cast<long long>(c0 + k0 + k) * a.H + h;
        const f32x4_t d = nxt[k];
        if (k0 + k + PF < nc) nxt[k] = load4(dbase + (o + static_cast<long long>(PF) * a.H) * size + e);
        *reinterpret_cast<f32x4_t*>(dbase + o * size + e) = s;
        const double fl = c.fl[o];
        if constexpr (STAB) {
          const double am = c.am[o];
          if (lead) c.m0[o] = m;
          const float m1 = static_cast<float>(fmax(fl + m, am));
          const float x = expf(static_cast<float>(fl + m - m1)), y = expf(static_cast<float>(am - m1));
          s = s * x + d * y;
          m = m1;
        } else {
          s = s * expf(static_cast<float>(fl)) + d;
        }
      }
    }
    *reinterpret_cast<f32x4_t*>(to + e) = s;
  }
}

// Weighted scores of 64 tokens as operands: [token][key].  bf16: both parts of `WideFrag`, made once where the four waves would each make them.
template <typename T, int SL> struct Weights;
template <int SL> struct Weights<bf16_t, SL> {
  static constexpr int BYTES = 2 * 64 * SL * 2, CH = SL / 8;
  static __device__ __forceinline__ int at(int t, int s) { return t * (SL * 2) + (((s >> 3) ^ (t & (CH - 1))) << 4) + (s & 7) * 2; }
  static __device__ __forceinline__ void put(unsigned char* p, int t, int s, const f32x4_t& w) {          // s % 4 == 0
    const u32x2_t hi = {pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3])};
    const u32x2_t lo = {pack_bf16x2(w[0] - bf16lo(hi[0]), w[1] - bf16hi(hi[0])), pack_bf16x2(w[2] - bf16lo(hi[1]), w[3] - bf16hi(hi[1]))};
    *reinterpret_cast<u32x2_t*>(p + at(t, s)) = hi;
    *reinterpret_cast<u32x2_t*>(p + 64 * SL * 2 + at(t, s)) = lo;
  }
  static __device__ __forceinline__ WideFrag<bf16_t> frag(const unsigned char* p, int t, int s) {         // s % 8 == 0
    return {__builtin_bit_cast(bf16x8_t, load16(p + at(t, s))), __builtin_bit_cast(bf16x8_t, load16(p + 64 * SL * 2 + at(t, s)))};
  }
};
template <int SL> struct Weights<float, SL> {
  static constexpr int PS = SL + 4, BYTES = 64 * PS * 4;
  static __device__ __forceinline__ void put(unsigned char* p, int t, int s, const f32x4_t& w) {
    *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p) + t * PS + s) = w;
  }
  static __device__ __forceinline__ WideFrag<float> frag(const unsigned char* p, int t, int s) {
    float x[8];
    load8(reinterpret_cast<const float*>(p) + t * PS + s, x);
    return wide_frag<float>(x);
  }
};

// Block: 64 value columns of one head and chunk.  Scores are computed transposed, a wave per sixteen keys of every
// 64, and meet in LDS (in the query tile's place); then a wave owns sixteen value rows for all tokens, so that the
// chunk's start state -- most of the bytes this kernel reads -- is read once.  Everything a step of 32 state columns reads
// is requested a step ahead, the first of them with the values; what is left is latency, so three blocks to a CU (168 registers a lane,
// under 54 KB of LDS).  To stay within those registers rows are offsets from a uniform base, 32 bits wide but for strides that need `Off`
// to be 64, and the values' operands are read behind the scores: with a pointer a lane and those operands early 13 registers of the
// instance with a maximum lay in scratch memory.  A weight's exponent is put together in double, as the sums it is the difference of are,
// and goes to v_exp_f32 in units of log2; expf of it, with the library's range checks, took most of the vector instructions.  (Sums kept as
// pairs of floats are as fast and lose bits from 2^30 on.)  4096 tokens, 134 MB of states: 8 heads of 512 x 256 with a maximum 87 us (105 out
// of scratch memory), 128 heads of 64 x 128 89, were both 174 with neither (state 48 and 53, were 74); the three launches 147 and 184, 100
// tokens of 4 heads 30.9 (163.6, 185.2 and 32.8 out of scratch memory).
template <typename T, bool STAB, int SL, typename Off>
__global__ __launch_bounds__(256, 3) void scan_chunk_out_kernel(ScanArgs a, ScanChunks c) {
  constexpr int NH = SL / 64, QS = 64 + 8, QV = sizeof(T) == 4 ? 2 : 1;
  using Tile = Columns<T, SL>;
  using Wgt = Weights<T, SL>;
  constexpr int Q_BYTES = SL * QS * sizeof(T);
  __shared__ __attribute__((aligned(16))) Tile vt;                                // values of the chunk's tokens
  __shared__ __attribute__((aligned(16))) unsigned char qp_lds[Q_BYTES > Wgt::BYTES ? Q_BYTES : Wgt::BYTES];
  T* qs = reinterpret_cast<T*>(qp_lds);                               // [token][64 of N]
  __shared__ __attribute__((aligned(16))) double F_s[SL];
  __shared__ __attribute__((aligned(16))) float in_s[SL];
  __shared__ float m_s[SL], inv_s[64], den_s[4][64];
  __shared__ __attribute__((aligned(16))) float nrm_s[64];            // the start state's normaliser, of the columns at hand
  const ScanTile tile(a.H);
  const int v0 = tile.v0, h = tile.h, ci = tile.chunk;
  const int row0 = c.chunks[ci * 4], len = min(c.chunks[ci * 4 + 1], SL);
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), fr = lane & 15, g = lane >> 4;
  const int nv = min(64, a.V - v0), hk = h / a.per_group;
  const long long ho = static_cast<long long>(ci) * a.H + h;
  const T* qp = static_cast<const T*>(a.q) + row0 * a.ldq + static_cast<long long>(hk) * a.N;
  const T* kp = static_cast<const T*>(a.k) + row0 * a.ldk + static_cast<long long>(hk) * a.N;
  const Off ldq = static_cast<Off>(a.ldq), ldk = static_cast<Off>(a.ldk);
  const float* S0 = c.dS + (ho * a.V + v0 + wid * 16) * a.N;
  const unsigned S_lane = fr * a.N + g * 8;
  const float* nrm = STAB ? c.dn + ho * a.N : nullptr;
  const bool rows_v = wid * 16 < nv;              // this wave has value rows
  const auto vr = Tile::request(static_cast<const T*>(a.v), a.ldv, row0, len, h * a.V + v0, nv);
  u32x4_t qr[2 * NH][QV];
  float nr = 0.f;
  auto request_q = [&](int n0) {
    if constexpr (STAB) nr = nrm[min(n0 + lane, a.N - 1)];
#pragma unroll
    for (int i = 0; i < 2 * NH; ++i) {
      const int idx = tid + i * 256, t = idx >> 3, c8 = (idx & 7) * 8;
      if (n0 + c8 < a.N) {
        const T* p = qp + (min(t, len - 1) * ldq + (n0 + c8));
#pragma unroll
        for (int v = 0; v < QV; ++v) qr[i][v] = load16(p + v * 4);
      }
    }
  };
  Frag<T> kn[NH];
  float xn[8];
  auto request_step = [&](int n) {
#pragma unroll
    for (int k = 0; k < NH; ++k) kn[k] = load_frag(kp + (min(k * 64 + wid * 16 + fr, len - 1) * ldk + (n + g * 8)));
    if (rows_v) load8(S0 + (S_lane + n), xn);
    else
#pragma unroll
      for (int j = 0; j < 8; ++j) xn[j] = 0.f;
  };
  request_q(0);
  request_step(0);
  const float m0 = STAB ? c.m0[ho] : 0.f;
  if (wid == 0) {
    double F[NH], top[NH];
    float li[NH];
    chunk_gates<NH, STAB>(a, row0, len, h, F, li, top);
#pragma unroll
    for (int i = 0; i < NH; ++i) {
      const int t = lane * NH + i;
      F_s[t] = F[i];
      in_s[t] = li[i];
      m_s[t] = STAB ? static_cast<float>(F[i] + fmax(static_cast<double>(m0), top[i])) : 0.f;
    }
    if constexpr (STAB) {
      const int last = c.chunks[ci * 4 + 3];
      if (v0 == 0 && lane == 0 && (last & 1))
        a.m[(static_cast<long long>(last >> 1 & 1) * a.slots + c.chunks[ci * 4 + 2]) * a.H + h] =
            static_cast<float>(fmax(c.fl[ho] + m0, c.am[ho]));
    }
  }
  vt.put(vr);
  f32x4_t st[NH][NH][4], inter[NH][4];            // [key half][token half][token tile]
  float nq[NH];
#pragma unroll
  for (int k = 0; k < NH; ++k) {
    nq[k] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      inter[k][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NH; ++j) st[k][j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }
  for (int n0 = 0; n0 < a.N; n0 += 64) {
    const int nn = min(64, a.N - n0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * NH; ++i) {
      const int idx = tid + i * 256, t = idx >> 3, c8 = (idx & 7) * 8;
      if (c8 < nn)
#pragma unroll
        for (int v = 0; v < QV; ++v) *reinterpret_cast<u32x4_t*>(qs + t * QS + c8 + v * 4) = qr[i][v];
    }
    if (STAB && wid == 0) nrm_s[lane] = nr;
    if (n0 + 64 < a.N) request_q(n0 + 64);
    __syncthreads();
    for (int n = 0; n < nn; n += 32) {
      Frag<T> kf[NH];
#pragma unroll
      for (int k = 0; k < NH; ++k) kf[k] = kn[k];
      const WideFrag<T> sf = wide_frag<T>(xn);
      if (n0 + n + 32 < a.N) request_step(n0 + n + 32);
#pragma unroll
      for (int th = 0; th < NH; ++th)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const Frag<T> qf = load_frag(qs + (th * 64 + j * 16 + fr) * QS + n + g * 8);
#pragma unroll
          for (int k = 0; k < NH; ++k)
            if (k < th || (k == th && j >= wid)) st[k][th][j] = mma(kf[k], qf, st[k][th][j]);
          inter[th][j] = mma(sf, qf, inter[th][j]);
        }
    }
    if constexpr (STAB) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int n = (tid & 3) * 16 + half * 8;
        if (n >= nn) break;
        float w[8], x[8];
        load8(nrm_s + n, w);
#pragma unroll
        for (int th = 0; th < NH; ++th) {
          load8(qs + (th * 64 + (tid >> 2)) * QS + n, x);
#pragma unroll
          for (int j = 0; j < 8; ++j) nq[th] += w[j] * x[j];
        }
      }
    }
  }
  const float skip = a.skip ? a.skip[h] : 0.f;
#pragma unroll
  for (int th = 0; th < NH; ++th) {
    if (th * 64 >= len) break;                    // block-uniform
    __syncthreads();                              // the query tile, or the scores of the half before, are no longer read
    float den[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k <= th; ++k) {
      // weighted scores of keys 64 k + 16 wid + 4 g + r and token 64 th + 16 j + fr
      const int s0 = k * 64 + wid * 16 + g * 4;
      const f32x4_t in = load4(in_s + s0);
      double Fs[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) Fs[r] = F_s[s0 + r];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = th * 64 + j * 16 + fr;
        const double Ft = F_s[t];
        const float mt = m_s[t];
        f32x4_t w = st[k][th][j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float e = STAB ? exp_of(Ft - Fs[r] + static_cast<double>(in[r] - mt)) : exp_of(Ft - Fs[r]) * in[r];
          w[r] = s0 + r <= t && t < len ? w[r] * (e * a.qscale) : 0.f;
          den[j] += w[r];
        }
        Wgt::put(qp_lds, j * 16 + fr, s0, w);
      }
    }
    if constexpr (STAB) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float d = den[j];
        d += __shfl_xor(d, 16, 64);
        d += __shfl_xor(d, 32, 64);
        if (g == 0) den_s[wid][j * 16 + fr] = d;
      }
    }
    __syncthreads();
    if constexpr (STAB) {
      const int tl = tid >> 2, t = th * 64 + tl;
      float d = nq[th];
      d += __shfl_xor(d, 1, 64);
      d += __shfl_xor(d, 2, 64);
      d = d * exp_of(F_s[t] + static_cast<double>(m0 - m_s[t])) * a.qscale + (den_s[0][tl] + den_s[1][tl] + den_s[2][tl] + den_s[3][tl]);
      if ((tid & 3) == 0) inv_s[tl] = 1.f / (fmaxf(fabsf(d), expf(-m_s[t])) + 1e-6f);
      __syncthreads();
    }
    if (!rows_v) continue;
    Frag<T> vf[SL / 32];                          // (here and not ahead of the scores, where there are no registers left)
#pragma unroll
    for (int kb = 0; kb < 2 * (th + 1); ++kb) vf[kb] = vt.frag(wid * 16, kb);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int tl = j * 16 + fr, t = th * 64 + tl;
      f32x4_t y = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < SL / 32; ++kb)
        if (kb < 2 * th || (kb < 2 * th + 2 && (kb - 2 * th) * 2 <= j)) y = mma(vf[kb], Wgt::frag(qp_lds, tl, kb * 32 + g * 8), y);
      if (t >= len) continue;
      y += inter[th][j] * (exp_of(F_s[t] + static_cast<double>(m0 - m_s[t])) * a.qscale);
      if constexpr (STAB) y *= inv_s[tl];
      const int v = wid * 16 + g * 4;
      if (a.skip) y += skip * vt.four(t, v);
      store4(static_cast<T*>(a.out) + (static_cast<long long>(row0 + t) * a.H + h) * a.V + v0 + v, y[0], y[1], y[2], y[3]);
    }
  }
}

template <typename T, bool STAB>
static void launch_scan(const ScanArgs& a, const ScanChunks& c, hipStream_t st) {
  constexpr int SL = sizeof(T) == 2 ? SCAN_CHUNK_BF16 : SCAN_CHUNK_F32;
  const dim3 g1((a.V + 63) / 64, a.H, c.C), block(256);
  const long long quads = static_cast<long long>(a.V) * a.N / 4;
  const dim3 g2(static_cast<unsigned>((quads + 255) / 256) + (STAB ? 1 : 0), a.H, c.nseq);
  hipLaunchKernelGGL((scan_chunk_state_kernel<T, STAB, SL>), g1, block, 0, st, a, c);
  hipLaunchKernelGGL(scan_chunk_pass_kernel<STAB>, g2, block, 0, st, a, c);
  if (std::max(a.ldq, a.ldk) < (1ll << 31) / SL - a.N)
    hipLaunchKernelGGL((scan_chunk_out_kernel<T, STAB, SL, unsigned>), g1, block, 0, st, a, c);
  else
    hipLaunchKernelGGL((scan_chunk_out_kernel<T, STAB, SL, long long>), g1, block, 0, st, a, c);
}
void launch_scan_prefill(const ScanArgs& a, const ScanChunks& c, bool f32, hipStream_t st) {
  const bool stab = a.log_in != nullptr;
  if (f32) {
    if (stab) launch_scan<float, true>(a, c, st);
    else launch_scan<float, false>(a, c, st);
  } else {
    if (stab) launch_scan<bf16_t, true>(a, c, st);
    else launch_scan<bf16_t, false>(a, c, st);
  }
}

}  // namespace evgpt
