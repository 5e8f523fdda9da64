// The part of a decode step between a mixer's input projection and its output projection, for one token per
// sequence, in one launch: attention heads (norm, rotation, cache append), the matrix memory and the
// state-space recurrence with its convolution.  Inputs are the projection's fp32 rows or split-K slabs;
// what a prompt would have stored in T is rounded to T here as well.
//
// A recurrent state is streamed once: sixteen lanes per state row read it, decay it, add the token, dot it with
// the query and write it back.  A block owns some rows of one head; it prepares the head's small vectors
// (query, key, convolution outputs, gates) itself in LDS rather than waiting for another launch.
#include <type_traits>

#include "src_rows.h"

namespace evgpt {

// The state rows a wave updates first (row wid * 4 + lane / 16 of the block, up to 256 columns): requested before the
// position, gates and small vectors they are combined with have arrived.  The kernels are a chain of such round trips on a
// few MB: one stream of 64 heads of 64 x 128 took 8.0 us with the rows requested behind the chain, 5.6 now
// (the convolution's operands are requested together as well); 4 heads of 512 x 256 with 20 attention heads 7.9, now 6.8.
constexpr int STATE_PRE = 4;
struct StateRows { f32x4_t v[STATE_PRE]; };
__device__ __forceinline__ StateRows request_state(const float* S, int N, int v0, int vb) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, i = wid * 4 + (lane >> 4);
  StateRows r;
  const float* Sr = S + static_cast<long long>(v0 + min(i, vb - 1)) * N;
#pragma unroll
  for (int u = 0; u < STATE_PRE; ++u) r.v[u] = load4(Sr + min((lane & 15) * 4 + u * 64, N - 4));
  return r;
}

// rows of S (of one head) from v0 on, vb of them, by the block's first four waves: S = decay S + add v k^T, y = S q.
// AHEAD: 256 columns of a row are requested while the ones before them are combined, for blocks of more than 16 rows, which have
// several such groups a wave and nothing else to hide their loads.  32 streams of 6 heads of 256 x 512 beside 16 attention heads:
// 46 us with a plain loop, 59 with only the first group requested early, 55 with the loads of a group together; a decode
// step there 685, 723, 709 and 686 us this way, of 64 streams, 8 heads of 512 x 256, eight layers, 2 853, 2 770, 2 763 and 2 724.
// Blocks of 16 rows do without its registers (80 and six blocks a CU, 64 and eight without; 16 streams of those
// 6 heads 575 us a step with it, 552 without, 564 with the plain loop).
template <bool AHEAD, typename Y>
__device__ __forceinline__ void stream_state(float* __restrict__ S, int N, int v0, int vb, bool fresh, float decay,
                                             const float* qs, const float* ks, const float* avs, const StateRows& first, Y&& put) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, l16 = lane & 15, rg = lane >> 4;
  if (wid >= 4) return;
  const auto request = [&](f32x4_t (&v)[STATE_PRE], int i, int e0) {
#pragma unroll
    for (int u = 0; u < STATE_PRE; ++u) v[u] = load4(S + static_cast<long long>(v0 + i) * N + min(e0 + l16 * 4 + u * 64, N - 4));
  };
  f32x4_t old[STATE_PRE], next[STATE_PRE];
  if constexpr (AHEAD) {
#pragma unroll
    for (int u = 0; u < STATE_PRE; ++u) old[u] = first.v[u];
  }
  for (int i = wid * 4 + rg; i < vb; i += 16) {
    float* Sr = S + static_cast<long long>(v0 + i) * N;
    const float av = avs[i];
    float y = 0.f;
    for (int e0 = 0; e0 < N; e0 += STATE_PRE * 64) {
      if constexpr (AHEAD) {
        if (e0 + STATE_PRE * 64 < N) request(next, i, e0 + STATE_PRE * 64);
        else if (i + 16 < vb) request(next, i + 16, 0);
      } else if (e0 == 0) {                        // (sixteen rows: the one a lane requested at the start)
#pragma unroll
        for (int u = 0; u < STATE_PRE; ++u) old[u] = first.v[u];
      } else {
        request(old, i, e0);
      }
#pragma unroll
      for (int u = 0; u < STATE_PRE; ++u) {
        const int e = e0 + l16 * 4 + u * 64;
        if (e >= N) continue;
        const f32x4_t kk = *reinterpret_cast<const f32x4_t*>(ks + e), qq = *reinterpret_cast<const f32x4_t*>(qs + e);
        f32x4_t s = kk * av;
        if (!fresh) s += old[u] * decay;
        *reinterpret_cast<f32x4_t*>(Sr + e) = s;
#pragma unroll
        for (int j = 0; j < 4; ++j) y += s[j] * qq[j];
      }
      if constexpr (AHEAD) {
#pragma unroll
        for (int u = 0; u < STATE_PRE; ++u) old[u] = next[u];
      }
    }
    y = group_sum<16>(y);
    if (l16 == 0) put(i, y);
  }
}

// (every operand of a thread's first element is requested before the sum of squares)
template <typename T, int M>
__device__ void head_step(const AttnPrepArgs& a, int b, int head, int p, bool live, float* red) {
  const bool is_q = head < a.Hq;
  const int h = is_q ? head : head - a.Hq;
  const int col = is_q ? a.q_col : a.k_col, width = (is_q ? a.Hq : a.Hkv) * a.D;
  const float* w = is_q ? a.qw : a.kw;
  const int half = a.rot >> 1;
  auto partner = [&](int d) { return h * a.D + (d < half ? d + half : d - half); };
  const int d0 = min(static_cast<int>(threadIdx.x), a.D - 1), c0 = h * a.D + d0, p0 = d0 < a.rot ? partner(d0) : c0;
  const float u0 = src1<M>(a.src, b, col + c0), o0 = src1<M>(a.src, b, col + p0);
  const float wu0 = w ? w[c0] : 1.f, wo0 = w ? w[p0] : 1.f;
  const float vv0 = is_q ? 0.f : src1<M>(a.src, b, a.v_col + c0);
  const int pt = min(max(p, 0), a.max_pos - 1);
  const float* cs = a.cos_tab + static_cast<long long>(pt) * half;
  const float* sn = a.sin_tab + static_cast<long long>(pt) * half;
  const int i0 = min(d0 < half ? d0 : d0 - half, half - 1);
  const float cs0 = half > 0 ? cs[i0] : 1.f, sn0 = half > 0 ? sn[i0] : 0.f;
  float r = 1.f;
  if (w) {
    float s = 0.f;
    for (int c = threadIdx.x * 8; c < width; c += 2048) {
      float t[8];
      src8<M>(a.src, b, col + c, t);
      s += sumsq8(t);
    }
    r = rsqrtf(block_sum<4>(s, red) / static_cast<float>(is_q ? a.nq : a.nk) + a.eps);
  }
  if (!is_q && !live) return;
  for (int d = threadIdx.x; d < a.D; d += 256) {
    const bool first = d < 256;
    const int c = h * a.D + d;
    float u = (first ? u0 : src1<M>(a.src, b, col + c)) * r;
    if (w) u *= first ? wu0 : w[c];
    if (d < a.rot) {
      const int i = d < half ? d : d - half, c2 = partner(d);
      float o = (first ? o0 : src1<M>(a.src, b, col + c2)) * r;
      if (w) o *= first ? wo0 : w[c2];
      const float ci = first ? cs0 : cs[i], si = first ? sn0 : sn[i];
      u = d < half ? u * ci - o * si : u * ci + o * si;
    }
    if (is_q) {
      static_cast<T*>(a.q_out)[static_cast<long long>(b) * width + c] = from_f32<T>(u);
    } else {
      const long long o = ((static_cast<long long>(b) * a.Hkv + h) * a.cap + max(p, 0) % a.cap) * a.D + d;
      static_cast<T*>(a.k_cache)[o] = from_f32<T>(u);
      static_cast<T*>(a.v_cache)[o] = from_f32<T>(first ? vv0 : src1<M>(a.src, b, a.v_col + c));
    }
  }
}

// Whatever a block combines with its state rows is requested with them, in both images where the position says which one is read: the
// kernel is the slowest of these loads, one barrier for the small vectors and one for the sum, instead of eight round trips one behind
// the other.  A chat of one stream, width 2048: 21.9 -> 21.35 ms with the state-space step below (6.3 and 5.4 us a launch before).
template <typename T, bool AHEAD, int M>
__device__ __forceinline__ void memory_step(const StepMemory& m, int b, int i0, int vb, int p, bool alive, float* lds, float* red) {
  const int per = m.V / vb, h = i0 / per, v0 = (i0 % per) * vb, tid = threadIdx.x;
  const int gi = b * m.H + h;
  float* out = m.out + static_cast<long long>(gi) * m.V + v0;
  float* S = m.S + static_cast<long long>(gi) * m.V * m.N;
  const StateRows rows = request_state(S, m.N, v0, vb);
  const int e0 = min(tid, m.N - 1);
  const long long image = static_cast<long long>(m.slots) * m.H;
  // (picked by a select below: an array indexed with the position is scratch memory)
  const float m_even = m.m[gi], m_odd = m.m[image + gi];
  const float n_even = m.n[static_cast<long long>(gi) * m.N + e0], n_odd = m.n[(image + gi) * m.N + e0];
  const float gi0 = src1<M>(m.src, b, m.i_col + h), gf0 = src1<M>(m.src, b, m.f_col + h), ib = m.ib[h], fb = m.fb[h];
  const float q0 = src1<M>(m.src, b, m.q_col + h * m.N + e0), k0 = src1<M>(m.src, b, m.k_col + h * m.N + e0);
  const float vr = src1<M>(m.src, b, m.v_col + h * m.V + v0 + min(tid, vb - 1));
  if (!alive) {                         // a parked sequence keeps its state
    for (int i = tid; i < vb; i += 256) out[i] = 0.f;
    return;
  }
  const bool fresh = p <= 0;
  float *qs = lds, *ks = lds + m.N, *avs = ks + m.N;
  const long long from = (static_cast<long long>(p & 1) * m.slots + b) * m.H + h;
  const long long to = (static_cast<long long>((p + 1) & 1) * m.slots + b) * m.H + h;
  const float li = m.cap * tanhf((gi0 + ib) / m.cap), lf = -softplus_f(-m.cap * tanhf((gf0 + fb) / m.cap));
  const float mt = fresh ? 0.f : p & 1 ? m_odd : m_even, m1 = fmaxf(lf + mt, li);
  const float decay = expf(lf + mt - m1), add = expf(li - m1);
  for (int i = tid; i < vb; i += 256) avs[i] = add * (i < 256 ? to_f32(from_f32<T>(vr)) : src_t<T, M>(m.src, b, m.v_col + h * m.V + v0 + i));
  float dot = 0.f;
  for (int e = tid; e < m.N; e += 256) {
    const bool first = e < 256;
    const float q = (first ? to_f32(from_f32<T>(q0)) : src_t<T, M>(m.src, b, m.q_col + h * m.N + e)) * m.qscale;
    const float k = first ? to_f32(from_f32<T>(k0)) : src_t<T, M>(m.src, b, m.k_col + h * m.N + e);
    qs[e] = q;
    ks[e] = k;
    const float n1 = (fresh ? 0.f : (first ? (p & 1 ? n_odd : n_even) : m.n[from * m.N + e]) * decay) + add * k;
    if (v0 == 0) m.n[to * m.N + e] = n1;
    dot += n1 * q;
  }
  dot = block_sum<4>(dot, red);         // (its barriers also publish the vectors)
  if (v0 == 0 && tid == 0) m.m[to] = m1;
  const float inv = 1.f / (fmaxf(fabsf(dot), expf(-m1)) + 1e-6f);
  stream_state<AHEAD>(S, m.N, v0, vb, fresh, decay, qs, ks, avs, rows, [&](int i, float y) { out[i] = y * inv; });
}
template <typename T, bool AHEAD, int M>
__global__ __launch_bounds__(256) void parallel_step_kernel(StepHeads sh, StepMemory m, const int* __restrict__ pos,
                                                            const int* __restrict__ live, int vb) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // [N] query, [N] key, [vb] weighted values
  __shared__ float red[16];
  const int b = blockIdx.y, p = pos[b];
  const bool alive = live == nullptr || live[b] != 0;
  const int n_heads = sh.on ? sh.a.Hq + sh.a.Hkv : 0;
  if (static_cast<int>(blockIdx.x) < n_heads) head_step<T, M>(sh.a, b, blockIdx.x, p, alive, red);
  else memory_step<T, AHEAD, M>(m, b, blockIdx.x - n_heads, vb, p, alive, lds, red);
}

// The same step with the attention over the cached keys in it, for a few sequences: a block takes a head's query (norm, rotation) and one
// of the splits of its keys, which are on their way meanwhile; the new key and value, which the cache will only hold afterwards,
// are made by the blocks of the first split and join there.  What is left of the attention is the merge of the splits.
// Partial results as attn_decode_split_kernel leaves them.
// A chat of one stream, width 2048, 100 + 64 tokens: 21.35 -> 20.9 ms (a launch of 4.1 us and its gap less in every second layer); 20.6 with
// the state's image picked by a select, 5.5 us a launch.
template <int D, int M>
__device__ __forceinline__ void attend_split(const AttnPrepArgs& a, const StepSplits& sp, int b, int h, int split, int p, bool live) {
  constexpr int LPK = D / 8, KPW = 64 / LPK, U = 4, NP = 4 * KPW;
  __shared__ __attribute__((aligned(16))) float s_o[NP][D];
  __shared__ float s_m[NP], s_l[NP], sums[8];
  __shared__ __attribute__((aligned(16))) bf16_t vec[3][D];        // query, new key, new value
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, sub = lane / LPK, dl = lane % LPK;
  const int hk = h / (a.Hq / a.Hkv), slot = max(p, 0) % a.cap;      // keys 0 .. slot - 1 are cached
  const int ngroups = (slot + KPW - 1) / KPW, gper = (ngroups + sp.nsplit - 1) / sp.nsplit;
  const int g0 = split * gper, g1 = min(g0 + gper, ngroups);
  const bf16_t* kb = static_cast<const bf16_t*>(a.k_cache) + (static_cast<long long>(b) * a.Hkv + hk) * a.cap * D + dl * 8;
  const bf16_t* vb = static_cast<const bf16_t*>(a.v_cache) + (static_cast<long long>(b) * a.Hkv + hk) * a.cap * D + dl * 8;
  u32x4_t kv[U], vv[U];
  int key[U];
  auto request = [&](int g) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      key[u] = (g + u) * KPW + sub;
      const bool ok = g + u < g1 && key[u] < slot;
      const int kk = ok ? key[u] : 0;
      kv[u] = load16(kb + static_cast<long long>(kk) * D);
      vv[u] = load16(vb + static_cast<long long>(kk) * D);
      if (!ok) key[u] = -1;
    }
  };
  request(g0 + wid * U);
  // a thread's element: of the query (first D threads), of the new key and value (next D)
  const bool is_q = tid < D;
  const int d = tid & (D - 1), half = a.rot >> 1;
  const int col = is_q ? a.q_col + h * D : a.k_col + hk * D, wrow = is_q ? h * D : hk * D;
  const float* w = is_q ? a.qw : a.kw;
  const int d2 = d < a.rot ? (d < half ? d + half : d - half) : d;
  const float u0 = src1<M>(a.src, b, col + d), o0 = src1<M>(a.src, b, col + d2);
  const float v0 = src1<M>(a.src, b, a.v_col + hk * D + d);
  const float wu = w ? w[wrow + d] : 1.f, wo = w ? w[wrow + d2] : 1.f;
  const int pt = min(max(p, 0), a.max_pos - 1), i = min(d < half ? d : d - half, half - 1);
  const float cs = half > 0 ? a.cos_tab[static_cast<long long>(pt) * half + max(i, 0)] : 1.f;
  const float sn = half > 0 ? a.sin_tab[static_cast<long long>(pt) * half + max(i, 0)] : 0.f;
  auto total = [&](const float* norm, int c0, int width) {
    float s = 0.f;
    if (norm)
      for (int c = tid * 8; c < width; c += 2048) {
        float t[8];
        src8<M>(a.src, b, c0 + c, t);
        s += sumsq8(t);
      }
    return wave_sum(s);
  };
  const float sq = total(a.qw, a.q_col, a.Hq * D), sk = total(a.kw, a.k_col, a.Hkv * D);
  if (lane == 0) { sums[wid] = sq; sums[4 + wid] = sk; }
  __syncthreads();
  const int at = is_q ? 0 : 4;
  const float r = w ? rsqrtf((sums[at] + sums[at + 1] + sums[at + 2] + sums[at + 3]) / static_cast<float>(is_q ? a.nq : a.nk) + a.eps) : 1.f;
  float u = u0 * r * wu;
  if (d < a.rot) {
    const float o = o0 * r * wo;
    u = d < half ? u * cs - o * sn : u * cs + o * sn;
  }
  if (tid < 2 * D) vec[is_q ? 0 : 1][d] = f32_to_bf16(u);
  if (tid >= D && tid < 2 * D) vec[2][d] = f32_to_bf16(v0);
  __syncthreads();
  if (split == 0 && live && h % (a.Hq / a.Hkv) == 0 && tid >= D && tid < 2 * D) {
    const long long o = ((static_cast<long long>(b) * a.Hkv + hk) * a.cap + slot) * D + d;
    static_cast<bf16_t*>(a.k_cache)[o] = vec[1][d];
    static_cast<bf16_t*>(a.v_cache)[o] = vec[2][d];
  }
  const u32x4_t qv = *reinterpret_cast<const u32x4_t*>(&vec[0][dl * 8]);
  float mx = -INFINITY, l = 0.f, o[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int g = g0 + wid * U; g < g1; g += 4 * U) {
    if (g != g0 + wid * U) request(g);
    float sc[U], mn = mx;
#pragma unroll
    for (int k = 0; k < U; ++k) {
      sc[k] = group_sum<LPK>(dot8_bf16(qv, kv[k], 0.f)) * sp.scale;
      if (key[k] >= 0) mn = fmaxf(mn, sc[k]);
    }
    const float al = mn == -INFINITY ? 1.f : __expf(mx - mn);
    l *= al;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= al;
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const float pr = key[k] >= 0 ? __expf(sc[k] - mn) : 0.f;
      l += pr;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] += pr * bf16lo(vv[k][e]);
        o[2 * e + 1] += pr * bf16hi(vv[k][e]);
      }
    }
    mx = mn;
  }
  if (split == 0 && wid == 0) {                       // the new key: the first group of lanes
    const float sc = group_sum<LPK>(dot8_bf16(qv, *reinterpret_cast<const u32x4_t*>(&vec[1][dl * 8]), 0.f)) * sp.scale;
    const u32x4_t nv = *reinterpret_cast<const u32x4_t*>(&vec[2][dl * 8]);
    if (sub == 0) {
      const float mn = fmaxf(mx, sc), al = __expf(mx - mn), pr = __expf(sc - mn);     // (mx = -inf: al = 0)
      l = l * al + pr;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[2 * e] = o[2 * e] * al + pr * bf16lo(nv[e]);
        o[2 * e + 1] = o[2 * e + 1] * al + pr * bf16hi(nv[e]);
      }
      mx = mn;
    }
  }
  const int pidx = wid * KPW + sub;
  *reinterpret_cast<f32x4_t*>(&s_o[pidx][dl * 8]) = f32x4_t{o[0], o[1], o[2], o[3]};
  *reinterpret_cast<f32x4_t*>(&s_o[pidx][dl * 8 + 4]) = f32x4_t{o[4], o[5], o[6], o[7]};
  if (dl == 0) { s_m[pidx] = mx; s_l[pidx] = l; }
  __syncthreads();
  if (tid < D) {
    float mm = s_m[0];
#pragma unroll
    for (int k = 1; k < NP; ++k) mm = fmaxf(mm, s_m[k]);
    float ll = 0.f, oo = 0.f;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const float c = s_m[k] == -INFINITY ? 0.f : __expf(s_m[k] - mm);
      ll += s_l[k] * c;
      oo += s_o[k][tid] * c;
    }
    const long long at_split = (static_cast<long long>(b) * a.Hq + h) * sp.nsplit + split;
    sp.part_o[at_split * D + tid] = oo;
    if (tid == 0) { sp.part_ml[at_split * 2] = mm; sp.part_ml[at_split * 2 + 1] = ll; }
  }
}
template <int D, bool AHEAD, int M>
__global__ __launch_bounds__(256) void attend_step_kernel(const int* __restrict__ pos, const int* __restrict__ live, int vb, StepHeads sh,
                                                          StepSplits sp, StepMemory m) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float red[16];
  const int b = blockIdx.y, p = pos[b], i = blockIdx.x, n_attend = sh.a.Hq * sp.nsplit;
  const bool alive = live == nullptr || live[b] != 0;
  if (i < n_attend) attend_split<D, M>(sh.a, sp, b, i % sh.a.Hq, i / sh.a.Hq, p, alive);
  else memory_step<bf16_t, AHEAD, M>(m, b, i - n_attend, vb, p, alive, lds, red);
}

// threads: one per convolution channel of the block where that is at most 512 (the state takes four waves).  As above, with all
// slots of the convolution's ring requested: the position picks among them.
template <typename T, bool AHEAD, int M>
__global__ __launch_bounds__(512) void ssd_step_kernel(StepSsd a, const int* __restrict__ pos, const int* __restrict__ live,
                                                       int vb) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // [N] C, [N] B, [vb] weighted x, [vb] x, [vb] silu(z)
  const int b = blockIdx.z, h = blockIdx.y, v0 = blockIdx.x * vb, p = pos[b];
  const int gi = b * a.H + h, per_group = a.H / a.G, g = h / per_group, nt = blockDim.x;
  float* out = a.out + static_cast<long long>(gi) * a.V + v0;
  float* S = a.S + static_cast<long long>(gi) * a.V * a.N;
  const StateRows rows = request_state(S, a.N, v0, vb);
  const float dt0 = src1<M>(a.src, b, a.dt_col + h), dt_bias = a.dt_bias[h], a_log = a.a_log[h], skip = a.skip[h];
  const bool parked = live && !live[b];
  float *cs = lds, *bs = lds + a.N, *avs = bs + a.N, *xs = avs + vb, *zs = xs + vb;
  const int C = a.H * a.V + 2 * a.G * a.N;
  T* ring = static_cast<T*>(a.ring) + static_cast<long long>(b) * a.taps * C;
  float dt = 0.f;
  for (int i = threadIdx.x; i < 2 * a.N + vb; i += nt) {
    const bool is_x = i >= 2 * a.N, first = i == static_cast<int>(threadIdx.x);
    const int c = is_x ? h * a.V + v0 + i - 2 * a.N
                       : a.H * a.V + (i < a.N ? g * a.N + i : (a.G + g) * a.N + i - a.N);     // B, then C
    const float* w = a.conv_w + static_cast<long long>(c) * a.taps;
    float acc = a.conv_b[c];
    const float now = src1<M>(a.src, b, a.x_col + c);
    const float z0 = is_x ? src1<M>(a.src, b, a.z_col + c) : 0.f;
    const T cur = from_f32<T>(now);
    if (a.taps == 4) {                  // (all operands on their way before the first product)
      const f32x4_t w4 = load4(w);
      T old[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) old[j] = ring[static_cast<long long>(j) * C + c];
      if (parked) break;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int at = max(p + j - 3, 0) & 3;
        const T o = at & 2 ? (at & 1 ? old[3] : old[2]) : (at & 1 ? old[1] : old[0]);
        acc = fmaf(w4[j], p + j - 3 < 0 ? 0.f : to_f32(o), acc);
      }
      acc = fmaf(w4[3], p < 0 ? 0.f : to_f32(cur), acc);
    } else {
      if (parked) break;
      for (int j = 0; j < a.taps; ++j) {
        const int d = a.taps - 1 - j;
        if (p - d < 0) continue;
        acc = fmaf(w[j], d == 0 ? to_f32(cur) : to_f32(ring[static_cast<long long>((p - d) % a.taps) * C + c]), acc);
      }
    }
    const float v = to_f32(from_f32<T>(acc * sigmoid_f(acc)));
    if (first) dt = softplus_f(dt0 + dt_bias);
    if (is_x) {
      const float z = to_f32(from_f32<T>(z0));
      xs[i - 2 * a.N] = v;
      avs[i - 2 * a.N] = dt * v;
      zs[i - 2 * a.N] = z * sigmoid_f(z);
    } else if (i < a.N) {
      bs[i] = v;
    } else {
      cs[i - a.N] = v;
    }
    // what is in the current input's slot is used by nobody in this step (requested with the others and dropped); one block per
    // channel stores it
    if (is_x || (v0 == 0 && h % per_group == 0)) ring[static_cast<long long>(max(p, 0) % a.taps) * C + c] = cur;
  }
  if (parked) {
    for (int i = threadIdx.x; i < vb; i += nt) out[i] = 0.f;
    return;
  }
  const float decay = expf(-expf(a_log) * softplus_f(dt0 + dt_bias));
  __syncthreads();
  stream_state<AHEAD>(S, a.N, v0, vb, p <= 0, decay, cs, bs, avs, rows, [&](int i, float y) { out[i] = (y + skip * xs[i]) * zs[i]; });
}

// state rows per block: sixteen keep a single stream's launch wide, more amortise the head's small vectors
static int rows_per_block(int heads, int V, int B) {
  int vb = 16;
  while (vb < 64 && V % (vb * 2) == 0 && static_cast<long long>(heads) * (V / vb) * B > 2048) vb *= 2;
  return vb;
}

void launch_parallel_step(const StepHeads& h, const StepMemory& m, const int* pos, const int* live, bool f32, int B,
                          hipStream_t st) {
  const int vb = rows_per_block(m.H, m.V, B);
  const dim3 grid((h.on ? h.a.Hq + h.a.Hkv : 0) + m.H * (m.V / vb), B);
  const size_t lds = (2 * m.N + vb) * 4;
  // (both halves read the same projection; fp32 storage has one instance)
  const bool same = !h.on || (h.a.src.p == m.src.p && src_mode(h.a.src) == src_mode(m.src));
  const int mode = f32 || !same ? SRC_ANY : src_mode(m.src);
  auto kernel = [&](auto ahead) {
    constexpr bool A = decltype(ahead)::value;
    if (f32) return &parallel_step_kernel<float, A, SRC_ANY>;
    return mode == SRC_ONE ? &parallel_step_kernel<bf16_t, A, SRC_ONE>
                           : mode == SRC_FOUR ? &parallel_step_kernel<bf16_t, A, SRC_FOUR> : &parallel_step_kernel<bf16_t, A, SRC_ANY>;
  };
  hipLaunchKernelGGL((vb > 16 ? kernel(std::true_type{}) : kernel(std::false_type{})), grid, dim3(256), lds, st, h, m, pos, live, vb);
}
// Where one launch is ahead of two.  us, two / one, 600 cached keys, 16 splits: 16 heads 10.3 / 7.9 for one stream, 12.1 / 9.3 for two, four splits
// 13.7 / 10.9 and 15.1 / 12.8 for three and four; 32 heads (the same order, four splits from three on) 11.7 / 9.2, 14.4 / 12.7, 17.6 / 14.5, 21.1 /
// 17.9.  Every block makes the norms of all heads anew, which is level around a thousand blocks and lost with more: 64 heads, 16 splits, one
// stream 14.9 / 13.6, two (2048 blocks) 20.2 / 20.6, four 32.7 / 34.0 (100 keys 25.0 / 27.9); 128 heads, one stream 17.8 / 19.5, but with two splits
// 17.9 / 16.5, four streams of those (1024 blocks) 24.8 / 22.0.  And it has fewer waves a CU to stream long caches with: 64 key heads of 2000 keys, two
// streams (131 MB) 35.6 / 34.2, three 50.4 / 54.0, four 62.7 / 69.4.
bool attend_step_ok(const StepHeads& h, const StepMemory& m, int B, int nsplit) {
  return B <= GEMV_ROWS_MAX && nsplit > 1 && nsplit <= 16 && (h.a.D == 64 || h.a.D == 128) && src_mode(m.src) == SRC_ONE && h.a.src.p == m.src.p &&
         static_cast<long long>(B) * h.a.Hq * nsplit <= 1024 && static_cast<long long>(B) * h.a.Hkv * h.a.cap * h.a.D <= 1ll << 25;
}
void launch_attend_step(const StepHeads& h, const StepMemory& m, const StepSplits& sp, const int* pos, const int* live, int B, hipStream_t st) {
  const int vb = rows_per_block(m.H, m.V, B);
  const dim3 grid(h.a.Hq * sp.nsplit + m.H * (m.V / vb), B);
  const size_t lds = (2 * m.N + vb) * 4;
  const bool ahead = vb > 16;
#define EVGPT_ATTEND_STEP(D, A) hipLaunchKernelGGL((attend_step_kernel<D, A, SRC_ONE>), grid, dim3(256), lds, st, pos, live, vb, h, sp, m)
  if (h.a.D == 128) { if (ahead) EVGPT_ATTEND_STEP(128, true); else EVGPT_ATTEND_STEP(128, false); }
  else { if (ahead) EVGPT_ATTEND_STEP(64, true); else EVGPT_ATTEND_STEP(64, false); }
#undef EVGPT_ATTEND_STEP
}
void launch_ssd_step(const StepSsd& a, const int* pos, const int* live, bool f32, int B, hipStream_t st) {
  const int vb = rows_per_block(a.H, a.V, B);
  const dim3 grid(a.V / vb, a.H, B);
  const size_t lds = (2 * a.N + 3 * vb) * 4;
  const int threads = min(512, max(256, (2 * a.N + vb + 63) / 64 * 64));
  const int mode = f32 ? SRC_ANY : src_mode(a.src);
  auto kernel = [&](auto ahead) {
    constexpr bool A = decltype(ahead)::value;
    if (f32) return &ssd_step_kernel<float, A, SRC_ANY>;
    return mode == SRC_ONE ? &ssd_step_kernel<bf16_t, A, SRC_ONE>
                           : mode == SRC_FOUR ? &ssd_step_kernel<bf16_t, A, SRC_FOUR> : &ssd_step_kernel<bf16_t, A, SRC_ANY>;
  };
  hipLaunchKernelGGL((vb > 16 ? kernel(std::true_type{}) : kernel(std::false_type{})), grid, dim3(threads), lds, st, a, pos, live, vb);
}

}  // namespace evgpt
