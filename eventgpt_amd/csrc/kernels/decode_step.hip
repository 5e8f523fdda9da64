// The part of a decode step between a mixer's input projection and its output projection, for one token per
// sequence, in one launch: attention heads (norm, rotation, cache append), the matrix memory and the
// state-space recurrence with its convolution.  Inputs are the projection's fp32 rows or split-K slabs;
// what a prompt would have stored in T is rounded to T here as well.
//
// A recurrent state is streamed once: sixteen lanes per state row read it, decay it, add the token, dot it with
// the query and write it back.  A block owns some rows of one head; it prepares the head's small vectors
// (query, key, convolution outputs, gates) itself in LDS rather than waiting for another launch.
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

template <typename T>
__device__ void head_step(const AttnPrepArgs& a, int b, int head, int p, bool live, float* red) {
  const bool is_q = head < a.Hq;
  const int h = is_q ? head : head - a.Hq;
  const int col = is_q ? a.q_col : a.k_col, width = (is_q ? a.Hq : a.Hkv) * a.D;
  const float* w = is_q ? a.qw : a.kw;
  float r = 1.f;
  if (w) {
    float s = 0.f;
    for (int c = threadIdx.x * 8; c < width; c += 2048) {
      float t[8];
      src8(a.src, b, col + c, t);
      s += sumsq8(t);
    }
    r = rsqrtf(block_sum<4>(s, red) / static_cast<float>(is_q ? a.nq : a.nk) + a.eps);
  }
  if (!is_q && !live) return;
  const int half = a.rot >> 1, pt = min(max(p, 0), a.max_pos - 1);
  const float* cs = a.cos_tab + static_cast<long long>(pt) * half;
  const float* sn = a.sin_tab + static_cast<long long>(pt) * half;
  for (int d = threadIdx.x; d < a.D; d += 256) {
    const int c = h * a.D + d;
    float u = src1(a.src, b, col + c) * r;
    if (w) u *= w[c];
    if (d < a.rot) {
      const int i = d < half ? d : d - half, c2 = d < half ? c + half : c - half;
      float o = src1(a.src, b, col + c2) * r;
      if (w) o *= w[c2];
      u = d < half ? u * cs[i] - o * sn[i] : u * cs[i] + o * sn[i];
    }
    if (is_q) {
      static_cast<T*>(a.q_out)[static_cast<long long>(b) * width + c] = from_f32<T>(u);
    } else {
      const long long o = ((static_cast<long long>(b) * a.Hkv + h) * a.cap + max(p, 0) % a.cap) * a.D + d;
      static_cast<T*>(a.k_cache)[o] = from_f32<T>(u);
      static_cast<T*>(a.v_cache)[o] = from_f32<T>(src1(a.src, b, a.v_col + c));
    }
  }
}

template <typename T, bool AHEAD>
__global__ __launch_bounds__(256) void parallel_step_kernel(StepHeads sh, StepMemory m, const int* __restrict__ pos,
                                                            const int* __restrict__ live, int vb) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // [N] query, [N] key, [vb] weighted values
  __shared__ float red[16], gates[2];
  const int b = blockIdx.y, p = pos[b];
  const bool alive = live == nullptr || live[b] != 0;
  const int n_heads = sh.on ? sh.a.Hq + sh.a.Hkv : 0;
  if (static_cast<int>(blockIdx.x) < n_heads) {
    head_step<T>(sh.a, b, blockIdx.x, p, alive, red);
    return;
  }
  const int per = m.V / vb, i0 = blockIdx.x - n_heads, h = i0 / per, v0 = (i0 % per) * vb;
  const int gi = b * m.H + h;
  if (!alive) {                         // a parked sequence keeps its state
    for (int i = threadIdx.x; i < vb; i += 256) m.out[static_cast<long long>(gi) * m.V + v0 + i] = 0.f;
    return;
  }
  float* S = m.S + static_cast<long long>(gi) * m.V * m.N;
  const StateRows rows = request_state(S, m.N, v0, vb);
  const bool fresh = p <= 0;
  float *qs = lds, *ks = lds + m.N, *avs = ks + m.N;
  const long long from = (static_cast<long long>(p & 1) * m.slots + b) * m.H + h;
  const long long to = (static_cast<long long>((p + 1) & 1) * m.slots + b) * m.H + h;
  const float m_old = m.m[from];
  const float n_old = m.n[from * m.N + min(static_cast<int>(threadIdx.x), m.N - 1)];
  if (threadIdx.x == 255) {
    gates[0] = m.cap * tanhf((src1(m.src, b, m.i_col + h) + m.ib[h]) / m.cap);
    gates[1] = -softplus_f(-m.cap * tanhf((src1(m.src, b, m.f_col + h) + m.fb[h]) / m.cap));
  }
  for (int e = threadIdx.x; e < m.N; e += 256) {
    qs[e] = src_t<T>(m.src, b, m.q_col + h * m.N + e) * m.qscale;
    ks[e] = src_t<T>(m.src, b, m.k_col + h * m.N + e);
  }
  __syncthreads();
  const float m0 = fresh ? 0.f : m_old;
  const float li = gates[0], lf = gates[1], m1 = fmaxf(lf + m0, li);
  const float decay = expf(lf + m0 - m1), add = expf(li - m1);
  for (int i = threadIdx.x; i < vb; i += 256) avs[i] = add * src_t<T>(m.src, b, m.v_col + h * m.V + v0 + i);
  float dot = 0.f;
  for (int e = threadIdx.x; e < m.N; e += 256) {
    const float n1 = (fresh ? 0.f : (e < 256 ? n_old : m.n[from * m.N + e]) * decay) + add * ks[e];
    if (v0 == 0) m.n[to * m.N + e] = n1;
    dot += n1 * qs[e];
  }
  dot = block_sum<4>(dot, red);            // (its barriers also publish avs)
  if (v0 == 0 && threadIdx.x == 0) m.m[to] = m1;
  const float inv = 1.f / (fmaxf(fabsf(dot), expf(-m1)) + 1e-6f);
  float* out = m.out + static_cast<long long>(gi) * m.V + v0;
  stream_state<AHEAD>(S, m.N, v0, vb, fresh, decay, qs, ks, avs, rows, [&](int i, float y) { out[i] = y * inv; });
}

// threads: one per convolution channel of the block where that is at most 512 (the state takes four waves)
template <typename T, bool AHEAD>
__global__ __launch_bounds__(512) void ssd_step_kernel(StepSsd a, const int* __restrict__ pos, const int* __restrict__ live,
                                                       int vb) {
  extern __shared__ __attribute__((aligned(16))) float lds[];      // [N] C, [N] B, [vb] weighted x, [vb] x, [vb] silu(z)
  __shared__ float gates[2];
  const int b = blockIdx.z, h = blockIdx.y, v0 = blockIdx.x * vb, p = pos[b];
  const int gi = b * a.H + h, per_group = a.H / a.G, g = h / per_group, nt = blockDim.x;
  float* out = a.out + static_cast<long long>(gi) * a.V + v0;
  if (live && !live[b]) {
    for (int i = threadIdx.x; i < vb; i += nt) out[i] = 0.f;
    return;
  }
  float* S = a.S + static_cast<long long>(gi) * a.V * a.N;
  const StateRows rows = request_state(S, a.N, v0, vb);
  const bool fresh = p <= 0;
  float *cs = lds, *bs = lds + a.N, *avs = bs + a.N, *xs = avs + vb, *zs = xs + vb;
  const int C = a.H * a.V + 2 * a.G * a.N;
  if (static_cast<int>(threadIdx.x) == nt - 1) {
    const float dt = softplus_f(src1(a.src, b, a.dt_col + h) + a.dt_bias[h]);
    gates[0] = expf(-expf(a.a_log[h]) * dt);
    gates[1] = dt;
  }
  T* ring = static_cast<T*>(a.ring) + static_cast<long long>(b) * a.taps * C;
  for (int i = threadIdx.x; i < 2 * a.N + vb; i += nt) {
    const bool is_x = i >= 2 * a.N;
    const int c = is_x ? h * a.V + v0 + i - 2 * a.N
                       : a.H * a.V + (i < a.N ? g * a.N + i : (a.G + g) * a.N + i - a.N);     // B, then C
    const float* w = a.conv_w + static_cast<long long>(c) * a.taps;
    float acc = a.conv_b[c];
    T cur;
    if (a.taps == 4) {                  // (all operands on their way before the first product)
      const f32x4_t w4 = load4(w);
      T old[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) old[j] = ring[static_cast<long long>(max(p + j - 3, 0) & 3) * C + c];
      cur = from_f32<T>(src1(a.src, b, a.x_col + c));
#pragma unroll
      for (int j = 0; j < 3; ++j) acc = fmaf(w4[j], p + j - 3 < 0 ? 0.f : to_f32(old[j]), acc);
      acc = fmaf(w4[3], p < 0 ? 0.f : to_f32(cur), acc);
    } else {
      cur = from_f32<T>(src1(a.src, b, a.x_col + c));
      for (int j = 0; j < a.taps; ++j) {
        const int d = a.taps - 1 - j;
        if (p - d < 0) continue;
        acc = fmaf(w[j], d == 0 ? to_f32(cur) : to_f32(ring[static_cast<long long>((p - d) % a.taps) * C + c]), acc);
      }
    }
    const float v = to_f32(from_f32<T>(acc * sigmoid_f(acc)));
    if (is_x) xs[i - 2 * a.N] = v;
    else if (i < a.N) bs[i] = v;
    else cs[i - a.N] = v;
    // the current input's slot is read by nobody in this step; one block per channel stores it
    if (is_x || (v0 == 0 && h % per_group == 0)) ring[static_cast<long long>(max(p, 0) % a.taps) * C + c] = cur;
  }
  __syncthreads();
  const float decay = gates[0], dt = gates[1];
  for (int i = threadIdx.x; i < vb; i += nt) {
    avs[i] = dt * xs[i];
    const float z = src_t<T>(a.src, b, a.z_col + h * a.V + v0 + i);
    zs[i] = z * sigmoid_f(z);
  }
  __syncthreads();
  const float skip = a.skip[h];
  stream_state<AHEAD>(S, a.N, v0, vb, fresh, decay, cs, bs, avs, rows, [&](int i, float y) { out[i] = (y + skip * xs[i]) * zs[i]; });
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
  const auto kernel = vb > 16 ? (f32 ? &parallel_step_kernel<float, true> : &parallel_step_kernel<bf16_t, true>)
                              : (f32 ? &parallel_step_kernel<float, false> : &parallel_step_kernel<bf16_t, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), lds, st, h, m, pos, live, vb);
}
void launch_ssd_step(const StepSsd& a, const int* pos, const int* live, bool f32, int B, hipStream_t st) {
  const int vb = rows_per_block(a.H, a.V, B);
  const dim3 grid(a.V / vb, a.H, B);
  const size_t lds = (2 * a.N + 3 * vb) * 4;
  const int threads = min(512, max(256, (2 * a.N + vb + 63) / 64 * 64));
  const auto kernel = vb > 16 ? (f32 ? &ssd_step_kernel<float, true> : &ssd_step_kernel<bf16_t, true>)
                              : (f32 ? &ssd_step_kernel<float, false> : &ssd_step_kernel<bf16_t, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, st, a, pos, live, vb);
}

}  // namespace evgpt
