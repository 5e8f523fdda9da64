// Fused AdamW update of one optimizer shard: a single pass over the gradient shard, the
// fp32 master weights and both moments that also writes the refreshed parameter shard in
// its storage type.  The unfused sequence is ten elementwise launches with fp32
// temporaries (~56 bytes of traffic per parameter); this is 30 (bf16 parameters).
//
//   g  = grad * clip                       m = b1 m + (1-b1) g      v = b2 v + (1-b2) g^2
//   w *= 1 - lr*wd                         w -= (lr / bc1) * m / (sqrt(v)/sqrt(bc2) + eps)
#include "common.h"
#include "../evgpt_kernels.h"

namespace evgpt {

template <typename T> __device__ __forceinline__ float ld_as_f32(const T* p);
template <> __device__ __forceinline__ float ld_as_f32<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ld_as_f32<bf16_t>(const bf16_t* p) { return bf16_to_f32(*p); }
template <typename T> __device__ __forceinline__ void st_from_f32(T* p, float v);
template <> __device__ __forceinline__ void st_from_f32<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void st_from_f32<bf16_t>(bf16_t* p, float v) { *p = f32_to_bf16(v); }

__device__ __forceinline__ float adamw_one(float g, float& m, float& v, float w, const AdamWArgs& a) {
  g *= a.clip;
  m = a.beta1 * m + (1.f - a.beta1) * g;
  v = a.beta2 * v + (1.f - a.beta2) * g * g;
  const float denom = sqrtf(v) * a.inv_sqrt_bc2 + a.eps;
  return w * a.decay - a.step_size * (m / denom);
}

template <typename T>
__global__ __launch_bounds__(256) void fused_adamw_kernel(const T* __restrict__ grad, float* __restrict__ master,
                                                          float* __restrict__ m, float* __restrict__ v,
                                                          T* __restrict__ param_out, long long n, AdamWArgs a) {
  if (a.clip_dev) a.clip *= *a.clip_dev;
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x * 4;
  for (long long i0 = (static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x) * 4; i0 < n; i0 += stride) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const long long i = i0 + k;
      if (i >= n) break;
      float mi = m[i], vi = v[i];
      const float w = adamw_one(ld_as_f32(grad + i), mi, vi, master[i], a);
      m[i] = mi; v[i] = vi; master[i] = w;
      st_from_f32(param_out + i, w);
    }
  }
}

// 8 elements per thread with 16-byte accesses (all pointers 16-byte aligned); block `block` of the shard's `blocks`
template <typename T>
__device__ __forceinline__ void adamw_vec(const T* __restrict__ grad, float* __restrict__ master, float* __restrict__ m,
                                          float* __restrict__ v, T* __restrict__ param_out, long long n8, const AdamWArgs& a, int block,
                                          int blocks) {
  const long long stride = static_cast<long long>(blocks) * 256;
  for (long long c = static_cast<long long>(block) * 256 + threadIdx.x; c < n8; c += stride) {
    float g[8], mm[8], vv[8], w[8];
    if constexpr (sizeof(T) == 2) {
      const u32x4_t gv = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(grad) + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) { g[2 * j] = bf16lo(gv[j]); g[2 * j + 1] = bf16hi(gv[j]); }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4_t t = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(grad) + 2 * c + h);
#pragma unroll
        for (int j = 0; j < 4; ++j) g[4 * h + j] = t[j];
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4_t tm = reinterpret_cast<const f32x4_t*>(m)[2 * c + h];
      const f32x4_t tv = reinterpret_cast<const f32x4_t*>(v)[2 * c + h];
      const f32x4_t tw = reinterpret_cast<const f32x4_t*>(master)[2 * c + h];
#pragma unroll
      for (int j = 0; j < 4; ++j) { mm[4 * h + j] = tm[j]; vv[4 * h + j] = tv[j]; w[4 * h + j] = tw[j]; }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = adamw_one(g[k], mm[k], vv[k], w[k], a);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      reinterpret_cast<f32x4_t*>(m)[2 * c + h] = f32x4_t{mm[4 * h], mm[4 * h + 1], mm[4 * h + 2], mm[4 * h + 3]};
      reinterpret_cast<f32x4_t*>(v)[2 * c + h] = f32x4_t{vv[4 * h], vv[4 * h + 1], vv[4 * h + 2], vv[4 * h + 3]};
      reinterpret_cast<f32x4_t*>(master)[2 * c + h] = f32x4_t{w[4 * h], w[4 * h + 1], w[4 * h + 2], w[4 * h + 3]};
    }
    if constexpr (sizeof(T) == 2) {
      u32x4_t o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = pack_bf16x2(w[2 * j], w[2 * j + 1]);
      reinterpret_cast<u32x4_t*>(param_out)[c] = o;
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        reinterpret_cast<f32x4_t*>(param_out)[2 * c + h] = f32x4_t{w[4 * h], w[4 * h + 1], w[4 * h + 2], w[4 * h + 3]};
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void fused_adamw_vec_kernel(const T* __restrict__ grad, float* __restrict__ master,
                                                              float* __restrict__ m, float* __restrict__ v,
                                                              T* __restrict__ param_out, long long n8, AdamWArgs a) {
  if (a.clip_dev) a.clip *= *a.clip_dev;
  adamw_vec(grad, master, m, v, param_out, n8, a, blockIdx.x, gridDim.x);
}

// All shards of a step: a small one (biases, a scalar) is a launch of 4 to 5 us by itself and a few blocks here.
constexpr int MANY = 32;
struct AdamWTable { AdamWShard s[MANY]; int first[MANY + 1]; };      // a shard's blocks: first[i] .. first[i + 1]

template <typename T>
__global__ __launch_bounds__(256) void fused_adamw_many_kernel(AdamWTable t, AdamWArgs a) {
  if (a.clip_dev) a.clip *= *a.clip_dev;
  int i = 0;
  while (static_cast<int>(blockIdx.x) >= t.first[i + 1]) ++i;
  const AdamWShard& s = t.s[i];
  const int block = blockIdx.x - t.first[i];
  const T* grad = static_cast<const T*>(s.grad);
  T* out = static_cast<T*>(s.out);
  adamw_vec(grad, s.master, s.m, s.v, out, s.n / 8, a, block, t.first[i + 1] - t.first[i]);
  const long long e = s.n / 8 * 8 + threadIdx.x;
  if (block == 0 && e < s.n) {
    float mi = s.m[e], vi = s.v[e];
    const float w = adamw_one(ld_as_f32(grad + e), mi, vi, s.master[e], a);
    s.m[e] = mi; s.v[e] = vi; s.master[e] = w;
    st_from_f32(out + e, w);
  }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <typename T>
static void launch_t(const T* grad, float* master, float* m, float* v, T* out, long long n,
                     const AdamWArgs& a, hipStream_t st) {
  if (n <= 0) return;
  if (n % 8 == 0 && aligned16(grad) && aligned16(master) && aligned16(m) && aligned16(v) && aligned16(out)) {
    const long long n8 = n / 8;
    long long vb = (n8 + 255) / 256;
    if (vb > 8192) vb = 8192;
    hipLaunchKernelGGL(fused_adamw_vec_kernel<T>, dim3(static_cast<unsigned int>(vb)), dim3(256), 0, st, grad,
                       master, m, v, out, n8, a);
    return;
  }
  long long blocks = (n + 1023) / 1024;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(fused_adamw_kernel<T>, dim3(static_cast<unsigned int>(blocks)), dim3(256), 0, st, grad,
                     master, m, v, out, n, a);
}

void launch_fused_adamw_bf16(const bf16_t* grad, float* master, float* m, float* v, bf16_t* out, long long n,
                             const AdamWArgs& a, hipStream_t st) {
  launch_t<bf16_t>(grad, master, m, v, out, n, a, st);
}
void launch_fused_adamw_f32(const float* grad, float* master, float* m, float* v, float* out, long long n,
                            const AdamWArgs& a, hipStream_t st) {
  launch_t<float>(grad, master, m, v, out, n, a, st);
}

void launch_fused_adamw_many(const AdamWShard* shards, int count, bool bf16, const AdamWArgs& a, hipStream_t st) {
  for (int at = 0; at < count; at += MANY) {
    AdamWTable t{};
    const int n = count - at < MANY ? count - at : MANY;
    for (int i = 0; i < n; ++i) {
      t.s[i] = shards[at + i];
      const long long want = (t.s[i].n / 8 + 255) / 256;
      t.first[i + 1] = t.first[i] + static_cast<int>(want > 8192 ? 8192 : (want < 1 && t.s[i].n > 0 ? 1 : want));
    }
    if (t.first[n] == 0) continue;
    if (bf16) hipLaunchKernelGGL(fused_adamw_many_kernel<bf16_t>, dim3(t.first[n]), dim3(256), 0, st, t, a);
    else hipLaunchKernelGGL(fused_adamw_many_kernel<float>, dim3(t.first[n]), dim3(256), 0, st, t, a);
  }
}

// ---- sum of squares of a gradient's shards (global-norm clipping), two deterministic stages: partial sums of blocks, then one block
// adds them.  Two launches in all instead of two a shard, each 4 to 5 us at the least.
template <typename T>
__device__ __forceinline__ float sumsq_block(const T* __restrict__ x, long long n, int block, int blocks, float* red) {
  float s = 0.f;
  const long long stride = static_cast<long long>(blocks) * 256 * 8;
  for (long long i0 = (static_cast<long long>(block) * 256 + threadIdx.x) * 8; i0 < n; i0 += stride) {
    if (i0 + 8 <= n) {
      if constexpr (sizeof(T) == 2) {
        const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(x + i0));
#pragma unroll
        for (int j = 0; j < 4; ++j) { const float a = bf16lo(v[j]), b = bf16hi(v[j]); s += a * a + b * b; }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(x + i0) + h);
          s += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
      }
    } else {
      for (long long i = i0; i < n; ++i) { const float a = ld_as_f32(x + i); s += a * a; }
    }
  }
  return block_sum(s, red);
}
struct SumsqTable { const void* x[MANY]; long long n[MANY]; int first[MANY + 1]; unsigned int bf16; };
__global__ __launch_bounds__(256) void sumsq_many_kernel(SumsqTable t, float* __restrict__ part) {
  __shared__ float red[4];
  int i = 0;
  while (static_cast<int>(blockIdx.x) >= t.first[i + 1]) ++i;
  const int block = blockIdx.x - t.first[i], blocks = t.first[i + 1] - t.first[i];
  const float s = t.bf16 >> i & 1 ? sumsq_block(static_cast<const bf16_t*>(t.x[i]), t.n[i], block, blocks, red)
                                  : sumsq_block(static_cast<const float*>(t.x[i]), t.n[i], block, blocks, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
__global__ __launch_bounds__(1024) void sumsq_many_final_kernel(const float* __restrict__ part, long long n, float* __restrict__ out) {
  __shared__ float red[16];
  float s = 0.f;
  for (long long i = threadIdx.x; i < n; i += 1024) s += part[i];
  s = block_sum<16>(s, red);
  if (threadIdx.x == 0) out[0] = s;
}
__global__ void clip_factor_kernel(const float* __restrict__ sq, float max_norm, float* __restrict__ norm, float* __restrict__ clip) {
  const float n = sqrtf(*sq), c = max_norm / (n + 1e-6f);
  *norm = n;
  *clip = c > 1.f ? 1.f : c;             // (not a number stays that)
}

static int sumsq_blocks(long long n) {
  long long b = (n + 256 * 8 * 4 - 1) / (256 * 8 * 4);   // at least four 16-byte loads per thread
  return static_cast<int>(b < 1 ? 1 : (b > 2048 ? 2048 : b));
}

long long sumsq_many_blocks(const SumsqShard* shards, int count) {
  long long n = 0;
  for (int i = 0; i < count; ++i) n += sumsq_blocks(shards[i].n);
  return n;
}
void launch_sumsq_many(const SumsqShard* shards, int count, float* part, float* out, hipStream_t st) {
  long long done = 0;
  for (int at = 0; at < count; at += MANY) {
    SumsqTable t{};
    const int n = count - at < MANY ? count - at : MANY;
    for (int i = 0; i < n; ++i) {
      t.x[i] = shards[at + i].x; t.n[i] = shards[at + i].n;
      t.bf16 |= static_cast<unsigned int>(shards[at + i].bf16) << i;
      t.first[i + 1] = t.first[i] + sumsq_blocks(t.n[i]);
    }
    hipLaunchKernelGGL(sumsq_many_kernel, dim3(t.first[n]), dim3(256), 0, st, t, part + done);
    done += t.first[n];
  }
  hipLaunchKernelGGL(sumsq_many_final_kernel, dim3(1), dim3(1024), 0, st, part, done, out);
}
void launch_clip_factor(const float* sq, float max_norm, float* norm, float* clip, hipStream_t st) {
  hipLaunchKernelGGL(clip_factor_kernel, dim3(1), dim3(1), 0, st, sq, max_norm, norm, clip);
}

}  // namespace evgpt
