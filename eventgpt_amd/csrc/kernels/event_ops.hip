// Event-stream front end on the GPU: rasterisation of polarity events into RGB
// frames, per-bin polarity histograms / voxel grids, and the fused CLIP
// preprocessing (antialiased bicubic resize + centre crop + normalise -> bf16).
//
// Rasterisation is a scatter with an ordering rule, so it is done with one
// 32-bit atomic per event and a colourise pass:
//   "last event wins"      atomicMax of (event_index << 1 | polarity)
//   "negative wins"        atomicOr  of a 2-bit {has_pos, has_neg} mask
// All T slices of a stream are handled by one launch (slice id from the event
// index via the equal-count boundaries).
#include "common.h"
#include "../evgpt_kernels.h"

namespace evgpt {

typedef __attribute__((ext_vector_type(4))) int i32x4_t;

// keys: [T][H*W] int32, pre-filled with -1 (last) or 0 (negative-wins mask)
__global__ __launch_bounds__(256) void raster_scatter_kernel(
    const int* __restrict__ x, const int* __restrict__ y, const int* __restrict__ p, int n_events,
    int n_slices, int per_slice, int H, int W, int* __restrict__ keys, int mode) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n_events; i += gridDim.x * 256) {
    int s = per_slice > 0 ? i / per_slice : 0;
    if (s >= n_slices) s = n_slices - 1;  // the last slice takes the remainder
    const int xi = x[i], yi = y[i];
    if (xi < 0 || xi >= W || yi < 0 || yi >= H) continue;
    int* cell = keys + static_cast<size_t>(s) * H * W + yi * W + xi;
    const int pol = p[i] != 0;
    if (mode == 0) atomicMax(cell, (i << 1) | pol);
    else atomicOr(cell, pol ? 1 : 2);
  }
}

__global__ __launch_bounds__(256) void raster_colorize_kernel(const int* __restrict__ keys,
                                                              unsigned char* __restrict__ img,
                                                              long long n_pix, int mode) {
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n_pix; i += gridDim.x * 256ll) {
    const int k = keys[i];
    unsigned char r = 255, g = 255, b = 255;
    if (mode == 0) {
      if (k >= 0) { if (k & 1) { g = 0; b = 0; } else { r = 0; g = 0; } }
    } else {
      if (k & 2) { r = 0; g = 0; } else if (k & 1) { g = 0; b = 0; }
    }
    img[i * 3] = r; img[i * 3 + 1] = g; img[i * 3 + 2] = b;
  }
}

void launch_event_raster(const int* x, const int* y, const int* p, int n_events, int n_slices,
                         int H, int W, int* keys, unsigned char* img, int mode, hipStream_t st) {
  const int per = n_events / n_slices;
  int blocks = (n_events + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks > 0)
    hipLaunchKernelGGL(raster_scatter_kernel, dim3(blocks), dim3(256), 0, st, x, y, p, n_events,
                       n_slices, per, H, W, keys, mode);
  const long long n_pix = static_cast<long long>(n_slices) * H * W;
  int cb = static_cast<int>((n_pix + 255) / 256);
  if (cb > 4096) cb = 4096;
  hipLaunchKernelGGL(raster_colorize_kernel, dim3(cb), dim3(256), 0, st, keys, img, n_pix, mode);
}

// Words out of pinned host memory, a 16-byte read a lane so that the bus has many of them at once.  (A copy command for them takes 11 us at 80 KB.)
__global__ __launch_bounds__(256) void copy_words_kernel(const int* __restrict__ src, int* __restrict__ dst, long long n) {
  const long long quads = n / 4;
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < quads; i += gridDim.x * 256ll)
    reinterpret_cast<i32x4_t*>(dst)[i] = reinterpret_cast<const i32x4_t*>(src)[i];
  if (blockIdx.x == 0 && threadIdx.x < (n & 3)) dst[quads * 4 + threadIdx.x] = src[quads * 4 + threadIdx.x];
}
void launch_copy_words(const int* src, int* dst, long long n, hipStream_t st) {
  if (n <= 0) return;
  const long long blocks = (n / 4 + 255) / 256;
  hipLaunchKernelGGL(copy_words_kernel, dim3(static_cast<unsigned>(blocks > 512 ? 512 : (blocks < 1 ? 1 : blocks))), dim3(256), 0, st, src, dst, n);
}

// Frames of a packed stream (x | y << 15 | positive << 30, one word an event) as one code a pixel: 0 untouched, 1 positive, 2
// negative.  A block owns some rows of one slice in LDS and scans the slice's events, so nothing is filled beforehand, no
// atomic leaves the CU and what the preprocessing reads is a third of an RGB frame.  Bound by the passes over LDS and the scan's
// round trips.  Five slices: 20 000 events on 160 x 120 4.4 us, 12.3 as a fill, a scatter of global atomics and a colour pass;
// 200 000 on 640 x 480 12.8 and 24.9; 2 500 000 there 101 and 108: from there on the atomics are as good.
__global__ __launch_bounds__(1024) void event_codes_kernel(const unsigned int* __restrict__ ev, int n_events, int n_slices, int H, int W,
                                                           int rows, unsigned char* __restrict__ codes, int mode) {
  extern __shared__ int cell[];        // [rows][W]: last (index << 1 | positive) or the mask of polarities seen
  const int s = blockIdx.y, y0 = blockIdx.x * rows, band = min(rows, H - y0), cells = band * W;
  for (int i = threadIdx.x; i < cells; i += 1024) cell[i] = mode == 0 ? -1 : 0;
  __syncthreads();
  const int per = n_events / n_slices;
  const int lo = s * per, hi = s + 1 < n_slices ? lo + per : n_events;      // the last slice takes the remainder
  for (int i0 = lo + threadIdx.x; i0 < hi; i0 += 4096) {
    unsigned int e[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) e[u] = ev[min(i0 + u * 1024, hi - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * 1024, x = e[u] & 0x7fff, r = static_cast<int>(e[u] >> 15 & 0x7fff) - y0, pol = e[u] >> 30;
      if (i >= hi || r < 0 || r >= band || x >= W) continue;
      if (mode == 0) atomicMax(&cell[r * W + x], (i - lo) << 1 | pol);
      else atomicOr(&cell[r * W + x], pol ? 1 : 2);
    }
  }
  __syncthreads();
  unsigned char* out = codes + (static_cast<size_t>(s) * H + y0) * W;
  for (int i = threadIdx.x; i < cells; i += 1024) {
    const int k = cell[i];
    out[i] = mode == 0 ? (k < 0 ? 0 : (k & 1 ? 1 : 2)) : (k & 2 ? 2 : (k & 1));
  }
}

// image rows of a block: about 160 blocks, at most 144 KB of cells (0: the image is too wide)
static int event_codes_rows(int n_slices, int H, int W) {
  const int most = 144 * 1024 / 4 / W;
  const int bands = (160 + n_slices - 1) / n_slices, rows = (H + bands - 1) / bands;
  return rows < most ? rows : most;
}
// every block of a slice scans all its events: worth it up to the 500 000 events a slice measured above (fewer events
// than slices are all of slice 0, which only the atomic kernel knows)
bool event_codes_ok(long long n_events, int n_slices, int H, int W) {
  if (n_slices < 1 || n_events < n_slices || n_slices > 65535 || H < 1 || W < 1 || H > 32768 || W > 32768) return false;
  const int rows = event_codes_rows(n_slices, H, W);
  return rows >= 1 && n_events / n_slices <= 500000 && (H + rows - 1) / rows * n_slices <= 1024;
}
void launch_event_codes(const unsigned int* ev, int n_events, int n_slices, int H, int W, unsigned char* codes, int mode, hipStream_t st) {
  const int rows = event_codes_rows(n_slices, H, W);
  static bool attr_set = false;
  if (!attr_set) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&event_codes_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 144 * 1024);
    attr_set = true;
  }
  hipLaunchKernelGGL(event_codes_kernel, dim3((H + rows - 1) / rows, n_slices), dim3(1024), static_cast<size_t>(rows) * W * 4, st, ev,
                     n_events, n_slices, H, W, rows, codes, mode);
}

// ------------------------------------------------------------ voxel / histogram
// Time-binned accumulation.  t is int64 microseconds; bin = floor((t - t0) * bins / span)
// clamped to bins-1.  out_hist: [bins][2][H][W] int32 counts (may be null);
// out_vox: [bins][H][W] fp32, +1/-1 (signed) or +1 per event (may be null).
__global__ __launch_bounds__(256) void voxel_kernel(
    const int* __restrict__ x, const int* __restrict__ y, const int* __restrict__ p,
    const long long* __restrict__ t, int n_events, long long t0, double span, int bins, int H,
    int W, int* __restrict__ out_hist, float* __restrict__ out_vox, int signed_mode, int by_count) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n_events; i += gridDim.x * 256) {
    const int xi = x[i], yi = y[i];
    if (xi < 0 || xi >= W || yi < 0 || yi >= H) continue;
    int b;
    if (by_count) b = static_cast<int>(static_cast<long long>(i) * bins / n_events);
    else b = static_cast<int>(static_cast<double>(t[i] - t0) / span * bins);
    b = b < 0 ? 0 : (b >= bins ? bins - 1 : b);
    const int pol = p[i] != 0;
    if (out_hist) atomicAdd(out_hist + ((static_cast<size_t>(b) * 2 + pol) * H + yi) * W + xi, 1);
    if (out_vox)
      atomicAdd(out_vox + (static_cast<size_t>(b) * H + yi) * W + xi,
                pol ? 1.f : (signed_mode ? -1.f : 1.f));
  }
}

void launch_event_voxel(const int* x, const int* y, const int* p, const long long* t, int n_events,
                        long long t0, long long span, int bins, int H, int W, int* out_hist,
                        float* out_vox, int signed_mode, int by_count, hipStream_t st) {
  int blocks = (n_events + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) return;
  const double dspan = static_cast<double>(span > 0 ? span : 1);
  hipLaunchKernelGGL(voxel_kernel, dim3(blocks), dim3(256), 0, st, x, y, p, t, n_events, t0,
                     dspan, bins, H, W, out_hist, out_vox, signed_mode, by_count);
}

// LDS-privatised variant for event streams whose bins are index ranges (binning by count, or by
// time on a time-sorted stream): bounds[b] .. bounds[b+1] are the events of bin b.  The
// per-polarity count image of one bin (2 x H x W int32) does not fit the 160 KB of LDS, so it is
// cut into bands of `rows` image rows; block (chunk, band, bin) scans its share of the bin's
// events, reads only `y` for every event (4 B) and `x`, `p` for the ~rows/H that fall into its
// band, counts them with LDS atomics, and flushes the non-zero counters: one global atomic per
// touched pixel and block instead of one per event.  Reading y once per band costs H/rows x 4 B
// per event, far less than an L2 atomic round trip per event.
constexpr int VL_THREADS = 1024;  // one block per CU (the band fills LDS): 16 waves hide the load latency
constexpr int VL_DEPTH = 4;       // y vectors in flight per thread

__global__ __launch_bounds__(VL_THREADS) void voxel_lds_kernel(
    const int* __restrict__ x, const int* __restrict__ y, const int* __restrict__ p,
    const int* __restrict__ bounds, int H, int W, int rows, int* __restrict__ out_hist,
    float* __restrict__ out_vox, int signed_mode) {
  extern __shared__ int cnt[];  // [2][rows][W]
  const int b = blockIdx.z, y0 = blockIdx.y * rows;
  const int band = min(rows, H - y0);
  const int cells = 2 * rows * W;
  for (int i = threadIdx.x; i < cells; i += VL_THREADS) cnt[i] = 0;
  __syncthreads();
  const int lo = bounds[b], hi = bounds[b + 1];
  // chunks of whole groups of 4 * VL_THREADS events: every load is a 16-byte aligned lane quad
  constexpr int GROUP = 4 * VL_THREADS;
  const int first = lo & ~3;
  const long long groups = (static_cast<long long>(hi) - first + GROUP - 1) / GROUP;
  const long long per = (groups + gridDim.x - 1) / gridDim.x;
  const long long g0 = per * blockIdx.x, g1 = min(groups, g0 + per);
  for (long long g = g0; g < g1; g += VL_DEPTH) {
    i32x4_t yv[VL_DEPTH];
    int base[VL_DEPTH];
#pragma unroll
    for (int d = 0; d < VL_DEPTH; ++d) {      // all y loads of this round first
      base[d] = first + static_cast<int>(g + d) * GROUP + threadIdx.x * 4;
      const bool in = g + d < g1 && base[d] < hi;
      if (in && base[d] + 3 < hi) {
        yv[d] = *reinterpret_cast<const i32x4_t*>(y + base[d]);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) yv[d][k] = (in && base[d] + k < hi) ? y[base[d] + k] : -1;
      }
    }
#pragma unroll
    for (int d = 0; d < VL_DEPTH; ++d) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int r = yv[d][k] - y0, i = base[d] + k;
        if (i < lo || r < 0 || r >= band) continue;
        const int xi = x[i];
        if (xi < 0 || xi >= W) continue;
        atomicAdd(&cnt[((p[i] != 0 ? rows : 0) + r) * W + xi], 1);
      }
    }
  }
  __syncthreads();
  const int band_cells = band * W;
  for (int i = threadIdx.x; i < band_cells; i += VL_THREADS) {
    const int neg = cnt[i], pos = cnt[rows * W + i];
    if ((neg | pos) == 0) continue;
    const size_t pix = static_cast<size_t>(y0) * W + i;
    if (out_hist) {
      if (neg) atomicAdd(out_hist + (static_cast<size_t>(b) * 2) * H * W + pix, neg);
      if (pos) atomicAdd(out_hist + (static_cast<size_t>(b) * 2 + 1) * H * W + pix, pos);
    }
    if (out_vox)
      atomicAdd(out_vox + static_cast<size_t>(b) * H * W + pix,
                static_cast<float>(signed_mode ? pos - neg : pos + neg));
  }
}

// rows of one band: as many as 150 KB of LDS hold for this width (0: image too wide)
int event_voxel_band_rows(int H, int W) {
  const int rows = (150 * 1024 / 4) / (2 * W);
  return rows < H ? rows : H;
}

void launch_event_voxel_ranges(const int* x, const int* y, const int* p, const int* bounds, int n_events,
                               int bins, int H, int W, int* out_hist, float* out_vox, int signed_mode,
                               hipStream_t st, int chunks_override) {
  const int rows = event_voxel_band_rows(H, W);
  const int bands = (H + rows - 1) / rows;
  // just under three full rounds of one block per CU (a partial extra round costs a whole one:
  // 240 / 480 / 720 blocks measured 0.59 ms at 1e7 events, 320 / 800 blocks 0.70-0.72 ms), but no
  // chunk below 64 K events (zeroing and flushing a band costs as much as scanning a few thousand)
  int chunks = (3 * 256) / (bands * bins);
  const int by_size = n_events / bins / 65536;
  if (chunks > by_size) chunks = by_size;
  if (chunks < 1) chunks = 1;
  if (chunks_override > 0) chunks = chunks_override;
  const size_t smem = static_cast<size_t>(2) * rows * W * sizeof(int);
  static bool attr_set = false;
  if (!attr_set) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&voxel_lds_kernel),
                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr_set = true;
  }
  hipLaunchKernelGGL(voxel_lds_kernel, dim3(chunks, bands, bins), dim3(VL_THREADS), smem, st, x, y, p, bounds, H, W,
                     rows, out_hist, out_vox, signed_mode);
}

// Counting without global atomics (what calls run on from 4 096 events: ops/event_ops.py), for streams in any order.  Three launches, no host round trip:
//   span   one pass over t: extent and whether it is sorted (binning by time only)
//   sort   a block orders its chunk of 8 192 events by (bin, band of `rows` image rows) in LDS and writes one 16-bit
//          record per event -- polarity and place within the band -- plus where each key's run starts
//   count  a block owns one (bin, band): it adds the runs of all chunks in LDS counters and writes both outputs whole
// The chunk of a sorted stream lies in one or two bins, so the sort reads t at its two ends only; the unsorted one
// reads it for every event.  Bound by memory: 12 B in, 2 B out, 2 B in per event (and 8 B for the span) plus 12 B out per
// pixel and bin.  1e7 clustered events, 480 x 640, 5 bins by time on a sorted stream, four recordings: span 15 to 18 us, sort 31,
// count 20 to 25 (by how the events cluster); the whole call 68 to 72 us in a row on one stream, 82 on another one each time (218 MB it cannot do
// without: 2.7 to 3.2 TB/s), 766 with voxel_lds_kernel above, which scans y once a band
// (506 us) behind host round trips for the extent and the order of t.
constexpr int VS_THREADS = 512, VS_PER = 16, VS_CHUNK = VS_THREADS * VS_PER, VS_KEYS = 4096, VS_SPANS = 256;

struct VoxelSpan { long long lo, hi; long long unsorted; };

struct VoxelArgs {
  const int *x, *y, *p;
  const long long* t;
  const VoxelSpan* span;         // [VS_SPANS] partial extents
  unsigned short* rec;           // [chunks][VS_CHUNK]
  unsigned short* off;           // [chunks][keys + 1]
  int2* range;                   // [chunks] first and last bin
  int n, bins, H, W, log_rows, bands, keys, chunks, by_count;
};

__global__ __launch_bounds__(1024) void voxel_span_kernel(const long long* __restrict__ t, int n, VoxelSpan* __restrict__ out) {
  constexpr int DEPTH = 8;
  __shared__ long long lo_s[16], hi_s[16];
  __shared__ int bad_s;
  if (threadIdx.x == 0) bad_s = 0;
  const int per = (static_cast<int>((static_cast<long long>(n) + VS_SPANS - 1) / VS_SPANS) + 1023) & ~1023;
  const long long first = static_cast<long long>(blockIdx.x) * per;
  const long long last = min(first + per, static_cast<long long>(n));
  long long lo = t[0], hi = lo;
  bool bad = false;
  for (long long i0 = first; i0 < last; i0 += 1024 * DEPTH) {
    long long v[DEPTH], w[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const long long i = min(i0 + d * 1024 + threadIdx.x, last - 1);
      v[d] = t[i];
      w[d] = (threadIdx.x & 63) == 63 ? t[min(i + 1, static_cast<long long>(n) - 1)] : 0;
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const long long next = __shfl_down(v[d], 1, 64);
      lo = min(lo, v[d]);
      hi = max(hi, v[d]);
      bad |= v[d] > ((threadIdx.x & 63) == 63 ? w[d] : next);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    lo = min(lo, static_cast<long long>(__shfl_xor(lo, off, 64)));
    hi = max(hi, static_cast<long long>(__shfl_xor(hi, off, 64)));
  }
  __syncthreads();
  if (bad) bad_s = 1;
  if ((threadIdx.x & 63) == 0) { lo_s[threadIdx.x >> 6] = lo; hi_s[threadIdx.x >> 6] = hi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 16; ++i) { lo = min(lo, lo_s[i]); hi = max(hi, hi_s[i]); }
    out[blockIdx.x] = {lo, hi, bad_s};
  }
}

__global__ __launch_bounds__(VS_THREADS) void voxel_sort_kernel(VoxelArgs a) {
  __shared__ int cnt[VS_KEYS];
  __shared__ __attribute__((aligned(16))) unsigned short rec[VS_CHUNK];
  __shared__ int wave_total[VS_THREADS / 64];
  __shared__ long long ends[2][VS_SPANS / 64];
  __shared__ int unsorted_s;
  const int c0 = blockIdx.x * VS_CHUNK, tid = threadIdx.x;
  const int in_chunk = min(VS_CHUNK, a.n - c0);
  // what the chunk's bins come from is requested ahead of the events: behind them it arrives behind them (1e7 events 34 -> 31 us)
  VoxelSpan ext{};
  long long t_end = 0;
  if (!a.by_count) {
    ext = a.span[tid & (VS_SPANS - 1)];
    t_end = a.t[c0 + ((tid & 63) == 0 ? 0 : in_chunk - 1)];
  }
  asm volatile("" ::: "memory");
  int xv[VS_PER], yv[VS_PER], pv[VS_PER];
#pragma unroll
  for (int e = 0; e < VS_PER; ++e) {
    const int i = c0 + min(e * VS_THREADS + tid, in_chunk - 1);
    xv[e] = a.x[i]; yv[e] = a.y[i]; pv[e] = a.p[i];
  }
  long long t0 = 0;
  double span = 1.0;
  const auto bin_at = [&](long long t) {
    const int b = static_cast<int>(static_cast<double>(t - t0) / span * a.bins);
    return b < 0 ? 0 : (b >= a.bins ? a.bins - 1 : b);
  };
  const auto bin_of = [&](int i) { return a.by_count ? static_cast<int>(static_cast<long long>(i) * a.bins / a.n) : bin_at(a.t[i]); };
  bool unsorted = false;
  if (!a.by_count) {
    if (tid == 0) unsorted_s = 0;
    __syncthreads();
    if (tid < VS_SPANS) {
      long long lo = ext.lo, hi = ext.hi;
      if (ext.unsorted) unsorted_s = 1;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        lo = min(lo, static_cast<long long>(__shfl_xor(lo, off, 64)));
        hi = max(hi, static_cast<long long>(__shfl_xor(hi, off, 64)));
      }
      if ((tid & 63) == 0) { ends[0][tid >> 6] = lo; ends[1][tid >> 6] = hi; }
    }
    __syncthreads();
    long long t1 = ends[1][0];
    t0 = ends[0][0];
    for (int i = 1; i < VS_SPANS / 64; ++i) { t0 = min(t0, ends[0][i]); t1 = max(t1, ends[1][i]); }
    span = static_cast<double>(t1 > t0 ? t1 - t0 : 1);
    unsorted = unsorted_s != 0;
  }
  int b0 = 0, b1 = a.bins - 1;
  if (a.by_count) {
    b0 = bin_of(c0);
    b1 = bin_of(c0 + in_chunk - 1);
  } else if (!unsorted) {
    const int b = bin_at(t_end);
    b0 = __builtin_amdgcn_readlane(b, 0);
    b1 = __builtin_amdgcn_readlane(b, 63);
  }
  const int keys = (b1 - b0 + 1) * a.bands, rows = 1 << a.log_rows;
  for (int k = tid; k < keys; k += VS_THREADS) cnt[k] = 0;
  __syncthreads();
  unsigned int item[VS_PER];                       // key << 16 | place; all ones: outside the image
  unsigned short rank[VS_PER];
#pragma unroll
  for (int e = 0; e < VS_PER; ++e) {
    const int j = e * VS_THREADS + tid;
    item[e] = 0xffffffffu;
    rank[e] = 0;
    if (j >= in_chunk || xv[e] < 0 || xv[e] >= a.W || yv[e] < 0 || yv[e] >= a.H) continue;
    const int key = (b0 == b1 ? 0 : bin_of(c0 + j) - b0) * a.bands + (yv[e] >> a.log_rows);
    const int place = ((pv[e] != 0 ? rows : 0) + (yv[e] & (rows - 1))) * a.W + xv[e];
    item[e] = static_cast<unsigned int>(key) << 16 | place;
    rank[e] = static_cast<unsigned short>(atomicAdd(&cnt[key], 1));
  }
  __syncthreads();
  // exclusive scan of the counts, VS_KEYS / VS_THREADS of them a thread
  constexpr int KT = VS_KEYS / VS_THREADS;
  int mine[KT], sum = 0;
#pragma unroll
  for (int k = 0; k < KT; ++k) {
    mine[k] = sum;
    sum += tid * KT + k < keys ? cnt[tid * KT + k] : 0;
  }
  int scan = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(scan, off, 64);
    if ((tid & 63) >= off) scan += v;
  }
  if ((tid & 63) == 63) wave_total[tid >> 6] = scan;
  __syncthreads();
  int before = scan - sum;
  for (int w = 0; w < (tid >> 6); ++w) before += wave_total[w];
  int total = 0;
  for (int w = 0; w < VS_THREADS / 64; ++w) total += wave_total[w];
  unsigned short* off = a.off + static_cast<size_t>(blockIdx.x) * (a.keys + 1);
#pragma unroll
  for (int k = 0; k < KT; ++k)
    if (tid * KT + k < keys) {
      cnt[tid * KT + k] = before + mine[k];
      off[tid * KT + k] = static_cast<unsigned short>(before + mine[k]);
    }
  if (tid == 0) {
    off[keys] = static_cast<unsigned short>(total);
    a.range[blockIdx.x] = make_int2(b0, b1);
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < VS_PER; ++e)
    if (item[e] != 0xffffffffu) rec[cnt[item[e] >> 16] + rank[e]] = static_cast<unsigned short>(item[e]);
  __syncthreads();
  u32x4_t* dst = reinterpret_cast<u32x4_t*>(a.rec + static_cast<size_t>(blockIdx.x) * VS_CHUNK);
  const u32x4_t* src = reinterpret_cast<const u32x4_t*>(rec);
  for (int i = tid; i * 8 < total; i += VS_THREADS) dst[i] = src[i];      // (the tail past `total` is never read)
}

// Every wave takes its own share of the chunks, a lane a chunk and neighbouring chunks in different waves (a bin of a sorted stream is a
// range of chunks), and has eight runs on their way, two records a load, before it counts the first: a run is some 70 records, and one
// after another they were as many round trips (1e7 events, four recordings: 28.7, 23.5, 28.5, 24.8 -> 25.1, 20.5, 24.0, 21.5 us; 5e6 events, one bin of 203 x 301: 34 -> 32).  What is left is the LDS adds, half
// of their lanes empty; runs filled up to 16 bytes, a lane a piece of one, took 2 us less here and cost the sort more.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void voxel_count_kernel(VoxelArgs a, int* __restrict__ out_hist, float* __restrict__ out_vox,
                                                              int signed_mode) {
  constexpr int WAVES = THREADS / 64, PASSES = 4, RUNS = 8;
  extern __shared__ __attribute__((aligned(16))) int cnt[];                     // [2][rows][W]
  const int band = blockIdx.x, b = blockIdx.y, rows = 1 << a.log_rows, tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = rows * a.W;
  for (int i = tid; i < 2 * half; i += THREADS) cnt[i] = 0;
  __syncthreads();
  const auto count = [&](unsigned int two, int at, int from, int to) {          // records `at`, `at` + 1 of a run that is from .. to
    if (at >= from && at < to) atomicAdd(&cnt[two & 0xffff], 1);
    if (at + 1 < to) atomicAdd(&cnt[two >> 16], 1);
  };
  const unsigned int* words = reinterpret_cast<const unsigned int*>(a.rec);
  for (int base = 0; base < a.chunks; base += THREADS * PASSES) {
    int start[PASSES], len[PASSES];
    int2 r[PASSES];
#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
      const int c = base + s * THREADS + lane * WAVES + wid;
      r[s] = c < a.chunks ? a.range[c] : make_int2(1, 0);
    }
#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
      const int c = base + s * THREADS + lane * WAVES + wid;
      start[s] = len[s] = 0;
      if (r[s].x <= b && b <= r[s].y) {
        const unsigned short* off = a.off + static_cast<size_t>(c) * (a.keys + 1) + (b - r[s].x) * a.bands + band;
        start[s] = off[0];
        len[s] = off[1];
      }
    }
#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
      len[s] -= start[s];
      start[s] = len[s] > 0 ? start[s] + (base + s * THREADS + lane * WAVES + wid) * VS_CHUNK : 0;      // (below 2^31: the events are)
    }
#pragma unroll 1
    for (int s = 0; s < PASSES; ++s) {
      const int at_s = s == 0 ? start[0] : s == 1 ? start[1] : s == 2 ? start[2] : start[3];
      const int len_s = s == 0 ? len[0] : s == 1 ? len[1] : s == 2 ? len[2] : len[3];
      unsigned long long todo = __builtin_amdgcn_ballot_w64(len_s > 0);
      while (todo) {
        int first[RUNS], odd[RUNS], end[RUNS];                                  // first word; the run among the words' records
        unsigned int v[RUNS][2];
#pragma unroll
        for (int u = 0; u < RUNS; ++u) {                                        // (lanes past the run, and runs past the last, read a word twice)
          const int l = __builtin_ctzll(todo | 1ull << 63);
          const int at = __builtin_amdgcn_readlane(at_s, l), n = todo ? __builtin_amdgcn_readlane(len_s, l) : 0;
          todo &= todo - 1;
          first[u] = at >> 1;
          odd[u] = at & 1;
          end[u] = odd[u] + n;
          const int last = max(end[u] - 1, 0) >> 1;
          v[u][0] = words[first[u] + min(lane, last)];
          v[u][1] = words[first[u] + min(64 + lane, last)];
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int u = 0; u < RUNS; ++u) {
          count(v[u][0], lane * 2, odd[u], end[u]);
          if (end[u] > 128) count(v[u][1], 128 + lane * 2, odd[u], end[u]);
          for (int i = 256 + lane * 2; i < end[u]; i += 512) {                  // four loads of a long run in flight
            unsigned int w[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) w[q] = words[first[u] + (min(i + q * 128, end[u] - 1) >> 1)];
#pragma unroll
            for (int q = 0; q < 4; ++q) count(w[q], i + q * 128, odd[u], end[u]);
          }
        }
      }
    }
  }
  __syncthreads();
  const int y0 = band << a.log_rows, cells = min(rows, a.H - y0) * a.W;
  const size_t plane = static_cast<size_t>(a.H) * a.W, at = static_cast<size_t>(y0) * a.W;
  int* hist = out_hist + static_cast<size_t>(b) * 2 * plane + at;
  float* vox = out_vox + static_cast<size_t>(b) * plane + at;
  if ((a.W & 3) == 0) {                            // (the outputs start on 16 bytes: they are allocated with the call)
    for (int i = tid * 4; i < cells; i += THREADS * 4) {
      const i32x4_t neg = *reinterpret_cast<const i32x4_t*>(cnt + i), pos = *reinterpret_cast<const i32x4_t*>(cnt + half + i);
      *reinterpret_cast<i32x4_t*>(hist + i) = neg;
      *reinterpret_cast<i32x4_t*>(hist + plane + i) = pos;
      f32x4_t v;
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = static_cast<float>(signed_mode ? pos[k] - neg[k] : pos[k] + neg[k]);
      *reinterpret_cast<f32x4_t*>(vox + i) = v;
    }
    return;
  }
  for (int i = tid; i < cells; i += THREADS) {
    const int neg = cnt[i], pos = cnt[half + i];
    hist[i] = neg;
    hist[plane + i] = pos;
    vox[i] = static_cast<float>(signed_mode ? pos - neg : pos + neg);
  }
}

// log2 of the rows of a band: as many as fill 48 KB of counters, fewer while there are not two blocks per CU; -1 where
// the image is too wide for a 16-bit place or the keys too many for the sort's counters
int event_voxel_log_rows(int bins, int H, int W) {
  if (W > 19200) return -1;
  int l = 0;
  while ((2ll << l) < H && (2ll << (l + 1)) * W * 4 <= 48 * 1024) ++l;
  const auto blocks = [&](int k) { return static_cast<long long>(bins) * ((H + (1 << k) - 1) >> k); };
  while (l > 0 && blocks(l) < 512 && blocks(l - 1) <= VS_KEYS) --l;
  return blocks(l) <= VS_KEYS ? l : -1;
}

EventVoxelPlan event_voxel_plan(int n, int bins, int H, int W) {
  EventVoxelPlan plan;
  plan.log_rows = event_voxel_log_rows(bins, H, W);
  plan.bands = plan.log_rows < 0 ? 0 : (H + (1 << plan.log_rows) - 1) >> plan.log_rows;
  plan.chunks = static_cast<int>((static_cast<long long>(n) + VS_CHUNK - 1) / VS_CHUNK);
  plan.off_bytes = 0;
  plan.range_bytes = static_cast<size_t>(plan.chunks) * sizeof(int2);
  plan.span_bytes = VS_SPANS * sizeof(VoxelSpan);
  plan.rec_bytes = static_cast<size_t>(plan.chunks) * VS_CHUNK * 2;
  plan.off_bytes = static_cast<size_t>(plan.chunks) * (bins * plan.bands + 1) * 2;
  return plan;
}

void launch_event_voxel_sorted(const int* x, const int* y, const int* p, const long long* t, int n, int bins, int H, int W,
                               const EventVoxelPlan& plan, unsigned char* work, int* out_hist, float* out_vox, int signed_mode,
                               int by_count, hipStream_t st) {
  VoxelArgs a;
  a.x = x; a.y = y; a.p = p; a.t = t;
  // records first: every chunk of them starts on 16 bytes
  a.rec = reinterpret_cast<unsigned short*>(work);
  VoxelSpan* span = reinterpret_cast<VoxelSpan*>(work + plan.rec_bytes);
  a.span = span;
  a.range = reinterpret_cast<int2*>(work + plan.rec_bytes + plan.span_bytes);
  a.off = reinterpret_cast<unsigned short*>(work + plan.rec_bytes + plan.span_bytes + plan.range_bytes);
  a.n = n; a.bins = bins; a.H = H; a.W = W; a.log_rows = plan.log_rows; a.bands = plan.bands; a.keys = bins * plan.bands;
  a.chunks = plan.chunks; a.by_count = by_count;
  if (!by_count) hipLaunchKernelGGL(voxel_span_kernel, dim3(VS_SPANS), dim3(1024), 0, st, t, n, span);
  hipLaunchKernelGGL(voxel_sort_kernel, dim3(plan.chunks), dim3(VS_THREADS), 0, st, a);
  const size_t smem = static_cast<size_t>(2) * (1 << plan.log_rows) * W * sizeof(int);
  const auto count = [&](auto threads) {
    constexpr int T = decltype(threads)::value;
    static bool attr_set = false;                       // (one a number of threads: the kernels' types are the same)
    if (!attr_set) {
      hipFuncSetAttribute(reinterpret_cast<const void*>(&voxel_count_kernel<T>), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);  // (W = 19 200)
      attr_set = true;
    }
    hipLaunchKernelGGL(voxel_count_kernel<T>, dim3(plan.bands, bins), dim3(T), smem, st, a, out_hist, out_vox, signed_mode);
  };
  // two blocks a CU and more of few events each: half as many threads, so that all are resident at once (600 blocks, 1e6 events 31.4 ->
  // 28.6 us, 2.4e6 40.2 -> 38.8); with more the block of the busiest band is
  // waited for, and its waves count (1e7 77.7 with 512 threads, 75.6 with 1 024; 4.3e6 0.98 to 1.03 of the time with 512)
  if (plan.bands * bins >= 512 && n / (plan.bands * bins) < 5000) count(std::integral_constant<int, 512>{});
  else count(std::integral_constant<int, 1024>{});
}

// --------------------------------------------------------- CLIP preprocessing
// img: [T][H][W][3] uint8.  Two-pass fixed-point resample identical to PIL's
// (horizontal pass with uint8 rounding, then vertical), restricted to the
// centre-crop window, then (v/255 - mean)/std -> bf16 [T][3][S][S].
// Tables (int32): start/count per output coordinate, weights [out][ksize] with
// 22 fractional bits.  One thread per output pixel; the source frame is
// L2-resident (0.9 MB), each thread touches ksize_v x ksize_h pixels.
struct PreprocParams {
  const unsigned char* img; bf16_t* out;
  const int* hstart; const int* hcount; const int* hweight;
  const int* vstart; const int* vcount; const int* vweight;
  int T, H, W, S, top, left, ksh, ksv, resize_h, resize_w;
  float mean[3], inv_std[3];
};

__device__ __forceinline__ int clip8_fix(long long acc) {
  const long long v = acc >> 22;
  return v < 0 ? 0 : (v > 255 ? 255 : static_cast<int>(v));
}

__global__ __launch_bounds__(256) void clip_preproc_kernel(PreprocParams p) {
  const long long total = static_cast<long long>(p.T) * p.S * p.S;
  const long long half = 1ll << 21;
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < total; i += gridDim.x * 256ll) {
    const int ox = static_cast<int>(i % p.S);
    const int oy = static_cast<int>((i / p.S) % p.S);
    const int t = static_cast<int>(i / (static_cast<long long>(p.S) * p.S));
    const int rx = ox + p.left, ry = oy + p.top;  // coordinates in the resized image
    const unsigned char* frame = p.img + static_cast<size_t>(t) * p.H * p.W * 3;
    int px[3];
    const bool need_h = p.resize_w != p.W, need_v = p.resize_h != p.H;
    const int hs = need_h ? p.hstart[rx] : rx, hc = need_h ? p.hcount[rx] : 1;
    const int vs = need_v ? p.vstart[ry] : ry, vc = need_v ? p.vcount[ry] : 1;
    long long vacc[3] = {half, half, half};
    for (int j = 0; j < vc; ++j) {
      const unsigned char* row = frame + static_cast<size_t>(vs + j) * p.W * 3;
      int hval[3];
      if (need_h) {
        long long hacc[3] = {half, half, half};
        for (int k = 0; k < hc; ++k) {
          const long long w = p.hweight[rx * p.ksh + k];
          const unsigned char* s = row + (hs + k) * 3;
          hacc[0] += w * s[0]; hacc[1] += w * s[1]; hacc[2] += w * s[2];
        }
        hval[0] = clip8_fix(hacc[0]); hval[1] = clip8_fix(hacc[1]); hval[2] = clip8_fix(hacc[2]);
      } else {
        const unsigned char* s = row + hs * 3;
        hval[0] = s[0]; hval[1] = s[1]; hval[2] = s[2];
      }
      if (need_v) {
        const long long w = p.vweight[ry * p.ksv + j];
        vacc[0] += w * hval[0]; vacc[1] += w * hval[1]; vacc[2] += w * hval[2];
      } else {
        px[0] = hval[0]; px[1] = hval[1]; px[2] = hval[2];
      }
    }
    if (need_v) { px[0] = clip8_fix(vacc[0]); px[1] = clip8_fix(vacc[1]); px[2] = clip8_fix(vacc[2]); }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float v = (static_cast<float>(px[c]) * (1.f / 255.f) - p.mean[c]) * p.inv_std[c];
      p.out[((static_cast<size_t>(t) * 3 + c) * p.S + oy) * p.S + ox] = f32_to_bf16(v);
    }
  }
}

// The same pixels in two passes over a tile of CP_ROWS x CP_COLS outputs: the source rows it needs are resized horizontally
// into LDS (one word a pixel), then vertically.  A pixel costs its horizontal taps once instead of once per vertical tap, and
// the sums fit 32 bits: weights of 22 fractional bits sum to one with magnitudes below 1.5, times 255.  Bound by that integer
// work: five frames of 160 x 120 to 336 x 336 9.9 us, 17.7 one pixel at a time in 64 bits; of
// 640 x 480 20.0 and 39.3.  Tiles of four rows where eight would leave CUs idle: one frame of 640 x 480 9.7, with eight 13.4, by
// pixels 11.1.
// CODES: the source is one code a pixel (event_codes_kernel) instead of three bytes.
// Tables whose rows reach over more than CP_SRC source rows (no resize's do) are followed without the first pass: a block
// then resizes each tap's row where it needs it.
constexpr int CP_COLS = 112, CP_SRC = 48;

__device__ __forceinline__ int clip8_fix32(int acc) { return min(max(acc >> 22, 0), 255); }

template <bool CODES, int CP_ROWS>
__global__ __launch_bounds__(256) void clip_preproc_tile_kernel(PreprocParams p) {
  __shared__ unsigned int mid[CP_SRC][CP_COLS];
  const int ox0 = blockIdx.x * CP_COLS, oy0 = blockIdx.y * CP_ROWS, t = blockIdx.z;
  const int cols = min(CP_COLS, p.S - ox0), rows = min(CP_ROWS, p.S - oy0);
  const bool need_h = p.resize_w != p.W, need_v = p.resize_h != p.H;
  const int first = oy0 + p.top, last = first + rows - 1;      // rows of the resized image
  int r0 = first, r1 = last + 1;                               // source rows; a lane looks at one row of the tile
  if (need_v) {
    const int mine = first + min(static_cast<int>(threadIdx.x) & 7, rows - 1);
    r0 = p.vstart[mine];
    r1 = r0 + p.vcount[mine];
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
      r0 = min(r0, __shfl_xor(r0, off, 64));
      r1 = max(r1, __shfl_xor(r1, off, 64));
    }
    r0 = __builtin_amdgcn_readfirstlane(r0);
    r1 = __builtin_amdgcn_readfirstlane(r1);
  }
  const int n_src = r1 - r0;
  const bool tall = n_src > CP_SRC;                            // (the same for the whole block)
  const unsigned char* frame = p.img + static_cast<size_t>(t) * p.H * p.W * (CODES ? 1 : 3);
  constexpr int half = 1 << 21;
  // column c of source row r0 + r, resized horizontally: one byte a channel
  const auto resized = [&](int r, int c) -> unsigned int {
    const int rx = ox0 + c + p.left, hs = need_h ? p.hstart[rx] : rx, hc = need_h ? p.hcount[rx] : 1;
    const unsigned char* src = frame + (static_cast<size_t>(r0 + r) * p.W + hs) * (CODES ? 1 : 3);
    int v[3] = {half, half, half};
    const int* w = p.hweight + rx * p.ksh;
    for (int k = 0; k < hc; ++k) {
      int px[3];
      if constexpr (CODES) {
        const int code = src[k];                   // white, red or blue
        px[0] = code == 2 ? 0 : 255; px[1] = code ? 0 : 255; px[2] = code == 1 ? 0 : 255;
      } else {
        px[0] = src[k * 3]; px[1] = src[k * 3 + 1]; px[2] = src[k * 3 + 2];
      }
      const int wk = need_h ? w[k] : 0;
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) v[ch] = need_h ? v[ch] + wk * px[ch] : px[ch];
    }
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) v[ch] = need_h ? clip8_fix32(v[ch]) : v[ch];
    return v[0] | v[1] << 8 | v[2] << 16;
  };
  // the outputs, from rows that `row(r, c)` gives
  const auto finish = [&](auto&& row) {
    for (int i = threadIdx.x; i < rows * CP_COLS; i += 256) {
      const int r = i / CP_COLS, c = i % CP_COLS;
      if (c >= cols) continue;
      const int ry = first + r, vs = (need_v ? p.vstart[ry] : ry) - r0;
      int px[3];
      if (need_v) {
        const int vc = p.vcount[ry];
        const int* w = p.vweight + ry * p.ksv;
        int v[3] = {half, half, half};
        for (int k = 0; k < vc; ++k) {
          const unsigned int m = row(vs + k, c);
          const int wk = w[k];
          v[0] += wk * static_cast<int>(m & 255); v[1] += wk * static_cast<int>(m >> 8 & 255); v[2] += wk * static_cast<int>(m >> 16);
        }
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) px[ch] = clip8_fix32(v[ch]);
      } else {
        const unsigned int m = row(vs, c);
        px[0] = m & 255; px[1] = m >> 8 & 255; px[2] = m >> 16;
      }
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) {
        const float v = (static_cast<float>(px[ch]) * (1.f / 255.f) - p.mean[ch]) * p.inv_std[ch];
        p.out[((static_cast<size_t>(t) * 3 + ch) * p.S + oy0 + r) * p.S + ox0 + c] = f32_to_bf16(v);
      }
    }
  };
  if (tall) {
    finish(resized);
    return;
  }
  for (int i = threadIdx.x; i < n_src * CP_COLS; i += 256) {
    const int r = i / CP_COLS, c = i % CP_COLS;
    if (c < cols) mid[r][c] = resized(r, c);
  }
  __syncthreads();
  finish([&](int r, int c) { return mid[r][c]; });
}

// source rows of a tile fit its LDS (a resize by less than about four)
bool clip_preproc_tiles_ok(int T, int H, int resize_h, int ksv) {
  const long long src = (7ll * H + resize_h - 1) / resize_h + ksv + 1;
  return src <= CP_SRC && T <= 65535;
}

void launch_clip_preproc(const unsigned char* img, bf16_t* out, const int* hstart,
                         const int* hcount, const int* hweight, const int* vstart,
                         const int* vcount, const int* vweight, int T, int H, int W, int S,
                         int resize_h, int resize_w, int top, int left, int ksh, int ksv,
                         const float* mean, const float* stdv, bool codes, hipStream_t st) {
  PreprocParams p;
  p.img = img; p.out = out; p.hstart = hstart; p.hcount = hcount; p.hweight = hweight;
  p.vstart = vstart; p.vcount = vcount; p.vweight = vweight;
  p.T = T; p.H = H; p.W = W; p.S = S; p.top = top; p.left = left; p.ksh = ksh; p.ksv = ksv;
  p.resize_h = resize_h; p.resize_w = resize_w;
  for (int c = 0; c < 3; ++c) { p.mean[c] = mean[c]; p.inv_std[c] = 1.f / stdv[c]; }
  // Outputs worth 160 full tiles of four rows take tiles, of eight rows from 256 full ones of those on; fewer pixels go one by one:
  // us by tiles / pixels, 112 x 112 from 336 x 336, five frames 23.8 / 22.4, eight 24.2 / 35.7; one frame of 224 x 224 from 720 x
  // 1280 27.0 / 24.7, two 27.3 / 40.3.  Thumbnails, of which a frame is a few blocks either way, share their taps' rows: 28 x 28 from
  // 90 x 120 20.7 / 27.1, 56 x 56 11.2 / 10.2.  (Codes are always in tiles.)
  const long long pixels = static_cast<long long>(T) * S * S;
  if (clip_preproc_tiles_ok(T, H, resize_h, ksv) && (codes || S <= 32 || pixels >= 160 * 4 * CP_COLS)) {
    const int cols = (S + CP_COLS - 1) / CP_COLS;
    if (pixels >= 256 * 8 * CP_COLS) {
      const dim3 grid(cols, (S + 7) / 8, T);
      if (codes) hipLaunchKernelGGL((clip_preproc_tile_kernel<true, 8>), grid, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((clip_preproc_tile_kernel<false, 8>), grid, dim3(256), 0, st, p);
    } else {
      const dim3 grid(cols, (S + 3) / 4, T);
      if (codes) hipLaunchKernelGGL((clip_preproc_tile_kernel<true, 4>), grid, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((clip_preproc_tile_kernel<false, 4>), grid, dim3(256), 0, st, p);
    }
    return;
  }
  const long long total = static_cast<long long>(T) * S * S;
  int blocks = static_cast<int>((total + 255) / 256);
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(clip_preproc_kernel, dim3(blocks), dim3(256), 0, st, p);
}

}  // namespace evgpt
