// bf16 GEMM over K-contiguous operands whose tiles are at most one round: eight waves and a deep ring, one workgroup per CU.
//
// A few hundred rows into a few thousand columns are fewer tiles than the CUs hold, and each of them is a serial chain of K-tiles whose
// staging loads come from memory.  The tiles of gemm.hip keep two K-tiles in flight and read a K-tile's operands from LDS only when its
// barrier has passed.  Here a workgroup has a CU's LDS to itself: three or four K-tiles are in flight, a wave reads its operands 32 k ahead
// of the products, and there is one barrier a K-tile.  us, weights from memory, the choice of gemm.hip -> this: 577 x 3072 x 1024 13.6 ->
// 10.3, 577 x 4096 x 1024 with quick-gelu 17.9 -> 13.9, 577 x 1024 x 4096 as three slabs 14.4 -> 11.9, 1154 x 3072 x 1024 19.9 -> 15.0,
// 300 x 4096 x 4096 35.6 -> 25.2, 2308 x 1024 x 1024 18.8 -> 12.2.  What is left is the operands' way into the CU (64 bytes a clock: 3 us of
// the first) and the launch.  Four waves: 13.2 instead of 10.6; three stages instead of five, two workgroups a CU: 15.7; six: level.
#include <type_traits>

#include "gemm_epilogue.h"
#include "gemm_ring.h"

namespace evgpt {

namespace {

template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

__device__ __forceinline__ void load_to_lds16(const unsigned char* src, int bytes, unsigned char* lds, int voff, int soff) {
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(src), 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)lds, 16, voff, soff, 0, 0);
}

// WGM x WGN waves, each TM x TN tiles of 16 x 16; S K-tiles of 64 in the ring
template <int TM, int TN, int WGM, int WGN, int S, int ACT>
__global__ __launch_bounds__(512) void gemm_ring_kernel(EVGPT_GEMM_ARGS) {
  EVGPT_GEMM_TAKE;
  constexpr int NW = WGM * WGN, WM = TM * 16, WN = TN * 16, BM = WM * WGM, BN = WN * WGN, A_BYTES = BM * 128, STAGE = (BM + BN) * 128;
  constexpr int IA = BM / (8 * NW), IW = BN / (8 * NW), G = IA + IW;           // staging instructions per wave and K-tile
  static_assert(NW == 8 && IA * 64 == BM && IW * 64 == BN && S >= 3, "eight waves stage whole groups of eight rows");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wid / WGN, wc = wid % WGN;
  const int bn_out = p.glu_half ? BN / 2 : BN;
  const int tiles_n = (p.N + bn_out - 1) / bn_out, tiles_m = (p.M + BM - 1) / BM, tiles = tiles_m * tiles_n;
  int tile = xcd_remap(blockIdx.x, tiles * p.splitk), ksplit = 0;
  if (p.splitk > 1) {                         // (an XCD inside one K range)
    ksplit = tile / tiles;
    tile -= ksplit * tiles;
  }
  // An XCD's tiles are consecutive ones.  They share the panels of the larger operand, so that it is read once into some L2 and the smaller
  // one into each (4 052 x 464 x 4480 by columns of tiles 44.2 us, the general tiles 31.6; by rows 4 011 x 496 x 4352 26.2 and 32.6).
  const bool tall = (p.glu_half ? p.M / 2 : p.M) > p.N;
  const int slow = tile / (tall ? tiles_n : tiles_m), fast = tile - slow * (tall ? tiles_n : tiles_m);
  const int tn = tall ? fast : slow, m0 = (tall ? slow : fast) * BM, n0 = tn * bn_out;
  const int k_begin = ksplit * p.k_per_split, nk = min(p.k_per_split, p.K - k_begin) / BK;

  int va[IA], vw[IW];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int r = (wid * IA + i) * 8 + (lane >> 3);
    va[i] = r * p.lda * 2 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < IW; ++i) {
    const int r = (wid * IW + i) * 8 + (lane >> 3);
    int src = r;
    if (p.glu_half) {      // a wave column's rows: first half gate, second half the matching up rows
      const int col = r / WN, within = r % WN;
      src = col * (WN / 2) + within + (within >= WN / 2 ? p.glu_half - WN / 2 : 0);
    }
    vw[i] = src * p.ldw * 2 + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
  }
  const unsigned char* A = reinterpret_cast<const unsigned char*>(p.A + static_cast<long long>(m0) * p.lda + k_begin);
  const unsigned char* W = reinterpret_cast<const unsigned char*>(p.W + static_cast<long long>(n0) * p.ldw + k_begin);
  // (rows past the operands' lie past the descriptors' ranges and arrive as zeros)
  const int bytes_a = (min(p.M - m0, BM) * p.lda - k_begin) * 2;
  const int bytes_w = ((p.glu_half ? 2 * p.glu_half - n0 : min(p.N - n0, BN)) * p.ldw - k_begin) * 2;
  int next = 0, into = 0;                     // K-tile staged next and the stage it goes to
  // Past the last one zero fills that nobody reads keep the counts uniform: an empty range, and with it no offset, so that range minus
  // offset is empty too.
  auto stage = [&]() {
    const int la = next < nk ? bytes_a : 0, lw = next < nk ? bytes_w : 0, off = next < nk ? next * (BK * 2) : 0;
    unsigned char* d = smem + into;
#pragma unroll
    for (int i = 0; i < IW; ++i) load_to_lds16(W, lw, d + A_BYTES + (wid * IW + i) * 1024, vw[i], off);
#pragma unroll
    for (int i = 0; i < IA; ++i) load_to_lds16(A, la, d + (wid * IA + i) * 1024, va[i], off);
    ++next;
    into = into == (S - 1) * STAGE ? 0 : into + STAGE;
  };

  const int frow = lane & 15, fq = lane >> 4, fsw = (frow >> 1) & 7;
  int ra[2], rw[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = ((h * 4 + fq) ^ fsw) << 4;
    ra[h] = (wr * WM + frow) * 128 + c;
    rw[h] = A_BYTES + (wc * WN + frow) * 128 + c;
  }
  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  bf16x8_t fa[2][TM], fw[2][TN];
  auto read = [&](auto hc, int st) {
    constexpr int h = decltype(hc)::value;
#pragma unroll
    for (int j = 0; j < TN; ++j) fw[h][j] = *reinterpret_cast<const bf16x8_t*>(smem + st + rw[h] + j * 2048);
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[h][i] = *reinterpret_cast<const bf16x8_t*>(smem + st + ra[h] + i * 2048);
  };
  auto multiply = [&](auto hc) {
    constexpr int h = decltype(hc)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[h][j], fa[h][i], acc[i][j], 0, 0, 0);
  };
  const std::integral_constant<int, 0> lower;
  const std::integral_constant<int, 1> upper;
#pragma unroll
  for (int s = 0; s < S - 1; ++s) stage();
  wait_loads<(S - 2) * G>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int st = 0;
  read(lower, st);
  for (int t = 0; t < nk; ++t) {
    read(upper, st);
    __builtin_amdgcn_sched_barrier(0);
    multiply(lower);
    __builtin_amdgcn_sched_barrier(0);
    // behind the barrier K-tile t + 1 has landed for every wave, and every wave has K-tile t - 1, whose stage is written next, in
    // registers (it multiplied its upper half before)
    wait_loads<(S - 3) * G>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    st = st == (S - 1) * STAGE ? 0 : st + STAGE;
    read(lower, st);
    __builtin_amdgcn_sched_barrier(0);
    stage();
    __builtin_amdgcn_sched_barrier(0);
    multiply(upper);
    __builtin_amdgcn_sched_barrier(0);
  }
  wait_loads<0>();
  gemm_epilogue<TM, TN, WM, WN, WGN, ACT>(p, acc, m0, n0, wr, wc, tn, tiles_n, ksplit, lane);
}

template <int TM, int TN, int WGM, int WGN, int S, int ACT>
void launch_act(const GemmParams& p, hipStream_t st) {
  constexpr int BM = TM * 16 * WGM, BN = TN * 16 * WGN, lds = S * (BM + BN) * 128;
  static const bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_ring_kernel<TM, TN, WGM, WGN, S, ACT>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
  (void)attr;
  const int bn_out = p.glu_half ? BN / 2 : BN;
  const int tiles = (p.M + BM - 1) / BM * ((p.N + bn_out - 1) / bn_out) * p.splitk;
  hipLaunchKernelGGL((gemm_ring_kernel<TM, TN, WGM, WGN, S, ACT>), dim3(tiles), dim3(512), lds, st, EVGPT_GEMM_PASS(p));
}
template <int TM, int TN, int WGM, int WGN, int S>
void launch(const GemmParams& p, hipStream_t st) {
  const int act = p.splitk > 1 || p.raw_partial ? ACT_NONE : p.act;       // (slabs: their consumer's)
  if (act == ACT_GELU) launch_act<TM, TN, WGM, WGN, S, ACT_GELU>(p, st);
  else if (act == ACT_QUICK_GELU) launch_act<TM, TN, WGM, WGN, S, ACT_QUICK_GELU>(p, st);
  else launch_act<TM, TN, WGM, WGN, S, ACT_NONE>(p, st);
}

}  // namespace

// The smallest tile that is one round: a CU's time goes with its tile's area (64 x 128 / 64 x 192 / 128 x 128 with 1024 k 10.7 / 13.7 /
// 15 us), and 128 x 64 reads the weights half as often as 64 x 128.  Against the tiles of gemm.hip over 22 900 products of 33 to 4 200
// rows, 64 to 16 384 columns and 64 to 12 288 k, each timed as both: 0.85 of their time at the mean where this rule takes them, same bits.
// The lines, this / the other choice:
//  * 64 x 64 from 128 tiles on; not with split K (64 x 1024 x 11008 in eight 12.4 / 10.3 us); under 256 rows up to 1024 k (160 x 3072 x
//    2048 14.5 / 12.3, x 1024 7.0 / 7.5)
//  * longer than 4096 k: not 160 tiles of 128 x 64 (636 x 2048 x 5632 39.4 / 36.2; 1000 x 2048, 256 tiles, ahead), not 64 x 192 (636 x
//    4096 x 5632 53.8 / 51.6; x 1024 ahead by 20 %)
//  * 128 x 64 over 512 k: from 200 rows on (160 x 5632 6.8 / 6.3)
//  * 128 x 128: up to 240 tiles (4039 x 1024, 256 of them, 25.8 / 24.8); gated with under 1024 rows from 170 tiles on (636 x 4096 x 4096,
//    160, 39.7 / 37.5; 400 x 5632 x 4096, 176, 35.4 / 48.1)
//  * short contractions, where filling the ring is what there is, by what the epilogue adds to both (this over the other at the mean):
//    64 x 64 plain 1.04 at 64 k under 600 rows, 0.95 over 1000, 0.93 at 192; a bias 0.97 and 0.92; a residual 1.05 to 1.13 up to 192 k
//    below 152 tiles, 0.96 above.  128 x 64 where the other choice is 64 x 64: plain 1.06 at 64, 0.96 at 320 (fp32 and slabs 1.0), a
//    residual 1.05 and 0.98, with a bias or activation ahead at any length.  Where it is 32 x 64 (under 300 tiles of 64 x 64): a bias
//    1.11 at 64, 1.0 at 512, quick-gelu 1.04 and 0.92, gelu 1.1 and 1.0, a residual 1.27, 1.09 and at 2048 0.96.
//    128 x 128: 1.0 to 1.1 up to 320 k, gated 1.02 at 128 and 0.98 at 192
//  * the eight waves of the 64 x 128 tile (`w8`), which share a CU with two other workgroups, take a bias or an activation sooner than
//    128 x 128 here (1.08 to 1.14), quick-gelu up to 192 k than 64 x 192 (1.1)
RingTile gemm_ring_tile(const GemmParams& p, bool w8) {
  const long long lim = 1ll << 31;
  if (p.act != ACT_NONE && p.act != ACT_GELU && p.act != ACT_QUICK_GELU) return RING_NONE;
  if (p.M <= 32 || p.k_cols || p.amax_val || p.rope_cos || p.grp_start) return RING_NONE;
  if (2ll * 128 * p.lda >= lim || 2ll * (p.glu_half ? 2ll * p.glu_half : 192) * p.ldw >= lim) return RING_NONE;
  auto tiles = [&](int bm, int bn) {
    const int out = p.glu_half ? bn / 2 : bn;
    return static_cast<long long>((p.M + bm - 1) / bm) * ((p.N + out - 1) / out) * p.splitk;
  };
  const bool gated = p.glu_half != 0, slabs = p.splitk > 1 || p.raw_partial;
  const bool act = !slabs && p.act != ACT_NONE, bias = !slabs && p.bias, res = !slabs && p.res;
  // longer than what the epilogue asks for
  auto longer = [&](int residual, int activation, int with_bias, int plain) {
    return p.k_per_split > (res ? residual : act ? activation : bias ? with_bias : plain);
  };
  const long long t64 = tiles(64, 64);
  if (t64 <= 256 && !gated) {
    if (t64 < 128 || p.splitk > 1 || (p.M < 256 && p.K > 1024)) return RING_NONE;
    return longer(t64 < 152 ? 512 : 192, 0, 128, 128) || (p.M > 600 && !res) ? RING_64x64 : RING_NONE;
  }
  for (const RingTile r : {RING_128x64, RING_64x128}) {
    const long long t = r == RING_128x64 ? tiles(128, 64) : tiles(64, 128);
    if (t > 256) continue;
    if (t < (p.K > 4096 && !gated ? 170 : 32) || (p.K <= 512 && p.M < 200 && !gated)) return RING_NONE;
    if (gated) return r;
    const int sums = p.Cf || slabs ? 320 : 192;
    return (t64 < 300 ? longer(2048, p.act == ACT_GELU ? 1024 : 512, 512, 512) : longer(320, 0, 0, sums)) ? r : RING_NONE;
  }
  if (!gated && tiles(64, 192) <= 256)
    return p.K <= 4096 && !(w8 && p.act == ACT_QUICK_GELU && p.K <= 192) ? RING_64x192 : RING_NONE;
  const long long t = tiles(128, 128);
  if (t > 240 || (gated && t < 170 && p.M < 1024) || (w8 && (act || bias))) return RING_NONE;
  return p.k_per_split > (gated ? 128 : 320) ? RING_128x128 : RING_NONE;
}

void launch_gemm_ring(const GemmParams& p, RingTile tile, hipStream_t st) {
  switch (tile) {
    case RING_64x64: launch<2, 1, 2, 4, 4>(p, st); break;
    case RING_128x64: launch<2, 2, 4, 2, 5>(p, st); break;
    case RING_64x128: launch<2, 2, 2, 4, 5>(p, st); break;
    case RING_64x192: launch<2, 3, 2, 4, 4>(p, st); break;
    default: launch<4, 2, 2, 4, 4>(p, st); break;
  }
}

}  // namespace evgpt
