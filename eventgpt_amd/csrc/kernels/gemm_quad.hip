// bf16 GEMM over K-contiguous operands with enough rows for 256 x 256 tiles: four waves a workgroup, each 128 x 128 of C, one
// workgroup per CU.
//
// The 8-wave kernel (gemm.hip) gives a wave 128 x 64 and runs two waves a SIMD half a phase apart; every K-tile costs it 192 KB of
// LDS reads and eight barriers.  Square wave tiles take 128 KB, and one wave a SIMD can keep the matrix core busy by itself when
// everything else is placed between its products: the 256 accumulators live in the accumulation registers, the operands of
// 32 k are multiplied (64 MFMAs) while those of the next 32 k are read into the other half of 128 vector registers, and
// the K-tile's order is fixed by sched_barrier.  Of the 128 MFMAs of a K-tile
//    0 .. 15    one LDS read each: the second 32 k of this K-tile
//    BAR1       every wave has this K-tile in registers: its stage may be written
//    BAR1 + 1.. one staging load (direct to LDS) every LOAD_EVERY: the K-tile after next
//    BAR2       the next K-tile has landed (counted vmcnt: the loads just issued stay out)
//    BAR2 + 1.. one LDS read each: the first 32 k of the next K-tile
// so a staging load has 134 to 209 MFMAs (128 + BAR2 less the slot it is issued at: 1.5 to 2.3 us) to land and there are two barriers a K-tile.  Spreading the loads matters
// most: one every two MFMAs 6688 x 22016 x 4096 944 us, every four or five 872 to 905, and reads at one every two MFMAs instead of
// one each 5 % behind.  The staging runs on over the ends of output tiles: during a tile's last two K-tiles it fetches the next
// one's first two, which land under the epilogue (32 KB of the LDS are the epilogue's own, so it needs no barrier).
//
// Against the 8-wave kernel, us, same operands: 23080 x 3072 x 1024 193 -> 151, 6688 x 22016 x 4096 957 -> 904, 6688 x 11008 x 4096
// 485 -> 458, 4643 x 12288 x 4096 388 -> 372, gated 4643 x 11008 x 4096 659 -> 627, 4096 x 4096 x 4096 103 -> 100.  The card's power limit
// holds the clock near 1.8 GHz on these (operands of zeros: 757 -> 719 us for the first of the 6688 rows, 2.4 GHz);
// per K-tile this takes 1.40 us, 1.02 with zeros, 0.85 is the matrix core's own at 2.4 GHz.  Results are bit for bit the 8-wave kernel's.
#include <type_traits>
#include <utility>

#include "gemm_common.h"
#include "gemm_quad.h"

namespace evgpt {

namespace {

constexpr int IMG = 32768, STAGE = 2 * IMG;       // one operand's 256 rows x 64 k; both of a K-tile
constexpr int SCRATCH = 8192;                     // a wave's rows of the output on their way out
constexpr int LDS_BYTES = 2 * STAGE + 4 * SCRATCH;

// where the 16 LDS reads, the 16 staging loads and the two barriers of a K-tile sit among its 128 MFMAs
constexpr int BAR1 = 24, LOAD_EVERY = 5, BAR2 = 106;
static_assert(BAR1 >= 16 && BAR1 + 15 * LOAD_EVERY < BAR2 && BAR2 + 16 < 128, "all of it within the 128, the loads ahead of BAR2");

__device__ __forceinline__ void load_to_lds16(const unsigned char* src, int bytes, unsigned char* lds, int voff, int soff) {
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(src), 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)lds, 16, voff, soff, 0, 0);
}

// f(0), f(1), ... with constants: accumulators are indexed by constants only, or they would live in memory
template <class F, int... I>
__device__ __forceinline__ void each_(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void each(F&& f) { each_(f, std::make_integer_sequence<int, N>{}); }

// An accumulator out of the matrix core's registers, here and not earlier: left to itself the compiler moves all 256 to
// vector registers ahead of the stores and spills what does not fit.
__device__ __forceinline__ f32x4_t take(const f32x4_t& a) {
  float x, y, z, w;
  asm volatile("v_accvgpr_read_b32 %0, %4\n\tv_accvgpr_read_b32 %1, %5\n\tv_accvgpr_read_b32 %2, %6\n\tv_accvgpr_read_b32 %3, %7"
               : "=&v"(x), "=&v"(y), "=&v"(z), "=&v"(w) : "a"(a[0]), "a"(a[1]), "a"(a[2]), "a"(a[3]));
  return f32x4_t{x, y, z, w};
}

// ACT: activation of a plain output (a constant: 256 run-time choices among the functions are 300 KB of instructions), or ROPE: a q | k | v
// projection whose heads of 128 columns are rotated and go to their places in q and the cache (gemm_rope_epilogue's rules and rounding).
// A wave's columns are one head and both halves of a pair are its own lane's, so the rotation costs the tables' values, from L2 and 16 rows
// ahead, and no exchange.  As a pass of its own over the packed rows it took 40 us a layer at 4643 rows (228 MB).  7B prompt, ms, so / now:
// 4643 tokens 57.9 / 57.1 (the card's power limit takes back half of it), 3000 36.1 / 35.2, 2115 27.8 / 27.4, 1300 20.96 / 20.57.
constexpr int ROPE = -2;
template <bool GRP, int ACT>
__global__ __launch_bounds__(256, 1) void gemm_quad_kernel(GemmParams p) {
  constexpr int BM = 256, BN = 256;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wid >> 1, wc = wid & 1;
  const int bn_out = p.glu_half ? BN / 2 : BN;
  const int tiles_n = (p.N + bn_out - 1) / bn_out, tiles_m = (p.M + BM - 1) / BM;
  int total = tiles_m * tiles_n * p.splitk;
  if constexpr (GRP) {
    total = group_tiles(p.grp_start, p.grp_count, BM, tiles_n);
    if (static_cast<int>(blockIdx.x) >= total) return;
  }
  struct Tile { int m0, n0, ksplit, nk, rows, first; const unsigned char *a, *w; int bytes_a, bytes_w; };

  // per-lane source offsets of the eight staging loads an operand's image takes from this wave: load j fetches rows
  // (4 j + wid) * 8 .. + 8, 128 bytes each, the 16-byte chunks of a row permuted by (row >> 1) & 7
  int va[8], vw[8];
  const int srow = wid * 8 + (lane >> 3), scol = ((lane & 7) ^ ((srow >> 1) & 7)) * 16;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int r = j * 32 + srow;
    va[j] = r * p.lda * 2 + scol;
    const int wrow = p.glu_half ? (r >> 7) * 64 + (r & 63) + ((r >> 6) & 1) * p.glu_half : r;
    vw[j] = wrow * p.ldw * 2 + scol;
  }
  auto locate = [&](int t, Tile& c) {
    const int bid = xcd_remap(t, total);
    int tm, tn;
    if constexpr (GRP) {
      int within = bid;
      const int e = max(group_of_tile(p.grp_start, p.grp_count, BM, tiles_n, within), 0);
      c.ksplit = 0;
      c.nk = p.K / BK;
      c.first = p.grp_start[e];
      c.rows = p.grp_start[e + 1] - c.first;
      tile_walk(within, (c.rows + BM - 1) / BM, tiles_n, p.group_m, tm, tn);
      c.m0 = tm * BM;
      c.n0 = tn * bn_out;
      c.a = reinterpret_cast<const unsigned char*>(p.A);
      c.bytes_a = 0x7fffffff;
      c.w = reinterpret_cast<const unsigned char*>(p.W + e * p.grp_wstride + static_cast<long long>(c.n0) * p.ldw);
#pragma unroll
      for (int j = 0; j < 8; ++j) {          // (rows past the group read its last one and are not stored)
        const int r = c.first + min(c.m0 + j * 32 + srow, c.rows - 1);
        va[j] = (p.grp_perm ? p.grp_perm[r] / p.grp_top : r) * p.lda * 2 + scol;
      }
    } else {
      const int tile = bid / p.splitk;
      c.ksplit = bid % p.splitk;
      const int k_begin = c.ksplit * p.k_per_split;
      c.nk = min(p.k_per_split, p.K - k_begin) / BK;
      tile_walk(tile, tiles_m, tiles_n, p.group_m, tm, tn);
      c.first = 0;
      c.rows = p.M;
      c.m0 = tm * BM;
      c.n0 = tn * bn_out;
      c.a = reinterpret_cast<const unsigned char*>(p.A + static_cast<long long>(c.m0) * p.lda + k_begin);
      c.bytes_a = (min(p.M - c.m0, BM) * p.lda - k_begin) * 2;
      c.w = reinterpret_cast<const unsigned char*>(p.W + static_cast<long long>(c.n0) * p.ldw + k_begin);
    }
    const int w_rows = p.glu_half ? 2 * p.glu_half - c.n0 : min(p.N - c.n0, BN);
    c.bytes_w = (w_rows * p.ldw - (GRP ? 0 : c.ksplit * p.k_per_split)) * 2;
  };

  const int frow = lane & 15, fq = lane >> 4, fsw = (frow >> 1) & 7;
  int ra[2], rw[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int c = ((ks * 4 + fq) ^ fsw) << 4;
    ra[ks] = (wr * 128 + frow) * 128 + c;
    rw[ks] = IMG + (wc * 128 + frow) * 128 + c;
  }
  f32x4_t acc[8][8];
  bf16x8_t fa[2][8], fw[2][8];

  // ---- the staging side runs two K-tiles ahead, over the ends of output tiles (nk >= 2)
  Tile cur, nxt;
  int t = blockIdx.x;
  locate(t, cur);
  const unsigned char *la = cur.a, *lw = cur.w;
  int lba = cur.bytes_a, lbw = cur.bytes_w, koff = 0;
  int stage = 0;                       // byte offset of the stage that is multiplied, then staged for two K-tiles later
  auto issue = [&](int l, int st) {
    unsigned char* dst = smem + st + (l >> 3) * IMG + (l & 7) * 4096 + wid * 1024;
    if (l < 8) load_to_lds16(la, lba, dst, va[l & 7], koff);
    else load_to_lds16(lw, lbw, dst, vw[l & 7], koff);
  };
  auto read_frag = [&](int h, int n, int st) {       // n: 0..7 W, 8..15 A
    if (n < 8) fw[h][n] = *reinterpret_cast<const bf16x8_t*>(smem + st + rw[h] + n * 2048);
    else fa[h][n - 8] = *reinterpret_cast<const bf16x8_t*>(smem + st + ra[h] + (n - 8) * 2048);
  };

#pragma unroll
  for (int l = 0; l < 16; ++l) issue(l, 0);
  koff = 128;
#pragma unroll
  for (int l = 0; l < 16; ++l) issue(l, STAGE);
  wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int n = 0; n < 16; ++n) read_frag(0, n, 0);

  for (;;) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const bool more = t + static_cast<int>(gridDim.x) < total;
    int left = cur.nk - 2;
    for (int part = 0; part < 2; ++part) {
      for (; left > 0; --left) {
        koff += 128;
        each<128>([&](auto mc) {
          constexpr int m = decltype(mc)::value, h = m >> 6, i = (m >> 3) & 7, j = m & 7;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[h][j], fa[h][i], acc[i][j], 0, 0, 0);
          // the second half of this K-tile, as soon as the first is being multiplied
          if constexpr (m < 16) read_frag(1, m, stage);
          // every wave has the K-tile in registers: its stage is free
          if constexpr (m == BAR1) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
          }
          if constexpr (m > BAR1 && (m - BAR1 - 1) % LOAD_EVERY == 0 && (m - BAR1 - 1) / LOAD_EVERY < 16)
            issue((m - BAR1 - 1) / LOAD_EVERY, stage);
          // the next K-tile has landed (the epilogue waits for a tile's second one)
          if constexpr (m == BAR2) {
            __builtin_amdgcn_sched_barrier(0);
            wait_vm<16>();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
          }
          if constexpr (m > BAR2 && m <= BAR2 + 16) read_frag(0, m - BAR2 - 1, stage ^ STAGE);
          __builtin_amdgcn_sched_barrier(0);
        });
        stage ^= STAGE;
      }
      // The last two K-tiles: staged meanwhile are the next output tile's first two, or what nobody uses: nearly all zeros, by a range
      // that ends with the first row's two K-tiles.  (Not an empty range: less the scalar offset of 128 it need not be empty.)
      left = part ? 0 : 2;
      koff = part ? 128 : -128;
      if (part == 0) {
        if (more) {
          locate(t + gridDim.x, nxt);
          la = nxt.a; lw = nxt.w; lba = nxt.bytes_a; lbw = nxt.bytes_w;
        } else {
          lba = 256; lbw = 256;
        }
      }
    }
    wait_vm<0>();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");     // the last products are in their registers
    // ---- epilogue
    const int M = cur.rows;
    bf16_t* C = p.C + (GRP ? static_cast<size_t>(cur.first) * p.ldc : 0);
    unsigned char* rows = smem + 2 * STAGE + wid * SCRATCH;
    if (!GRP && ACT != ROPE && (p.splitk > 1 || p.raw_partial || p.Cf)) {
      const bool whole = p.splitk == 1 && !p.raw_partial;              // the fp32 output itself
      float* slab = whole ? p.Cf : p.partial + static_cast<size_t>(cur.ksplit) * p.M * p.N;
      const size_t ld = whole ? p.ldc : p.N;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int m = cur.m0 + wr * 128 + i * 16 + frow;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int n = cur.n0 + wc * 128 + j * 16 + fq * 4;
          if (m < M && n < p.N) *reinterpret_cast<f32x4_t*>(slab + m * ld + n) = take(acc[i][j]);
        }
      }
    } else if constexpr (ACT == ROPE) {
      const int head = (cur.n0 >> 7) + wc + p.rope_head0, pos0 = p.rope_pos0 ? p.rope_pos0[0] : 0;
      const bool to_cache = head >= p.rope_hq, is_v = head >= p.rope_hq + p.rope_hkv, inside = cur.n0 + wc * 128 < p.N;
      // the head's rows: of q, one after another by token; of k and v by position
      bf16_t* dst = !to_cache ? p.rope_q + head * 128
                              : (is_v ? p.rope_v : p.rope_k) + static_cast<size_t>(head - p.rope_hq - (is_v ? p.rope_hkv : 0)) * p.rope_lmax * 128;
      const int ld = to_cache ? 128 : p.rope_hq * 128, most = to_cache ? p.rope_lmax : M;
      const auto heads = [&](auto rotated) {      // (one head a wave)
        constexpr bool TURN = decltype(rotated)::value;
        f32x4_t cs[2][4], sn[2][4];        // the tables of 16 rows, and of the next 16 on their way
        const auto request = [&](int i) {
          const int pos = min(max(pos0 + min(cur.m0 + wr * 128 + i * 16 + frow, M - 1), 0), p.rope_lmax - 1);
          const unsigned int at = static_cast<unsigned int>(pos) * 256 + fq * 16;      // (rope_lmax * 256 is below 2^32: gemm_quad_serves)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            cs[i & 1][j] = *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const char*>(p.rope_cos) + at + j * 64);
            sn[i & 1][j] = *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const char*>(p.rope_sin) + at + j * 64);
          }
        };
        if constexpr (TURN) request(0);
        each<4>([&](auto pc) {
          constexpr int pass = decltype(pc)::value;
          each<2>([&](auto ic) {
            constexpr int il = decltype(ic)::value, i = pass * 2 + il;
            if constexpr (TURN && i < 7) request(i + 1);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              f32x4_t a = take(acc[i][j]), b = take(acc[i][j + 4]);
              if constexpr (TURN) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {          // (sums rounded as rope_kv_prefill_kernel's)
                  const float x = bf16_to_f32(f32_to_bf16(a[r])), y = bf16_to_f32(f32_to_bf16(b[r])), c = cs[i & 1][j][r], t = sn[i & 1][j][r];
                  a[r] = fmaf(c, x, -(t * y));
                  b[r] = fmaf(c, y, t * x);
                }
              }
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const f32x4_t v = h ? b : a;
                const u32x2_t w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                const int chunk = ((j + h * 4) * 2 + (fq >> 1)) ^ frow;
                *reinterpret_cast<u32x2_t*>(rows + (il * 16 + frow) * 256 + chunk * 16 + (fq & 1) * 8) = w;
              }
            }
          });
          asm volatile("" ::: "memory");
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int r = q * 4 + (lane >> 4), c = lane & 15;
            const u32x4_t d = *reinterpret_cast<const u32x4_t*>(rows + r * 256 + ((c ^ (r & 15)) << 4));
            const int m = cur.m0 + wr * 128 + pass * 32 + r, row = to_cache ? pos0 + m : m;
            if (m < M && inside && row >= 0 && row < most) *reinterpret_cast<u32x4_t*>(dst + static_cast<long long>(row) * ld + c * 8) = d;
          }
          asm volatile("" ::: "memory");
        });
      };
      if (is_v) heads(std::false_type{});
      else heads(std::true_type{});
    } else if (ACT == ACT_NONE && p.glu_half) {
      each<4>([&](auto pc) {
        constexpr int pass = decltype(pc)::value;
#pragma unroll
        for (int il = 0; il < 2; ++il)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x4_t g = take(acc[pass * 2 + il][j]), u = take(acc[pass * 2 + il][j + 4]);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
              v[r] = glu_gate(bf16_to_f32(f32_to_bf16(g[r])), p.glu_act) * bf16_to_f32(f32_to_bf16(u[r]));
            const u32x2_t w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            const int chunk = (j * 2 + (fq >> 1)) ^ (frow & 7);
            *reinterpret_cast<u32x2_t*>(rows + (il * 16 + frow) * 256 + chunk * 16 + (fq & 1) * 8) = w;
          }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = q * 8 + (lane >> 3), c = lane & 7;
          const u32x4_t d = *reinterpret_cast<const u32x4_t*>(rows + r * 256 + ((c ^ (r & 7)) << 4));
          const int m = cur.m0 + wr * 128 + pass * 32 + r, n = cur.n0 + wc * 64 + c * 8;
          if (m < M && n < p.N) *reinterpret_cast<u32x4_t*>(C + static_cast<size_t>(m) * p.ldc + n) = d;
        }
        asm volatile("" ::: "memory");
      });
    } else {
      each<4>([&](auto pc) {
        constexpr int pass = decltype(pc)::value;
        u32x4_t rv[8];                       // the residual's rows, on their way while the tile's are packed
        if (!GRP && p.res) {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int m = cur.m0 + wr * 128 + pass * 32 + q * 4 + (lane >> 4), n = cur.n0 + wc * 128 + (lane & 15) * 8;
            rv[q] = load16(p.res + (m < M && n < p.N ? static_cast<size_t>(m) * p.ldc + n : 0));
          }
        }
        each<8>([&](auto jc) {
          constexpr int j = decltype(jc)::value;
          const int n = cur.n0 + wc * 128 + j * 16 + fq * 4;
          float b[4] = {0.f, 0.f, 0.f, 0.f};
          if (p.bias && n < p.N) {
            const u32x2_t bb = *reinterpret_cast<const u32x2_t*>(p.bias + n);
            b[0] = bf16lo(bb[0]); b[1] = bf16hi(bb[0]); b[2] = bf16lo(bb[1]); b[3] = bf16hi(bb[1]);
          }
#pragma unroll
          for (int il = 0; il < 2; ++il) {
            const f32x4_t o = take(acc[pass * 2 + il][j]);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = ACT <= ACT_NONE ? o[r] + b[r] : apply_act(o[r] + b[r], ACT);
            const u32x2_t w = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            const int chunk = (j * 2 + (fq >> 1)) ^ frow;
            *reinterpret_cast<u32x2_t*>(rows + (il * 16 + frow) * 256 + chunk * 16 + (fq & 1) * 8) = w;
          }
        });
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int r = q * 4 + (lane >> 4), c = lane & 15;
          u32x4_t d = *reinterpret_cast<const u32x4_t*>(rows + r * 256 + ((c ^ (r & 15)) << 4));
          const int m = cur.m0 + wr * 128 + pass * 32 + r, n = cur.n0 + wc * 128 + c * 8;
          if (m < M && n < p.N) {
            const size_t o = static_cast<size_t>(m) * p.ldc + n;
            if (!GRP && p.res) {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                d[e] = pack_bf16x2(bf16lo(d[e]) + bf16lo(rv[q][e]), bf16hi(d[e]) + bf16hi(rv[q][e]));
            }
            *reinterpret_cast<u32x4_t*>(C + o) = d;
          }
        }
        asm volatile("" ::: "memory");
      });
    }
    if (!more) break;
    t += gridDim.x;
    cur = nxt;
  }
}

}  // namespace

template <bool GRP, int ACT = ACT_NONE>
static void launch(const GemmParams& p, int grid, hipStream_t st) {
  static const bool attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_quad_kernel<GRP, ACT>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) == hipSuccess;
  (void)attr;
  hipLaunchKernelGGL((gemm_quad_kernel<GRP, ACT>), dim3(grid), dim3(256), LDS_BYTES, st, p);
}

bool gemm_quad_serves(const GemmParams& p) {
  const long long lim = 1ll << 31;
  const int tail = p.K % p.k_per_split;
  if (p.k_per_split < 2 * BK || (tail && tail < 2 * BK)) return false;
  if (p.k_cols || p.amax_val) return false;
  if (2ll * 256 * p.lda >= lim || 2ll * (p.glu_half ? 2ll * p.glu_half : 256) * p.ldw >= lim) return false;
  if (p.grp_start && (2ll * p.M * p.lda >= lim || p.res || p.bias || p.act != ACT_NONE)) return false;
  if (p.splitk > 1 || p.raw_partial) return !p.glu_half && p.partial && p.N % 4 == 0;
  if (p.rope_cos)
    return !p.grp_start && p.rope_lmax < (1 << 24) && ((reinterpret_cast<uintptr_t>(p.rope_q) | reinterpret_cast<uintptr_t>(p.rope_k) | reinterpret_cast<uintptr_t>(p.rope_v) |
                             reinterpret_cast<uintptr_t>(p.rope_cos) | reinterpret_cast<uintptr_t>(p.rope_sin)) & 15) == 0;
  if (p.Cf)
    return !p.C && !p.grp_start && !p.glu_half && !p.bias && !p.res && p.act == ACT_NONE && p.N % 4 == 0 && p.ldc % 4 == 0 &&
           (reinterpret_cast<uintptr_t>(p.Cf) & 15) == 0;
  if (p.N % 8 || p.ldc % 8 || !p.C || (reinterpret_cast<uintptr_t>(p.C) & 15) || (reinterpret_cast<uintptr_t>(p.res) & 15)) return false;
  if (p.glu_half) return !p.bias && !p.res && p.act == ACT_NONE;
  return (reinterpret_cast<uintptr_t>(p.bias) & 7) == 0 && (p.act == ACT_NONE || p.act == ACT_GELU || p.act == ACT_QUICK_GELU);
}

// Over short contractions its ends, longer than the 8-wave kernel's, are what there is; that kernel's own end is the longer one with a bias or
// an activation (a choice among all of them).  Its time over the 8-wave kernel's at the mean of 13 200 products of 768 to 9 000 rows, up to 256
// tiles and more, K = 128 / 448 / 768 / 1024 / 1536 / 2048:
//  * plain 1.08 / 1.04 / 1.00 / 0.98 / 0.97 / 0.97 and 1.00 / 0.97 / 0.96 / 0.96 / 0.96 / 0.96
//  * slabs 1.06 / 1.04 / 1.03 / 1.02 / 1.00 / 0.97 and 1.00 / 0.96 / 0.96 / 0.96 / 0.94 / 0.94
//  * gated 1.08 / 1.05 / 1.04 / 1.03 / 1.00 / 0.98 and 1.06 / 1.02 / 1.01 / 0.99 / 0.98 / 0.97
//  * an fp32 output, us before (the 8-wave kernel with its general epilogue) / now: 4096 x 4096 x 4096 104 / 96, x 2048 63 / 56, 6688 x 4096 x
//    1024 71 / 58, 4096 x 11008 x 320 67 / 52; the line is the slabs'
//  * a residual 1.00 to 0.96 and 0.96 to 0.94, a bias 0.80 to 0.86, gelu 0.88 to 0.94, quick-gelu 0.70 to 0.80
bool gemm_quad_ahead(const GemmParams& p, int tiles) {
  const int k = p.k_per_split;
  const bool many = tiles > 256;
  if (p.glu_half) return k > (many ? 768 : 1024);
  if (p.splitk > 1 || p.raw_partial || p.Cf) return k > (many ? 192 : 1024);
  return p.bias || p.res || p.act != ACT_NONE || k > (many ? 192 : 576);
}

void launch_gemm_quad(const GemmParams& p, int grid, hipStream_t st) {
  if (p.rope_cos && p.splitk == 1) launch<false, ROPE>(p, grid, st);
  else if (p.grp_start) launch<true>(p, grid, st);
  else if (p.splitk > 1 || p.raw_partial || p.Cf || p.act == ACT_NONE) launch<false>(p, grid, st);
  else if (p.act == ACT_GELU) launch<false, ACT_GELU>(p, grid, st);
  else launch<false, ACT_QUICK_GELU>(p, grid, st);
}

}  // namespace evgpt
