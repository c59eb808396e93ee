// Uniform groups (matmul, bmm) on tiles whose wavefronts split K: 16 to 64 tokens x 128 columns, the same packed layout,
// dequantisation and sparse-MFMA operand mapping as sparse24_grouped_kernel.
//
// Between decode and prefill a launch has few tiles and each is a chain of K steps, so what counts is how little a step
// costs the CU and how much of it is in flight:
//   * activations go to LDS by direct loads of 4 rows x 256 bytes, whole cache lines.  Loaded as operands, as the streaming kernel
//     does, four neighbouring lanes read four rows, and a KB takes the address unit 64 cycles instead of 19: 5 of the 9 us of
//     640 such requests a CU on 4096 x 4096 with 64 tokens;
//   * every wavefront has its own steps, its own place in LDS for a step's activations and two steps of weights in registers: no
//     barrier before the end.  The place is free once the step's last operands have been read, half a step ahead of its end;
//   * a dequantised weight meets up to 64 tokens (the streaming kernel gives tokens to workgroups 16 at a time to fill the chip
//     and dequantises for each of them anew);
//   * K is split further over workgroups where the tiles do not fill the chip (splitk_reduce_kernel adds the shares).
// Measured (before -> now): 37 tokens on 11008 x 4096 20.4 -> 14.3 us, 192 on 4096 x 11008 46.8 -> 21.1, 384 on 4096 x 4096 26.6 -> 14.4,
// 256 on 13824 x 5120 72 -> 33, 48 on each of 8 matrices of 4096 x 4096 26.2 -> 15.9, 16 on each of 4 of 11008 x 4096 24.3 -> 17.3.
// Needs k % 128 == 0 and 16-byte aligned activations.
#pragma once
#include "sparse24_gemm.hip.h"

namespace triteia_hip {

// NT: 16-token tiles of a workgroup; KW: its wavefronts.
template <int NT, int KW>
struct KTile {
  static constexpr int kTokens = 16 * NT;
  static constexpr int kXBytes = KW * NT * 4096;                      // a step's activations for every wavefront
  static constexpr int kRedBytes = KW * 16 * kRedStride * 4;
  static constexpr int kLdsBytes = kXBytes > kRedBytes ? kXBytes : kRedBytes;
};

// One tile: up to 16 NT tokens x column block `cb` of matrix `delta`, on this workgroup's KW wavefronts.
// PLAN: the tokens are rows of a routing plan's list, s_off[i] the byte offset of the i-th token's row in x (past the last token: the last
// one's) and s_rows[i] its row in the output, which the sums may be added to; the walk over K starts at step `rot` and wraps
// around, as in the streaming kernel.  With its four wavefronts the sums are then the streaming kernel's to the bit: a routed
// token does not depend on the size of its batch.
// Otherwise: tokens first .. of a uniform group of `count` rows from row0, steps s0 .. s0 + n_all - 1, share z of K.
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));
template <int NT, int KW, bool PLAN>
__device__ __forceinline__ void ktile_run(const Sparse24Args& p, unsigned char* smem, int wave, int delta, int cb, int s0, int n_all, int rot, int first,
                                          int count, long row0, int z, int splits, const uint32_t* s_off, const int* s_rows) {
  // (the lane's number afresh: a caller's loop carries neither it nor the offsets made of it in registers)
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  const int tid = wave * 64 + lane;
  const int r = lane & 15, q = lane >> 4;
  // A 16-token tile that would run past the group's last token starts earlier instead: its first rows are another tile's,
  // computed again and not stored, and every tile reads whole rows at the same distances.
  auto tile_start = [&](int nt) { return max(0, min(first + 16 * nt, count - 16)); };
  const int n = max(0, (n_all - wave + KW - 1) / KW);                // this wavefront's steps: wave, + KW, ...
  auto phys = [&](int i) {
    const int st = wave + KW * i;
    if (!PLAN) return s0 + st;
    return st + rot < n_all ? st + rot : st + rot - n_all;
  };

  const long qrow = p.m >> 1, mrow = p.m >> 2;
  const char* qw = reinterpret_cast<const char*>(p.qweight + (long)delta * p.qweight_stride + (long)cb * 64);
  const char* mt = reinterpret_cast<const char*>(p.meta + (long)delta * p.meta_stride + (long)cb * 32);
  const uint32_t woff = (uint32_t)(q * qrow + 4 * r) * 16, moff = (uint32_t)(q * mrow + (r >> 3) * 16 + (r & 7)) * 16;
  struct WFrag {
    uint4_t wq[4], mt[2];
  };
  auto load_w = [&](WFrag& f, int i) {                               // (past the end: the last step again, from cache)
    const long tr = n > 0 ? (long)phys(min(i, n - 1)) << 2 : 0;
#pragma unroll
    for (int a = 0; a < 4; a++) f.wq[a] = *reinterpret_cast<const uint4_t*>(qw + tr * qrow * 16 + woff + 16 * a);
    f.mt[0] = *reinterpret_cast<const uint4_t*>(mt + tr * mrow * 16 + moff);
    f.mt[1] = *reinterpret_cast<const uint4_t*>(mt + tr * mrow * 16 + moff + 128);
  };

  // activations: a request covers 4 rows x 256 bytes; lane l fills position l % 16 of row l / 16 with the row's 16-byte piece
  // (l % 16) ^ (row % 16).  (a group of fewer than 16 tokens repeats its last row)
  const uint32_t lds_x = (uint32_t)(uintptr_t)smem + wave * (NT * 4096);
  uint32_t xoff[4];                                                  // bytes from a 16-token tile's first row; PLAN: from a row
#pragma unroll
  for (int i = 0; i < 4; i++) xoff[i] = (PLAN ? 0 : (uint32_t)min(4 * i + q, count - 1) * (uint32_t)(p.x_stride * 2)) + 16 * (r ^ (4 * i + q));
  auto issue_x = [&](int i) {
    const _Float16* x0 = p.x + (PLAN ? 0 : row0 * p.x_stride) + (long)phys(i) * 128;
    uint32x4 rows = {0, 0, 0, 0};
    uint32_t x_lane = xoff[0];
    if (PLAN) asm volatile("" : "+v"(x_lane));                       // (one register: the exclusive ors below are made where they are used)
#pragma unroll
    for (int j = 0; j < 4 * NT; j++) {
      if (PLAN && (j & 3) == 0) rows = *reinterpret_cast<const uint32x4*>(s_off + 4 * j + 4 * q);
      const _Float16* base = PLAN ? x0 : x0 + (long)tile_start(j >> 2) * p.x_stride;
      const uint32_t off = PLAN ? rows[j & 3] + (x_lane ^ (64 * (j & 3))) : xoff[j & 3];
      const uint32_t d = __builtin_amdgcn_readfirstlane(lds_x + 1024 * j);
      direct_load(off, base, d);
    }
  };

  float4_t acc[8][NT];
#pragma unroll
  for (int cc = 0; cc < 8; cc++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[cc][nt] = float4_t{0.f, 0.f, 0.f, 0.f};

  const unsigned char* xw = smem + wave * (NT * 4096) + r * 256;
  auto read_b = [&](int nt, int u) {
    const int c = 4 * (q >> 1) + (q & 1) + 2 * u;
    typedef uint32_t uint8_t_v __attribute__((ext_vector_type(8)));
    const uint4_t lo = *reinterpret_cast<const uint4_t*>(xw + nt * 4096 + ((c ^ r) << 4));
    const uint4_t hi = *reinterpret_cast<const uint4_t*>(xw + nt * 4096 + (((c + 8) ^ r) << 4));
    const uint8_t_v bb = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(half16_t, bb);
  };
  auto step = [&](const WFrag& f, int i) {
    // Requests complete in order and come as: a step's activations (in the middle of the step before), then the weights of
    // the step after it, six requests.  All but the newest six done: this step's activations have landed.  (The compiler
    // waits for this step's weights by the same count.)
    asm volatile("s_waitcnt vmcnt(6)" : : : "memory");
#pragma unroll
    for (int u = 0; u < 2; u++) {
      half16_t b[NT];
#pragma unroll
      for (int nt = 0; nt < NT; nt++) b[nt] = read_b(nt, u);
      if (u == 1) {
        // the step's last operands are in registers: its place takes the next step's activations
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < n) issue_x(i + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int b2 = 0; b2 < 2; b2++) {
        half8_t A[4];
#pragma unroll
        for (int w = 0; w < 4; w++) {
          uint4_t av;
#pragma unroll
          for (int a = 0; a < 4; a++) {
            uint32_t word = f.wq[a][w];
            if (b2) word >>= 8;
            av[a] = u ? dequant_odd(word) : dequant_even(word);
          }
          A[w] = __builtin_bit_cast(half8_t, av);
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
          for (int w = 0; w < 4; w++) {
            const int cc = 4 * b2 + w;
            const int idx = (int)f.mt[(cc >> 1) & 1][(cc & 1) * 2 + u];
            if (b2) acc[cc][nt] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A[w], b[nt], acc[cc][nt], idx, 0, 1);
            else acc[cc][nt] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A[w], b[nt], acc[cc][nt], idx, 0, 0);
          }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // The scales of this thread's 8 columns (the same ones for every 16 tokens), for the epilogue of an unsplit uniform launch: among the sums
  // they are a round trip to memory for every 16 tokens (loads are not moved across a barrier).  Tiles of up to 48 tokens request them
  // ahead of the loop (1315 tokens on 3328 x 640, in tiles of 32, 12.5 -> 12.3 us); tiles of 64 have no registers to keep them in and request them once,
  // behind it (100 tokens on 4096 x 11008 14.3 -> 13.4).  A plan's tiles, mostly of 16 or 32 tokens, lost 0.7 - 1.3 % by either.
  const _Float16* sc = p.scales + (long)delta * p.scales_stride + cb * 128;
  half8_t scales = {0, 0, 0, 0, 0, 0, 0, 0};
  if (!PLAN && NT < 4 && splits == 1) scales = *reinterpret_cast<const half8_t*>(sc + (tid & 15) * 8);
  WFrag ring[2];
  if (n > 0) issue_x(0);
  __builtin_amdgcn_sched_barrier(0);
  load_w(ring[0], 0);
  load_w(ring[1], 1);
  __builtin_amdgcn_sched_barrier(0);
  for (int i = 0; i < n; i += 2) {
    step(ring[0], i);
    load_w(ring[0], i + 2);
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < n) step(ring[1], i + 1);
    load_w(ring[1], i + 3);
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
  if (!PLAN && NT == 4 && splits == 1) scales = *reinterpret_cast<const half8_t*>(sc + (tid & 15) * 8);

  // the wavefronts' sums, added in order, 16 tokens at a time, each of the first 256 threads 8 columns of one (as a loop over such pieces,
  // which ran once, 2436 tokens over 8 plan deltas of 1280 x 1536 took 21.3 us instead of 20.8)
  float(*red)[16][kRedStride] = reinterpret_cast<float(*)[16][kRedStride]>(smem);
  static_assert(64 * KW >= 256, "a thread for every 8 columns of 16 tokens");
  const int tok = tid >> 4, f0 = (tid & 15) * 8;
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    if (first + 16 * nt >= count) break;
    const int t = PLAN ? 16 * nt + tok : tile_start(nt) + tok;
    const bool live = tid < 256 && t < count && (PLAN || t >= first + 16 * nt);
    lds_barrier();
    float* dst = &red[wave][r][32 * q];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      *reinterpret_cast<float4_t*>(dst + 8 * j) = float4_t{acc[0][nt][j], acc[1][nt][j], acc[2][nt][j], acc[3][nt][j]};
      *reinterpret_cast<float4_t*>(dst + 8 * j + 4) = float4_t{acc[4][nt][j], acc[5][nt][j], acc[6][nt][j], acc[7][nt][j]};
    }
    lds_barrier();
    if (!live) continue;
    const long row = PLAN ? s_rows[t] : row0 + t;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = 0.f;
#pragma unroll
    for (int w = 0; w < KW; w++) {
      const float4_t a0 = *reinterpret_cast<const float4_t*>(&red[w][tok][f0]);
      const float4_t a1 = *reinterpret_cast<const float4_t*>(&red[w][tok][f0 + 4]);
#pragma unroll
      for (int i = 0; i < 4; i++) { v[i] += a0[i]; v[4 + i] += a1[i]; }
    }
    if (!PLAN && splits > 1) {
      float* pp = p.partial + ((long)z * p.partial_rows + row) * p.m + cb * 128 + f0;
      *reinterpret_cast<float4_t*>(pp) = float4_t{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<float4_t*>(pp + 4) = float4_t{v[4], v[5], v[6], v[7]};
      continue;
    }
    const half8_t sv = PLAN ? *reinterpret_cast<const half8_t*>(sc + f0) : scales;
    _Float16* op = p.out + row * p.out_stride + cb * 128 + f0;
    half8_t old = {0, 0, 0, 0, 0, 0, 0, 0};
    if (PLAN && p.accumulate) old = *reinterpret_cast<const half8_t*>(op);
    half8_t o;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = scaled_sum_f16(old[i], v[i], sv[i]);
    *reinterpret_cast<half8_t*>(op) = o;
  }
}

template <int NT, int KW>
__global__ __launch_bounds__(64 * KW, 2) void sparse24_ktile_kernel(const Sparse24Args p, int splits) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  // Units in the order (group, column block, share of K, token tile), token tiles fastest; an XCD (workgroup u runs on XCD
  // u % 8) takes a run of them: the token tiles of a column block read its weights through one L2.
  const int col_blocks = p.m >> 7, ttiles = (p.uniform_count + 16 * NT - 1) / (16 * NT);
  const int units = p.n_groups * col_blocks * splits * ttiles;
  const int per_xcd = (units + 7) >> 3;
  const int unit = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || unit >= units) return;
  const int tt = unit % ttiles, z = (unit / ttiles) % splits;
  const int gcb = unit / (ttiles * splits), cb = gcb % col_blocks, grp = gcb / col_blocks;
  const int steps = p.k >> 7;                                        // (k % 128 == 0)
  const int s0 = (int)((long)z * steps / splits), n_all = (int)((long)(z + 1) * steps / splits) - s0;
  ktile_run<NT, KW, false>(p, smem, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), grp * p.delta_step, cb, s0, n_all, 0, tt * 16 * NT, p.uniform_count,
                           (long)grp * p.uniform_stride + p.uniform_first, z, splits, nullptr, nullptr);
}

// A routing plan's list of tiles {delta, start, count} of at most 16 MAXNT tokens: p.tiles, p.perm, p.n_groups_dev[0] of them (at most
// p.n_groups), on the same body: a tile runs on the build for its own number of 16-token tiles, its rows gathered by byte offsets
// from LDS.  Four wavefronts and no split of K over workgroups: the sums are the streaming kernel's to the bit.
// Bound by the weights' way through L2 on a batch of small tiles (32 deltas of 4096 x 4096 with 513 tokens 48 us, 4.9 TB/s of
// weights), by the activations' (16 KB a step and 64 tokens, for 128 columns) on one of full tiles.  The streaming kernel that it
// replaces there reads activations in operand order, 16 rows x 64 bytes at 37 GB/s a CU, these whole lines at 110 - 125: 22 deltas of
// 8192 x 1024 with 500 tokens 58 -> 23 us, 5 of 11008 x 4096 with 279 63 -> 41, 16 of 4096 x 4096 with 513 37 -> 30.
// (Measured and not taken: runs of even work instead of even length, cut by a scan of the list in every workgroup, cost 1 - 9 %, as
// much as they gave back under a skewed routing; 16 lane offsets in registers instead of LDS spill at 64 tokens.)
constexpr int kKTilePlanWaves = 4;
template <int MAXNT>
constexpr int ktile_plan_lds() { return 1024 + KTile<MAXNT, kKTilePlanWaves>::kLdsBytes; }   // (the tables in front: a 16-bit offset reaches them)
template <int MAXNT>
__global__ __launch_bounds__(64 * kKTilePlanWaves, 2) void sparse24_ktile_plan_kernel(const Sparse24Args p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  // p.xcd_cgs = 1, 2, 4 or 8: column blocks in that many parts of even width; the units of a part -- tile by tile, its column
  // blocks side by side -- in 8 / xcd_cgs runs of even length, one for each XCD (workgroup u runs on XCD u % 8): the tiles of a
  // delta follow each other in the list and read its weights through one L2.
  const int col_blocks = p.m >> 7, tiles = min(p.n_groups, p.n_groups_dev[0]);
  const int parts = p.xcd_cgs, runs = 8 / parts;
  const int xcd = blockIdx.x & 7, part = xcd % parts, run = xcd / parts;
  const int c0 = part * col_blocks / parts, width = (part + 1) * col_blocks / parts - c0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long total = (long)width * tiles;
  const int u = (int)(run * total / runs) + (blockIdx.x >> 3);
  if (u >= (run + 1) * total / runs) return;
  const int tile = u / width, cb = c0 + u - tile * width;
  const int4 d = p.tiles[tile];
  const int delta = d.x, count = min(d.z, 16 * MAXNT);
  if (delta < 0 || delta >= p.n_deltas || count <= 0) return;
  uint32_t* s_off = reinterpret_cast<uint32_t*>(smem);
  int* s_rows = reinterpret_cast<int*>(s_off + 16 * MAXNT);
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  if (wave == 0 && lane < 16 * MAXNT) {
    const int i = lane, row = p.perm[d.y + min(i, count - 1)];
    s_rows[i] = row;
    s_off[(i & ~15) + 4 * (i & 3) + ((i >> 2) & 3)] = (uint32_t)((long)row * p.x_stride * 2);   // (the launcher sends activations of 4 GiB and more elsewhere)
  }
  __syncthreads();
  const int steps = p.k >> 7;
  const int rot = (int)(((unsigned)delta * (unsigned)p.rot_spread) % (unsigned)steps);
  const int nt = (count + 15) >> 4;
  if (nt == 1) ktile_run<1, kKTilePlanWaves, true>(p, smem + 1024, wave, delta, cb, 0, steps, rot, 0, count, 0, 0, 1, s_off, s_rows);
  else if (nt == 2) ktile_run<2, kKTilePlanWaves, true>(p, smem + 1024, wave, delta, cb, 0, steps, rot, 0, count, 0, 0, 1, s_off, s_rows);
  else if (MAXNT >= 3 && nt == 3) ktile_run<MAXNT >= 3 ? 3 : 1, kKTilePlanWaves, true>(p, smem + 1024, wave, delta, cb, 0, steps, rot, 0, count, 0, 0, 1, s_off, s_rows);
  else ktile_run<MAXNT >= 4 ? 4 : 1, kKTilePlanWaves, true>(p, smem + 1024, wave, delta, cb, 0, steps, rot, 0, count, 0, 0, 1, s_off, s_rows);
}

}  // namespace triteia_hip
