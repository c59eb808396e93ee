// y[T, m] = x[T, k] W[m, k]^T in fp16 with fp32 sums: a layer's dense base weight for the tokens of a routed batch, which
// the deltas' kernels then add to.
//
// A dozen to a few hundred tokens: the launch is bound by W's way from HBM, and past 64 tokens by the tiles' way from L2
// into the CUs.  What that asks for:
//   * both operands go to LDS by direct loads, 8 rows x 128 bytes a request (whole cache lines).  Loaded as operands, 16 rows
//     x 64 bytes a request, four neighbouring lanes read four rows and a CU takes in 37 GB/s from L2 instead of 118;
//   * a ring of chunks of 64 k in LDS, all but one of them in flight.  One barrier a chunk, behind which the stage read in the
//     chunk before is requested anew, request by request between the MFMAs (in one burst the wavefronts stand at the
//     address unit's queue with their MFMAs behind it);
//   * one set of sums per result, added to in the order of K (where the walk starts at the first chunk): the bits of a plain MFMA
//     product.  (Two sets of wavefronts on the halves of a chunk need fewer operand reads and measured the same.)
//   * feature groups may start their walk over K spread around its chunks: rows of W lie a power of two apart, and in
//     lockstep all workgroups read the same few channels (13 tokens on 8192 x 8192 31.6 -> 27.8 us);
//   * K split over workgroups where a layer has too few tiles; a second launch adds the shares in order.
#pragma once
#include "sparse24_gemm.hip.h"

namespace triteia_hip {

struct DenseArgs {
  const _Float16* x;      // [tokens, k]
  long x_stride;
  const _Float16* w;      // [m, k]
  long w_stride;
  _Float16* out;          // [tokens, m]
  long out_stride;
  int tokens, m, k;       // k a multiple of 64, m of 8
  int splits;             // shares of K over workgroups; 1: the result goes to `out`
  int rotate;             // 1: feature groups start their walks over K spread around its chunks, 0: at the first
  float* partial;         // [splits][tokens][m] fp32 sums (splits > 1)
};

// NT x F: 16-token by 16-feature tiles of a wavefront; TW x FW wavefronts side by side.
template <int NT, int TW, int F, int FW, int STAGES>
struct DenseTile {
  static constexpr int kTokens = 16 * NT * TW, kFeatures = 16 * F * FW;
  static constexpr int kWaves = TW * FW, kThreads = 64 * kWaves;
  static constexpr int kStageBytes = 128 * (kTokens + kFeatures);
  static constexpr int kRedStride = kFeatures + 4;
  static constexpr int kRedBytes = kTokens * kRedStride * 4;
  static constexpr int kLdsBytes = STAGES * kStageBytes > kRedBytes ? STAGES * kStageBytes : kRedBytes;
};

template <int NT, int TW, int F, int FW, int STAGES>
__global__ __launch_bounds__(64 * TW * FW) void dense_base_kernel(const DenseArgs p) {
  using Tile = DenseTile<NT, TW, F, FW, STAGES>;
  constexpr int TT = Tile::kTokens, FF = Tile::kFeatures, WAVES = Tile::kWaves;
  constexpr int kXLoads = (TT / 8 + WAVES - 1) / WAVES, kWLoads = (FF / 8 + WAVES - 1) / WAVES;
  constexpr int kLoads = kXLoads + kWLoads;      // a wavefront's requests per chunk: the same in all of them (a few are made twice)
  constexpr int AHEAD = STAGES - 1;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int tw = wave / FW, fw = wave % FW;

  // Units in the order (feature group, share of K, token tile), token tiles fastest; an XCD (workgroup u runs on XCD u % 8)
  // takes a run of them: the token tiles of a feature group read its weights through one L2.
  const int ttiles = (p.tokens + TT - 1) / TT, groups = (p.m + FF - 1) / FF;
  const int units = ttiles * groups * p.splits;
  const int per_xcd = (units + 7) >> 3;
  const int u = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (u >= units) return;
  const int tt = u % ttiles, z = (u / ttiles) % p.splits, fg = u / (ttiles * p.splits);
  const int t0 = tt * TT, f0 = fg * FF;
  const int chunks = p.k >> 6;                   // (splits <= chunks: every share has one)
  const int c0 = (int)((long)z * chunks / p.splits), n = (int)((long)(z + 1) * chunks / p.splits) - c0;
  const int rot = p.rotate ? (int)((long)fg * n / groups) : 0;

  // A request: 8 rows x 128 bytes; lane l takes 16 bytes of row l / 8, the piece (l % 8) ^ (l / 8) to position l % 8.
  // (rows past the end repeat the last one: their sums are not stored)
  const _Float16* src[kLoads];
  uint32_t dst[kLoads];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
#pragma unroll
  for (int i = 0; i < kLoads; i++) {
    const bool is_x = i < kXLoads;
    const int g = min(wave + WAVES * (is_x ? i : i - kXLoads), (is_x ? TT : FF) / 8 - 1), row = 8 * g + (lane >> 3);
    const _Float16* base = is_x ? p.x + (long)min(t0 + row, p.tokens - 1) * p.x_stride : p.w + (long)min(f0 + row, p.m - 1) * p.w_stride;
    src[i] = base + 8 * ((lane & 7) ^ (lane >> 3)) + (long)c0 * 64;
    dst[i] = lds0 + (is_x ? 0 : 128 * TT) + 1024 * g;
  }
  // (inline assembly: the compiler takes a direct load for an LDS write and would wait for all of them at every barrier;
  // no other vector memory request is made between the first of these and the last wait)
  auto issue = [&](int i, int c, int stage) {
    const uint32_t d = __builtin_amdgcn_readfirstlane(dst[i] + stage * Tile::kStageBytes);
    const _Float16* s = src[i] + (long)(c + rot < n ? c + rot : c + rot - n) * 64;
    direct_load(s, d);
  };

  float4_t acc[F][NT];
#pragma unroll
  for (int f = 0; f < F; f++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[f][t] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int piece = (q ^ (r & 7)) * 16;                    // (of the chunk's second half: ^ 64)
  const uint32_t xrow = (16 * NT * tw + r) * 128;
  const uint32_t wrow = 128 * TT + (16 * F * fw + r) * 128;
  auto compute = [&](int stage, auto&& request) {
    const unsigned char* s = smem + stage * Tile::kStageBytes;
    half8_t x[2][NT], w[2][F];
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int t = 0; t < NT; t++) x[h][t] = *reinterpret_cast<const half8_t*>(s + xrow + (piece ^ (64 * h)) + 2048 * t);
#pragma unroll
      for (int f = 0; f < F; f++) w[h][f] = *reinterpret_cast<const half8_t*>(s + wrow + (piece ^ (64 * h)) + 2048 * f);
    }
    __builtin_amdgcn_sched_barrier(0);
    constexpr int kMfmas = 2 * F * NT, kGroup = (kMfmas + kLoads - 1) / kLoads;
#pragma unroll
    for (int e = 0; e < kMfmas; e++) {
      const int h = e / (F * NT), f = e % (F * NT) / NT, t = e % NT;
      acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[h][f], x[h][t], acc[f][t], 0, 0, 0);
      if ((e + 1) % kGroup == 0 || e + 1 == kMfmas) {
        __builtin_amdgcn_sched_barrier(0);
        request(e / kGroup);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int i = (kMfmas + kGroup - 1) / kGroup; i < kLoads; i++) request(i);
  };

  for (int c = 0; c < AHEAD && c < n; c++)
#pragma unroll
    for (int i = 0; i < kLoads; i++) issue(i, c, c);
  int stage = 0, c = 0;
  // AHEAD chunks are in flight at the top, kLoads requests each, and complete in order: all but the newest AHEAD - 1 sets done
  // means that this wavefront's part of chunk c has landed.  The barrier makes all parts visible and says that every wavefront
  // has read the chunk before, whose stage takes chunk c + AHEAD.
  for (; c + AHEAD <= n; c++) {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"((AHEAD - 1) * kLoads) : "memory");
    lds_barrier();
    const int free_stage = stage == 0 ? STAGES - 1 : stage - 1;
    if (c + AHEAD < n) compute(stage, [&](int i) { issue(i, c + AHEAD, free_stage); });
    else compute(stage, [](int) {});
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  }
  for (; c < n; c++) {
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    lds_barrier();
    compute(stage, [](int) {});
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  }

  // through LDS, from where whole rows go out
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);
  // D: lane (token r, q) holds features 4q .. 4q + 3 of a tile
  float* mine = red + (16 * NT * tw + r) * Tile::kRedStride + 16 * F * fw + 4 * q;
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int f = 0; f < F; f++) *reinterpret_cast<float4_t*>(mine + 16 * t * Tile::kRedStride + 16 * f) = acc[f][t];
  __syncthreads();
  constexpr int kPieces = FF / 8;
  for (int e = tid; e < TT * kPieces; e += Tile::kThreads) {
    const int tok = e / kPieces, f = (e - tok * kPieces) * 8;
    if (t0 + tok >= p.tokens || f0 + f >= p.m) continue;
    const float4_t a = *reinterpret_cast<const float4_t*>(red + tok * Tile::kRedStride + f);
    const float4_t b = *reinterpret_cast<const float4_t*>(red + tok * Tile::kRedStride + f + 4);
    if (p.splits > 1) {
      float* o = p.partial + ((long)z * p.tokens + t0 + tok) * p.m + f0 + f;
      *reinterpret_cast<float4_t*>(o) = a;
      *reinterpret_cast<float4_t*>(o + 4) = b;
    } else {
      half8_t o;
#pragma unroll
      for (int i = 0; i < 4; i++) { o[i] = (_Float16)a[i]; o[4 + i] = (_Float16)b[i]; }
      *reinterpret_cast<half8_t*>(p.out + (long)(t0 + tok) * p.out_stride + f0 + f) = o;
    }
  }
}

// The shares of K, added in order and rounded once; 8 features a thread.
__global__ __launch_bounds__(256) void dense_reduce_kernel(const float* __restrict__ partial, int splits, int tokens, int m,
                                                          _Float16* __restrict__ out, long out_stride) {
  const int per_row = m >> 3;
  const long e = (long)blockIdx.x * 256 + threadIdx.x, row = e / per_row;
  if (row >= tokens) return;
  const int c = (int)(e - row * per_row) * 8;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = 0.f;
#pragma unroll 4
  for (int z = 0; z < splits; z++) {
    const float* s = partial + ((long)z * tokens + row) * m + c;
    const float4_t a = *reinterpret_cast<const float4_t*>(s), b = *reinterpret_cast<const float4_t*>(s + 4);
#pragma unroll
    for (int i = 0; i < 4; i++) { v[i] += a[i]; v[4 + i] += b[i]; }
  }
  half8_t o;
#pragma unroll
  for (int i = 0; i < 8; i++) o[i] = (_Float16)v[i];
  *reinterpret_cast<half8_t*>(out + row * out_stride + c) = o;
}

}  // namespace triteia_hip
