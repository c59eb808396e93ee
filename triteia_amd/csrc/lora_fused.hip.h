// The LoRA product of lora_routed.hip.h in ONE launch:
//
//   y[t] (+)= scale * (x[t] @ A[i]) @ B[i],   i = indices[t] in [0, M);  other tokens: nothing added, or zeros stored
//
// A workgroup takes one tile (16 NT tokens of one adapter) and a chunk of output columns: it routes by itself, multiplies the
// tile's rows by the whole of A, keeps the intermediate in LDS, and multiplies that by its columns of B.  Workgroups of a tile
// repeat its first product, which costs them x and A once more from L2; what it saves is the second launch, with its own chain of round
// trips (tile -> rows and shares of K -> operands) and the shares' way to memory and back, and on the host a launch and a scratch.
// So the rule that picks it (lora_fused_takes) bounds what a workgroup reads, and how many columns it has.  Measured against the pair, in a
// graph / called one by one: 16 tokens over 16 adapters of rank 16 on 1024 x 2048 7.0 -> 5.6 / 8.3 -> 5.8 us, 600 over 8 of rank 32 on
// 2048 x 2048 11.9 -> 10.7 / 11.9 -> 10.6.  Of the 5 us, 2 are the routing, 0.8 the first operands, 0.7 the sums, 0.6 the columns of B.
//   * The wavefronts split K in steps of 64.  A step's rows of A (128 r consecutive bytes) and pieces of x (8 rows x 128 bytes a
//     request, whole lines) come by direct loads to a place in LDS that is the wavefront's own: no barrier in the loop.  A step's operands
//     are read into registers, the next step's requests go out, then come the MFMAs.
//   * Behind its last step a wavefront's place takes the first of its columns of B, 64 at a time, while the wavefronts' sums
//     are added (in a fixed order; rounded to T once).
//   * Both contractions as in lora_routed.hip.h: out^T = W^T x^T on the matrix cores, W transposed on its way out of LDS.  The 16-byte
//     pieces of a row are exchanged so that the four rows of a transposing read fall into different banks: no conflicts.
// Needs k % 64 == 0 and a rank of at most 64.
#pragma once
#include "lora_routed.hip.h"
#include "sparse24_gemm.hip.h"

namespace triteia_hip {

template <class T>
struct LoraFusedArgs {
  LoraArgs<T> l;           // (its scratch is not used)
  int tiles;               // the host's bound on the tiles
  int chunks, columns;     // chunks of `columns` output columns (a multiple of 64)
};

template <int R16, int NT>
struct LoraFusedTile {
  static constexpr int kTokens = 16 * NT, kRanks = 16 * R16;
  static constexpr int kWaves = 8, kThreads = 64 * kWaves;
  static constexpr int kDepth = R16 == 1 && NT == 1 ? 4 : R16 + NT <= 3 ? 2 : 1;         // steps in flight per wavefront
  static constexpr int kStageBytes = 2048 * (R16 + NT);
  static constexpr int kWaveBytes = kDepth * kStageBytes;
  static constexpr int kStrips = kWaveBytes / (2048 * R16);          // pieces of 64 columns of B that fit a wavefront's place
  static constexpr int kRedStride = kRanks + 4;
  static constexpr bool kPairs = R16 * NT > 4;                       // the wavefronts' sums do not all fit: first those of the halves
  static constexpr int kSums = kPairs ? kWaves / 2 : kWaves, kRedBytes = kSums * kTokens * kRedStride * 4;
  static constexpr int kVStride = kRanks + 8, kVBytes = kTokens * kVStride * 2;
  static constexpr int kRingBytes = kWaves * kWaveBytes;
  static constexpr int kLdsBytes = kRingBytes + kRedBytes + kVBytes + 4 * kTokens + 4 * kWaves;
  static_assert(kLdsBytes > 81920 && kLdsBytes <= 163840, "one workgroup on a CU");
  static_assert(kRingBytes >= 2 * kLoraMaxTokens + 4 * (kLoraMaxAdapters + 1), "the routing's tables lie in the ring");
};

template <class T, int R16, int NT>
__global__ __launch_bounds__((LoraFusedTile<R16, NT>::kThreads), (LoraFusedTile<R16, NT>::kWaves / 4)) void lora_fused_kernel(const LoraFusedArgs<T> p) {
  using Tile = LoraFusedTile<R16, NT>;
  constexpr int TT = Tile::kTokens, WAVES = Tile::kWaves, DEPTH = Tile::kDepth, STRIPS = Tile::kStrips;
  constexpr int kLoads = 2 * R16 + 2 * NT;                           // requests of a step
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float* red = reinterpret_cast<float*>(smem + Tile::kRingBytes);
  T* v = reinterpret_cast<T*>(smem + Tile::kRingBytes + Tile::kRedBytes);
  int* s_rows = reinterpret_cast<int*>(smem + Tile::kRingBytes + Tile::kRedBytes + Tile::kVBytes);
  const LoraArgs<T>& a = p.l;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // The chunks of a tile on one XCD (workgroup u runs on XCD u % 8), whose L2 then fetches the tile's A and x once; fewer than eight
  // tiles: spread.
  const int u = blockIdx.x, i8 = u >> 3;
  const int tile = p.tiles >= 8 ? (u & 7) + 8 * (i8 / p.chunks) : u / p.chunks;
  const int chunk = p.tiles >= 8 ? i8 % p.chunks : u % p.chunks;
  if (tile >= p.tiles) return;
  const LoraTile found = lora_find_tile<Tile::kThreads, TT>(
      a, tile, {reinterpret_cast<uint16_t*>(smem), reinterpret_cast<int*>(smem + 2 * kLoraMaxTokens), s_rows + TT, s_rows});
  const int bin = found.bin, cnt = found.count;
  if (bin < 0) return;
  const int c0 = chunk * p.columns, c1 = min(a.m, c0 + p.columns);
  if (bin == a.n_adapters) {
    const int pieces = (c1 - c0) >> 3;
    for (int e = tid; e < cnt * pieces; e += Tile::kThreads) {
      const int tok = e / pieces, c = e - tok * pieces;
      *reinterpret_cast<lvec8<T>*>(a.y + (long)s_rows[tok] * a.y_stride + c0 + 8 * c) = lvec8<T>{0, 0, 0, 0, 0, 0, 0, 0};
    }
    return;
  }

  const int j = lane & 15, q = lane >> 4;
  const int r = a.r, per_row = r >> 3;                               // 16-byte pieces of a row of A
  // Pieces of a row of A change places by twos, so that the four rows x 32 bytes of a transposing read cover 128 bytes of banks: rows
  // of 128 bytes alternate between two halves of them by themselves.  (ranks below 64 need none, others that are no power of two get none)
  auto swap_a = [&](int row) { return r == 64 ? 2 * ((row >> 1) & 3) : 0; };
  const char* wa = reinterpret_cast<const char*>(a.a + (long)bin * a.k * r);
  uint32_t asrc[2 * R16];                                            // byte offset inside a step's rows of this lane's part of each KB
#pragma unroll
  for (int i = 0; i < 2 * R16; i++) {
    const int piece = min(lane + 64 * i, 8 * r - 1);                 // (past the step's 64 rows: the last piece again)
    const int row = piece / per_row, c = piece - row * per_row;
    asrc[i] = (uint32_t)(row * per_row + (c ^ swap_a(row))) * 16;
  }
  const T* xsrc[2 * NT];                                             // lane l takes position l % 8 of row l / 8
#pragma unroll
  for (int i = 0; i < 2 * NT; i++) {
    const int row = 8 * i + (lane >> 3);
    xsrc[i] = a.x + (long)s_rows[min(row, cnt - 1)] * a.x_stride + 8 * ((lane & 7) ^ (row & 7));
  }
  unsigned char* mine = smem + wave * Tile::kWaveBytes;
  const uint32_t mine_lds = (uint32_t)(uintptr_t)mine;
  const int steps = a.k >> 6, n = max(0, (steps - wave + WAVES - 1) / WAVES);
  auto issue = [&](int i) {
    const int st = wave + WAVES * i;
    const uint32_t lds = mine_lds + (DEPTH == 1 ? 0 : (i % DEPTH) * Tile::kStageBytes);
#pragma unroll
    for (int ii = 0; ii < 2 * R16; ii++) {
      const uint32_t d = __builtin_amdgcn_readfirstlane(lds + 1024 * ii);
      direct_load(asrc[ii], wa + (long)st * 128 * r, d);
    }
#pragma unroll
    for (int ii = 0; ii < 2 * NT; ii++) {
      const uint32_t d = __builtin_amdgcn_readfirstlane(lds + 2048 * R16 + 1024 * ii);
      direct_load(xsrc[ii] + (long)st * 64, d);
    }
  };
  lm_float4 acc[R16][NT];
#pragma unroll
  for (int rt = 0; rt < R16; rt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[rt][nt] = lm_float4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int i = 0; i < DEPTH; i++)
    if (i < n) issue(i);
  for (int i = 0; i < n; i++) {
    // requests complete in order: all but the DEPTH - 1 steps behind this one
    if (DEPTH > 1 && i + DEPTH <= n) asm volatile("s_waitcnt vmcnt(%0)" : : "n"((DEPTH - 1) * kLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    const unsigned char* s = mine + (DEPTH == 1 ? 0 : (i % DEPTH) * Tile::kStageBytes);
    lvec8<T> xv[2][NT];
    lvec4<T> lo[2][R16], hi[2][R16];
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
        xv[h][nt] = *reinterpret_cast<const lvec8<T>*>(s + 2048 * R16 + (16 * nt + j) * 128 + ((4 * h + q) ^ (j & 7)) * 16);
#pragma unroll
      for (int rt = 0; rt < R16; rt++) {
        // rows 8 q .. + 3 and + 4 .. + 7, columns 16 rt .. + 15 (columns past r hold other weights: dropped below)
        const int c = 2 * rt + ((j & 3) >> 1), row = 32 * h + 8 * q + (j >> 2);
        lo[h][rt] = lds_read_transposed<T>(s + (row * per_row + (c ^ swap_a(row))) * 16 + 8 * (j & 1));
        hi[h][rt] = lds_read_transposed<T>(s + ((row + 4) * per_row + (c ^ swap_a(row + 4))) * 16 + 8 * (j & 1));
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");             // the place has been read
    __builtin_amdgcn_sched_barrier(0);
    if (i + DEPTH < n) issue(i + DEPTH);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int rt = 0; rt < R16; rt++) {
        const typename LoraMfma<T>::v8 A = {lo[h][rt][0], lo[h][rt][1], lo[h][rt][2], lo[h][rt][3], hi[h][rt][0], hi[h][rt][1], hi[h][rt][2], hi[h][rt][3]};
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[rt][nt] = LoraMfma<T>::run(A, xv[h][nt], acc[rt][nt]);
      }
  }

  // The first columns of B: 64 of them a piece, 128 bytes of each rank; a request covers 8 ranks.  Columns past m repeat the last ones
  // (they are not stored).  Ranks past r (a multiple of 8) are cleared: a weight there that is not finite would turn the product with
  // the zero intermediate into a NaN.
  const T* b = a.b + (long)bin * r * a.m;
  auto swap_b = [](int rank) { return (rank >> 1) & 7; };
  const int strips = (c1 - c0 + 63) >> 6;
  auto issue_b = [&](int first) {
#pragma unroll
    for (int i = 0; i < STRIPS; i++) {
      const int strip = first + WAVES * i;
      if (strip >= strips) break;
#pragma unroll
      for (int g = 0; g < 2 * R16; g++) {
        if (8 * g >= r) break;
        const int rank = 8 * g + (lane >> 3);
        const uint32_t d = __builtin_amdgcn_readfirstlane(mine_lds + 2048 * R16 * i + 1024 * g);
        direct_load(b + (long)rank * a.m + min(c0 + 64 * strip + 8 * ((lane & 7) ^ swap_b(rank)), a.m - 8), d);
      }
    }
  };
  issue_b(wave);
#pragma unroll
  for (int i = 0; i < STRIPS; i++)
#pragma unroll
    for (int g = 0; g < 2 * R16; g++)
      if (8 * g >= r) *reinterpret_cast<lvec8<T>*>(mine + 2048 * R16 * i + 1024 * g + 16 * lane) = lvec8<T>{0, 0, 0, 0, 0, 0, 0, 0};

  // the wavefronts' sums, added in order
  auto at = [&](int w, int tok) { return red + (w * TT + tok) * Tile::kRedStride; };
  if (!Tile::kPairs || wave >= WAVES / 2) {
#pragma unroll
    for (int rt = 0; rt < R16; rt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++) *reinterpret_cast<lm_float4*>(at(wave % Tile::kSums, 16 * nt + j) + 16 * rt + 4 * q) = acc[rt][nt];
  }
  lds_barrier();
  if (Tile::kPairs) {
    if (wave < WAVES / 2) {
#pragma unroll
      for (int rt = 0; rt < R16; rt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
          lm_float4* s = reinterpret_cast<lm_float4*>(at(wave, 16 * nt + j) + 16 * rt + 4 * q);
          const lm_float4 o = *s;
#pragma unroll
          for (int i = 0; i < 4; i++) acc[rt][nt][i] += o[i];
          *s = acc[rt][nt];
        }
    }
    lds_barrier();
  }
  for (int e = tid; e < TT * 4 * R16; e += Tile::kThreads) {
    const int tok = e / (4 * R16), f = (e - tok * (4 * R16)) * 4;
    lm_float4 s = *reinterpret_cast<const lm_float4*>(at(0, tok) + f);
#pragma unroll
    for (int w = 1; w < Tile::kSums; w++) {
      const lm_float4 o = *reinterpret_cast<const lm_float4*>(at(w, tok) + f);
#pragma unroll
      for (int i = 0; i < 4; i++) s[i] += o[i];
    }
    lvec4<T> o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = f < r ? (T)s[i] : (T)0.f;
    *reinterpret_cast<lvec4<T>*>(v + tok * Tile::kVStride + f) = o;
  }
  lds_barrier();

  int rows[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) rows[nt] = s_rows[min(16 * nt + j, cnt - 1)];
  for (int first = wave; first < strips; first += WAVES * STRIPS) {
    if (first != wave) issue_b(first);
    lvec8<T> old[STRIPS][NT][2];
#pragma unroll
    for (int i = 0; i < STRIPS; i++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          old[i][nt][h] = lvec8<T>{0, 0, 0, 0, 0, 0, 0, 0};
          const int col = c0 + 64 * (first + WAVES * i) + 16 * q + 8 * h;
          if (a.accumulate && col < c1) old[i][nt][h] = *reinterpret_cast<const lvec8<T>*>(a.y + (long)rows[nt] * a.y_stride + col);
        }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
#pragma unroll
    for (int i = 0; i < STRIPS; i++) {
      const int strip = first + WAVES * i;
      if (strip >= strips) break;
      const unsigned char* patch = mine + 2048 * R16 * i;
      lm_float4 sum[4][NT];
#pragma unroll
      for (int cc = 0; cc < 4; cc++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) sum[cc][nt] = lm_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int rt = 0; rt < R16; rt++) {
        lvec4<T> V[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) V[nt] = *reinterpret_cast<const lvec4<T>*>(v + (16 * nt + j) * Tile::kVStride + 16 * rt + 4 * q);
        const int rank = 16 * rt + 4 * q + (j >> 2);
#pragma unroll
        for (int cc = 0; cc < 4; cc++) {
          // A row 4 q' + i of MFMA cc = column 16 q' + 4 cc + i of the piece: a lane of D ends up with 16 adjacent columns
          const int c = 2 * (j & 3) + (cc >> 1);
          const lvec4<T> A = lds_read_transposed<T>(patch + rank * 128 + ((c ^ swap_b(rank)) * 16) + 8 * (cc & 1));
#pragma unroll
          for (int nt = 0; nt < NT; nt++) sum[cc][nt] = LoraMfma16<T>::run(A, V[nt], sum[cc][nt]);
        }
      }
      const int col = c0 + 64 * strip + 16 * q;
#pragma unroll
      for (int nt = 0; nt < NT; nt++) {
        if (16 * nt + j >= cnt) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          if (col + 8 * h >= c1) continue;
          lvec8<T> o;
#pragma unroll
          for (int e = 0; e < 8; e++) o[e] = (T)__builtin_fmaf(sum[2 * h + (e >> 2)][nt][e & 3], a.scale, (float)old[i][nt][h][e]);
          *reinterpret_cast<lvec8<T>*>(a.y + (long)rows[nt] * a.y_stride + col + 8 * h) = o;
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");             // the pieces have been read: the next ones may come
  }
}

}  // namespace triteia_hip
