// LoRA pair for tokens in any order, on adapters as a program holds them (A [M, k, r], B [M, r, m] row-major):
//
//   y[t] (+)= scale * (x[t] @ A[i]) @ B[i],   i = indices[t] in [0, M);  other tokens: nothing added, or zeros stored
//
// in two launches and nothing else: no routing launch, no transposed copies of the adapters, no segment table from the
// host, no clearing of the output or of the intermediate.
//
// Bound by latency: a chain of dependent round trips (indices -> rows and adapter -> operands -> partial sums -> output)
// over a few MB that mostly come from cache.  So
//   * every workgroup of the shrink routes by itself: the batch's indices (at most 4096) go to LDS with a histogram of
//     the adapters, a scan over that finds the workgroup's tile (16 NT tokens of one adapter), ballots list its tokens in
//     batch order.  About 2 us, against a launch of its own (5 - 7 us with its gap).  The workgroups of a tile's
//     first share of K leave the tile and its token rows behind for the expand;
//   * K is split over gridDim.y so that a few tiles still fill the chip and a wavefront has all of its operands in flight at
//     once: the adapter's rows by direct-to-LDS loads (a step of 32 k is 64 r consecutive bytes), activations straight into
//     the B operand.  The fp32 shares are added in order by the expand, which rounds the intermediate to T once;
//   * both contractions run on the matrix cores as out^T = W^T x^T.  W has its output index fastest, the operand wants
//     k fastest: ds_read_b64_tr_b16 transposes on the way out of LDS (lane i of 16 gives the address of row i / 4, columns
//     4 (i % 4) ..; it receives column i of the four rows: measured on the device).  16-byte chunks are XOR-swizzled by row.
// Measured: 100 Zipf-routed tokens over 32 adapters of rank 16 on 4096 x 11008, two transposing copies and the BGMV pair
// 48 us -> 9.2 us a call, 8.4 in a graph; 1000 tokens over 8 of rank 64 on 4096 x 4096 in bf16, 31 + 9 us of kernels behind 250 us of
// host round trips -> 19.2 us a call, 17.9 in a graph, of which 8 MB each in and out take 4.
#pragma once
#include "lora_mfma.hip.h"

namespace triteia_hip {

constexpr int kLoraMaxTokens = 4096;      // indices in LDS
constexpr int kLoraMaxAdapters = 1024;    // histogram in LDS
constexpr int kLoraMaxSplits = 8;         // shares of K
constexpr int kLoraExpandCols = 256;      // output columns of an expand workgroup

template <class T>
struct LoraArgs {
  const T* x;
  long x_stride;
  const T* a;              // [M, k, r]
  const T* b;              // [M, r, m]
  T* y;
  long y_stride;
  const void* indices;     // int32 or int64 per token
  int index64;
  int n_tokens, n_adapters, k, r, m;
  int splits;              // shares of K (gridDim.y of the shrink)
  float scale;
  int accumulate;          // 1: y += result; 0: y = result, and tokens without an adapter get zeros
  int4* tiles;             // scratch: {adapter (-1: none), first list position, tokens, 0}; 0 tokens = no tile
  int* perm;               // scratch: token of each list position
  float* partial;          // scratch: [splits][list position][r]
};

// at most this many tiles of `tt` tokens: one partial tile per group (the tokens without an adapter are one) in use
__host__ __device__ inline int lora_max_tiles(int n_tokens, int n_adapters, int tt) {
  const int groups = n_adapters + 1 < n_tokens ? n_adapters + 1 : n_tokens;
  return groups + n_tokens / tt;
}

template <class T> struct LoraMfma16;      // 16 x 16 x 16: 4 elements of k per lane
template <> struct LoraMfma16<_Float16> {
  static __device__ __forceinline__ lm_float4 run(lvec4<_Float16> a, lvec4<_Float16> b, lm_float4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  }
};
template <> struct LoraMfma16<__bf16> {
  static __device__ __forceinline__ lm_float4 run(lvec4<__bf16> a, lvec4<__bf16> b, lm_float4 c) {
    typedef short short4_v __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(short4_v, a), __builtin_bit_cast(short4_v, b), c, 0, 0, 0);
  }
};

// four rows x 16 columns, transposed: see the head of this file
template <class T>
__device__ __forceinline__ lvec4<T> lds_read_transposed(const unsigned char* p) {
  typedef short short4_v __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(lvec4<T>, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_v*)p));
}

// 16 bytes per lane from global memory to LDS at `dst` (the same in every lane) + 16 * lane
__device__ __forceinline__ void load_to_lds(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(uintptr_t)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
__device__ __forceinline__ void wait_for_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Inclusive sum over a wavefront's lanes (six additions on the vector ALU; through shuffles, which go by LDS, they took 0.3 us).
__device__ __forceinline__ int lane_sums(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);     // row_shr:1, 2, 4, 8: inside rows of 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);     // row_bcast:15: a row's last lane to the row behind (rows 1 and 3)
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);     // row_bcast:31: the first half's sum to rows 2 and 3
  return v;
}

// Every workgroup routes by itself: the tile (TT tokens of one adapter, in batch order) that is number `tile` of the batch, its
// token rows in s_rows.  All of the workgroup's wavefronts call it; all wavefronts are past their last use of s.idx and s.hist when it
// returns a tile.
struct LoraTile {
  int bin;        // adapter; n_adapters: tokens without one; -1: no such tile
  int start;      // first list position: adapters in ascending order, their tokens in the batch's
  int count;      // tokens
};
template <int THREADS, int TT>
struct LoraRouteTables {
  uint16_t* idx;      // [tokens]
  int* hist;          // [adapters + 1]
  int* wave_count;    // [THREADS / 64]
  int* rows;          // [TT]
};
template <int THREADS, int TT, class T>
__device__ __forceinline__ LoraTile lora_find_tile(const LoraArgs<T>& a, const int tile, const LoraRouteTables<THREADS, TT>& s) {
  constexpr int WAVES = THREADS / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int none = a.n_adapters;                               // bin of the tokens without an adapter

  auto count = [&](int t, long v) {
    const int d = v >= 0 && v < none ? (int)v : none;
    s.idx[t] = (uint16_t)d;
    atomicAdd(&s.hist[d], 1);                                  // (integer counts: the order does not matter)
  };
  auto count_all = [&](auto* indices) {
    if (a.n_tokens <= THREADS) {
      const long v = tid < a.n_tokens ? (long)indices[tid] : 0;   // (on its way while the bins are cleared)
      for (int i = tid; i <= none; i += THREADS) s.hist[i] = 0;
      __syncthreads();
      if (tid < a.n_tokens) count(tid, v);
      return;
    }
    for (int i = tid; i <= none; i += THREADS) s.hist[i] = 0;
    __syncthreads();
    // (four requests a lane in flight: the pair, 1000 tokens over 8 adapters of rank 64 19.25 -> 18.95 us, 2000 over 16 of rank 16 23.5 -> 22.5;
    // level at 257 .. 512 tokens, which have two)
    for (int t = tid; t < a.n_tokens; t += 4 * THREADS) {
      long v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = indices[min(t + THREADS * i, a.n_tokens - 1)];
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (t + THREADS * i < a.n_tokens) count(t + THREADS * i, v[i]);
    }
  };
  if (a.index64) count_all(static_cast<const long*>(a.indices));
  else count_all(static_cast<const int*>(a.indices));
  __syncthreads();

  // the bin that the tile belongs to, its tokens' first list position and the tile's number inside the bin
  int bin = -1, bin_tokens = 0, start = 0, in_bin = 0;
  for (int base = 0, before = 0; base <= none; base += 64) {   // (before: tiles << 16 | tokens of the bins so far)
    const int b = base + lane;
    const int c = b > none || (b == none && a.accumulate) ? 0 : s.hist[b];
    const int own = ((c + TT - 1) / TT) << 16 | c;
    const int incl = lane_sums(own) + before, excl = incl - own;
    const unsigned long long hit = __ballot(tile >= (excl >> 16) && tile < (incl >> 16));
    if (hit) {
      const int src = __ffsll((long long)hit) - 1;
      bin = base + src;
      bin_tokens = __builtin_amdgcn_readlane(c, src);
      const int e = __builtin_amdgcn_readlane(excl, src);
      start = e & 0xffff;
      in_bin = tile - (e >> 16);
      break;
    }
    before = __builtin_amdgcn_readlane(incl, 63);
  }
  if (bin < 0) return {-1, 0, 0};
  const int rank0 = in_bin * TT;
  const int cnt = min(TT, bin_tokens - rank0);
  const int pieces = (a.n_tokens + 63) >> 6, per_wave = (pieces + WAVES - 1) / WAVES;
  const int first = wave * per_wave, last = min(pieces, first + per_wave);
  int rank = -rank0;
  if (per_wave == 1) {
    // one piece a wavefront: each counts the pieces before its own itself
#pragma unroll
    for (int w = 0; w < WAVES - 1; w++)
      if (w < wave) rank += __popcll(__ballot(64 * w + lane < a.n_tokens && s.idx[64 * w + lane] == bin));
  } else {
    int mine = 0;
    for (int ch = first; ch < last; ch++) {
      const int t = ch * 64 + lane;
      mine += __popcll(__ballot(t < a.n_tokens && s.idx[t] == bin));
    }
    if (lane == 0) s.wave_count[wave] = mine;
    __syncthreads();
    for (int w = 0; w < wave; w++) rank += s.wave_count[w];
  }
  for (int ch = first; ch < last; ch++) {
    const int t = ch * 64 + lane;
    const bool member = t < a.n_tokens && s.idx[t] == bin;
    const unsigned long long members = __ballot(member);
    const int at = rank + __popcll(members & ((1ull << lane) - 1ull));
    if (member && at >= 0 && at < cnt) s.rows[at] = t;
    rank += __popcll(members);
  }
  __syncthreads();
  return {bin, start + rank0, cnt};
}

// R16: 16-rank tiles (r <= 16 R16); NT: 16-token tiles.  grid (tiles, shares of K), block 256.
template <class T, int R16, int NT>
__global__ __launch_bounds__(256) void lora_shrink_kernel(const LoraArgs<T> a) {
  constexpr int TT = 16 * NT;
  constexpr int S = R16 == 8 ? 2 : (R16 == 1 ? 8 : 4);        // steps of 32 k that a wavefront requests together
  constexpr int kSlab = 1024 * R16;                            // bytes of a step's adapter rows
  constexpr int kRedStride = 16 * R16 + 4;
  constexpr int kRedBytes = 4 * TT * kRedStride * 4, kSlabBytes = 4 * S * kSlab;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kSlabBytes > kRedBytes ? kSlabBytes : kRedBytes];
  __shared__ uint16_t s_idx[kLoraMaxTokens];
  __shared__ int s_hist[kLoraMaxAdapters + 1];
  __shared__ int s_wave_count[4];
  __shared__ int s_rows[TT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int none = a.n_adapters, tile = blockIdx.x;
  const LoraTile found = lora_find_tile<256, TT>(a, tile, {s_idx, s_hist, s_wave_count, s_rows});
  const int bin = found.bin, start = found.start, cnt = found.count;
  if (bin < 0) {
    if (blockIdx.y == 0 && tid == 0) a.tiles[tile] = make_int4(0, 0, 0, 0);
    return;
  }
  if (blockIdx.y == 0) {
    if (tid == 0) a.tiles[tile] = make_int4(bin == none ? -1 : bin, start, cnt, 0);
    if (tid < cnt) a.perm[start + tid] = s_rows[tid];
  }
  if (bin == none) return;

  const int j = lane & 15, kq = lane >> 4;
  const int r = a.r, chunks_per_row = r >> 3;
  const int swizzle = (r & (r - 1)) == 0 ? chunks_per_row - 1 : 0;
  const char* w = reinterpret_cast<const char*>(a.a + (long)bin * a.k * r);
  int src[R16];                        // byte offset inside a step's rows of this lane's piece of each 1 KB
#pragma unroll
  for (int i = 0; i < R16; i++) {
    const int p = min(lane + 64 * i, 4 * r - 1);
    const int row = p / chunks_per_row, c = p - row * chunks_per_row;
    src[i] = (row * chunks_per_row + (c ^ (row & swizzle))) * 16;
  }
  const T* xr[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) xr[nt] = a.x + (long)s_rows[min(16 * nt + j, cnt - 1)] * a.x_stride + 8 * kq;

  lm_float4 acc[R16][NT];
#pragma unroll
  for (int rt = 0; rt < R16; rt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[rt][nt] = lm_float4{0.f, 0.f, 0.f, 0.f};

  const int steps = a.k >> 5, per = (steps + a.splits - 1) / a.splits;
  const int s0 = blockIdx.y * per, s1 = min(steps, s0 + per);
  unsigned char* slabs = smem + wave * S * kSlab;
  for (int base = s0 + wave; base < s1; base += 4 * S) {
    lvec8<T> xv[S][NT];
#pragma unroll
    for (int i = 0; i < S; i++) {
      const int st = base + 4 * i;
      if (st >= s1) break;                                     // (the same for the whole wavefront)
#pragma unroll
      for (int ii = 0; ii < R16; ii++) load_to_lds(w + (long)st * 64 * r + src[ii], slabs + i * kSlab + ii * 1024);
#pragma unroll
      for (int nt = 0; nt < NT; nt++) xv[i][nt] = *reinterpret_cast<const lvec8<T>*>(xr[nt] + st * 32);
    }
    wait_for_loads();
#pragma unroll
    for (int i = 0; i < S; i++) {
      if (base + 4 * i >= s1) break;
#pragma unroll
      for (int rt = 0; rt < R16; rt++) {
        // rows 8 kq .. + 3 and + 4 .. + 7, columns 16 rt .. + 15 (columns past r hold other weights: dropped below)
        const int c = 2 * rt + ((j & 3) >> 1);
        const int row = 8 * kq + (j >> 2);
        const lvec4<T> lo = lds_read_transposed<T>(slabs + i * kSlab + (row * chunks_per_row + (c ^ (row & swizzle))) * 16 + 8 * (j & 1));
        const lvec4<T> hi = lds_read_transposed<T>(slabs + i * kSlab + ((row + 4) * chunks_per_row + (c ^ ((row + 4) & swizzle))) * 16 + 8 * (j & 1));
        const typename LoraMfma<T>::v8 A = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[rt][nt] = LoraMfma<T>::run(A, xv[i][nt], acc[rt][nt]);
      }
    }
  }

  // the wavefronts' sums, added in order, to this share's rows of the partial buffer
  __syncthreads();                     // the slabs have been read for the last time
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int rt = 0; rt < R16; rt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
      *reinterpret_cast<lm_float4*>(red + (wave * TT + 16 * nt + j) * kRedStride + 16 * rt + 4 * kq) = acc[rt][nt];
  __syncthreads();
  const int quads = r >> 2;
  float* out = a.partial + ((long)blockIdx.y * a.n_tokens + start) * r;
  for (int e = tid; e < cnt * quads; e += 256) {
    const int tok = e / quads, f = (e - tok * quads) * 4;
    lm_float4 s = *reinterpret_cast<const lm_float4*>(red + tok * kRedStride + f);
#pragma unroll
    for (int v = 1; v < 4; v++) {
      const lm_float4 o = *reinterpret_cast<const lm_float4*>(red + (v * TT + tok) * kRedStride + f);
#pragma unroll
      for (int q = 0; q < 4; q++) s[q] += o[q];
    }
    *reinterpret_cast<lm_float4*>(out + (long)tok * r + f) = s;
  }
}

// grid (tiles, ceil(m / 256)), block 256: a wavefront takes 64 columns.
template <class T, int R16, int NT>
__global__ __launch_bounds__(256) void lora_expand_kernel(const LoraArgs<T> a) {
  constexpr int TT = 16 * NT, R = 16 * R16;
  constexpr int kVStride = R + 8;
  __shared__ __attribute__((aligned(1024))) unsigned char patch[R * 512];      // [rank][256 columns]
  __shared__ __attribute__((aligned(16))) T v[TT * kVStride];
  const int4 d = a.tiles[blockIdx.x];
  const int cnt = d.z;
  if (cnt <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c0 = blockIdx.y * kLoraExpandCols;
  if (d.x < 0) {
    const int chunks = min(kLoraExpandCols, a.m - c0) >> 3;
    for (int e = tid; e < cnt * chunks; e += 256) {
      const int tok = e / chunks, c = e - tok * chunks;
      *reinterpret_cast<lvec8<T>*>(a.y + (long)a.perm[d.y + tok] * a.y_stride + c0 + 8 * c) = lvec8<T>{0, 0, 0, 0, 0, 0, 0, 0};
    }
    return;
  }
  // the adapter's patch: a request covers two rank rows; columns past m repeat the last ones (they are not stored).  Rows
  // past r (r is a multiple of 8: both rows of a request) are cleared: a weight there that is not finite would turn the
  // product with the zero intermediate into a NaN.
  const T* b = a.b + (long)d.x * a.r * a.m;
#pragma unroll
  for (int i = 0; i < 2 * R16; i++) {
    const int piece = (wave + 4 * i) * 64 + lane, row = piece >> 5, c = (piece & 31) ^ (row & 31);
    if (2 * (wave + 4 * i) < a.r) load_to_lds(b + (long)row * a.m + min(c0 + 8 * c, a.m - 8), patch + (wave + 4 * i) * 1024);
    else *reinterpret_cast<lvec8<T>*>(patch + piece * 16) = lvec8<T>{0, 0, 0, 0, 0, 0, 0, 0};
  }
  const int j = lane & 15, q = lane >> 4;
  const int col = c0 + 64 * wave + 8 * q;            // this lane's output columns: col .. + 7 and col + 32 .. + 39
  int rows[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) rows[nt] = a.perm[d.y + min(16 * nt + j, cnt - 1)];
  // the intermediate: the shares of K in order, rounded once (eight ranks of a token at a time, all shares requested together:
  // against four at a time the pair with eight shares, 400 tokens over 32 adapters of rank 16 on 4096 x 4096 10.0 -> 9.6 us, 512 over 8 of rank 64
  // in bf16 18.0 -> 17.7, 1000 18.1 -> 17.9; launches of up to four, 100 over 32 of rank 16 on 4096 x 11008 among them, are level)
  for (int e = tid; e < TT * 2 * R16; e += 256) {
    const int tok = e / (2 * R16), f = (e - tok * (2 * R16)) * 8;
    lvec8<T> o = {0, 0, 0, 0, 0, 0, 0, 0};
    if (tok < cnt && f < a.r) {
      const float* p = a.partial + (long)(d.y + tok) * a.r + f;
      lm_float4 part[kLoraMaxSplits][2];
#pragma unroll
      for (int z = 0; z < kLoraMaxSplits; z++) {
        if (z >= a.splits) break;
        part[z][0] = *reinterpret_cast<const lm_float4*>(p);
        part[z][1] = *reinterpret_cast<const lm_float4*>(p + 4);
        p += (long)a.n_tokens * a.r;
      }
      lm_float4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int z = 0; z < kLoraMaxSplits; z++) {
        if (z >= a.splits) break;
#pragma unroll
        for (int i = 0; i < 4; i++) { lo[i] += part[z][0][i]; hi[i] += part[z][1][i]; }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) { o[i] = (T)lo[i]; o[4 + i] = (T)hi[i]; }
    }
    *reinterpret_cast<lvec8<T>*>(v + tok * kVStride + f) = o;
  }
  lvec8<T> old[NT][2];
#pragma unroll
  for (int nt = 0; nt < NT; nt++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      old[nt][h] = lvec8<T>{0, 0, 0, 0, 0, 0, 0, 0};
      if (a.accumulate) old[nt][h] = *reinterpret_cast<const lvec8<T>*>(a.y + (long)rows[nt] * a.y_stride + min(col + 32 * h, a.m - 8));
    }
  wait_for_loads();
  __syncthreads();

  lm_float4 acc[4][NT];
#pragma unroll
  for (int cc = 0; cc < 4; cc++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[cc][nt] = lm_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int rt = 0; rt < R16; rt++) {
    lvec4<T> B[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) B[nt] = *reinterpret_cast<const lvec4<T>*>(v + (16 * nt + j) * kVStride + 16 * rt + 4 * q);
    const int row = 16 * rt + 4 * q + (j >> 2);
#pragma unroll
    for (int cc = 0; cc < 4; cc++) {
      // A row 4 q' + i of MFMA cc = column 32 (cc / 2) + 8 q' + 4 (cc % 2) + i of the wavefront's 64: a lane of D ends up with two runs of
      // 8 columns, and a store of four lanes with 64 consecutive bytes of a token
      const int c = 8 * wave + 4 * (cc >> 1) + (j & 3);
      const lvec4<T> A = lds_read_transposed<T>(patch + row * 512 + ((c ^ (row & 31)) * 16) + 8 * (cc & 1));
#pragma unroll
      for (int nt = 0; nt < NT; nt++) acc[cc][nt] = LoraMfma16<T>::run(A, B[nt], acc[cc][nt]);
    }
  }
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    if (16 * nt + j >= cnt) continue;
    T* yp = a.y + (long)rows[nt] * a.y_stride + col;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (col + 32 * h >= a.m) continue;
      lvec8<T> o;
#pragma unroll
      for (int i = 0; i < 8; i++) o[i] = (T)__builtin_fmaf(acc[2 * h + (i >> 2)][nt][i & 3], a.scale, (float)old[nt][h][i]);
      *reinterpret_cast<lvec8<T>*>(yp + 32 * h) = o;
    }
  }
}

}  // namespace triteia_hip
