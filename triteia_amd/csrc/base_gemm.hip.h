// The dense base product of a small batch: y[t] = x[t] @ W^T, W [m, k] fp16 or bf16 with rows `w_stride` apart, at most 64
// tokens.
//
// Bound by reading W once.  A workgroup takes 16 MT rows of W (output features) over all of K; its eight wavefronts take
// steps of 64 k in turn, every lane loads its 16-byte pieces of W and x straight into the MFMA operands (out^T = W x^T:
// lane l = row l % 16, k 8 (l / 16) .. + 7), and a ring of DEPTH steps per wavefront keeps the requests in flight.
// Nothing is staged: a piece of W is used by one lane once, and x (at most 64 rows) comes from L2.  The wavefronts' fp32
// sums are added in order through LDS and rounded once.
// BASE_MEASURED
#pragma once
#include "lora_mfma.hip.h"

namespace triteia_hip {

constexpr int kBaseWaves = 8;
constexpr int kBaseMaxTokens = 64;

template <class T>
struct BaseArgs {
  const T* x;         // [tokens][k], dense
  const T* w;         // [m][k], rows w_stride elements apart
  long w_stride;
  T* y;               // [tokens][m], dense
  int tokens, m, k;   // m % 16 == 0, k % 64 == 0
};

// MT: 16-feature tiles of a workgroup; NT: 16-token tiles (tokens <= 16 NT).  grid ceil(m / (16 MT)), block 512.
template <class T, int MT, int NT, int DEPTH>
__global__ __launch_bounds__(64 * kBaseWaves) void base_gemm_kernel(const BaseArgs<T> a) {
  constexpr int kStride = 16 * MT + 4;
  __shared__ __attribute__((aligned(16))) float red[kBaseWaves][16 * NT][kStride];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, q = lane >> 4;
  const int f0 = blockIdx.x * 16 * MT;
  const int steps = a.k >> 6;

  const T* wr[MT];
  const T* xr[NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) wr[mt] = a.w + (long)min(f0 + 16 * mt + j, a.m - 1) * a.w_stride + 8 * q;
#pragma unroll
  for (int nt = 0; nt < NT; nt++) xr[nt] = a.x + (long)min(16 * nt + j, a.tokens - 1) * a.k + 8 * q;   // (repeats are not stored)

  struct Frag {
    lvec8<T> w[MT][2], x[NT][2];
  };
  // (steps past the end read the last one and are not multiplied: every iteration issues the same requests)
  auto load = [&](Frag& f, int st) {
    const int k0 = min(st, steps - 1) << 6;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int u = 0; u < 2; u++) f.w[mt][u] = *reinterpret_cast<const lvec8<T>*>(wr[mt] + k0 + 32 * u);
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
      for (int u = 0; u < 2; u++) f.x[nt][u] = *reinterpret_cast<const lvec8<T>*>(xr[nt] + k0 + 32 * u);
  };
  lm_float4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[mt][nt] = lm_float4{0.f, 0.f, 0.f, 0.f};

  Frag ring[DEPTH];
#pragma unroll
  for (int i = 0; i < DEPTH; i++) load(ring[i], wave + i * kBaseWaves);
  for (int st = wave; st < steps; st += DEPTH * kBaseWaves) {
#pragma unroll
    for (int i = 0; i < DEPTH; i++) {
      const int cur = st + i * kBaseWaves;
      if (cur < steps) {
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) acc[mt][nt] = LoraMfma<T>::run(ring[i].w[mt][u], ring[i].x[nt][u], acc[mt][nt]);
      }
      load(ring[i], cur + DEPTH * kBaseWaves);
    }
  }

  // D: lane (token j, features 4 q ..)
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) *reinterpret_cast<lm_float4*>(&red[wave][16 * nt + j][16 * mt + 4 * q]) = acc[mt][nt];
  __syncthreads();
  for (int e = tid; e < a.tokens * 2 * MT; e += 64 * kBaseWaves) {
    const int t = e / (2 * MT), f = (e - t * 2 * MT) * 8;
    if (f0 + f >= a.m) continue;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = red[0][t][f + i];
#pragma unroll
    for (int w = 1; w < kBaseWaves; w++)
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] += red[w][t][f + i];
    lvec8<T> o;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = (T)v[i];
    *reinterpret_cast<lvec8<T>*>(a.y + (long)t * a.m + f0 + f) = o;
  }
}

}  // namespace triteia_hip
