// Quantise + prune + pack a dense fp16 weight [k, m] into the 2:4 int4 layout (sparse24_gemm.hip.h) in one pass.
//
// Per output column and aligned group of 4 along k: the two entries of largest magnitude are kept (of equal ones the
// later, i.e. what a stable ascending sort leaves; a NaN counts as larger than everything), each becomes
// clamp(round(fp16(w / scale)) + 8, 0, 15), and their positions the 4-bit code lo | hi << 2.  Every rounding is the
// torch codec's (fp32 division, rounded to fp16, round to nearest even), so the bytes are the codec's
// (triteia/python/nn/linear.py:79-141, triteia/python/ops/utils/sparsity.py:35-61,99-118,134-161).
//
// Bound by memory: 2 B read and 0.5 B written per weight.  A wavefront takes one packed row (32 dense k) x 128 columns, a
// lane two adjacent columns: its 32 loads are independent dwords (256 contiguous bytes per wavefront) and all in
// flight together.  A 32-bit word of the layout interleaves the columns c and c + 4, which are two lanes apart: one
// exchange with lane ^ 2 gives each lane whole words, and the packed row's 1 KB of weights and 512 B of metadata are
// written by the wavefront that read it.  The workgroup's eight wavefronts are eight packed rows below each other,
// which makes the pieces of the logical metadata (row = column, stride k / 8 B) 32 B long.
// 4096 x 4096: 6442 us as some two hundred torch kernels (4.9 ms of them a segmented sort of groups of four) -> 11.8 us
// (3.5 TB/s; the vector ALUs and memory are about even: with comparisons by rank and the compiler's divisions 22 us).
#pragma once
#include "sparse24_gemm.hip.h"

namespace triteia_hip {

constexpr int kPackRows = 8;       // packed rows (wavefronts) per workgroup
constexpr int kPackCols = 128;     // columns per workgroup

// One column's 8 groups.  word[a]: the column's share of word (a, w) of the layout (before the shift by 8 of the upper
// four columns of a block); meta: the codes of its first / second 16 dense k in the lower / upper half.
struct PackedColumn {
  uint32_t word[4];
  uint32_t meta;
};

// fp16(fp32 v / s) rounded to an integer in [-8, 7], as half(1024 + 8 + integer).  The quotient is v * (1 / s) and one
// correction by its remainder, within 2^-24 (1 + 2^-20) of the exact one: v and s have 11-bit mantissas, so an exact
// quotient that is not itself a midpoint between two halves (12 bits) is at least 2^-23 away from every such midpoint,
// and one that is a midpoint comes out exactly: the integer is that of a correctly rounded division (the GPU test compares
// all 2^32 pairs of fp16 values), for 4 instructions instead of its 12.  The first estimate is bounded so that the
// remainder of an infinite quotient is not a NaN; `s_rem` is s, or 0 for an infinite s (whose product with the estimate 0
// would be one).  NaNs (0 / 0) count as zero.  The sum with 1032 in fp16 rounds to whole numbers, ties to even.
__device__ __forceinline__ _Float16 pack_quotient(_Float16 v, float s_rem, float inv) {
  const float x = (float)v;
  const float estimate = __builtin_amdgcn_fmed3f(x * inv, -16.f, 16.f);
  float q = __builtin_fmaf(__builtin_fmaf(-estimate, s_rem, x), inv, estimate);
  q = q == q ? q : 0.f;
  return (_Float16)__builtin_amdgcn_fmed3f(q, -8.f, 7.f);
}

// `key[i]`: magnitude of entry i in the upper 16 bits, i in bits 15:14, its sign in bit 0 -- all different, ordered by
// magnitude and then by position, so that the two kept entries are the two largest.
__device__ __forceinline__ void pack_group(const uint32_t (&key)[4], float s_rem, float inv, uint32_t* pair, uint32_t* code) {
  const uint32_t a = max(key[0], key[1]), b = min(key[0], key[1]), c = max(key[2], key[3]), d = min(key[2], key[3]);
  const uint32_t first = max(a, c), second = max(max(min(a, c), b), d);
  const uint32_t i1 = (first >> 14) & 3u, i2 = (second >> 14) & 3u;
  const uint32_t lo = i1 < i2 ? first : second, hi = i1 < i2 ? second : first;
  *code = min(i1, i2) | (max(i1, i2) << 2);
  auto value = [](uint32_t k) { return __builtin_bit_cast(_Float16, (uint16_t)((k >> 16) | (k << 15))); };
  const half2_t q = {pack_quotient(value(lo), s_rem, inv), pack_quotient(value(hi), s_rem, inv)};
  *pair = h2_bits(q + half2_t{(_Float16)1032.0f, (_Float16)1032.0f}) & 0x000f000fu;
}

// grid (ceil(m / 128), ceil(k / 256)), block 512.  m % 64 == 0, k % 32 == 0.
__global__ __launch_bounds__(64 * kPackRows) void pack_2_4_kernel(const _Float16* __restrict__ w, const _Float16* __restrict__ scales,
                                                                 int k, int m, uint32_t* __restrict__ qweight,
                                                                 uint32_t* __restrict__ meta, uint32_t* __restrict__ meta_raw) {
  const int lane = threadIdx.x & 63;
  const int tr = blockIdx.y * kPackRows + (threadIdx.x >> 6);
  const int col = blockIdx.x * kPackCols + 2 * lane;
  if (tr >= (k >> 5) || col >= m) return;   // (columns end at a multiple of 64: a quad of lanes is inside or outside as one)
  const uint32_t* wp = reinterpret_cast<const uint32_t*>(w + (long)tr * 32 * m + col);
  uint32_t x[32];
#pragma unroll
  for (int i = 0; i < 32; i++) x[i] = wp[(long)i * (m >> 1)];
  const half2_t s = *reinterpret_cast<const half2_t*>(scales + col);
  float inv[2], s_rem[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    s_rem[c] = (float)s[c];
    inv[c] = __builtin_amdgcn_rcpf(s_rem[c]);
    if (__builtin_fabsf(s_rem[c]) == __builtin_inff()) s_rem[c] = 0.f;
  }
  PackedColumn c0, c1;
  c0.meta = c1.meta = 0;
#pragma unroll
  for (int g = 0; g < 8; g++) {
    uint32_t k0[4], k1[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      // both columns' magnitudes, every NaN as the same one above infinity
      typedef uint16_t ushort2_t __attribute__((ext_vector_type(2)));
      const uint32_t v = x[4 * g + i];
      const uint32_t mag = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(ushort2_t, v & 0x7fff7fffu),
                                                                                 ushort2_t{0x7c01, 0x7c01}));
      k0[i] = (mag << 16) | (uint32_t)(i << 14) | ((v >> 15) & 1u);
      k1[i] = (mag & 0xffff0000u) | (uint32_t)(i << 14) | (v >> 31);
    }
    uint32_t p0, p1, code0, code1;
    pack_group(k0, s_rem[0], inv[0], &p0, &code0);
    pack_group(k1, s_rem[1], inv[1], &p1, &code1);
    c0.word[g & 3] = g < 4 ? p0 : c0.word[g & 3] | (p0 << 4);
    c1.word[g & 3] = g < 4 ? p1 : c1.word[g & 3] | (p1 << 4);
    c0.meta |= code0 << (4 * g);
    c1.meta |= code1 << (4 * g);
  }

  // lane = 4 i4 + l: l = 0, 1 hold the lower four columns (words w = 2 l, 2 l + 1) of block i4, l = 2, 3 the upper four.
  // The lower lanes finish vectors a = 0, 1 and the upper lanes a = 2, 3.
  const bool upper = lane & 2;
  const int half = lane & 1;
  uint32_t* qp = qweight + (long)tr * 2 * m + (long)(col >> 6) * 128 + ((col & 63) >> 3) * 16 + 2 * half;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const uint32_t send0 = upper ? c0.word[j] : c0.word[j + 2], send1 = upper ? c1.word[j] : c1.word[j + 2];
    const uint32_t got0 = __shfl_xor(send0, 2, 64), got1 = __shfl_xor(send1, 2, 64);
    const uint32_t own0 = upper ? c0.word[j + 2] : c0.word[j], own1 = upper ? c1.word[j + 2] : c1.word[j];
    uint2 out;
    out.x = upper ? got0 | (own0 << 8) : own0 | (got0 << 8);
    out.y = upper ? got1 | (own1 << 8) : own1 | (got1 << 8);
    *reinterpret_cast<uint2*>(qp + 4 * (upper ? j + 2 : j)) = out;
  }
  // metadata, 16-bit index [b1 b5 b4 b3 b0 h b2] inside 64 columns: a dword holds b2 = 0, 1 of one (column pair, h); the
  // lower lane finishes b0 = 0, the upper one b0 = 1
  {
    const uint32_t send = upper ? c0.meta : c1.meta;
    const uint32_t got = __shfl_xor(send, 2, 64);
    const uint32_t low = upper ? got : c0.meta, high = upper ? c1.meta : got;   // b2 = 0 / b2 = 1
    uint2 out;
    out.x = (low & 0xffffu) | (high << 16);             // h = 0
    out.y = (low >> 16) | (high & 0xffff0000u);         // h = 1
    const int b1 = lane & 1, b543 = (lane >> 2) & 7, b0 = upper ? 1 : 0;
    *reinterpret_cast<uint2*>(meta + (long)tr * m + (long)(col >> 6) * 64 + 32 * b1 + 4 * b543 + 2 * b0) = out;
  }
  const long raw_row = k >> 5;   // dwords per column
  meta_raw[(long)col * raw_row + tr] = c0.meta;
  meta_raw[(long)(col + 1) * raw_row + tr] = c1.meta;
}

}  // namespace triteia_hip
