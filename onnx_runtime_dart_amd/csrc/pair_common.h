// Products of fp32 operands carried as pairs of fp16 digits: what the weight
// Gemm (pair.hip) and the convolution (conv_pair.hip) share.
#pragma once

#include "mg_internal.h"

typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

constexpr int kMarked = 1 << 29;  // exponent of a scope with Inf or NaN

// A scope of one scale (a row of A, a column of B) in one word: its exponent e
// and how many of its elements are small, scaled magnitudes in (0, 2^-13).  The
// digits of the others are within 2^-23 of the element, those of a small one
// only within 2^-36, which can be all of it (1 beside 1e20).  Such errors come
// to at most 2^-21 (na + nb) in a sum of products, the other factors being below
// 2^15.  So an output keeps them below 2^-21 of its sum of magnitudes where that
// is at least na + nb; where it may not be, the output is computed on fp32 MFMA
// (pair_mask).  Ordinary data meets none: its partial sums are some 2^23 sqrt(K).
// In the place of the count stand kPairInf for a scope with Inf or NaN, whose
// digits are zeros, so that all its outputs are redone, and kPairZero for one of
// zeros, whose outputs (exact zeros) are not, unless the other is kPairInf.
constexpr int kPairMaxSmall = 1 << 18, kPairZero = -(1 << 19), kPairInf = 1 << 20;

__device__ inline int pair_word(int e, unsigned mx, int small) {
  if (e == kMarked) return kPairInf * 1024 + 512;
  return (mx ? min(small, kPairMaxSmall) : kPairZero) * 1024 + e + 512;
}
__device__ inline int pair_word_exp(int w) { return (w & 1023) - 512; }
__device__ inline int pair_word_small(int w) { return w >> 10; }

// Magnitudes below this (as bits, less one) are small in a scope of exponent e.
__device__ inline unsigned pair_small_below(int e) {
  return max(__builtin_bit_cast(unsigned, ldexpf(1.f, -13 - e)), 1u) - 1u;
}
// v's magnitude as bits, less one: zeros come out largest.
__device__ inline unsigned pair_bits1(float v) {
  return (__builtin_bit_cast(unsigned, v) & 0x7fffffffu) - 1u;
}

// Exponent that puts the largest magnitude (its bits, mx) in [2^14, 2^15).
__device__ inline int pair_exponent(unsigned mx) {
  if (mx >= 0x7f800000u) return kMarked;
  if (!mx) return 0;
  int xp;
  frexpf(__builtin_bit_cast(float, mx), &xp);
  return 15 - xp;
}

// The pair of eight fp32 values scaled by 2^e; zeros in a marked row.
__device__ inline void pair_split8(const float v[8], int e, half8 *hi, half8 *lo) {
  *hi = *lo = (half8){};
  if (e == kMarked) return;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float x = ldexpf(v[i], e);
    const _Float16 h = (_Float16)x;
    (*hi)[i] = h;
    (*lo)[i] = (_Float16)((x - (float)h) * 2048.f);
  }
}

// Sums of one wave over n 16-k steps of a 64 x 64 tile: load(d, k) fills a[d]
// and b[d] ([32-row block][hi, lo]) with step k's fragments, k < n.
template <class Load>
__device__ inline void pair_sums(const half8 (&a)[2][2][2], const half8 (&b)[2][2][2], int n,
                                 float16v (&s1)[2][2], Load load) {
  constexpr int D = 2;
  float16v s2[2][2];
#pragma unroll
  for (int i = 0; i < 4; i++) s1[i >> 1][i & 1] = s2[i >> 1][i & 1] = (float16v){};
  auto step = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < 3; g++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
          float16v &s = g == 0 ? s1[i][j] : s2[i][j];
          s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[d][i][g == 2], b[d][j][g == 1], s, 0, 0, 0);
        }
  };
#pragma unroll
  for (int d = 0; d < D; d++) load(d, min(d, n - 1));
  int k = 0;
  for (; k + D <= n; k += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      step(d);
      load(d, min(k + D + d, n - 1));
    }
  }
#pragma unroll
  for (int d = 0; d < D; d++)
    if (k + d < n) step(d);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) s1[i][j][v] = fmaf(s2[i][j][v], 1.f / 2048.f, s1[i][j][v]);
}

// The four waves' sums added in wave order: wave q gets block q (rows 32 (q /
// 2), columns 32 (q % 2)) of the tile.  part is read after a barrier.
__device__ inline float16v pair_reduce(float4v (*part)[4][4][64], int wave, int lane,
                                       const float16v (&s1)[2][2]) {
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const float16v &s = s1[q >> 1][q & 1];
      part[wave][q][v][lane] = (float4v){s[4 * v], s[4 * v + 1], s[4 * v + 2], s[4 * v + 3]};
    }
  __syncthreads();
  float16v sum;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    float4v x = part[0][wave][v][lane];
#pragma unroll
    for (int w = 1; w < 4; w++) x += part[w][wave][v][lane];
#pragma unroll
    for (int e = 0; e < 4; e++) sum[4 * v + e] = x[e];
  }
  return sum;
}

// Which of a lane's 16 outputs (bits v) of block `wave` are to be redone: those
// whose words (wa[v], wb) count small elements and whose sums of magnitudes, of
// which the waves' partial sums are a lower bound, may be too small beside them.
__device__ inline unsigned pair_mask(const float4v (*part)[4][4][64], int wave, int lane,
                                     const int (&wa)[16], int wb) {
  unsigned mask = 0;
#pragma unroll
  for (int v = 0; v < 16; v++) {
    float mag = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) mag += __builtin_fabsf(part[w][wave][v >> 2][lane][v & 3]);
    mask |= (unsigned)(mag < (float)(pair_word_small(wa[v]) + pair_word_small(wb))) << v;
  }
  return mask;
}

// The blocks of a workgroup's tile that have outputs to be redone (mask, for this
// wave's block): for each, the four waves share the products, tile(q, wave)
// giving this wave's part of block q's sums on fp32 MFMA, and wave q takes
// their sums: store(sums).
template <class Tile, class Store>
__device__ inline void pair_redo(float4v (*part)[4][4][64], int wave, int lane, unsigned mask,
                                 Tile tile, Store store) {
  __shared__ int redo[4];
  const bool mine = __ballot(mask != 0) != 0;
  if (lane == 0) redo[wave] = mine;
  __syncthreads();
  for (int q = 0; q < 4; q++) {
    if (!redo[q]) continue;  // uniform
    const float16v s = tile(q, wave);
#pragma unroll
    for (int v = 0; v < 4; v++)
      part[wave][q][v][lane] = (float4v){s[4 * v], s[4 * v + 1], s[4 * v + 2], s[4 * v + 3]};
    __syncthreads();
    if (wave != q) continue;
    float16v sum;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      float4v x = part[0][q][v][lane];
#pragma unroll
      for (int w = 1; w < 4; w++) x += part[w][q][v][lane];
#pragma unroll
      for (int e = 0; e < 4; e++) sum[4 * v + e] = x[e];
    }
    store(sum);
  }
}
