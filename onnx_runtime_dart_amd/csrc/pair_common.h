// Products of fp32 operands carried as pairs of fp16 digits: what the weight
// Gemm (pair.hip) and the convolution (conv_pair.hip) share.
#pragma once

#include "mg_internal.h"

typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

constexpr int kMarked = 1 << 29;  // exponent of a row with Inf or NaN

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
