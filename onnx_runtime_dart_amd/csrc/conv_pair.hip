// fp32 Conv (one group) as an implicit GEMM on fp16 digit pairs
// (pair_common.h): lib/src/onnx_nn_ops.dart:179-817.
//
// Rows of the product are the output channels (the filters, scaled by a power
// of two per channel), columns the output positions of all images (the input,
// scaled per image), k = (16-channel block, tap).  Two launches lay the
// operands out:
//   * k_conv_pair_prep: the filters' pair fragments, [m32][step][hi|lo][lane]
//     with step = block * taps + tap, and the largest magnitude of each chunk
//     of each image;
//   * k_conv_pair_x: the input as [image][block][hi|lo][position][16] with the
//     padding written out as zeros, a position being one of the padded window,
//     and the number of small elements of each image (pair_common.h).
// So a step's operand of 32 consecutive output positions is 32-byte pieces
// at the positions' window origins (one 32-bit offset per lane, the same in
// every step) plus the step's own offset, a scalar: the products' loop has
// no gather arithmetic, no masks and no LDS.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pair_common.h"

namespace {

constexpr int kMaxChunks = 64;  // chunk maxima per image (one per lane of a wave)

// Ints between the counters that workgroups add to: a line each (32 images'
// counters in one line, added to by every wave: 15 us).
constexpr int kCountStride = 64;

struct ConvPair {
  const float *x, *w, *bias;
  float *y;
  int n, c, m, taps, cb, ns;      // images, channels, 16-channel blocks, steps (padded to 4)
  int in[3], out[3], ker[3], str[3], dil[3], pad[3], win[3];  // win: padded window dims
  int in_sp, out_sp, win_sp;
  int chunks, chunk;              // maxima chunks of an image, elements of each
  uint4 *wi, *xi;                 // images of the filters and of the input
  int *we, *xe;                   // their words (pair_word) without the counts
  int *wn;                        // small elements of filter m: four counts at 4 m
  int *xn;                        // small elements of image i at i * kCountStride
  unsigned *part;                 // [n][chunks] largest magnitudes (bits)
  int nx, pr, pc;                 // tile grid and its XCD cut
  int wvec;                       // the filters' rows are 16-byte aligned
};

// Bound by latency (a few loads per thread, one round trip each way): the
// filters' rows and the input's maxima share one launch.
__global__ __launch_bounds__(256) void k_conv_pair_prep(const ConvPair p) {
  const int t = threadIdx.x;
  const int mp = (p.m + 63) / 64 * 64;
  const bool filt = (int)blockIdx.x < mp;
  const int m = blockIdx.x, K = p.c * p.taps;
  const int q = (int)blockIdx.x - mp, img = filt ? 0 : q / p.chunks, ch = q - img * p.chunks;
  const int64_t xn = (int64_t)p.c * p.in_sp;
  const float *src = filt ? p.w + (int64_t)m * K : p.x + img * xn + (int64_t)ch * p.chunk;
  const int len = filt ? (m < p.m ? K : 0)
                       : (int)std::min<int64_t>(p.chunk, xn - (int64_t)ch * p.chunk);
  unsigned mx = 0;
  for (int i = t; i < len; i += 8 * 256) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = src[min(i + 256 * u, len - 1)];
#pragma unroll
    for (int u = 0; u < 8; u++) mx = max(mx, __builtin_bit_cast(unsigned, v[u]) & 0x7fffffffu);
  }
  for (int o = 32; o > 0; o >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, o));
  __shared__ unsigned wmx[4];
  if ((t & 63) == 0) wmx[t >> 6] = mx;
  __syncthreads();
  mx = max(max(wmx[0], wmx[1]), max(wmx[2], wmx[3]));
  if (!filt) {
    if (t == 0) p.part[q] = mx;
    if (t == 0 && ch == 0) p.xn[img * kCountStride] = 0;
    return;
  }
  const int e = pair_exponent(mx);
  if (t == 0) p.we[m] = pair_word(e, mx, 0);
  const unsigned below = pair_small_below(e);
  int small = 0;
  // Octet o: channels 8 c8 .. +7 of tap r, then the padding steps' zeros.
  const int real = p.cb * p.taps;
  for (int o = t; o < 2 * p.ns; o += 256) {
    const int c8 = o / p.taps, r = o - c8 * p.taps;
    float v[8] = {};
    if (o < 2 * real && m < p.m)
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (8 * c8 + j < p.c) v[j] = src[(8 * c8 + j) * p.taps + r];
#pragma unroll
    for (int j = 0; j < 8; j++) small += pair_bits1(v[j]) < below;
    half8 hi, lo;
    pair_split8(v, e, &hi, &lo);
    const int s = o < 2 * real ? (c8 >> 1) * p.taps + r : o >> 1, h = o < 2 * real ? c8 & 1 : o & 1;
    uint4 *d = p.wi + ((int64_t)(m >> 5) * p.ns + s) * 128 + 32 * h + (m & 31);
    d[0] = __builtin_bit_cast(uint4, hi);
    d[64] = __builtin_bit_cast(uint4, lo);
  }
  // A count of each wave: no barrier, and few have any to add up.
  if (__ballot(small != 0))
    for (int o = 32; o > 0; o >>= 1) small += __shfl_xor(small, o);
  if ((t & 63) == 0) p.wn[4 * m + (t >> 6)] = small;
}

// Thread = one position of the padded window, 16 channels (grid: positions,
// channel blocks, images).  Bound by memory at large inputs.
__global__ __launch_bounds__(256) void k_conv_pair_x(const ConvPair p) {
  const int t = threadIdx.x, lane = t & 63;
  const int pos = (int)blockIdx.x * 256 + t, cb = blockIdx.y, img = blockIdx.z;
  const int zx = pos % p.win[2], zy = pos / p.win[2] % p.win[1], zz = pos / p.win[2] / p.win[1];
  const int ix = zx - p.pad[2], iy = zy - p.pad[1], iz = zz - p.pad[0];
  const bool in = pos < p.win_sp && (unsigned)ix < (unsigned)p.in[2] &&
                  (unsigned)iy < (unsigned)p.in[1] && (unsigned)iz < (unsigned)p.in[0];
  const int c0 = 16 * cb;
  const float *src = p.x + ((int64_t)img * p.c + c0) * p.in_sp +
                     (in ? (iz * p.in[1] + iy) * p.in[2] + ix : 0);
  float v[2][8];
#pragma unroll
  for (int j = 0; j < 16; j++) v[j >> 3][j & 7] = src[(int64_t)min(j, p.c - 1 - c0) * p.in_sp];
  unsigned mx = lane < p.chunks ? p.part[img * p.chunks + lane] : 0;
  for (int o = 32; o > 0; o >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, o));
  const int e = pair_exponent(mx);
  if (pos == 0 && cb == 0) p.xe[img] = pair_word(e, mx, 0);
#pragma unroll
  for (int j = 0; j < 16; j++)
    if (!in || c0 + j >= p.c) v[j >> 3][j & 7] = 0.f;
  const unsigned below = pair_small_below(e);
  unsigned mn = ~0u;
#pragma unroll
  for (int j = 0; j < 16; j++) mn = min(mn, pair_bits1(v[j >> 3][j & 7]));
  if (__ballot(mn < below)) {  // uniform; few waves of ordinary data
    int small = 0;
#pragma unroll
    for (int j = 0; j < 16; j++) small += pair_bits1(v[j >> 3][j & 7]) < below;
    for (int o = 32; o > 0; o >>= 1) small += __shfl_xor(small, o);
    if (lane == 0) atomicAdd(&p.xn[img * kCountStride], small);
  }
  if (pos >= p.win_sp) return;
  uint4 *d = p.xi + ((int64_t)img * p.cb + cb) * p.win_sp * 4 + 2 * pos;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    half8 hi, lo;
    pair_split8(v[h], e, &hi, &lo);
    d[h] = __builtin_bit_cast(uint4, hi);
    d[2 * p.win_sp + h] = __builtin_bit_cast(uint4, lo);
  }
}

// One wave's quarter of the sums of the 32 x 32 block of channels m0 .. and
// columns of which lane l's is (img, window origin oz, oy, ox), on fp32 MFMA
// straight from the tensors.  Lanes 0-31 take the first half of the quarter's k =
// (channel, tap) and 32-63 the second, each in order, so that eight k of a filter
// are two 16-byte loads (wvec: rows are aligned for it) and the tap advances by
// counting; the next eight are on their way during the products.  Channels past m
// repeat the last one; nobody stores their sums.  ResNet-50's 3 x 3 takes 202 us
// where one of its 32 images has a NaN and 248 where each has (steps of 16 channels
// at one tap, whose filter loads touch a line per lane: 200 / 346; the same with the
// tap advanced by selects in place of branches: 230 / 306).
__device__ inline float16v conv_f32_tile(const ConvPair &p, int m0, int img, int oz, int oy, int ox,
                                         int wave, int lane) {
  const int K = p.c * p.taps, half = (K + 63) / 64 * 8, steps = half / 8;
  int k = (2 * wave + (lane >> 5)) * half;  // of the next load
  const float *w = p.w + (int64_t)min(m0 + (lane & 31), p.m - 1) * K;
  const float *x = p.x + (int64_t)img * p.c * p.in_sp;
  const int ch = k / p.taps, tap = k - ch * p.taps;
  int kx = tap % p.ker[2], ky = tap / p.ker[2] % p.ker[1], kz = tap / p.ker[2] / p.ker[1];
  int ix = ox + kx * p.dil[2], iy = oy + ky * p.dil[1], iz = oz + kz * p.dil[0];
  int64_t xc = (int64_t)ch * p.in_sp;
  float a[2][8], b[2][8];
  auto load = [&](int d) __attribute__((always_inline)) {
    if (p.wvec) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const float4v v =
            k + 4 * q < K ? *reinterpret_cast<const float4v *>(w + k + 4 * q) : (float4v){};
#pragma unroll
        for (int i = 0; i < 4; i++) a[d][4 * q + i] = v[i];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) a[d][j] = k + j < K ? w[k + j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 8; j++, k++) {
      const bool ok = k < K && (unsigned)iz < (unsigned)p.in[0] &&
                      (unsigned)iy < (unsigned)p.in[1] && (unsigned)ix < (unsigned)p.in[2];
      b[d][j] = ok ? x[xc + (iz * p.in[1] + iy) * p.in[2] + ix] : 0.f;
      ix += p.dil[2];
      if (++kx == p.ker[2]) {
        kx = 0, ix = ox, iy += p.dil[1];
        if (++ky == p.ker[1]) {
          ky = 0, iy = oy, iz += p.dil[0];
          if (++kz == p.ker[0]) kz = 0, iz = oz, xc += p.in_sp;
        }
      }
    }
  };
  float16v acc = {};
  auto step = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; j++)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[d][j], b[d][j], acc, 0, 0, 0);
  };
  load(0);
  for (int s = 0; s < steps; s += 2) {
    if (s + 1 < steps) load(1);
    step(0);
    if (s + 1 == steps) break;
    if (s + 2 < steps) load(0);
    step(1);
  }
  return acc;
}

// 64 channels x 64 output positions per workgroup, the four waves a quarter
// of the steps each (pair_sums).  Bound by the rate at which a CU takes in
// fragments.  ResNet-50 3 x 3 (32 x 256 x 14 x 14 -> 256): 30 us and 47 with
// the two launches ahead of it (153 on k_conv's fp32 MFMA, whose gather and
// fp32 matrix rate bounded it); 16 x 240 x 28 x 28 -> 240: 256 -> 70 us.
__global__ __launch_bounds__(256, 2) void k_conv_pair(const ConvPair p) {
  __shared__ float4v part[4][4][4][64];
  __shared__ int exps[64];
  __shared__ float bias[64];
  __shared__ int count;
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int tr, tc;
  {
    const int L = (int)blockIdx.x;
    if (p.pr == 0) {
      tr = L / p.nx;
      tc = L % p.nx;
    } else {
      const int ny = (p.m + 63) / 64;
      const int x = L & 7, i = L >> 3, br = x / p.pc, bcol = x % p.pc;
      const int rlo = br * ny / p.pr, rhi = (br + 1) * ny / p.pr;
      const int clo = bcol * p.nx / p.pc, chi = (bcol + 1) * p.nx / p.pc;
      const int w = chi - clo;
      if (i >= (rhi - rlo) * w) return;  // uniform: the whole workgroup leaves
      tr = rlo + i / w;
      tc = clo + i % w;
    }
  }
  const int m0 = tr * 64, cols = p.n * p.out_sp, ns = p.ns, per = ns / 4;
  if (t < 64) {
    const int4 n = reinterpret_cast<const int4 *>(p.wn)[m0 + t];
    const int w = p.we[m0 + t];
    exps[t] = pair_word_small(w) ? w : w + (n.x + n.y + n.z + n.w) * 1024;
    const bool some = __ballot(pair_word_small(exps[t]) > 0) != 0;
    if (t == 0) count = some;
    bias[t] = p.bias && m0 + t < p.m ? p.bias[m0 + t] : 0.f;
  }
  // The lane's column in each of the tile's two 32-column blocks: image,
  // output position and window origin.
  int col[2], img[2], pos[2], oz[2], oy[2], ox[2], eb[2], nb[2];
  unsigned vb[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    col[j] = tc * 64 + 32 * j + l32;
    const int cc = min(col[j], cols - 1);
    img[j] = cc / p.out_sp;
    pos[j] = cc - img[j] * p.out_sp;
    ox[j] = pos[j] % p.out[2] * p.str[2];
    oy[j] = pos[j] / p.out[2] % p.out[1] * p.str[1];
    oz[j] = pos[j] / p.out[2] / p.out[1] * p.str[0];
    eb[j] = p.xe[img[j]];
    nb[j] = p.xn[img[j] * kCountStride];
    vb[j] = (unsigned)(img[j] * p.cb * p.win_sp * 64 +
                       ((oz[j] * p.win[1] + oy[j]) * p.win[2] + ox[j]) * 32 + 16 * h);
  }
  auto rsrc = [](const void *base) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, 0x7ffffff0,
                                             0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rw = rsrc(p.wi + (int64_t)(m0 >> 5) * ns * 128), rx = rsrc(p.xi);
  // This wave's next step: 16-channel block and tap; a padding step reads the
  // last real one (its filters are zero).
  const int s0 = min(wave * per, p.cb * p.taps - 1);
  int kb = s0 / p.taps, r0 = s0 % p.taps;
  int kx = r0 % p.ker[2], ky = r0 / p.ker[2] % p.ker[1], kz = r0 / p.ker[2] / p.ker[1];
  int at = -1;
  half8 a[2][2][2], b[2][2][2];
  auto load = [&](int d, int k) __attribute__((always_inline)) {
    if (k != at && at >= 0) {
      if (++kx == p.ker[2]) {
        kx = 0;
        if (++ky == p.ker[1]) {
          ky = 0;
          if (++kz == p.ker[0]) kz = 0, kb = min(kb + 1, p.cb - 1);
        }
      }
    }
    at = k;
    const int so = (kb * 2 * p.win_sp +
                    (kz * p.dil[0] * p.win[1] + ky * p.dil[1]) * p.win[2] + kx * p.dil[2]) * 32;
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        a[d][i][g] = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(
                       rw, lane * 16 + g * 1024, (i * ns + wave * per + k) * 2048, 0));
        b[d][i][g] = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(rx, vb[i], so + g * p.win_sp * 32, 0));
      }
  };
  float16v s1[2][2];
  pair_sums(a, b, per, s1, load);
  // (The barrier of the sum also publishes exps, bias and count.)
  const float16v sum = pair_reduce(part, wave, lane, s1);
  const int i = wave >> 1, j = wave & 1;
  const bool mine = m0 + 32 * i < p.m && tc * 64 + 32 * j < cols;
  const int cj = j ? col[1] : col[0], ij = j ? img[1] : img[0], pj = j ? pos[1] : pos[0];
  // A window has at most its own products' number of the image's small elements.
#pragma unroll
  for (int k = 0; k < 2; k++)
    if (pair_word_small(eb[k]) == 0) eb[k] += min(nb[k], p.c * p.taps) * 1024;
  const int wj = j ? eb[1] : eb[0];
  int wa[16];
#pragma unroll
  for (int v = 0; v < 16; v++) wa[v] = exps[32 * i + 4 * h + 8 * (v >> 2) + (v & 3)];
  // Without small elements in the tile's filters and images no output is redone.
  const bool check =  // uniform: every wave holds the tile's columns
      count != 0 || __ballot(pair_word_small(eb[0]) > 0 || pair_word_small(eb[1]) > 0) != 0;
  const __amdgpu_buffer_rsrc_t ry = rsrc(p.y);
  // The outputs in `which`; stores of the others go past the resource and are
  // dropped in hardware.
  auto finish = [&](const float16v &s, unsigned which) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int lr = 32 * i + 4 * h + 8 * (v >> 2) + (v & 3);
      const float y = p.bias ? s[v] + bias[lr] : s[v];
      __builtin_amdgcn_raw_buffer_store_b32(
          __builtin_bit_cast(unsigned, y), ry,
          m0 + lr < p.m && cj < cols && (which >> v & 1)
              ? (unsigned)((ij * p.m + m0 + lr) * p.out_sp + pj) * 4u
              : 0x80000000u,
          0, 0);
    }
  };
  float16v s;
#pragma unroll
  for (int v = 0; v < 16; v++) s[v] = ldexpf(sum[v], -(pair_word_exp(wa[v]) + pair_word_exp(wj)));
  if (!check) {
    if (mine) finish(s, ~0u);
    return;
  }
  const unsigned mask = mine ? pair_mask(part, wave, lane, wa, wj) : 0u;
  if (mine) finish(s, ~mask);
  // (Copies: arrays indexed by a lambda's argument would be kept in LDS.)
  const int i0 = img[0], i1 = img[1], z0 = oz[0], z1 = oz[1], y0 = oy[0], y1 = oy[1], x0 = ox[0],
            x1 = ox[1];
  pair_redo(
      part, wave, lane, mask,
      [=](int q, int w) __attribute__((always_inline)) {
        const bool k = q & 1;
        return conv_f32_tile(p, m0 + 32 * (q >> 1), k ? i1 : i0, (k ? z1 : z0) - p.pad[0],
                             (k ? y1 : y0) - p.pad[1], (k ? x1 : x0) - p.pad[2], w, lane);
      },
      [&](const float16v &e) __attribute__((always_inline)) { finish(e, mask); });
}

struct Plan {
  bool ok = false;
  ConvPair q{};
  int64_t nb = 0;  // images per round of launches
  size_t off_we = 0, off_wn = 0, off_xi = 0, off_xe = 0, off_xn = 0, off_part = 0, total = 0;
};

Plan plan(const mg_conv_problem &p) {
  Plan r;
  if (p.xk != MG_CONV_F32 || p.trans || p.phased || p.group != 1) return r;
  // Elements of a round's output: its resource ends 16 bytes below 2^31.
  const int64_t lim = (int64_t)1 << 29, out_max = lim - 4;
  int64_t win = 1, out = 1, in = 1, taps = 1;
  ConvPair &q = r.q;
  for (int d = 0; d < 3; d++) {
    const int64_t e = (p.out[d] - 1) * p.str[d] + (p.ker[d] - 1) * p.dil[d] + 1;
    if (p.dil[d] < 1 || p.str[d] < 1 || p.ker[d] < 1 || p.in[d] < 1 || p.out[d] < 1 || e >= lim ||
        p.in[d] >= lim || p.pad[d] >= lim || p.pad[d] <= -lim || p.dil[d] >= lim || p.str[d] >= lim)
      return r;
    win *= e, out *= p.out[d], in *= p.in[d], taps *= p.ker[d];
    if (win >= lim || out >= lim || in >= lim || taps >= lim) return r;
    q.in[d] = (int)p.in[d], q.out[d] = (int)p.out[d], q.ker[d] = (int)p.ker[d];
    q.str[d] = (int)p.str[d], q.dil[d] = (int)p.dil[d], q.pad[d] = (int)p.pad[d];
    q.win[d] = (int)e;
  }
  if (p.c < 1 || p.c >= lim || p.m < 1 || p.m >= lim || p.n < 1) return r;
  const int64_t cb = (p.c + 15) / 16, ns = (cb * taps + 3) / 4 * 4, mp = (p.m + 63) / 64 * 64;
  const int64_t img = cb * win * 64;  // bytes of one image's pairs
  // Where it pays (us a call here / on k_conv; input [n, c, size, size], m
  // channels, kernel).  Short sums stay on k_conv, whose one launch costs a
  // stage per 32 k: [4, 24, 28] 3 x 3 to 64 channels 16.1 / 15.3, [4, 64, 14]
  // 1 x 1 18 / 13, [2, 256, 14] 1 x 1 16.0 / 16.3, [1, 512, 7] 1 x 1 16.0 /
  // 28.1.  So do inputs of several times the caches' reach that meet few
  // products (they pass through memory three times here): [32, 256, 56] 1 x 1
  // to 64 channels 99 / 67, to 256 of [32, 1024, 14] 35 / 74; and channel
  // counts that the blocks of 16 more than double ([32, 3, 224] 7 x 7: 206 /
  // 153).  And so do large inputs that a stride mostly skips, unless k_conv would
  // have a long chain over k on few tiles (lines from 280 sizes of stride 2 to 4):
  // 1 x 1 stride 3 to 256 channels of [32, 512, 56] 172 / 91, stride 2 of [1, 256,
  // 112] 28 / 18.5; 4 x 4 stride 4 to 64 channels of [32, 512, 56] 497 / 393, but of
  // [8, 512, 56] 0.31 of its time.
  const int64_t mib = p.n * p.c * in * 4 >> 20;
  const int64_t tiles = mp / 64 * ((p.n * out + 63) / 64);
  if (p.c * taps < 256 || 16 * cb > 2 * p.c || (p.m * taps < 128 && mib >= 8) ||
      (mib >= 8 && 30 * 256 * mib > p.c * taps * std::max<int64_t>(256, tiles)) ||
      (mib >= 128 && p.m * taps * out < 128 * in))
    return r;
  // 32-bit offsets throughout, and the filter rows as laid out.
  if (p.w_ms != p.c * taps || p.w_cs != taps || p.c * taps > kPairMaxSmall || p.c * in >= lim ||
      mp * ns * 64 >= 4 * lim || ns * 2048 * 2 >= 4 * lim || img >= 4 * lim || p.m * out > out_max ||
      (win + 255) / 256 > 0x7fffff || cb > 65535)
    return r;
  const int64_t fit = std::min<int64_t>((64ll << 20) / img, out_max / (p.m * out));
  r.nb = std::max<int64_t>(1, std::min<int64_t>(p.n, std::min<int64_t>(fit, 65535)));
  q.c = (int)p.c, q.m = (int)p.m, q.taps = (int)taps, q.cb = (int)cb, q.ns = (int)ns;
  q.in_sp = (int)in, q.out_sp = (int)out, q.win_sp = (int)win;
  // Chunks of at least 4096 elements, at most kMaxChunks of them.
  q.chunks = (int)std::min<int64_t>(kMaxChunks, (p.c * in + 4095) / 4096);
  q.chunk = (int)((p.c * in + q.chunks - 1) / q.chunks);
  q.chunks = (int)((p.c * in + q.chunk - 1) / q.chunk);
  if (mp + r.nb * q.chunks >= 0x7fffffff) return r;
  size_t off = mg_align((size_t)(mp * ns * 64));
  r.off_we = off;
  off += mg_align((size_t)mp * 4);
  r.off_wn = off;
  off += (size_t)mp * 16;
  r.off_xi = off;
  off += mg_align((size_t)(r.nb * img));
  r.off_xe = off;
  off += mg_align((size_t)r.nb * 4);
  r.off_xn = off;
  off += (size_t)r.nb * kCountStride * 4;
  r.off_part = off;
  off += mg_align((size_t)(r.nb * q.chunks) * 4);
  r.total = off;
  r.ok = true;
  return r;
}

}  // namespace

size_t mg_conv_pair_bytes(const mg_conv_problem &p) {
  const Plan r = plan(p);
  return r.ok ? r.total : 0;
}

mg_status mg_conv_pair_run(mg_ctx *ctx, const mg_conv_problem &p, void *ws) {
  Plan r = plan(p);
  ConvPair &q = r.q;
  char *base = static_cast<char *>(ws);
  q.w = static_cast<const float *>(p.w);
  q.bias = static_cast<const float *>(p.bias);
  q.wi = reinterpret_cast<uint4 *>(base);
  q.we = reinterpret_cast<int *>(base + r.off_we);
  q.wn = reinterpret_cast<int *>(base + r.off_wn);
  q.xi = reinterpret_cast<uint4 *>(base + r.off_xi);
  q.xe = reinterpret_cast<int *>(base + r.off_xe);
  q.xn = reinterpret_cast<int *>(base + r.off_xn);
  q.part = reinterpret_cast<unsigned *>(base + r.off_part);
  q.wvec = q.c * q.taps % 4 == 0 && reinterpret_cast<uintptr_t>(p.w) % 16 == 0;
  const int mp = (q.m + 63) / 64 * 64;
  for (int64_t n0 = 0; n0 < p.n; n0 += r.nb) {
    q.n = (int)std::min(r.nb, p.n - n0);
    q.x = static_cast<const float *>(p.x) + n0 * q.c * q.in_sp;
    q.y = static_cast<float *>(p.y) + n0 * q.m * q.out_sp;
    hipLaunchKernelGGL(k_conv_pair_prep, dim3((unsigned)(mp + q.n * q.chunks)), dim3(256), 0,
                       ctx->stream, q);
    MG_TRY(mg_launch_check("k_conv_pair_prep"));
    hipLaunchKernelGGL(k_conv_pair_x,
                       dim3((unsigned)((q.win_sp + 255) / 256), (unsigned)q.cb, (unsigned)q.n),
                       dim3(256), 0, ctx->stream, q);
    MG_TRY(mg_launch_check("k_conv_pair_x"));
    const int64_t nx = ((int64_t)q.n * q.out_sp + 63) / 64, ny = mp / 64;
    int64_t per = 0;
    q.nx = (int)nx;
    const bool cut = mg_f32_xcd_cut(ny, nx, &q.pr, &q.pc, &per);
    if (!cut) q.pr = q.pc = 0;
    hipLaunchKernelGGL(k_conv_pair, dim3((unsigned)(cut ? 8 * per : nx * ny)), dim3(256), 0,
                       ctx->stream, q);
    MG_TRY(mg_launch_check("k_conv_pair"));
  }
  return MG_OK;
}
