// fp32 products on fp16 MFMA: operands as pairs of fp16 digits.
//
// Every operand row (a row of A, a column of B) is scaled by a power of two
// that puts its largest magnitude in [2^14, 2^15) and each element x is
// carried as hi = fp16(x) and lo = fp16((x - hi) 2^11).  hi and lo are within
// 2^-23 of x (fp32's 24 bits less half a bit on average) for every element down
// to 2^-28 of the row's largest; rows with smaller ones count them.
// The product is hi hi' + 2^-11 (hi lo' + lo hi'), each sum in an
// fp32 accumulator of its own; lo lo' (2^-22 of the product at most) is left
// out.  Three v_mfma_f32_32x32x16_f16 take the place of eight
// v_mfma_f32_32x32x2_f32 on 1/5 of their matrix-core time, and the leading
// sum is rounded once per 16 k instead of once per 2.
//
// Outputs that this cannot give to fp32's accuracy are computed on fp32 MFMA
// from the fp32 operands (f32_tile): those of rows that hold Inf or NaN, and sums
// of products so small that the lost parts of small elements could show in them
// (pair_mask).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pair_common.h"

namespace {

// Pair images of X [R, K] (row-major, K contiguous): per 32 rows and 16 k a
// hi and a lo fragment of 1 KiB in MFMA operand order, [r32][k16][hi|lo][32 h
// + r][8] for row r and k = 16 k16 + 8 h .. +7; zeros past R and K.  ex[row]
// is the row's exponent and count of small elements (pair_word).
// TPR threads per row, 256 / TPR rows per workgroup; UL > 0: a thread keeps
// its UL octets in registers between the row maximum and the split (K <= 8
// TPR UL), UL = 0 reads the row twice.  Bound by memory at large R (4096 x 1536:
// 25 MB in, 25 MB out, 10.4 us, 4.8 TB/s) and by its launch and one round trip at small ones, so
// rows of few workgroups take a whole workgroup each (long rows in eights, whose
// pieces fill whole lines: 4096 x 4096 -> 512 140 -> 115 us a call).
template <int TPR, int UL>
__global__ __launch_bounds__(256) void k_pair_split(const float *__restrict__ X, int64_t R,
                                                    int64_t K, int nk, int vec,
                                                    uint4 *__restrict__ img,
                                                    int *__restrict__ ex) {
  const int t = threadIdx.x, u = t % TPR;
  const int64_t row = (int64_t)blockIdx.x * (256 / TPR) + t / TPR;
  const float *x = X + row * K;
  auto load = [&](int o, float v[8]) __attribute__((always_inline)) {
    const int64_t k0 = (int64_t)o * 8;
    if (row < R && vec && k0 + 8 <= K) {
      const float4v a = *reinterpret_cast<const float4v *>(x + k0);
      const float4v b = *reinterpret_cast<const float4v *>(x + k0 + 4);
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = a[i], v[4 + i] = b[i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = row < R && k0 + i < K ? x[k0 + i] : 0.f;
    }
  };
  // Largest and smallest nonzero magnitude as bits: ordered as integers, Inf
  // and NaN largest.
  unsigned mx = 0, mn = ~0u;
  auto amax = [&](const float v[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      mx = max(mx, __builtin_bit_cast(unsigned, v[i]) & 0x7fffffffu);
      mn = min(mn, pair_bits1(v[i]));
    }
  };
  const int no = 2 * nk;
  float v[UL ? UL : 1][8];
  if constexpr (UL > 0) {
#pragma unroll
    for (int j = 0; j < UL; j++) load(u + TPR * j, v[j]);
#pragma unroll
    for (int j = 0; j < UL; j++) amax(v[j]);
  } else {
    for (int o = u; o < no; o += TPR) {
      load(o, v[0]);
      amax(v[0]);
    }
  }
  for (int o = std::min(TPR, 64) / 2; o > 0; o >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, o));
  if constexpr (TPR > 64) {
    __shared__ unsigned wmx[4];
    if ((t & 63) == 0) wmx[t >> 6] = mx;
    __syncthreads();
    mx = max(max(wmx[0], wmx[1]), max(wmx[2], wmx[3]));
  }
  const int e = pair_exponent(mx);
  // (The thread's own smallest spares the count where there is none.)
  const unsigned below = pair_small_below(e);
  int small = 0;
  auto store = [&](int o, const float w[8]) __attribute__((always_inline)) {
    if (o >= no) return;
    if (mn < below)
#pragma unroll
      for (int i = 0; i < 8; i++) small += pair_bits1(w[i]) < below;
    half8 hi, lo;
    pair_split8(w, e, &hi, &lo);
    uint4 *d = img + (((row >> 5) * nk + (o >> 1)) * 2) * 64 + 32 * (o & 1) + (row & 31);
    d[0] = __builtin_bit_cast(uint4, hi);
    d[64] = __builtin_bit_cast(uint4, lo);
  };
  if constexpr (UL > 0) {
#pragma unroll
    for (int j = 0; j < UL; j++) store(u + TPR * j, v[j]);
  } else {
    for (int o = u; o < no; o += TPR) {
      load(o, v[0]);
      store(o, v[0]);
    }
  }
  for (int o = std::min(TPR, 64) / 2; o > 0; o >>= 1) small += __shfl_xor(small, o);
  if constexpr (TPR > 64) {
    __shared__ int wsm[4];
    if ((t & 63) == 0) wsm[t >> 6] = small;
    __syncthreads();
    small = wsm[0] + wsm[1] + wsm[2] + wsm[3];
  }
  if (u == 0) ex[row] = pair_word(e, mx, small);
}

// One wave's quarter of the sums of a 32 x 32 output tile of A [M, K] . B [N,
// K]^T on fp32 MFMA, operands read straight from memory: MFMA i of eight k holds
// k = i (lanes 0-31) and 4 + i (lanes 32-63), so that a lane's four k are one
// 16-byte load (vec: rows are aligned for it).  The next 32 k are on their way
// during the products.  Rows past M and columns past N repeat the last one;
// nobody stores their sums.
__device__ inline float16v f32_tile(const float *__restrict__ A, const float *__restrict__ B,
                                    int64_t M, int64_t N, int64_t K, int vec, int64_t r0,
                                    int64_t c0, int wave, int lane) {
  const float *pa = A + min(r0 + (lane & 31), M - 1) * K, *pb = B + min(c0 + (lane & 31), N - 1) * K;
  const int64_t per = (K + 127) / 128 * 32, kend = min(K, (wave + 1) * per);
  const int64_t k0 = 4 * (lane >> 5);
  float4v a[2][4], b[2][4];
  auto load = [&](int d, int64_t kb) __attribute__((always_inline)) {
    if (vec && kb + 32 <= kend) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        a[d][j] = *reinterpret_cast<const float4v *>(pa + kb + 8 * j + k0);
        b[d][j] = *reinterpret_cast<const float4v *>(pb + kb + 8 * j + k0);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int64_t k = kb + 8 * j + k0 + i;
          a[d][j][i] = k < kend ? pa[k] : 0.f;
          b[d][j][i] = k < kend ? pb[k] : 0.f;
        }
    }
  };
  float16v acc = {};
  auto step = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[d][j][i], b[d][j][i], acc, 0, 0, 0);
  };
  load(0, wave * per);
  for (int64_t kb = wave * per; kb < kend; kb += 64) {
    load(1, kb + 32);
    step(0);
    load(0, kb + 64);
    step(1);
  }
  return acc;
}

struct PairArgs {
  const uint4 *ai, *bi;     // pair images
  const int *ae, *be;       // row exponents and counts (pair_word)
  const float *a, *b;       // the fp32 operands (f32_tile)
  int64_t M, N, K;
  int vec;                  // their rows are 16-byte aligned
  int nk, nx, pr, pc;       // 16-k steps; tile grid and its XCD cut
  float alpha, beta;
  const float *c;
  int64_t c_rs, c_cs, ldy;
  float *y;
};

// A 64 x 64 workgroup tile, the four waves a quarter of the 16-k steps each,
// their sums added in wave order through LDS.  Fragments stream from L2
// straight into registers, two steps in flight.
// What bounds it is the rate at which a CU takes fragments in (8 KiB per wave
// and 12 MFMAs; a workgroup alone on a CU gets ~90 GB/s), with launch, first
// loads and epilogue around it at small sizes.  Measured (4096 x 384 -> 1536
// / 4096 x 1536 -> 384 / 256 x 2048 -> 512, us a call with the split of A;
// fp32 MFMA kernel 58 / 57 / 30): this form 30.7 / 31.6 / 19.6; 128 x 128
// tiles without the K shares 32.1 / 45.8 / 44.8; fragments through an LDS
// ring of 4 steps, 128 x 128 tiles 31.3 / 45.1 / 46.7 and 64 x 64 tiles 48.3 /
// 38.9 / 23.2; three steps in flight 31.8 / 32.1 / 19.8.  One form for all
// sizes also keeps an output's sums independent of M and N: rows and column
// slices that take it (mg_pair_pays) agree bitwise.
__global__ __launch_bounds__(256, 2) void k_pair_gemm(const PairArgs p) {
  constexpr int T = 64, KW = 4;
  __shared__ float4v part[KW][4][4][64];  // [wave][32 x 32 block][v / 4][lane]
  __shared__ __attribute__((aligned(16))) int exps[2 * T];
  __shared__ int counts[2];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int tr, tc;
  {
    const int L = (int)blockIdx.x;
    if (p.pr == 0) {
      tr = L / p.nx;
      tc = L % p.nx;
    } else {
      const int ny = (int)((p.M + T - 1) / T);
      const int x = L & 7, i = L >> 3, br = x / p.pc, bcol = x % p.pc;
      const int rlo = br * ny / p.pr, rhi = (br + 1) * ny / p.pr;
      const int clo = bcol * p.nx / p.pc, chi = (bcol + 1) * p.nx / p.pc;
      const int w = chi - clo;
      if (i >= (rhi - rlo) * w) return;  // uniform: the whole workgroup leaves
      tr = rlo + i / w;
      tc = clo + i % w;
    }
  }
  const int nk = p.nk, per = nk / KW;  // steps; of each wave (nk is a multiple of 4)
  const int64_t r0 = (int64_t)tr * T, c0 = (int64_t)tc * T;
  auto rsrc = [](const void *base) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, 0x7ffffff0,
                                             0x00020000);
  };
  const __amdgpu_buffer_rsrc_t ra = rsrc(p.ai + (r0 >> 5) * nk * 128);
  const __amdgpu_buffer_rsrc_t rb = rsrc(p.bi + (c0 >> 5) * nk * 128);
  half8 a[2][2][2], b[2][2][2];
  auto load = [&](int d, int k) __attribute__((always_inline)) {
    k += wave * per;
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        a[d][i][g] = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(ra, lane * 16 + g * 1024,
                                                         (i * nk + k) * 2048, 0));
        b[d][i][g] = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(rb, lane * 16 + g * 1024,
                                                         (i * nk + k) * 2048, 0));
      }
  };
  // The tile's words (images reach to whole 64-row blocks) and a column's
  // C where C is a row: read here, not in the epilogue, where each would be a
  // round trip of its own.
  const int l32 = lane & 31, h = lane >> 5;
  if (t < 2 * T) {  // waves 0 and 1
    exps[t] = t < T ? p.ae[r0 + t] : p.be[c0 + t - T];
    const bool some = __ballot(pair_word_small(exps[t]) > 0) != 0;
    if (lane == 0) counts[wave] = some;
  }
  float cb[2] = {0.f, 0.f};
  if (p.c && p.c_rs == 0)
#pragma unroll
    for (int j = 0; j < 2; j++) cb[j] = p.c[min(c0 + 32 * j + l32, p.N - 1) * p.c_cs];
  float16v s1[2][2];
  pair_sums(a, b, per, s1, load);
  // (The barrier of the sum also publishes exps and counts.)
  const float16v sum = pair_reduce(part, wave, lane, s1);
  // This wave's 32 x 32 block (i, j) of the tile: lane l holds column l % 32
  // and rows 8 (v / 4) + 4 (l / 32) + v % 4.
  const int i = wave >> 1, j = wave & 1;
  const int64_t tr0 = r0 + 32 * i, tc0 = c0 + 32 * j;
  const bool mine = tr0 < p.M && tc0 < p.N;
  const int wb = exps[T + 32 * j + l32];
  int wa[16];
#pragma unroll
  for (int v = 0; v < 16; v += 4) {
    const int4 x = *reinterpret_cast<const int4 *>(&exps[32 * i + 4 * h + 2 * v]);
    wa[v] = x.x, wa[v + 1] = x.y, wa[v + 2] = x.z, wa[v + 3] = x.w;
  }
  // Without small elements in the tile's rows and columns no output is redone (a
  // barrier at the end of every workgroup took 3 us of FFN1's 32).
  const bool check = (counts[0] | counts[1]) != 0;  // uniform
  // y = alpha sum + beta C of the outputs in `which`.  Stores of the others, and
  // past M or N, go past the resource and are dropped in hardware.
  auto finish = [&](const float16v &s, unsigned which) __attribute__((always_inline)) {
    const int64_t col = tc0 + l32, rw = tr0 + 4 * h;
    float cv[16];
#pragma unroll
    for (int v = 0; v < 16; v++) cv[v] = cb[j];
    if (p.c && p.c_rs) {
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int64_t row = rw + 8 * (v >> 2) + (v & 3);
        cv[v] = p.c[row < p.M && col < p.N ? row * p.c_rs + col * p.c_cs : 0];
      }
    }
    const __amdgpu_buffer_rsrc_t ry = rsrc(p.y + tr0 * p.ldy + tc0);
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int lr = 4 * h + 8 * (v >> 2) + (v & 3);
      float y = s[v];
      if (p.alpha != 1.f) y = p.alpha * y;
      if (p.c) y = y + (p.beta != 1.f ? p.beta * cv[v] : cv[v]);
      const bool st = tr0 + lr < p.M && col < p.N && (which >> v & 1);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, y), ry,
                                            st ? (unsigned)(lr * (int)p.ldy + l32) * 4u : 0x80000000u,
                                            0, 0);
    }
  };
  float16v s;
#pragma unroll
  for (int v = 0; v < 16; v++) s[v] = ldexpf(sum[v], -(pair_word_exp(wa[v]) + pair_word_exp(wb)));
  if (!check) {
    if (mine) finish(s, ~0u);
    return;
  }
  const unsigned mask = mine ? pair_mask(part, wave, lane, wa, wb) : 0u;
  if (mine) finish(s, ~mask);
  pair_redo(
      part, wave, lane, mask,
      [&](int q, int w) __attribute__((always_inline)) {
        return f32_tile(p.a, p.b, p.M, p.N, p.K, p.vec, r0 + 32 * (q >> 1), c0 + 32 * (q & 1), w,
                        lane);
      },
      [&](const float16v &e) __attribute__((always_inline)) { finish(e, mask); });
}

}  // namespace

// 16-k steps of the images: K padded with zeros to a multiple of 64 k, so
// that the K shares of a tile's waves are equal.
static int64_t mg_pair_steps(int64_t K) { return (K + 63) / 64 * 4; }

size_t mg_pair_bytes(int64_t R, int64_t K) {
  const int64_t r = (R + 63) / 64 * 64, nk = mg_pair_steps(K);
  return mg_align((size_t)(r * nk * 64)) + mg_align((size_t)r * 4);
}

// N: 32-bit offsets within an output tile.  K: the images of 64 rows of A, the
// least that a call takes, within a chunk, which is at most 2^18 - 64 (the
// fragments' 32-bit offsets would reach 2^23).  And no more than twice the
// weight's own bytes (N >= 32 always), or a MiB, go into the images, whose rows are
// padded to 64: a 1 x 2^20 weight of 4 MiB would take 256.
bool mg_pair_keeps(int64_t N, int64_t K) {
  return N > 0 && K >= 192 && N < ((int64_t)1 << 22) && K < ((int64_t)1 << 18) &&
         (int64_t)mg_pair_bytes(64, K) <= MG_PAIR_CHUNK_BYTES &&
         (int64_t)mg_pair_bytes(N, K) <= 8 * N * K + (1 << 20);
}

// Where the pairs pay: the split of A (a launch, and 12 bytes of traffic per
// element beside the 4 that fp32 products read) against products at two to three
// times the rate.  us a call on fp32 MFMA / on pairs, rows x K -> N:
// - Short sums do not: 1024 x 128 -> 1024 7.5 / 9.4, 4096 x 64 -> 4096 33 / 40.
//   At K = 192 only few rows (64 -> 64 7.7 / 7.9; K = 224 to 256 0.97 to 0.9 of the
//   time) and many outputs (4096 -> 1024 22.2 / 21.1, 8192 -> 768 0.80).
// - Few rows are bound by the chain over K, which the pairs' four waves share,
//   whatever N is: 1024 x 256 -> 1 9.1 / 9.1, 16 x 512 -> 64 14.7 / 8.8, 2048 x
//   384 -> 64 12.9 / 12.1, 1024 x 8192 -> 64 0.74, 2048 x 8192 -> 64 1.46; 1536 x
//   256 -> 512 1.12, -> 768 0.90.
// - Many rows are bound by the traffic of A at few columns: 32768 x 1024 -> 64
//   50 / 86, -> 128 88 / 98, -> 256 151 / 123, -> 1024 564 / 321; 8192 x 384 -> 128
//   1.40, 8192 x 1024 -> 128 0.80, 16384 x 384 -> 128 1.16, -> 192 0.91; 8192 x 256 ->
//   256 1.11, -> 384 0.99; 8192 x 4096 -> 128 1.53, -> 192 1.12, -> 256 0.90; 4096 x
//   8192 -> 384 1.04, -> 512 0.87.
// A column slice of a weight gives bitwise the whole one's columns where both are
// on one side of these lines: up to 1024 rows they read rows and K only (K >= 256).
bool mg_pair_pays(int64_t M, int64_t N, int64_t K) {
  if (K < 256) return K >= 192 && (M <= 128 || (N >= 768 && M * N >= (int64_t)1 << 22));
  if (M <= 2048 && M * K <= (int64_t)1 << 23 && K >= (M <= 1024 ? 256 : 384)) return true;
  if (K < 384) return N >= (M <= 2048 ? 768 : 384);
  if (K <= 2048) return N >= (M <= 8192 ? 128 : 192);
  return K <= 4096 ? N >= 256 : K <= 8192 && N >= 512;
}

mg_status mg_pair_split(mg_ctx *ctx, const float *x_dev, int64_t R, int64_t K, void *img) {
  const int64_t rp = (R + 63) / 64 * 64;
  const int nk = (int)mg_pair_steps(K);
  uint4 *im = static_cast<uint4 *>(img);
  int *ex = reinterpret_cast<int *>(static_cast<char *>(img) + mg_align((size_t)(rp * nk * 64)));
  const int vec = reinterpret_cast<uintptr_t>(x_dev) % 16 == 0 && K % 4 == 0;
#define MG_SPLIT(TPR, UL)                                                                    \
  hipLaunchKernelGGL((k_pair_split<TPR, UL>), dim3((unsigned)(rp / (256 / TPR))), dim3(256), 0, \
                     ctx->stream, x_dev, R, K, nk, vec, im, ex)
  if (rp * K >= (int64_t)1 << 20 && (K <= 2048 || rp >= 2048)) {
    if (K <= 512) MG_SPLIT(32, 2);
    else if (K <= 1024) MG_SPLIT(32, 4);
    else if (K <= 2048) MG_SPLIT(32, 8);
    else MG_SPLIT(32, 0);
  } else {
    if (K <= 2048) MG_SPLIT(256, 1);
    else if (K <= 8192) MG_SPLIT(256, 4);
    else MG_SPLIT(256, 0);
  }
#undef MG_SPLIT
  return mg_launch_check("k_pair_split");
}

mg_status mg_pair_run(mg_ctx *ctx, const mg_f32_problem &p, const float *a_dev,
                      const void *a_img, const float *b_dev, const void *b_img, float *y_dev) {
  const int64_t mp = (p.M + 63) / 64 * 64, np = (p.N + 63) / 64 * 64;
  PairArgs q{};
  q.nk = (int)mg_pair_steps(p.K);
  q.ai = static_cast<const uint4 *>(a_img);
  q.bi = static_cast<const uint4 *>(b_img);
  q.ae = reinterpret_cast<const int *>(static_cast<const char *>(a_img) + mg_align((size_t)(mp * q.nk * 64)));
  q.be = reinterpret_cast<const int *>(static_cast<const char *>(b_img) + mg_align((size_t)(np * q.nk * 64)));
  q.a = a_dev;
  q.b = b_dev;
  q.vec = p.K % 4 == 0 && reinterpret_cast<uintptr_t>(a_dev) % 16 == 0 &&
          reinterpret_cast<uintptr_t>(b_dev) % 16 == 0;
  q.M = p.M;
  q.N = p.N;
  q.K = p.K;
  q.alpha = p.alpha;
  q.beta = p.beta;
  q.c = p.c;
  q.c_rs = p.c_rs;
  q.c_cs = p.c_cs;
  q.ldy = p.ldy ? p.ldy : p.N;
  q.y = y_dev;
  const int64_t nx = np / 64, ny = mp / 64;
  q.nx = (int)nx;
  int64_t per = 0;
  const bool cut = mg_f32_xcd_cut(ny, nx, &q.pr, &q.pc, &per);
  if (!cut) q.pr = q.pc = 0;
  const unsigned gx = (unsigned)(cut ? 8 * per : nx * ny);
  hipLaunchKernelGGL(k_pair_gemm, dim3(gx), dim3(256), 0, ctx->stream, q);
  return mg_launch_check("k_pair_gemm");
}
