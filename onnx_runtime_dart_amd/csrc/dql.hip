// DynamicQuantizeLinear on device (lib/src/onnx_ops.dart:3556-3583):
//   mn = min(0, min x), mx = max(0, max x)       (NaN never updates either)
//   scale = fl32((mx - mn) / 255)                 computed in f64
//   zp = roundHalfEven(clamp(fl32(-mn / scale), 0, 255))
//   y = clamp(roundHalfEven(fl32(x / scale)) + zp, 0, 255), or zp if scale==0
// fl32 of an f64 quotient of two floats equals the correctly rounded f32
// quotient, but the f64 form is kept to follow the reference literally.
// Two kernels: per-workgroup min/max partials, then every workgroup of the
// quantising kernel reduces the (few) partials itself and quantises its
// slice, so no host round trip sits between them.
#include <hip/hip_runtime.h>

#include <cmath>

#include "mg_internal.h"

namespace {

constexpr int DQL_PARTS = 512;

typedef float float4v __attribute__((ext_vector_type(4)));

// The workgroup's smallest and largest value and bad flag, in every thread:
// within the waves by shuffles, across them through LDS with one barrier (a
// tree over 256 LDS slots took eight).
__device__ inline void dql_reduce(float &mn, float &mx, int &bad) {
  __shared__ float smn[4], smx[4];
  __shared__ int sbad[4];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o));
    mx = fmaxf(mx, __shfl_xor(mx, o));
  }
  bad = __ballot(bad) != 0;
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) smn[w] = mn, smx[w] = mx, sbad[w] = bad;
  __syncthreads();
  mn = fminf(fminf(smn[0], smn[1]), fminf(smn[2], smn[3]));
  mx = fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3]));
  bad = sbad[0] | sbad[1] | sbad[2] | sbad[3];
}

// Both kernels take x in quads (16-byte loads where x is aligned; y in 4-byte
// stores) and n % 4 elements by the first threads; with one element per load
// and store 512 x 1024 took 4.0 + 5.0 us (now 2.5 + 3.6), bound by latency and instruction
// count, not by the 2 MB.
__global__ __launch_bounds__(256) void k_dql_partial(const float *__restrict__ x,
                                                     int64_t n, int vec, float *__restrict__ pmn,
                                                     float *__restrict__ pmx,
                                                     int *__restrict__ pbad) {
  float mn = 0.f, mx = 0.f;
  int bad = 0;
  auto take = [&](float v) __attribute__((always_inline)) {
    if (v < mn) mn = v;
    if (v > mx) mx = v;
    if (!isfinite(v)) bad = 1;
  };
  const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  const int64_t n4 = vec ? n / 4 : 0;
  for (int64_t i = i0; i < n4; i += step) {
    const float4v v = reinterpret_cast<const float4v *>(x)[i];
#pragma unroll
    for (int j = 0; j < 4; j++) take(v[j]);
  }
  for (int64_t i = 4 * n4 + i0; i < n; i += step) take(x[i]);
  dql_reduce(mn, mx, bad);
  if (threadIdx.x == 0) {
    pmn[blockIdx.x] = mn;
    pmx[blockIdx.x] = mx;
    pbad[blockIdx.x] = bad;
  }
}

__device__ inline double round_even(double v) { return rint(v); }

__global__ __launch_bounds__(256) void k_dql_quant(
    const float *__restrict__ x, int64_t n, int vec, const float *__restrict__ pmn,
    const float *__restrict__ pmx, const int *__restrict__ pbad, int nparts,
    uint8_t *__restrict__ y, void *__restrict__ scale_zp) {
  // The first quad is on its way while the partials are reduced.
  const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  const int64_t n4 = vec ? n / 4 : 0;
  float4v first = {};
  if (i0 < n4) first = reinterpret_cast<const float4v *>(x)[i0];
  float mn = 0.f, mx = 0.f;
  int bad = 0;
  for (int i = threadIdx.x; i < nparts; i += 256) {
    mn = fminf(mn, pmn[i]);
    mx = fmaxf(mx, pmx[i]);
    bad |= pbad[i];
  }
  dql_reduce(mn, mx, bad);
  const double dmn = mn, dmx = mx;
  const float scale_f = (float)((dmx - dmn) / 255.0);
  const double scale = scale_f;
  const float zpf = scale == 0.0 ? 0.f : (float)(-dmn / scale);
  double zc = zpf;
  zc = zc < 0.0 ? 0.0 : (zc > 255.0 ? 255.0 : zc);
  const int zp = (int)round_even(zc);
  auto quant = [&](float v) __attribute__((always_inline)) {
    int q;
    if (scale == 0.0) {
      q = zp;
    } else {
      const float r = (float)((double)v / scale);
      q = isfinite(r) ? (int)round_even((double)r) + zp : zp;
    }
    return (uint32_t)(q < 0 ? 0 : (q > 255 ? 255 : q));
  };
  for (int64_t i = i0; i < n4; i += step) {
    const float4v v = i == i0 ? first : reinterpret_cast<const float4v *>(x)[i];
    reinterpret_cast<uint32_t *>(y)[i] =
        quant(v[0]) | quant(v[1]) << 8 | quant(v[2]) << 16 | quant(v[3]) << 24;
  }
  for (int64_t i = 4 * n4 + i0; i < n; i += step) y[i] = (uint8_t)quant(x[i]);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    float *sp = static_cast<float *>(scale_zp);
    int *ip = static_cast<int *>(scale_zp);
    sp[0] = scale_f;
    ip[1] = zp;
    ip[2] = (bad && scale != 0.0) ? 1 : 0;
  }
}

}  // namespace

size_t mg_dql_ws_bytes(int64_t) { return 3 * mg_align(DQL_PARTS * 4); }

mg_status mg_dql_run(mg_ctx *ctx, const float *x_dev, int64_t n,
                     uint8_t *y_dev, void *scale_zp_dev, void *ws) {
  char *p = static_cast<char *>(ws);
  float *pmn = reinterpret_cast<float *>(p);
  float *pmx = reinterpret_cast<float *>(p + mg_align(DQL_PARTS * 4));
  int *pbad = reinterpret_cast<int *>(p + 2 * mg_align(DQL_PARTS * 4));
  // Quads need x on 16 and y on 4 bytes.
  const int vec = reinterpret_cast<uintptr_t>(x_dev) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(y_dev) % 4 == 0;
  int64_t parts = (n + (vec ? 1023 : 255)) / (vec ? 1024 : 256);
  if (parts > DQL_PARTS) parts = DQL_PARTS;
  if (parts < 1) parts = 1;
  hipLaunchKernelGGL(k_dql_partial, dim3((unsigned)parts), dim3(256), 0, ctx->stream, x_dev, n,
                     vec, pmn, pmx, pbad);
  MG_TRY(mg_launch_check("k_dql_partial"));
  hipLaunchKernelGGL(k_dql_quant, dim3((unsigned)parts), dim3(256), 0, ctx->stream, x_dev, n,
                     vec, pmn, pmx, pbad, (int)parts, y_dev, scale_zp_dev);
  return mg_launch_check("k_dql_quant");
}
