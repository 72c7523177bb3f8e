// GELU (erf form) on the way from an fp32 accumulator to bf16.
#pragma once
#include "rt_common.h"

namespace rt {

__device__ __forceinline__ float gelu_erf(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }

// Two GELU results in bf16, the bits of gelu_erf's. erff computes two ranges per lane, which in the epilogue of a 768 -> 3072
// product took nearly as long as the product. Here erf(x / sqrt 2) is x P(x^2) on |x| <= 5.2 (degree 13 in v = x^2 / 13.52 - 1, least
// squares reweighted towards the maximum) and 1 beyond: 3.3e-7 from erff at most, over all x. The results with 5e-7 more and
// 5e-7 less enclose gelu_erf's fp32 result; both rounding to the same bf16, that is the answer, else erff decides: about 1 pair of
// 2500 for x around 0, every second one at -3.8. 41.5k rows, 768 -> 3072, inputs of
// standard deviation 0.55 / 1.1: 389 / 467 -> 290 / 307 us (without GELU 242); 24k rows, 384 -> 1536: 108 / 144 -> 82 / 82 (49).
// gelu2_fast: the packed results and whether they are the answer.
__device__ __forceinline__ bool gelu2_fast(float x0, float x1, uint32_t& y) {
  float hi[2], lo[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float x = k ? x1 : x0;
    const float z = __builtin_amdgcn_fmed3f(x, -5.2f, 5.2f);
    const float v = fmaf(z * z, 2.f / (5.2f * 5.2f), -1.f);
    float q = -0.0009625543607398868f;
    q = fmaf(q, v, 0.0025370221119374037f);
    q = fmaf(q, v, -0.0024429871700704098f);
    q = fmaf(q, v, 0.0036002453416585922f);
    q = fmaf(q, v, -0.009578078053891659f);
    q = fmaf(q, v, 0.017119934782385826f);
    q = fmaf(q, v, -0.0250102411955595f);
    q = fmaf(q, v, 0.03590957447886467f);
    q = fmaf(q, v, -0.04944726079702377f);
    q = fmaf(q, v, 0.06397991627454758f);
    q = fmaf(q, v, -0.07985963672399521f);
    q = fmaf(q, v, 0.10004904121160507f);
    q = fmaf(q, v, -0.13548733294010162f);
    q = fmaf(q, v, 0.2718999981880188f);
    const float h = 0.5f * x;
    hi[k] = h * fmaf(z, q, 1.f + 5e-7f);
    lo[k] = fmaf(h, -1e-6f, hi[k]);
  }
  y = pack2bf(hi[0], hi[1]);
  return y == pack2bf(lo[0], lo[1]);
}
__device__ __forceinline__ uint32_t gelu2_bf16(float x0, float x1) {
  uint32_t y;
  if (__builtin_expect(!gelu2_fast(x0, x1, y), 0)) y = pack2bf(gelu_erf(x0), gelu_erf(x1));
  return y;
}

// The pairs of x[0 .. 2 N) whose results gelu2_fast left open (a bit each), by erff in ONE copy of its code: each lane picks its
// next one.
template <int N>
__device__ __forceinline__ void gelu2_settle(const float (&x)[2 * N], uint32_t (&y)[N], unsigned open) {
  while (__any(open != 0)) {
    float a = 0.f, b = 0.f;
    const int k0 = open ? __ffs(open) - 1 : N;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      a = k == k0 ? x[2 * k] : a;
      b = k == k0 ? x[2 * k + 1] : b;
    }
    const uint32_t v = pack2bf(gelu_erf(a), gelu_erf(b));
#pragma unroll
    for (int k = 0; k < N; ++k) y[k] = k == k0 ? v : y[k];
    open &= open - 1;
  }
}

}  // namespace rt
