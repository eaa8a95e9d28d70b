// The projections' epilogues, shared by the GEMM kernels.
#pragma once

#include <type_traits>

#include "mb_internal.h"

namespace mb {

// GELU with the tanh approximation, 0.5 v (1 + tanh(u)) with
// u = 0.7978845608 (v + 0.044715 v^3) (kernels-decode.ts:373-385), evaluated
// as v / (1 + exp(-2u)): 0.5 (1 + tanh(u)) is the logistic function of 2u, so
// the two forms are equal, and this one needs one exponential and no
// cancellation (exp(-2u) overflowing to inf gives -0, the limit).
__device__ __forceinline__ float gelu_tanh(float v) {
  const float u = 0.7978845608028654f * (v + 0.044715f * v * v * v);
  return v / (1.f + __expf(-2.f * u));
}

// Exact GELU 0.5 v (1 + erf(v / sqrt 2)), the codec decoder's activation,
// with erf from Abramowitz & Stegun 7.1.26 (|error| <= 1.5e-7), the form
// GELU_ERF evaluates (kernels-decode.ts:392-415).
__device__ __forceinline__ float erf_as(float x) {
  const float sgn = x >= 0.f ? 1.f : -1.f;
  const float ax = fabsf(x);
  const float t = 1.f / (1.f + 0.3275911f * ax);
  const float poly =
      ((((1.061405429f * t + -1.453152027f) * t + 1.421413741f) * t + -0.284496736f) * t +
       0.254829592f) * t;
  return sgn * (1.f - poly * expf(-ax * ax));
}
__device__ __forceinline__ float gelu_erf(float v) {
  return 0.5f * v * (1.f + erf_as(v * 0.7071067811865476f));
}

// Compile-time epilogue dispatch: f(std::integral_constant<int, EPI>{}).
template <class F>
static void with_epi(int epi, F f) {
  switch (epi) {
    case EPI_GELU: f(std::integral_constant<int, EPI_GELU>{}); break;
    case EPI_ADD: f(std::integral_constant<int, EPI_ADD>{}); break;
    case EPI_SCALE_ADD: f(std::integral_constant<int, EPI_SCALE_ADD>{}); break;
    case EPI_GELU_ERF: f(std::integral_constant<int, EPI_GELU_ERF>{}); break;
    default: f(std::integral_constant<int, EPI_STORE>{}); break;
  }
}

// Four adjacent outputs of one row: bias (or the scale of EPI_SCALE_ADD) at
// columns n .. n + 3, activation, residual (the old values at cp).
template <int EPI>
__device__ __forceinline__ float4 epilogue4(float4 v, const float* __restrict__ bias, int n,
                                            const float* cp) {
  if (EPI == EPI_SCALE_ADD) {  // bias holds the per-column scale
    const float4 c = *(const float4*)cp, sc = *(const float4*)(bias + n);
    return make_float4(c.x + sc.x * v.x, c.y + sc.y * v.y, c.z + sc.z * v.z, c.w + sc.w * v.w);
  }
  if (bias) {
    const float4 b = *(const float4*)(bias + n);
    v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
  }
  if (EPI == EPI_GELU) {
    v.x = gelu_tanh(v.x); v.y = gelu_tanh(v.y); v.z = gelu_tanh(v.z); v.w = gelu_tanh(v.w);
  }
  if (EPI == EPI_GELU_ERF) {
    v.x = gelu_erf(v.x); v.y = gelu_erf(v.y); v.z = gelu_erf(v.z); v.w = gelu_erf(v.w);
  }
  if (EPI == EPI_ADD) {
    const float4 c = *(const float4*)cp;
    v.x = c.x + v.x; v.y = c.y + v.y; v.z = c.z + v.z; v.w = c.w + v.w;
  }
  return v;
}

}  // namespace mb
