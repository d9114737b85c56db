// exp, sigmoid, tanh and square root for kernels that are bound by vector work: the hardware's approximations (1 unit in the last place) with what
// the argument loses to rounding put back, or one Newton step. About as exact as the library's functions, at a third to a half of
// their instructions: no division expansion, no second case that a wave runs beside the first.
#pragma once
#include "common.h"

namespace dlia {

// x log2(e) rounds; the rest of the product is a factor close to 1. Saturates at exp(88) and exp(-104) ~ 0; no number stays no number.
__device__ __forceinline__ float exp_c(float x) {
  x = x > 88.f ? 88.f : (x < -104.f ? -104.f : x);
  const float t = x * 1.44269502162933349609f;                     // log2(e) = 1.442695021629333 (its nearest float) + 1.925963e-8
  const float lost = __builtin_fmaf(x, 1.925963e-8f, __builtin_fmaf(x, 1.44269502162933349609f, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return __builtin_fmaf(e * 0.6931471805599453f, lost, e);
}

__device__ __forceinline__ float rcp_c(float d) {                  // (d a normal number)
  const float r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, r, 1.f), r, r);
}

// e / (1 + e) of e = exp(-|x|), or 1 minus that: the rounding of 1 + e and of its inverse does not reach values near 1
__device__ __forceinline__ float sigmoid_c(float x) {
  const float e = exp_c(-fabsf(x)), q = e * rcp_c(1.f + e);
  return x > 0.f ? 1.f - q : q;
}

// The instruction takes no input below the normal range (it would be 0, and its inverse infinite): small ones are scaled by 2^32 and back.
// x no negative number, finite. 0.50 / 0.29 either way.
__device__ __forceinline__ float sqrt_c(float x) {
  const bool low = x < 0x1p-96f;
  const float y = low ? x * 0x1p32f : x;
  const float s = __builtin_amdgcn_sqrtf(y);
  const float r = __builtin_fmaf(__builtin_fmaf(-s, s, y), 0.5f * __builtin_amdgcn_rcpf(s), s);
  const float v = y > 0.f ? r : s;
  return low ? v * 0x1p-16f : v;
}

// (1 - e) / (1 + e), e = exp(-2 |y|); below 1/4, where 1 - e cancels, the odd series (what it leaves out is under 2^-26 there)
__device__ __forceinline__ float tanh_c(float y) {
  const float e = exp_c(-2.f * fabsf(y)), y2 = y * y;
  const float big = copysignf((1.f - e) * rcp_c(1.f + e), y);
  const float small = y * __builtin_fmaf(y2, __builtin_fmaf(y2, __builtin_fmaf(y2, __builtin_fmaf(y2, 62.f / 2835.f, -17.f / 315.f), 2.f / 15.f), -1.f / 3.f), 1.f);
  return y2 < 0.0625f ? small : big;
}

// 1 - exp(x) for x <= 0, given e = exp(x / 2): the series above -1/2 (what it leaves out is under 2^-27 of the value), else 1 - e^2
__device__ __forceinline__ float one_minus_exp_c(float x, float e) {
  float c = 1.f / 40320.f;
  const float inv[7] = {1.f / 5040.f, 1.f / 720.f, 1.f / 120.f, 1.f / 24.f, 1.f / 6.f, 0.5f, 1.f};
#pragma unroll
  for (int i = 0; i < 7; ++i) c = __builtin_fmaf(c, x, inv[i]);
  return x > -0.5f ? -x * c : __builtin_fmaf(-e, e, 1.f);
}

// exp(v) - 1 - v for v <= 0: the series above -1/2 (what it leaves out is under 2^-29 of the value; expm1f(v) - v cancels there). Both cases are
// evaluated, some 16 instructions in all.
__device__ __forceinline__ float exp_rest(float v) {
  float c = 1.f / 362880.f;
  const float inv[7] = {1.f / 40320.f, 1.f / 5040.f, 1.f / 720.f, 1.f / 120.f, 1.f / 24.f, 1.f / 6.f, 0.5f};
#pragma unroll
  for (int i = 0; i < 7; ++i) c = __builtin_fmaf(c, v, inv[i]);
  return v > -0.5f ? v * v * c : exp_c(v) - (1.f + v);
}

// ap = softplus(p), aq = 1/2 + softplus(q)
__device__ __forceinline__ float xielu(float v, float ap, float aq) {
  return v > 0.f ? ap * v * v + 0.5f * v : aq * exp_rest(v) + 0.5f * v;
}

}  // namespace dlia
