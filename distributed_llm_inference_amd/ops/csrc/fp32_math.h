// exp, sigmoid, tanh and square root for kernels that are bound by vector work: the hardware's approximations (1 unit in the last place) of
// reduced arguments, quotients and roots with one correction. As exact as the library's functions to a tenth of a unit or two (the figures are
// over all floats of the ranges given, against 64 bits: largest error / root mean square in units in the last place, library -> these), without
// the division's expansion and a second case that a wave runs beside the first.
#pragma once
#include "common.h"

namespace dlia {

// x <= 0, or positive and below the overflow's 88.7 (infinite from there to 2e38). 2^round(x log2 e) times exp2 of the rest, which the fused multiply-adds
// leave exact: log2(e) = 1.442695021629333 (its nearest float) + 1.925963e-8. Results below the normal range keep what bits there are; no number
// stays no number. 0.86 / 0.30 -> 0.97 / 0.31.
__device__ __forceinline__ float exp_c(float x) {
  x = x < -104.f ? -104.f : x;                                     // (exp(-104) is 0, and so is exp(-inf))
  const float n = __builtin_rintf(x * 1.44269502162933349609f);
  const float rest = __builtin_fmaf(x, 1.925963e-8f, __builtin_fmaf(x, 1.44269502162933349609f, -n));
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(rest), (int)n);
}

// e / (1 + e) for e from 0 to 1, with what 1 + e loses to rounding
__device__ __forceinline__ float share_c(float e) {
  const float d = 1.f + e, lost = e - (d - 1.f);
  const float r = __builtin_amdgcn_rcpf(d), q = e * r;
  return __builtin_fmaf(__builtin_fmaf(-q, lost, __builtin_fmaf(-q, d, e)), r, q);
}

// e / (1 + e) of e = exp(-|x|), or 1 minus that. Negative x: 2.62 / 0.63 -> 1.71 / 0.34.
__device__ __forceinline__ float sigmoid_c(float x) {
  const float q = share_c(exp_c(-fabsf(x)));
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

// 1 - 2 e / (1 + e), e = exp(-2 |y|); below 3/4, where that cancels, y + y^3 P(y^2): P is the polynomial of degree 5 whose largest relative error in tanh
// is least (1.7e-9), found by repeated weighted least squares. 1.41 / 0.115 -> 1.03 / 0.113.
__device__ __forceinline__ float tanh_c(float y) {
  const float z = y * y;
  const float big = copysignf(__builtin_fmaf(-2.f, share_c(exp_c(-2.f * fabsf(y))), 1.f), y);
  const float k[5] = {-0.0076572527177631855f, 0.021452032029628754f, -0.053892724215984344f, 0.1333269476890564f, -0.33333316445350647f};
  float c = 0.0017369342967867851f;
#pragma unroll
  for (int i = 0; i < 5; ++i) c = __builtin_fmaf(c, z, k[i]);
  return z < 0.5625f ? __builtin_fmaf(y * z, c, y) : big;
}

// 1 - exp(x) for x <= 0, given e = exp(x / 2): -x - x^2 (1/2 + x/6 + ...) above -1 (what the series leaves out is under 2^-28 of the value), else
// 1 - e^2. 0.89 / 0.155 -> 1.45 / 0.156 (with the error of e).
__device__ __forceinline__ float one_minus_exp_c(float x, float e) {
  float c = 1.f / 39916800.f;
  const float inv[9] = {-1.f / 3628800.f, 1.f / 362880.f, -1.f / 40320.f, 1.f / 5040.f, -1.f / 720.f, 1.f / 120.f, -1.f / 24.f, 1.f / 6.f, -0.5f};
#pragma unroll
  for (int i = 0; i < 9; ++i) c = __builtin_fmaf(c, -x, inv[i]);
  return x > -1.f ? __builtin_fmaf(x * x, c, -x) : __builtin_fmaf(-e, e, 1.f);
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
