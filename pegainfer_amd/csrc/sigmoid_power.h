// Decay functions that more than one recurrence uses (recurrent.hip, gated_linear.hip, recurrent_step.hip).
#pragma once

#include "common.h"

namespace pk {

__device__ __forceinline__ float softplus_f(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

// sigmoid(z)^p through x = p (min(z, 0) - log(1 + e^-|z|)).  A decay near one multiplies hundreds of tokens, so its error must not lean to
// one side: there the logarithm comes from the series of 2 artanh(t / (2 + t)) and e^x from its own series around 1, whose last step is
// the only rounding that counts; a decay further down is forgotten before the hardware exponential's last bit shows.
__device__ __forceinline__ float sigmoid_power(float z, float p) {
  constexpr float kLog2e = 1.44269504088896341f;
  const float t = __builtin_amdgcn_exp2f(-fabsf(z) * kLog2e);
  const float s = t / (2.0f + t), q = s * s;           // s <= 1/3
  float l = 2.0f / 15.0f;
  l = fmaf(l, q, 2.0f / 13.0f);
  l = fmaf(l, q, 2.0f / 11.0f);
  l = fmaf(l, q, 2.0f / 9.0f);
  l = fmaf(l, q, 2.0f / 7.0f);
  l = fmaf(l, q, 2.0f / 5.0f);
  l = fmaf(l, q, 2.0f / 3.0f);
  l = fmaf(l, q, 2.0f);
  const float x = (fminf(z, 0.f) - l * s) * p;
  float e = 1.0f / 362880.0f;                          // (e^x - 1) / x for -1/2 < x <= 0
  e = fmaf(e, x, 1.0f / 40320.0f);
  e = fmaf(e, x, 1.0f / 5040.0f);
  e = fmaf(e, x, 1.0f / 720.0f);
  e = fmaf(e, x, 1.0f / 120.0f);
  e = fmaf(e, x, 1.0f / 24.0f);
  e = fmaf(e, x, 1.0f / 6.0f);
  e = fmaf(e, x, 0.5f);
  e = fmaf(e, x, 1.0f);
  return x > -0.5f ? fmaf(e, x, 1.0f) : __builtin_amdgcn_exp2f(x * kLog2e);
}

}  // namespace pk
