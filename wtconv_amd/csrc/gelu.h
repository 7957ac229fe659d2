// The erf form of GELU and its derivative.
#pragma once

#include "common.h"

namespace wt {

// erf form of GELU: x * Phi(x) = x / 2 + |x| * (1 / 2 - Phi(-|x|)).  log2 of Phi(-a) is a smooth, nearly quadratic function, so
// Phi(-a) is 2 to a polynomial in a (degree 7, fitted to the error of the result weighted by a * Phi(-a)): |error| <=
// 3.9e-7 over all x (x / 2 * (1 + erf) in float32: 1.2e-6), for 28 cycles of the vector pipe a value instead of the 44 of
// a rational times an exponential.  (The last two terms see x itself: infinities and NaNs come out as they do of erf.)  Beyond
// the range of the fit, [0, 16], the polynomial falls on and on, as its first coefficient does at infinity: 2 to it is 0, which
// is what Phi(-a) is there in float32, and needs no clamp (two instructions of sixteen).
__device__ __forceinline__ float gelu_erf(float x) {
  const float a = fabsf(x);
  float p = fmaf(a, -1.09032517e-06f, 4.60320700e-05f);
  p = fmaf(a, p, -8.13045196e-04f);
  p = fmaf(a, p, 8.10905740e-03f);
  p = fmaf(a, p, -5.33128628e-02f);
  p = fmaf(a, p, -4.58948432e-01f);
  p = fmaf(a, p, -1.15110632f);
  p = fmaf(a, p, -1.00000798f);
  return fmaf(fabsf(x), 0.5f - __builtin_amdgcn_exp2f(p), 0.5f * x);
}

// Phi(-a), a >= 0, the same way to a degree more and fitted to the errors of both Phi(-a) and a * Phi(-a): <= 5e-8 each.
// (Training needs Phi by itself, for the derivative.)
__device__ __forceinline__ float phi_of_minus(float a) {
  float p = fmaf(a, -2.293375708e-06f, 3.306769568e-05f);
  p = fmaf(a, p, -1.571017356e-04f);
  p = fmaf(a, p, -2.048604372e-04f);
  p = fmaf(a, p, 7.149047006e-03f);
  p = fmaf(a, p, -5.255343381e-02f);
  p = fmaf(a, p, -4.591896931e-01f);
  p = fmaf(a, p, -1.151107504f);
  p = fmaf(a, p, -9.999999444e-01f);
  return __builtin_amdgcn_exp2f(p);
}

__device__ __forceinline__ float gelu_train(float x) {
  return fmaf(fabsf(x), 0.5f - phi_of_minus(fabsf(x)), 0.5f * x);
}

// d/dx x Phi(x) = Phi(x) + x phi(x)
__device__ __forceinline__ float gelu_derivative(float x) {
  const float low = phi_of_minus(fabsf(x));
  const float density = 0.3989422804f * __builtin_amdgcn_exp2f(-0.7213475204f * x * x);
  return fmaf(x, density, x < 0.f ? low : 1.f - low);
}

}  // namespace wt
