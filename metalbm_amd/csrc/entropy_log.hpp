// entropy_log.hpp -- quotient and logarithms of the entropic root solve.
#pragma once

#include <cmath>

#include <hip/hip_runtime.h>

namespace lbm {

// The mantissa of v in [1/2, 1), its exponent and a reciprocal of v good to 2^-24 or
// better: instructions on the device, the library's elsewhere.
__host__ __device__ __forceinline__ double mantissa_of(double v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_frexp_mant(v);
#else
  int k;
  return std::frexp(v, &k);
#endif
}
__host__ __device__ __forceinline__ int exponent_of(double v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_frexp_exp(v);
#else
  int k;
  (void)std::frexp(v, &k);
  return k;
#endif
}
__host__ __device__ __forceinline__ double reciprocal_estimate(double v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcp(v);
#else
  return double(float(1.0 / v));
#endif
}

// n / v to about an ulp for v > 0 in the normal range: the hardware reciprocal
// with one Newton-Raphson correction (to 2^-48 or better) and the quotient's
// residual through it.
__host__ __device__ __forceinline__ double quotient(double n, double v) {
  double r = reciprocal_estimate(v);
  r = fma(r, fma(-v, r, 1.0), r);
  const double q = n * r;
  return fma(r, fma(-v, q, n), q);
}

// log(2^k m) for m = 1 + m1 in [sqrt(1/2), sqrt(2)): log m = 2 atanh(s), s = m1 /
// (m + 1), s^2 <= 0.02944.  The atanh series beyond its first term is replaced by the
// polynomial through seven Chebyshev nodes of that interval (relative error of the
// logarithm below 5e-18), so the result is within two ulps, at a third of the
// library's instructions.
__host__ __device__ __forceinline__ double log_reduced(double m1, int k) {
  const double s = quotient(m1, m1 + 2.0);
  const double z = s * s;
  double p = 0.146167211662876;
  p = fma(p, z, 0.15331699634642276);
  p = fma(p, z, 0.1818288978615799);
  p = fma(p, z, 0.22222211125723262);
  p = fma(p, z, 0.28571428626031065);
  p = fma(p, z, 0.3999999999989938);
  p = fma(p, z, 0.666666666666667);
  // ln 2 in two parts, the first short enough for k ln2_hi to be exact
  constexpr double ln2_hi = 0x1.62e42fee00000p-1, ln2_lo = 0x1.a39ef35793c76p-33;
  const double dk = double(k);
  return fma(dk, ln2_hi, fma(dk, ln2_lo, fma(s * z, p, s + s)));
}

// log(1 + y) for 1 + y positive and normal.  Where 1 + y needs no scaling m1 is y itself,
// so nothing is lost for small y.
__host__ __device__ __forceinline__ double log1p_positive(double y) {
  const double v = 1.0 + y;
  double m = mantissa_of(v);
  int k = exponent_of(v);
  const bool low = m < 0.70710678118654752440;
  m = low ? m + m : m;
  k = low ? k - 1 : k;
  return log_reduced(k == 0 ? y : m - 1.0, k);
}

// log(v) for finite v > 0, however small (m - 1 is exact); not a number for v <= 0 (the
// library's -inf at 0 enters G as 0 times infinity).
__host__ __device__ __forceinline__ double log_or_nan(double v) {
  double m = mantissa_of(v);
  int k = exponent_of(v);
  const bool low = m < 0.70710678118654752440;
  m = low ? m + m : m;
  k = low ? k - 1 : k;
  const double l = log_reduced(m - 1.0, k);
  return v > 0.0 ? l : __builtin_nan("");
}

}  // namespace lbm
