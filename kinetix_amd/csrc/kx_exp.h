// FP64 exp2, exp and log2 for the production-rate kernels, without the library functions' range
// handling (a third of their instructions): results beyond the double range come out of ldexp as
// infinity or zero, a NaN stays NaN; infinite arguments, and of exp2 and exp those whose binary
// exponent is no int (|x| above 2^31, 1.4e9), are the caller's to avoid.
//
// Method: reduction to |r| <= 1/2 (exp2) or |r| <= ln 2 / 2 (exp; ln 2 in two parts, the first of
// 24 bits, so that n ln2_hi is exact), a degree-11 polynomial, and the power of two by ldexp. log2:
// mantissa m in [sqrt 1/2, sqrt 2), 2/ln 2 atanh(s) with s = (m - 1) / (m + 1), degree 7 in s^2. The
// polynomials interpolate the functions at Chebyshev nodes (computed in 60 digits, rounded once):
// relative error below 2.1e-17 before the arithmetic's own rounding. With it exp2 and exp are within 1
// ulp; log2, through a rounded quotient, within 6.6 2^-53 of its value (3.2 ulp seen), exact on powers
// of two (kx_selftest_exp on the device).
#pragma once
#include <hip/hip_runtime.h>
#include "kx_rcp.h"

__device__ __forceinline__ double kx_exp2(double y)
{
  const double n = __builtin_rint(y), r = y - n;
  double p = 4.4558179083360645e-10;
  p = fma(p, r, 7.074194297288521e-09);
  p = fma(p, r, 1.0178057087733941e-07);
  p = fma(p, r, 1.3215432535912375e-06);
  p = fma(p, r, 1.5252733841556773e-05);
  p = fma(p, r, 0.00015403530463724353);
  p = fma(p, r, 0.001333355814640647);
  p = fma(p, r, 0.009618129107587256);
  p = fma(p, r, 0.055504108664821625);
  p = fma(p, r, 0.24022650695910158);
  p = fma(p, r, 0.6931471805599453);
  p = fma(p, r, 1.0);
  return __builtin_ldexp(p, (int)n);
}

__device__ __forceinline__ double kx_exp(double x)
{
  const double n = __builtin_rint(x * 1.4426950408889634);
  const double r = fma(-n, 5.7699990475432854e-08, fma(-n, 0.6931471228599548, x));
  double p = 2.5110049204818658e-08;
  p = fma(p, r, 2.763265472252779e-07);
  p = fma(p, r, 2.755724088722987e-06);
  p = fma(p, r, 2.4801485441561313e-05);
  p = fma(p, r, 0.00019841269890076403);
  p = fma(p, r, 0.0013888888952352863);
  p = fma(p, r, 0.008333333333319589);
  p = fma(p, r, 0.04166666666648795);
  p = fma(p, r, 0.1666666666666668);
  p = fma(p, r, 0.5000000000000019);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return __builtin_ldexp(p, (int)n);
}

// x normal; NaN for x <= 0 (log2(0) is the caller's to avoid)
__device__ __forceinline__ double kx_log2(double x)
{
  double m = __builtin_amdgcn_frexp_mant(x);                  // [1/2, 1)
  int e = __builtin_amdgcn_frexp_exp(x);
  const bool low = m < 0.7071067811865476;
  m = low ? m + m : m;
  e = low ? e - 1 : e;
  const double s = (m - 1.0) * kx_rcp(m + 1.0), z = s * s;
  double p = 0.21368163909696675;
  p = fma(p, z, 0.2209109142370262);
  p = fma(p, z, 0.2623344335728468);
  p = fma(p, z, 0.3205985334227465);
  p = fma(p, z, 0.41219858585486296);
  p = fma(p, z, 0.5770780163454586);
  p = fma(p, z, 0.9617966939259899);
  p = fma(p, z, 2.8853900817779268);
  return x > 0.0 ? fma(s, p, (double)e) : __builtin_nan("");
}

// 2^y with an FP32 exponent: hardware exp2 of the fraction, the power of two in FP64
__device__ __forceinline__ double kx_exp2_f32(float y)
{
  const float n = __builtin_rintf(y);
  return __builtin_ldexp((double)__builtin_amdgcn_exp2f(y - n), (int)n);
}
