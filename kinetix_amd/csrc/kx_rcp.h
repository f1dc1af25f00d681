// FP64 reciprocal for the transport and rate kernels: 1/y for |y| and 1/|y| in the normal range,
// within 1 ulp of the quotient: v_rcp_f64 (relative error e of about 2^-24) refined by one
// third-order step r (1 + e + e^2), error e^3. Four dependent instructions instead of the IEEE
// division's ~10 (scaling, Newton, fmas, fixup). No special cases: y = 0, infinities, NaN and
// results in the subnormal range give NaN or lose digits. Its callers: the transport fits (positive,
// moderate exponents) and products of eight of them; exp(g) of the rates, whose exponent is some
// hundreds (|g| < 708 above ~140 K for the mechanisms here); 1 + Pr and the Troe denominators.
// kx_selftest_rcp checks the bound on the device from 2^-1000 to 2^1000.
#pragma once
#include <hip/hip_runtime.h>

__device__ __forceinline__ double kx_rcp(double y)
{
  const double r = __builtin_amdgcn_rcp(y);
  const double e = fma(-y, r, 1.0);
  return fma(r, fma(e, e, e), r);
}
