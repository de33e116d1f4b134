// quot.h -- division by a tabulated divisor.
#pragma once
#include <hip/hip_runtime.h>

#include "dual.h"

namespace fv3 {

// a / b from y = 1/b (rounded): two residual corrections of a*y.  The first
// leaves q within one unit in the last place, so that the second is a/b
// correctly rounded (Markstein, IBM J. Res. Dev. 34, 1990), in five instructions:
// the value of the division it replaces where a, b and a / b are finite, b is not
// zero and the residual (about a 2^-24 in FP32, a 2^-53 in FP64) is no subnormal.
template <typename R>
__host__ __device__ __forceinline__ R quot(R a, R b, R y) {
  R q = a * y;
  q = fma(fma(-b, q, a), y, q);
  return fma(fma(-b, q, a), y, q);
}
// of a (value, tangent) pair: each component's quotient, as Dual's division (whose
// tangent is a NaN where the value is not finite: the divisor's is 0, times it)
__host__ __device__ __forceinline__ Dual<1> quot(const Dual<1> &a, double b, double y) {
  Dual<1> r(quot(a.v, b, y));
  r.d[0] = quot(a.d[0] - r.v * 0.0, b, y);
  return r;
}

// the same for any operands: infinities, NaNs and zero divisors as the division
// has them (one instruction more)
__host__ __device__ __forceinline__ double quot_any(double a, double b, double y) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_div_fixup(quot(a, b, y), b, a);
#else
  (void)y;
  return a / b;
#endif
}
__host__ __device__ __forceinline__ Dual<1> quot_any(const Dual<1> &a, double b, double y) {
  Dual<1> r(quot_any(a.v, b, y));
  r.d[0] = quot_any(a.d[0] - r.v * 0.0, b, y);
  return r;
}

}  // namespace fv3
