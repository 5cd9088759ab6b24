// Division by a divisor known in advance, rounded exactly like a / b.
//
// With y = RN(1/b), q = RN(a y) is within one unit of a / b, the remainder
// r = a - b q is exact in one fma, and RN(q + r y) is RN(a / b) (Markstein's
// theorem), so three operations replace the division's dozen.  It holds
// while nothing under- or overflows: callers take it for divisors in
// [1e-60, 1e60] and dividends that are zero or in [1e-200, 1e200], and divide
// otherwise.  (A dividend of -0 gives +0.)
#pragma once

#include <math.h>

namespace lsamd {

__host__ __device__ inline bool div_known_divisor(double b) { return b >= 1e-60 && b <= 1e60; }

__host__ __device__ inline bool div_known_dividend(double a) {
  const double m = fabs(a);
  return (m >= 1e-200 && m <= 1e200) || a == 0.0;
}

// a / b for y = 1.0 / b
__host__ __device__ inline double div_known(double a, double b, double y) {
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}

}  // namespace lsamd
