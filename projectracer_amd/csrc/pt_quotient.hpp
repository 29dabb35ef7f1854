// pt_quotient.hpp -- quotients by grid constants without a division.
#pragma once
#include <cmath>
#include <hip/hip_runtime.h>

namespace pt {

// s / d, correctly rounded, from rd = RN(1/d).  PW2: d is a power of two and
// the product is the quotient.  Otherwise two residual corrections: the first
// leaves q within one unit of the quotient, and then the second rounds it
// correctly (Markstein's theorem), as long as the residuals are representable:
// from |s| = 2^-969 on.  Below, their low bits underflow and the quotient may be
// one unit in the last place off.  A quotient that overflows is returned as
// it is (the correction of an infinity would be NaN).  5 (1) instructions
// against about 14 of the hardware's division sequence.
template <bool PW2>
__device__ __forceinline__ double quot(double s, double d, double rd) {
  const double q0 = s * rd;
  if constexpr (PW2) return q0;
  const double q1 = __fma_rn(__fma_rn(-q0, d, s), rd, q0);
  const double q2 = __fma_rn(__fma_rn(-q1, d, s), rd, q1);
  return fabs(q0) < INFINITY ? q2 : q0;
}

inline bool pow2(double x) {
  int e;
  return std::frexp(x, &e) == 0.5;
}

}  // namespace pt
