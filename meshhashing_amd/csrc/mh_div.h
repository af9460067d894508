// mh_div.h -- correctly rounded FP32 division by a constant (host and device).
#pragma once
#include <math.h>

#if defined(__HIPCC__)
#define MH_DIV_HD __host__ __device__ __forceinline__
#else
#define MH_DIV_HD inline
#endif

namespace mh {

// a / d, correctly rounded, given inv = the correctly rounded 1 / d: Markstein
// (P. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", 1990): with q within one ulp of a / d, the residual
// a - q d is exact in one fused multiply-add, and q + residual * inv is the
// correctly rounded quotient.  a * inv can be two ulp off; a first correction
// brings it within one.  Five instructions, where the IEEE division, which
// also handles every exponent, takes about twice as many.  Holds while nothing
// under- or overflows (2^-100 <= |a| <= 2^100, 2^-20 <= d <= 2^20; also a = 0,
// up to the sign of the zero); below that range the result is off by a
// rounding of a number under 2^-80, above it and for infinities it is not
// usable (tests/test_quotient_cpu.py).
MH_DIV_HD float quotient(float a, float d, float inv) {
  const float q0 = a * inv;
  const float q1 = fmaf(fmaf(-q0, d, a), inv, q0);
  return fmaf(fmaf(-q1, d, a), inv, q1);
}

}  // namespace mh
