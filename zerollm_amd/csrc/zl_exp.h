// The exponential of the attention softmax: plain f64 arithmetic, the same on the host and on the device (where the HIP
// runtime header comes first).
#pragma once
#include <cmath>

#ifdef __HIPCC__
#define ZL_EXP_FN __host__ __device__ __forceinline__
#else
#define ZL_EXP_FN inline
#endif

namespace zl {

constexpr double LN2_HI = 2977044472.0 / 4294967296.0;     // ln 2 to 32 fractional bits (n LN2_HI is exact)
constexpr double LN2_LO = -4.2009150726810846e-11;          // ln 2 - LN2_HI

// exp of x <= 0 in f64 (NaN and -inf included): x = n ln 2 + r with |r| <= ln 2 / 2 (ln 2 in two parts, n exact), the
// Taylor polynomial of degree 13 in Horner form (remainder r^14 / 14! < 5e-18), scaled by 2^n. Within an ulp of the
// exact value (0.85 at most of 4 million arguments). 21 VALU instructions where the device library's exp, which serves
// every argument, takes about 45: the softmax of a 12K-position prefill row is bound by them.
ZL_EXP_FN double exp_neg(double x) {
  const double y = x < -1000.0 ? -1000.0 : x;  // (2^n underflows to 0 long before; a NaN stays one)
  const double n = rint(y * 1.4426950408889634);
  double r = fma(n, -LN2_HI, y);
  r = fma(n, -LN2_LO, r);
  double p = 1.0 / 6227020800.0;
  p = fma(p, r, 1.0 / 479001600.0);
  p = fma(p, r, 1.0 / 39916800.0);
  p = fma(p, r, 1.0 / 3628800.0);
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return ldexp(p, (int)n);
}

}  // namespace zl
