// FP64 reciprocal square root to rounding from an estimate (the hardware's, good
// to 2^-24), without a division on the chain.
#ifndef MBA_RSQRT_H_
#define MBA_RSQRT_H_

#include <cmath>

#if defined(__HIPCC__)
#define MBA_RSQRT __host__ __device__ __forceinline__
#else
#define MBA_RSQRT inline
#endif

namespace mba {

// 1 / (2 sqrt(s)), 0.25 <= s <= 4, from an estimate y of 1 / sqrt(s): a
// Goldschmidt step (g -> sqrt(s), h -> 1 / (2 sqrt(s))), then a correction by
// the residual 1/2 - 2 s h^2, formed with 2 s h in two parts (g and what g
// misses of it), so that the last rounding is the only one left.  Six dependent
// operations.
MBA_RSQRT double refine_half_rsqrt(double s, double y) {
  double g = s * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  const double lo = fma(s + s, h, -g);
  return fma(h, fma(-lo, h, fma(-g, h, 0.5)), h);
}

}  // namespace mba

#endif  // MBA_RSQRT_H_
