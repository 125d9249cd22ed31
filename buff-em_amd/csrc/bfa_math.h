// bfa_math.h -- device arithmetic shared by the cubature kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace bfa {

// 1/sqrt(x): the hardware estimate y (v_rsq_f64, ~23 correct bits) and one
// step of third order, y <- y (1 + e/2 + 3/8 e^2) with e = 1 - x y^2: what the
// series leaves off is 5/16 e^3 < 2^-65.  Replaces a correctly rounded sqrt and
// a division in the pair loops, and two Newton steps (5 instructions after the
// estimate instead of 8).
__device__ __forceinline__ double rsqrt_nr(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// sin and cos of a phase k r: reduced by multiples n of pi/2, which two doubles
// hold to 2^-109, then the Taylor polynomials on |f| <= pi/4, whose first
// dropped terms are f^17/17! <= 5e-17 and f^18/18! <= 2e-18.  That |f| takes
// n = x 2/pi to within rounding of the nearest: true to 0.002 for |x| < 2^44.
// Above, the product's rounding moves n, |f| reaches 0.95 and the dropped term
// 1.2e-15 at 2^50, where x's own last place is already 0.25; larger phases
// carry no digits and get none here.  About 30 instructions, no table and no branch,
// against some 80 and twice the registers with the library's sincos and its
// reduction for huge arguments.
__device__ __forceinline__ void sincos_mod(double x, double *sn, double *cs)
{
  const double n = rint(x * 0.63661977236758134308);
  const double f = fma(n, -6.12323399573676603587e-17, fma(n, -1.57079632679489655800, x));
  const double z = f * f;
  double s = -1.0 / 1307674368000.0;
  s = fma(s, z, 1.0 / 6227020800.0);
  s = fma(s, z, -1.0 / 39916800.0);
  s = fma(s, z, 1.0 / 362880.0);
  s = fma(s, z, -1.0 / 5040.0);
  s = fma(s, z, 1.0 / 120.0);
  s = fma(s, z, -1.0 / 6.0);
  s = fma(s * z, f, f);
  double c = 1.0 / 20922789888000.0;
  c = fma(c, z, -1.0 / 87178291200.0);
  c = fma(c, z, 1.0 / 479001600.0);
  c = fma(c, z, -1.0 / 3628800.0);
  c = fma(c, z, 1.0 / 40320.0);
  c = fma(c, z, -1.0 / 720.0);
  c = fma(c, z, 1.0 / 24.0);
  c = fma(c, z, -0.5);
  c = fma(c, z, 1.0);
  const int q = (int)(n - 4.0 * floor(0.25 * n));
  const double a = q & 1 ? c : s, b = q & 1 ? s : c;
  *sn = q & 2 ? -a : a;
  *cs = (q + 1) & 2 ? -b : b;
}

}  // namespace bfa
