// sin and cos of one FP64 argument, for the phases exp(-i gamma D) that the
// kernels evaluate per amplitude.
//
// Argument reduction by multiples of pi/2 with pi/2 split into two doubles
// (Cody and Waite, "Software Manual for the Elementary Functions", 1980),
// then the Taylor series of sin and cos on [-pi/4, pi/4] (first dropped terms
// x^19/19! < 1e-19 and x^18/18! < 3e-18).  For |x| < 2^26 the first reduction
// step x - k (pi/2)_hi is exact in one FMA (both are multiples of 2^-52 and
// the difference is below 1), and the parts that later roundings drop are
// carried to first order: the largest error over 2e7 arguments up to 2^26 is
// 8.3e-17 (0.75 ulp of the values above 1/2).  Larger, infinite and NaN
// arguments take the library's sincos.
//
// The library's sincos carries a reduction for arguments of any size in every
// instance; sixteen instances in a row (one per amplitude of a thread) spilled
// registers in the pass kernels and overran the instruction cache in the
// whole-circuit kernel.
#pragma once
#include <hip/hip_runtime.h>

namespace qg {

__host__ __device__ __forceinline__ void sincos_reduced(double x, double* sn, double* cs) {
  const double k = __builtin_rint(x * 0.63661977236758134308);  // 2 / pi
  const double r0 = __builtin_fma(-k, 1.5707963267948965580, x);     // (pi / 2)_hi, exact
  const double r = __builtin_fma(-k, 6.1232339957367658e-17, r0);    // (pi / 2)_lo
  const double rl = __builtin_fma(-k, 6.1232339957367658e-17, r0 - r);  // what r's rounding dropped
  const double z = r * r, zl = __builtin_fma(r, r, -z);
  // sin(r) = r + r z S(z), S = -1/3! + z/5! - ... ; cos(r) = 1 - z/2 + z z C(z), C = 1/4! - z/6! + ...
  double s = 1.0 / 355687428096000.0;
  s = __builtin_fma(s, z, -1.0 / 1307674368000.0);
  s = __builtin_fma(s, z, 1.0 / 6227020800.0);
  s = __builtin_fma(s, z, -1.0 / 39916800.0);
  s = __builtin_fma(s, z, 1.0 / 362880.0);
  s = __builtin_fma(s, z, -1.0 / 5040.0);
  s = __builtin_fma(s, z, 1.0 / 120.0);
  s = __builtin_fma(s, z, -1.0 / 6.0);
  double c = 1.0 / 20922789888000.0;
  c = __builtin_fma(c, z, -1.0 / 87178291200.0);
  c = __builtin_fma(c, z, 1.0 / 479001600.0);
  c = __builtin_fma(c, z, -1.0 / 3628800.0);
  c = __builtin_fma(c, z, 1.0 / 40320.0);
  c = __builtin_fma(c, z, -1.0 / 720.0);
  c = __builtin_fma(c, z, 1.0 / 24.0);
  // the dropped parts of r, z and 1 - z/2 enter to first order
  const double h = 0.5 * z, w = 1.0 - h;
  const double sr = r + __builtin_fma(r * z, s, __builtin_fma(-h, rl, rl));
  const double cr = w + (((1.0 - w) - h) + __builtin_fma(z * z, c, __builtin_fma(-0.5, zl, -r * rl)));
  const int q = (int)k;
  const double a = (q & 1) ? cr : sr, b = (q & 1) ? sr : cr;
  *sn = (q & 2) ? -a : a;
  *cs = ((q + 1) & 2) ? -b : b;
}

constexpr double kSincosMax = 67108864.0;  // 2^26

__device__ __forceinline__ void sincos_phase(double x, double* sn, double* cs) {
  if (__builtin_fabs(x) < kSincosMax) sincos_reduced(x, sn, cs);
  else sincos(x, sn, cs);
}

}  // namespace qg
