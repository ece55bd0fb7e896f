// Scalar FP64 math for the sweep kernels, written so every result that feeds a
// position or a decision is the one the reference computes on Linux.
//
//  * hmc_cbrt: Rust's f64::cbrt calls the C library's cbrt; this restates
//    glibc 2.35's sysdeps/ieee754/dbl-64/s_cbrt.c (IBM Accurate Mathematical
//    Library lineage; LGPL-2.1+): frexp, the rational polynomial, one
//    Newton-like step, then scaling by 2^(e/3).  It matches the host library
//    bit for bit on the inputs the 3D ball sampler produces.
//  * glibc_exp, glibc_log, glibc_sincos (glibc_math.hpp): the library's exp,
//    log and sincos, for the normal sampler's tail and wedge test, Metropolis,
//    and the rotation sampler.
//
// Everything here is compiled with -ffp-contract=off; fma() appears only where
// the restated library fuses a product.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#define HMC_HD __host__ __device__ __forceinline__

namespace hmc {

// ------------------------------------------------- division by a constant --
// a / b, correctly rounded, for a constant b with y = 1 / b correctly rounded.
// Two residual corrections of a y: the first leaves q within an ulp of a / b, so
// the second residual a - b q is exact and its correction rounds a / b
// (Markstein: correctly rounded when q is that close and b's significand is
// not all ones, for which inv_const gives 0).  Holds for 2^-900 <= |a| <=
// 2^900, where the residuals are exact.  Five operations for the compiler's
// division's dozen with a reciprocal estimate: 25 cycles for 77 in a dependent
// chain.
HMC_HD double div_const_fast(double a, double b, double y) {
  double q = a * y;
  q = fma(fma(-q, b, a), y, q);
  return fma(fma(-q, b, a), y, q);
}
// The y of div_const_fast for b, or 0 where it does not apply.
HMC_HD double inv_const(double b) {
  int e;
  const double f = frexp(fabs(b), &e);  // [1/2, 1)
  if (!(f < 1.0 - 0x1p-53) || e < -100 || e > 100) return 0.0;
  return 1.0 / b;
}

// ---------------------------------------------------------------- cube root --
HMC_HD double hmc_cbrt(double x) {
  const double kCbrt2 = 1.2599210498948731648;      // 2^(1/3)
  const double kSqrCbrt2 = 1.5874010519681994748;   // 2^(2/3)
  int xe;
  double xm = frexp(fabs(x), &xe);
  double u = (0.354895765043919860 +
              ((1.50819193781584896 +
                ((-2.11499494167371287 +
                  ((2.44693122563534430 +
                    ((-1.83469277483613086 + (0.784932344976639262 - 0.145263899385486377 * xm) * xm) * xm)) *
                   xm)) *
                 xm)) *
               xm));
  double t2 = u * u * u;
  const int r = xe % 3;
  double factor = r == -2 ? 1.0 / kSqrCbrt2 : r == -1 ? 1.0 / kCbrt2 : r == 0 ? 1.0 : r == 1 ? kCbrt2 : kSqrCbrt2;
  double ym = u * (t2 + 2.0 * xm) / (2.0 * t2 + xm) * factor;
  const double y = ldexp(x > 0.0 ? ym : -ym, xe / 3);
  return x == 0.0 || !isfinite(x) ? x + x : y;
}

}  // namespace hmc

#include "glibc_math.hpp"
