// FP64 elementary functions of the kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace h2hip {

// sin and cos of |r| <= 0.80: r + r^3 S(r^2) and 1 - r^2/2 + r^4 C(r^2) with
// S and C of degree 5, the best approximations in the maximum norm on
// |r| <= 1.02 pi/4 (exchange algorithm of Remez in 60 digits; they miss
// sin and cos by 2.1e-18 and 6.4e-20 before the coefficients are rounded).
// Absolute errors 0.35 and 0.43 times 2^-52 (4e6 arguments against
// long-double sinl / cosl, the same operations in C).
__device__ __forceinline__ void sincos_poly(double r, double &s, double &c) {
  const double r2 = r * r;
  double ps = 1.5881735738984916e-10;
  ps = fma(ps, r2, -2.5050476368259563e-08);
  ps = fma(ps, r2, 2.755731170446063e-06);
  ps = fma(ps, r2, -0.00019841269823307647);
  ps = fma(ps, r2, 0.0083333333333128);
  ps = fma(ps, r2, -0.16666666666666582);
  s = fma(r * r2, ps, r);
  double pc = -1.1355204972150358e-11;
  pc = fma(pc, r2, 2.087563880745057e-09);
  pc = fma(pc, r2, -2.7557313742707853e-07);
  pc = fma(pc, r2, 2.4801587287420472e-05);
  pc = fma(pc, r2, -0.0013888888888870916);
  pc = fma(pc, r2, 0.04166666666666658);
  pc = fma(pc, r2, -0.5);
  c = fma(r2, pc, 1.0);
}

// sin and cos of |r| <= 0.255, as sincos_poly with S and C of degree 3 (they
// miss sin and cos by 1.0e-17 and 1.4e-19 before the coefficients are
// rounded).
__device__ __forceinline__ void sincos_poly_tiny(double r, double &s,
                                                 double &c) {
  const double r2 = r * r;
  double ps = 2.751519574989631e-06;
  ps = fma(ps, r2, -0.0001984124490180426);
  ps = fma(ps, r2, 0.008333333327309867);
  ps = fma(ps, r2, -0.16666666666661845);
  s = fma(r * r2, ps, r);
  double pc = -2.752053385775909e-07;
  pc = fma(pc, r2, 2.4801564162277738e-05);
  pc = fma(pc, r2, -0.001388888888282356);
  pc = fma(pc, r2, 0.0416666666666612);
  pc = fma(pc, r2, -0.5);
  c = fma(r2, pc, 1.0);
}

// sin and cos of x: Cody and Waite's reduction by pi/2 in three parts
// (n the integer next to 2x / pi, r = x - n pi/2 with fused products) to |r| <= pi/4,
// then sincos_poly (Taylor polynomials of degree 17 and 16, which the code
// had before, took three operations more for the same error).  Absolute
// error below 0.59 * 2^-52 for |x| < 2^45 (the same operations in C with
// fma, against long-double sinl / cosl on 4e6 arguments, a quarter of them
// next to multiples of pi/2); beyond, where k r of a coupling never comes,
// the error grows with the rounding of 2x / pi; NaN and infinities give NaN.
// No branches, so the evaluations of the coupling kernels stay branch-free
// (the library's sincos carries a large-argument path).
__device__ __forceinline__ void sincos_cw(double x, double &s, double &c) {
  constexpr double TWO_OVER_PI = 0.6366197723675814;
  constexpr double P1 = 1.5707963267948966, P2 = 6.123233995736766e-17,
                   P3 = -1.4973849048591698e-33;
  // adding 1.5 * 2^52 rounds to an integer and leaves its low bits in the
  // low mantissa bits (the conversion to a 64-bit integer took eight
  // operations)
  constexpr double MAGIC = 6755399441055744.0;
  const double m = fma(x, TWO_OVER_PI, MAGIC);
  const double n = m - MAGIC;
  double r = fma(-n, P1, x);
  r = fma(-n, P2, r);
  r = fma(-n, P3, r);
  double sr, cr;
  sincos_poly(r, sr, cr);
  // quadrant n mod 4: (sin, cos) = (sr, cr), (cr, -sr), (-sr, -cr), (-cr, sr)
  const uint32_t q = (uint32_t)__builtin_bit_cast(uint64_t, m);
  const double s0 = (q & 1u) ? cr : sr, c0 = (q & 1u) ? sr : cr;
  const uint64_t ss = (uint64_t)(q & 2u) << 62,
                 cs = (uint64_t)((q + 1u) & 2u) << 62;
  s = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, s0) ^ ss);
  c = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, c0) ^ cs);
}

// e^x: n the integer next to x / ln 2, r = x - n ln 2 with ln 2 in two parts
// and fused products, |r| <= 0.3466, the Taylor polynomial of degree 13 (the
// first term left out is 4.2e-18 at most) and a scaling by 2^n.  Relative
// error below 0.63 * 2^-52 (4e6 arguments against long-double expl, the same
// operations in C); NaN gives NaN.  No branches, for the damping of the coupling values
// (the library's exponential breaks up the evaluations of a lane).
__device__ __forceinline__ double exp_cw(double x) {
  constexpr double LOG2E = 1.4426950408889634;
  constexpr double L1 = 0.6931471805599453, L2 = 2.3190468138462996e-17;
  constexpr double MAGIC = 6755399441055744.0;
  // beyond, the result is 0 or infinite (selections, which keep a NaN)
  x = x < -1100.0 ? -1100.0 : x;
  x = x > 1100.0 ? 1100.0 : x;
  const double m = fma(x, LOG2E, MAGIC);
  const double n = m - MAGIC;
  double r = fma(-n, L1, x);
  r = fma(-n, L2, r);
  double p = 1.0 / 6227020800.0;  // 1 / 13!
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
  return __builtin_amdgcn_ldexp(p, (int)(uint32_t)__builtin_bit_cast(uint64_t, m));
}

}  // namespace h2hip
