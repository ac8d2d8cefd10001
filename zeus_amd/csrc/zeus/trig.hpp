// trig.hpp -- sine and cosine of whole turns, sin(2 pi x) and cos(2 pi x), for
// the objectives that are sums of them (Rastrigin, Ackley).
//
// The reduction to a quarter turn is exact in the argument x itself (x minus
// its nearest integer), so there is no rounded product 2 pi x, no branch for
// large arguments and no table: about 20 instructions against about 190 of the
// library's cosine, and several evaluations interleave.  The sine of a quarter
// turn is its Taylor series in 2 pi u to u^21 (remainder below 1.3e-18 at u =
// 1/4), in two chains of u^4.  Error against 128-bit over |x| <= 6: cosine
// 9.7e-17 at most (2.9e-17 rms), sine 2.7e-16 (3.8e-17); of the rounded product
// 2 pi x the functions' values are off by up to 5.0e-15 (9.8e-16).
#pragma once

#include "config.hpp"

#include <cmath>

namespace zeus::dev {

// sin(2 pi u), |u| <= 1/4
ZEUS_HD ZEUS_FI double
sin_quarter(double u)
{
  const double w = u * u, w2 = w * w;
  double a = -0.012031585942120627;           // -(2 pi)^19 / 19!
  double b = 0.0011309237482517963;           //  (2 pi)^21 / 21!
  a = ::fma(a, w2, -0.7181223017785006);      // 15
  b = ::fma(b, w2, 0.10422916220813984);      // 17
  a = ::fma(a, w2, -15.09464257682299);       // 11
  b = ::fma(b, w2, 3.819952584848282);        // 13
  a = ::fma(a, w2, -76.70585975306139);       // 7
  b = ::fma(b, w2, 42.058693944897655);       // 9
  a = ::fma(a, w2, -41.34170224039976);       // 3
  b = ::fma(b, w2, 81.60524927607506);        // 5
  const double p = ::fma(w, b, a);            // (sin(2 pi u) / u - 2 pi) / u^2
  // 2 pi = 6.283185307179586 + 2.449e-16
  return ::fma(u, 6.283185307179586, u * ::fma(w, p, 2.4492935982947064e-16));
}

// cos(2 pi x), r = x - its nearest integer; NaN for an infinite x.  Within an
// eighth of a turn of an extremum +-(1 - 2 sin^2 of half the angle), which
// keeps the value's last bits there, else the sine of the complement.
ZEUS_HD ZEUS_FI double
cos_turns(double x)
{
  const double r = ::fabs(x - ::rint(x));
  const double m = ::fmin(r, 0.5 - r);
  const bool near = m <= 0.125;
  const double s = sin_quarter(near ? 0.5 * m : 0.25 - r);
  const double c = ::fma(-2.0 * s, s, 1.0);
  return near ? (r <= 0.25 ? c : -c) : s;
}

// sin(2 pi x): beyond a quarter turn the mirror image
ZEUS_HD ZEUS_FI double
sin_turns(double x)
{
  const double r = x - ::rint(x);
  const double m = ::copysign(0.5, r) - r;
  return sin_quarter(::fabs(r) <= 0.25 ? r : m);
}

} // namespace zeus::dev
