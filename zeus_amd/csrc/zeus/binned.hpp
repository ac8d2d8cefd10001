// binned.hpp -- the binned spectrum's expected counts without a power
// function per evaluation.
//
// mu = a (1 - x)^b / x^(c + d ln x) is a exp(b ln(1 - x) - q ln x), q = c + d
// ln x: of the parameters being fitted only the exponent's coefficients
// change, so the logarithms of x and of 1 - x are taken once per call, in
// double-double (the table below), and an evaluation of a bin is one
// exponential; ln mu, which the Poisson likelihood needs as well, is ln a plus
// the exponent.  With two powers, two logarithms and a division per bin the
// evaluation was bound by VALU issue (two powers of about 270 instructions, two
// logarithms of about 120; now about 110 in all).
//
// Accuracy: the products are kept with their rounding errors (fma) and the
// exponent is a sum of two doubles, so that mu is off by the rounding of q and
// of the last operations, as with the power functions.
#pragma once

#include "config.hpp"

#include <cmath>

namespace zeus::dev {

struct DD { // unevaluated sum hi + lo
  double hi, lo;
};

ZEUS_HD ZEUS_FI DD
two_sum(double a, double b)
{
  const double s = a + b, t = s - a;
  return {s, (a - (s - t)) + (b - t)};
}
ZEUS_HD ZEUS_FI DD
two_prod(double a, double b)
{
  const double p = a * b;
  return {p, ::fma(a, b, -p)};
}

constexpr double kLog2e = 1.4426950408889634074;
constexpr double kLn2Hi = 0.69314718055994530942;   // ln 2 rounded
constexpr double kLn2Lo = 2.3190468138462996155e-17; // ln 2 - kLn2Hi

// exp(h + l), |h| <= 700, |l| tiny: r = h - k ln 2 in [-0.35, 0.35], the
// Taylor series of exp to r^13 (remainder r^14 / 14! < 5e-18) as two chains
// in r^2, times 2^k.
ZEUS_HD ZEUS_FI double
exp_sum(double h, double l)
{
  const double k = ::rint(h * kLog2e);
  const double r = ::fma(-k, kLn2Lo, ::fma(-k, kLn2Hi, h)) + l;
  const double r2 = r * r;
  double e = 1.0 / 479001600.0;         // 1/12!
  double o = 1.0 / 6227020800.0;        // 1/13!
  e = ::fma(e, r2, 1.0 / 3628800.0);    // 1/10!
  o = ::fma(o, r2, 1.0 / 39916800.0);   // 1/11!
  e = ::fma(e, r2, 1.0 / 40320.0);      // 1/8!
  o = ::fma(o, r2, 1.0 / 362880.0);     // 1/9!
  e = ::fma(e, r2, 1.0 / 720.0);        // 1/6!
  o = ::fma(o, r2, 1.0 / 5040.0);       // 1/7!
  e = ::fma(e, r2, 1.0 / 24.0);         // 1/4!
  o = ::fma(o, r2, 1.0 / 120.0);        // 1/5!
  e = ::fma(e, r2, 0.5);                // 1/2!
  o = ::fma(o, r2, 1.0 / 6.0);          // 1/3!
  // 1 + r + r^2 (e + r o): the small terms are summed first
  const double p = ::fma(r2, ::fma(o, r, e), r) + 1.0;
  return ::ldexp(p, int(k));
}

// log x - l for l = log(x) rounded (x finite, > 0): x exp(-l) - 1, good to
// 1e-19: the first four terms of the series in double-double, the rest of it
// (below 6e-4) in double.
ZEUS_HD inline double
log_rest(double x, double l)
{
  const double k = ::rint(-l * kLog2e);
  const DD kl = two_prod(k, kLn2Hi);
  const DD s = two_sum(-l, -kl.hi);
  const DD r = two_sum(s.hi, s.lo - kl.lo - k * kLn2Lo);
  double t = 1.0 / 6227020800.0; // 1/13!
  const double c[9] = {1.0 / 479001600.0, 1.0 / 39916800.0, 1.0 / 3628800.0,
                       1.0 / 362880.0,    1.0 / 40320.0,    1.0 / 5040.0,
                       1.0 / 720.0,       1.0 / 120.0,      1.0 / 24.0};
  for (int n = 0; n < 9; ++n)
    t = ::fma(t, r.hi, c[n]);
  DD e{t, 0.0};
  const DD head[4] = {{1.0 / 6.0, 9.2518585385429707e-18}, {0.5, 0.0}, {1.0, 0.0}, {1.0, 0.0}};
  for (int n = 0; n < 4; ++n) { // e = head + r e
    const DD p = two_prod(r.hi, e.hi);
    const DD q = two_sum(head[n].hi, p.hi);
    e = two_sum(q.hi, q.lo + (p.lo + (r.hi * e.lo + r.lo * e.hi) + head[n].lo));
  }
  const double sc = ::ldexp(1.0, int(k));
  const DD m = two_prod(x, e.hi * sc);
  return ((m.hi - 1.0) + m.lo) + x * (e.lo * sc);
}

// One bin's logarithms: ln x and ln(1 - x), rounded and the rest.  A bin whose
// x or rounded 1 - x is not inside (0, 1) has l1 = NaN and is evaluated with
// the power functions.
struct BinLogs {
  double lx, lx_lo, l1, l1_lo;
};
constexpr int kBinLogs = 4;

ZEUS_HD ZEUS_FI bool
bin_plain(double x)
{
  return x > 0.0 && x < 1.0 && 1.0 - x < 1.0;
}
ZEUS_HD inline DD
bin_log_x(double x)
{
  const double l = ::log(x);
  return {l, bin_plain(x) ? log_rest(x, l) : 0.0};
}
ZEUS_HD inline DD
bin_log_1mx(double x)
{
  if (!bin_plain(x))
    return {__builtin_nan(""), 0.0};
  const double y = 1.0 - x, l = ::log(y);
  return {l, log_rest(y, l)};
}

// Expected count of a bin, its logarithm, and whether the plain exponent gave
// them (else the power functions or their limits did, in the reference's order
// of operations, with its overflows).
struct BinMean {
  double mean, log_mean;
  bool plain;
  double ratio; // (1 - x)^b / x^q when !plain
};

// y^p = exp(h + l) with the limits of the power function, |h| outside
// (700, 746); y in (0, 1).
ZEUS_HD ZEUS_FI double
pow_limit(double h, double l)
{
  if (h > 700.0)
    return __builtin_huge_val();
  if (h < -700.0)
    return 0.0;
  return exp_sum(h, l);
}

// The power functions themselves, out of line: next to overflow and in the
// denormal range, for NaN parameters and for bins outside (0, 1).  (Inlined,
// their constants and temporaries took the fit kernel to one wavefront per
// SIMD.)
#if defined(__HIP_DEVICE_COMPILE__)
__attribute__((noinline))
#else
inline
#endif
ZEUS_HD DD
bin_pows(double b, double q, double x)
{
  return {::pow(1.0 - x, b), ::pow(x, q)};
}
#if defined(__HIP_DEVICE_COMPILE__)
__attribute__((noinline))
#else
inline
#endif
ZEUS_HD double
pow_any(double y, double p)
{
  return ::pow(y, p);
}

// la = log(a); a_plain: a in [1e-30, 1e30].
ZEUS_HD ZEUS_FI BinMean
bin_mean(double a, double b, double c, double d, double la, bool a_plain, double x,
         const BinLogs& t)
{
  const double q = c + d * t.lx;
  const DD p1 = two_prod(b, t.l1);
  const DD p2 = two_prod(q, t.lx);
  const double r1 = ::fma(b, t.l1_lo, p1.lo), r2 = ::fma(q, t.lx_lo, p2.lo);
  const DD s = two_sum(p1.hi, -p2.hi);
  const double lo = s.lo + (r1 - r2);
  const double h1 = ::fabs(p1.hi), h2 = ::fabs(p2.hi);
  // neither power nor the products with a leave the normal range
  if (a_plain && h1 <= 300.0 && h2 <= 300.0) {
    const DD lm = two_sum(la, s.hi);
    return {a * exp_sum(s.hi, lo), lm.hi + (lm.lo + lo), true, 0.0};
  }
  const bool limits = (h1 <= 700.0 || h1 >= 746.0) && (h2 <= 700.0 || h2 >= 746.0);
  const DD w = limits ? DD{pow_limit(p1.hi, r1), pow_limit(p2.hi, r2)} : bin_pows(b, q, x);
  const double mean = a * w.hi / w.lo;
  return {mean, ::log(mean), false, w.hi / w.lo};
}

// The bin in the fit itself keeps the power functions and their order of
// operations, so that a fit's trajectory (along which the likelihood's flat
// directions amplify a rounding error up to 1e9 times, in 0.3 % of the fits) does
// not depend on this file; only powers that are certain to overflow or vanish, as
// in most trials of a first line search, are not evaluated.
struct BinPow {
  double mean, ratio;
};
// y^p for p ln y = h, rounded (NaN: unknown).  Where h is known y is positive and
// finite and so is p, and the compiler drops the library's selections for other
// operands: 30 of its 224 instructions, the same bits.  64 fits of 256 starts, 100
// bins: BFGS 1.66 -> 1.54 ms.
ZEUS_HD ZEUS_FI double
pow_or_limit(double y, double p, double h)
{
  if (h > 711.0)
    return __builtin_huge_val();
  if (h < -747.0)
    return 0.0;
  if (!(h == h))
    return pow_any(y, p);
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_assume(!__builtin_isnan(y));
  __builtin_assume(!__builtin_isinf(y));
  __builtin_assume(!__builtin_isnan(p));
  __builtin_assume(!__builtin_isinf(p));
  __builtin_assume(y > 0.0);
#endif
  return ::pow(y, p);
}
ZEUS_HD ZEUS_FI BinPow
bin_pow(double a, double b, double c, double d, double x, const BinLogs& t)
{
  const double q = c + d * t.lx;
  const double h1 = b * t.l1;
  // t.l1 is NaN for a bin outside (0, 1): both powers are evaluated
  const double h2 = t.l1 == t.l1 ? q * t.lx : t.l1;
  const double pw = pow_or_limit(1.0 - x, b, h1);
  const double qw = pow_or_limit(x, q, h2);
  return {a * pw / qw, pw / qw};
}

} // namespace zeus::dev
