// The likelihood's bin without power functions (zeus/binned.hpp) against the
// formula with them, on the host: ordinary parameters, and every mixture of
// zeros, signs, overflowing and non-finite parameters and bin centers.  Prints
// one line and returns 0 when all agree.
#include "zeus/binned.hpp"

#include <cfloat>
#include <cstdio>

using namespace zeus::dev;

int
main()
{
  const double inf = HUGE_VAL, nan = std::nan("");
  const double as[] = {0.0,  -1.0, 1e-300, 9e-31, 1e-30, 0.5,
                       10.0, 1e30, 1.1e30, 1e300, inf,   nan};
  const double ps[] = {0.0,    -0.1, 0.1,  -5.0, 5.0,  -99.0, 99.0, -299.0, 301.0, -699.0,
                       701.0,  -1e3, 1e3,  -1e6, 1e6,  1e300, -inf, inf,    nan};
  const double xs[] = {0.0768, 0.31, 0.5, 0.532, 0.999, 1e-20, 1e-300, 0.0, -0.5, 1.0, 1.5, nan};
  long n = 0, bad = 0;
  auto same = [](double u, double v, double tol) {
    if (u != u || v != v)
      return u != u && v != v;
    if (std::isinf(u) || std::isinf(v) || u == 0.0 || v == 0.0)
      return u == v;
    return std::fabs(u - v) <= tol * std::fabs(v) + 4 * DBL_TRUE_MIN;
  };
  for (double x : xs)
    for (double a : as)
      for (double b : ps)
        for (double c : ps)
          for (double d : {0.0, 0.1, -3.0, 1e6, inf}) {
            const DD lx = bin_log_x(x), l1 = bin_log_1mx(x);
            const BinLogs t{lx.hi, lx.lo, l1.hi, l1.lo};
            const BinMean m =
              bin_mean(a, b, c, d, std::log(a), a >= 1e-30 && a <= 1e30, x, t);
            const double q = c + d * std::log(x);
            const double pw = std::pow(1.0 - x, b), qw = std::pow(x, q);
            const double mean = a * pw / qw, lm = std::log(mean);
            // a few roundings; a denormal mean or power carries one of its own
            const double tiny = std::fmin(std::fmin(std::fabs(mean), std::fabs(pw)),
                                          std::fmin(std::fabs(qw), std::fabs(a * pw)));
            const double tol =
              32 * DBL_EPSILON + (tiny > 0 && tiny < 1e-290 ? 4 * DBL_TRUE_MIN / tiny : 0.0);
            const bool ok = same(m.mean, mean, tol) &&
                            (same(m.log_mean, lm, 8 * DBL_EPSILON) ||
                             std::fabs(m.log_mean - lm) <= tol);
            ++n;
            if (!ok && ++bad <= 10)
              std::printf("x %g a %g b %g c %g d %g: mean %.17g want %.17g, log %.17g want %.17g\n",
                          x, a, b, c, d, m.mean, mean, m.log_mean, lm);
          }
  std::printf("%ld bins, %ld differ\n", n, bad);
  return bad != 0;
}
