// Hyperbolic tangent (zeus/tanh.hpp) against long double, on the host: the
// whole range, its ends, zeros, NaN.  Prints one line and returns 0 when every
// error is within an ulp.
#include "zeus/tanh.hpp"

#include <cstdio>

using namespace zeus::dev;

int
main()
{
  double worst = 0.0;
  auto check = [&](double x) {
    const long double t = ::tanhl(x);
    int e;
    (void)std::frexp(double(t), &e);
    const double ulp = std::fmax(std::ldexp(1.0, e - 53), 4.9e-324);
    worst = std::fmax(worst, double(::fabsl(tanh_unit(x) - t)) / ulp);
  };
  for (double r : {1e-300, 1e-9, 1e-3, 0.1, 0.36, 1.0, 4.0, 23.0})
    for (int i = 0; i < 40000; ++i)
      check(r * (2.0 * (i + 0.31) / 40000 - 1.0));
  for (int k = 0; k <= 64; ++k) // the edges of the reduction by ln 2 / 2
    for (double d : {-1e-15, 0.0, 1e-15})
      check(0.34657359027997264 * (k + 0.5) / 2.0 * (1.0 + d));
  for (double x : {0.0, 5e-324, 1e-310, 22.0, 700.0, 1e308, HUGE_VAL})
    check(x), check(-x);
  const bool rest = std::signbit(tanh_unit(-0.0)) && tanh_unit(std::nan("")) != tanh_unit(std::nan("")) &&
                    tanh_unit(HUGE_VAL) == 1.0 && tanh_unit(-1e308) == -1.0;
  std::printf("worst %.3f ulp, special values %d\n", worst, rest);
  return !(rest && worst <= 1.0);
}
