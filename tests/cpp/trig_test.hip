// Sine and cosine of whole turns (zeus/trig.hpp) against long double, on the
// host: the octant edges, quarter turns, large and non-finite arguments.
// Prints one line and returns 0 when every error is within the bound.
#include "zeus/trig.hpp"

#include <cstdio>

using namespace zeus::dev;

int
main()
{
  const long double tau = 6.283185307179586476925286766559005768L;
  double worst_c = 0.0, worst_s = 0.0;
  auto check = [&](double x) {
    const long double r = (long double)(x) - ::rintl(x); // exact
    worst_c = std::fmax(worst_c, std::fabs(double(cos_turns(x) - ::cosl(tau * r))));
    worst_s = std::fmax(worst_s, std::fabs(double(sin_turns(x) - ::sinl(tau * r))));
  };
  for (int o = -64; o <= 64; ++o) // octants of a turn and their neighbours
    for (double e : {0.0, 1e-17, 1e-9, -1e-9, 1e-3, -1e-3})
      check(o / 8.0 + e);
  for (int i = 0; i < 200000; ++i)
    check(-6.0 + 12.0 * (i + 0.37) / 200000);
  for (double x : {1e3 + 0.3, 1e8 + 0.125, 4503599627370497.0, 1e300})
    check(x);
  const bool nans = cos_turns(HUGE_VAL) != cos_turns(HUGE_VAL) &&
                    sin_turns(-HUGE_VAL) != sin_turns(-HUGE_VAL) &&
                    cos_turns(std::nan("")) != cos_turns(std::nan(""));
  std::printf("cosine %.3g sine %.3g nan %d\n", worst_c, worst_s, nans);
  // a rounding of the result, the series' roundings below it, long double's
  return !(nans && worst_c <= 2.0 * 1.11e-16 && worst_s <= 3.0 * 1.11e-16);
}
