// obj::Gaussian passed to zeus::Zeus as a functor: its cooperative evaluator
// reads the prepared symmetric matrix.  Every start of a well-conditioned
// quadratic converges to the origin.  Prints one line per case; returns 0 when
// all do.
#include "zeus/zeus.hpp"

#include <cmath>
#include <cstdio>
#include <vector>

template <std::size_t D>
int
run(zeus::Gradient gradient)
{
  std::vector<double> c(D * D);
  for (std::size_t i = 0; i < D; ++i)
    for (std::size_t j = 0; j < D; ++j) // not symmetric: the value takes (C + C^T) / 2
      c[i * D + j] = (i == j ? 2.0 : 0.0) + 0.5 / double(D) * (i < j ? 1.5 : 0.5);
  zeus::DoubleBuffer dev(c.size());
  if (zeus_memcpy_h2d(dev.data(), c.data(), 8 * c.size()) != ZEUS_OK)
    return 1;
  const int N = 40;
  const zeus::obj::Gaussian<D> f{dev.data()};
  const auto r = zeus::Zeus(f, -5.0, 5.0, N, 200, 2, N + 1, "gaussian", 1e-7, 7, 0, true,
                            zeus::PRNGType::PHILOX, {}, 0, gradient);
  bool ok = r.status == 1 && r.c.claimed == N && std::fabs(r.fval) < 1e-14;
  for (std::size_t d = 0; d < D; ++d)
    ok = ok && std::fabs(r.coordinates[d]) < 1e-7; // the smallest eigenvalue is above 1
  std::printf("D %d gradient %d: status %d claimed %d f %g%s\n", int(D), int(gradient), r.status,
              r.c.claimed, r.fval, ok ? "" : " BAD");
  std::fflush(stdout);
  return !ok;
}

int
main()
{
  zeus::set_results_table(false);
  int bad = 0;
  for (auto g : {zeus::Gradient::Adjoint, zeus::Gradient::Dual})
    bad += run<3>(g) + run<32>(g) + run<100>(g) + run<150>(g);
  bad += run<300>(zeus::Gradient::Adjoint); // beyond 256: the pair list
  return bad != 0;
}
