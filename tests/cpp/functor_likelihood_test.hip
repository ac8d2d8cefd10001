// obj::LogLikelihood passed to zeus::Zeus as a functor (no built-in: its
// kernels are instantiated here, with no parameters in the problem descriptor)
// against the same fit through zeus_run_batch: starts drawn in the box, no PSO,
// two iterations, so that rounding has no time to grow.  Bin counts below and
// above the 128 that the per-workgroup form keeps in LDS.  Prints one line per
// case; returns 0 when all agree.
#include "zeus/zeus.hpp"

#include <cmath>
#include <cstdio>
#include <vector>

int
main()
{
  zeus::set_results_table(false);
  int bad = 0;
  for (int bins : {1, 63, 128, 129, 200})
    for (auto gradient : {zeus::Gradient::Adjoint, zeus::Gradient::Dual}) {
      std::vector<double> p(3 * bins);
      if (zeus_make_dijet(42, 3, bins, p.data()) != ZEUS_OK)
        return 1;
      zeus::DoubleBuffer dev(p.size());
      if (zeus_memcpy_h2d(dev.data(), p.data(), 8 * p.size()) != ZEUS_OK)
        return 1;
      const int N = 300;
      const zeus::obj::LogLikelihood f{dev.data(), bins};
      const auto r = zeus::Zeus(f, 0.0, 10.0, N, 2, -1, N + 1, "dijet", 1e-8, 7, 0, true,
                                zeus::PRNGType::PHILOX, {}, 0, gradient);
      zeus_problem q{};
      q.objective = ZEUS_OBJ_LOGLIK;
      q.dim = 4;
      q.lower = 0.0;
      q.upper = 10.0;
      q.n_starts = N;
      q.max_iter = 2;
      q.pso_iter = -1;
      q.required = N + 1;
      q.seed = 7;
      q.prng = ZEUS_PRNG_PHILOX;
      q.tol = 1e-8;
      q.params = dev.data();
      q.n_params = 3 * bins;
      zeus_options o{};
      o.gradient = gradient == zeus::Gradient::Dual ? ZEUS_GRAD_DUAL : ZEUS_GRAD_ADJOINT;
      o.form = ZEUS_FORM_GROUP;
      o.group_threads = 64;
      zeus_result w{};
      double x[4];
      if (zeus_run_batch(&q, 1, &o, &w, x, nullptr, nullptr) != ZEUS_OK)
        return 1;
      // the same kernel on the same bins: a few roundings at most
      bool ok = r.idx == w.idx && r.status == w.status && r.iter == w.iter &&
                std::isfinite(w.fval) && std::fabs(r.fval - w.fval) <= 1e-12 * std::fabs(w.fval);
      for (int d = 0; d < 4; ++d)
        ok = ok && std::fabs(r.coordinates[d] - x[d]) <= 1e-10 * (1.0 + std::fabs(x[d]));
      bad += !ok;
      std::printf("bins %d gradient %d: idx %d f %.17g, want %d %.17g%s\n", bins, o.gradient,
                  r.idx, r.fval, int(w.idx), w.fval, ok ? "" : " BAD");
      std::fflush(stdout);
    }
  return bad != 0;
}
