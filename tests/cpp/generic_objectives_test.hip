// The likelihood and the network objective in numbers of a caller's own (a
// templated operator() takes any with the functions it needs) and in float,
// against double, on the host.  Prints one line and returns 0 when all agree.
#include "zeus/objectives.hpp"

#include <array>
#include <cmath>
#include <cstdio>
#include <vector>

namespace user {
struct Num { // a double that counts nothing: its functions are found by its namespace
  double v;
  ZEUS_HD Num(double x = 0.0) : v(x) {}
  ZEUS_HD Num operator+(Num o) const { return v + o.v; }
  ZEUS_HD Num operator-(Num o) const { return v - o.v; }
  ZEUS_HD Num operator*(Num o) const { return v * o.v; }
  ZEUS_HD Num operator/(Num o) const { return v / o.v; }
  ZEUS_HD Num& operator+=(Num o) { v += o.v; return *this; }
  ZEUS_HD Num& operator-=(Num o) { v -= o.v; return *this; }
  ZEUS_HD Num& operator/=(Num o) { v /= o.v; return *this; }
};
ZEUS_HD inline Num log(Num x) { return ::log(x.v); }
ZEUS_HD inline Num pow(Num x, Num y) { return ::pow(x.v, y.v); }
ZEUS_HD inline Num tanh(Num x) { return ::tanh(x.v); }
} // namespace user

static int bad = 0;
static void
near(const char* what, double a, double b, double tol)
{
  const bool ok = std::fabs(a - b) <= tol * std::fabs(b);
  bad += !ok;
  if (!ok)
    std::printf("%s: %.17g, want %.17g\n", what, a, b);
}

int
main()
{
  const int n = 40, m = 30;
  std::vector<double> p(3 * n), q(2 * m);
  for (int i = 0; i < n; ++i) {
    p[i] = 0.05 + 0.02 * i;
    p[n + i] = (i * 7) % 23;
    p[2 * n + i] = std::lgamma(p[n + i] + 1.0);
  }
  for (int i = 0; i < m; ++i) {
    q[i] = -1.0 + 2.0 * i / m;
    q[m + i] = std::sin(3.0 * q[i]);
  }
  const zeus::obj::LogLikelihood f{p.data(), n};
  const double t[4] = {0.5, 3.0, 1.5, 0.1};
  const double want = f(std::array<double, 4>{t[0], t[1], t[2], t[3]});
  // the same operations: a few roundings; float: 2^-24 in each of 40 terms of
  // exponents up to ten
  near("likelihood, own numbers", f(std::array<user::Num, 4>{t[0], t[1], t[2], t[3]}).v, want, 1e-13);
  near("likelihood, float",
       f(std::array<float, 4>{float(t[0]), float(t[1]), float(t[2]), float(t[3])}), want, 1e-4);
  double s = 0.0;
  for (int i = 0; i < n; ++i)
    s += f.bin_value(t, i);
  near("likelihood, bin by bin", s, want, 1e-13);

  constexpr std::size_t D = zeus::obj::Mlp::arity;
  std::array<double, D> th;
  std::array<user::Num, D> tu;
  std::array<float, D> tf;
  for (std::size_t k = 0; k < D; ++k) {
    th[k] = std::sin(1.0 + 0.7 * double(k));
    tu[k] = th[k];
    tf[k] = float(th[k]);
  }
  const zeus::obj::Mlp g{q.data(), m};
  const double w = g(th);
  near("network, own numbers", g(tu).v, w, 1e-12);
  near("network, float", g(tf), w, 1e-4);
  std::printf("%d differ\n", bad);
  return bad != 0;
}
