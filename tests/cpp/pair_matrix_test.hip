// PairMatrix (zeus/block.hpp) on the GPU: products after n appended rank-2
// pairs, across the folds, against the explicit matrix on the host.  Prints one
// line per case; returns 0 when all agree.
#include "zeus/block.hpp"

#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

using namespace zeus::dev;

// one workgroup: appends the n pairs (n x 2 x D), then out = H g
template <int D, int NT>
__global__ __launch_bounds__(NT) void
run(const double* pairs, int n, const double* g, double* slab, double* out)
{
  __shared__ double s[D], a[D], gl[D], part[pair_parts<D, NT>() * D];
  PairMatrix<D, NT> H;
  H.slab = slab;
  H.set_identity();
  for (int i = threadIdx.x; i < D; i += NT)
    gl[i] = g[i];
  for (int j = 0; j < n; ++j) {
    for (int i = threadIdx.x; i < D; i += NT) {
      s[i] = pairs[int64_t(j) * 2 * D + i];
      a[i] = pairs[int64_t(j) * 2 * D + D + i];
    }
    H.append(s, a);
    __syncthreads();
  }
  __syncthreads();
  H.apply(gl, part);
  for (int i = threadIdx.x; i < D; i += NT)
    out[i] = H.total(part, gl, i);
}

#define CHECK(x) \
  if ((x) != hipSuccess) \
    return std::printf("hip error\n"), 1;

template <int D, int NT>
int
cases(std::initializer_list<int> counts)
{
  int bad = 0, n_max = 0;
  for (int n : counts)
    n_max = n > n_max ? n : n_max;
  std::mt19937_64 rng(D);
  std::normal_distribution<double> N(0.0, 0.1);
  std::vector<double> pairs(size_t(n_max) * 2 * D), g(D), out(D);
  for (auto& v : pairs)
    v = N(rng);
  for (auto& v : g)
    v = N(rng);
  double *dp, *dg, *ds, *dout;
  CHECK(hipMalloc(&dp, pairs.size() * 8 + 8));
  CHECK(hipMalloc(&dg, D * 8));
  CHECK(hipMalloc(&dout, D * 8));
  CHECK(hipMalloc(&ds, group_slab_doubles<D, NT, false>() * 8));
  CHECK(hipMemcpy(dp, pairs.data(), pairs.size() * 8, hipMemcpyHostToDevice));
  CHECK(hipMemcpy(dg, g.data(), D * 8, hipMemcpyHostToDevice));
  for (int n : counts) {
    run<D, NT><<<1, NT>>>(dp, n, dg, ds, dout);
    CHECK(hipGetLastError());
    CHECK(hipMemcpy(out.data(), dout, D * 8, hipMemcpyDeviceToHost));
    // H g = g + sum s (a.g) + a (s.g); the size of the terms bounds the error
    std::vector<double> want(g), size(D);
    for (int i = 0; i < D; ++i)
      size[i] = std::fabs(g[i]);
    for (int j = 0; j < n; ++j) {
      const double* s = &pairs[size_t(j) * 2 * D];
      const double* a = s + D;
      double ag = 0.0, sg = 0.0, aa = 0.0, sa = 0.0;
      for (int i = 0; i < D; ++i) {
        ag += a[i] * g[i];
        sg += s[i] * g[i];
        aa += std::fabs(a[i] * g[i]);
        sa += std::fabs(s[i] * g[i]);
      }
      for (int i = 0; i < D; ++i) {
        want[i] += s[i] * ag + a[i] * sg;
        size[i] += std::fabs(s[i]) * aa + std::fabs(a[i]) * sa;
      }
    }
    double worst = 0.0;
    for (int i = 0; i < D; ++i)
      worst = std::fmax(worst, std::fabs(out[i] - want[i]) / size[i]);
    const double tol = (D + 2.0 * n + 8) * 2.2e-16; // a rounding per addition
    const bool ok = worst <= tol;
    bad += !ok;
    std::printf("D %d NT %d pairs %d: %.2g (%.2g)%s\n", D, NT, n, worst, tol, ok ? "" : " BAD");
  }
  return bad;
}

int
main()
{
  int bad = 0;
  bad += cases<321, 256>({0, 1, 2, 5, 7, 8, 159, 160, 161, 191, 192, 193, 300});
  bad += cases<300, 512>({3, 149, 150, 151, 183});
  bad += cases<520, 512>({1, 9, 160, 170});
  return bad != 0;
}
