// Hyperbolic tangent (zeus/tanh.hpp) on the GPU, where its reciprocal is the
// hardware's, against long double: over each range no further off than the
// library's tanh on the same points, at the worst and in the mean.  Prints one
// line per range; returns 0 when all hold.
#include "zeus/tanh.hpp"

#include <hip/hip_runtime.h>

#include <cstdio>
#include <random>
#include <vector>

__global__ void
run(const double* x, double* own, double* lib, int n)
{
  const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < n) {
    own[i] = zeus::dev::tanh_unit(x[i]);
    lib[i] = ::tanh(x[i]);
  }
}

int
main()
{
  constexpr int n = 1 << 20;
  std::vector<double> x(n), own(n), lib(n);
  double *dx, *d_own, *d_lib;
  if (hipMalloc(&dx, 8 * n) != hipSuccess || hipMalloc(&d_own, 8 * n) != hipSuccess ||
      hipMalloc(&d_lib, 8 * n) != hipSuccess)
    return 1;
  std::mt19937_64 rng(1);
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  int bad = 0;
  for (double range : {0.1, 0.36, 1.0, 4.0, 23.0}) {
    for (auto& v : x)
      v = range * u(rng);
    if (hipMemcpy(dx, x.data(), 8 * n, hipMemcpyHostToDevice) != hipSuccess)
      return 1;
    run<<<n / 256, 256>>>(dx, d_own, d_lib, n);
    if (hipMemcpy(own.data(), d_own, 8 * n, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(lib.data(), d_lib, 8 * n, hipMemcpyDeviceToHost) != hipSuccess)
      return 1;
    double worst[2] = {}, square[2] = {};
    for (int i = 0; i < n; ++i) {
      const long double t = ::tanhl(x[i]);
      int e;
      (void)std::frexp(double(t), &e);
      const double ulp = std::ldexp(1.0, e - 53);
      for (int k = 0; k < 2; ++k) {
        const double err = double(::fabsl((k == 0 ? own : lib)[i] - t)) / ulp;
        worst[k] = std::fmax(worst[k], err);
        square[k] += err * err;
      }
    }
    const bool ok = worst[0] <= worst[1] && square[0] <= square[1];
    bad += !ok;
    std::printf("|x| < %g: %.3f ulp at most (library %.3f), rms %.3f (%.3f)%s\n", range, worst[0],
                worst[1], std::sqrt(square[0] / n), std::sqrt(square[1] / n), ok ? "" : " BAD");
    std::fflush(stdout);
  }
  return bad != 0;
}
