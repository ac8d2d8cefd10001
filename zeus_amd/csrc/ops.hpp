// ops.hpp -- the launch table of one (objective, D) class, as a template that
// each instantiation unit expands for its dimensions.
#pragma once

#include "runtime.hpp"
#include "zeus/bfgs_solo.hpp"

#include <algorithm>

namespace zeus::rt {

template <class F, int D, Gradient G>
__global__ void
eval_kernel(dev::ProblemDesc P, const double* x, int64_t n, double* f, double* g)
{
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  const F fn = dev::BuiltinProvider{}.template get<F>(P);
  f[i] = dev::lane_value<F, D>(fn, x + i * D);
  if (g)
    dev::lane_gradient<F, D, G>(fn, x + i * D, g + i * D);
}

// Values and gradients of the binned likelihood: a team of 16 lanes per point
// splits the bins.  A lane per point walked 100 bins with the power functions
// on 250 wavefronts for 16000 points (254 us, value and gradient in two
// passes); the teams make one pass over 4000 wavefronts.
constexpr int kEvalTeam = 16, kEvalTeams = 256 / kEvalTeam;

template <Gradient G>
__global__ __launch_bounds__(256) void
eval_bins_kernel(dev::ProblemDesc P, const double* x, int64_t n, double* f, double* g)
{
  using F = obj::LogLikelihood;
  const int r = threadIdx.x % kEvalTeam;
  const F fn = dev::BuiltinProvider{}.template get<F>(P);
  const bool adjoint = g != nullptr && G == Gradient::Adjoint;
  for (int64_t i = int64_t(blockIdx.x) * kEvalTeams + threadIdx.x / kEvalTeam; i < n;
       i += int64_t(gridDim.x) * kEvalTeams) {
    const double th[4] = {x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
    const F::Theta h(th);
    const double ra = 1.0 / h.a;
    double v = 0.0, d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int b = r; b < fn.n; b += kEvalTeam) {
      const F::Bin e = fn.bin(b);
      v += adjoint ? F::bin_gradient(h, ra, e, d) : F::bin_term(h, e);
      if constexpr (G == Gradient::Dual)
        if (g != nullptr)
#pragma unroll
          for (int k = 0; k < 4; ++k)
            d[k] -= fn.bin_dual(obj::SeededView{th, k}, b).dual;
    }
    v = dev::team_sum<kEvalTeam>(v);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      d[k] = dev::team_sum<kEvalTeam>(d[k]);
    if (r == 0)
      f[i] = v;
    if (g != nullptr && r < 4)
      g[4 * i + r] = r == 0 ? d[0] : r == 1 ? d[1] : r == 2 ? d[2] : d[3];
  }
}

template <class F, int D>
struct Ops {
  static constexpr bool kMfmaPso = F::id == obj::kGaussian && D >= 16;
  static constexpr bool kThreadOk = F::id != obj::kMlp && D <= 64;
  // workgroup sizes of the group form (the MLP's cooperative evaluator: eight
  // wavefronts of 16 points)
  static constexpr int kNGroup = F::id == obj::kMlp ? 1 : group_nt_count(D);
  static constexpr int nt_at(int k) { return F::id == obj::kMlp ? 512 : group_nt_at(D, k); }
  // tile form: Gaussian classes whose PSO already runs in tiles of 16
  static constexpr bool kTileOk = kMfmaPso;
  // PSO with a workgroup per particle: objectives whose one evaluation is
  // worth a workgroup (the MLP loss over its data points)
  static constexpr bool kGroupPso = F::id == obj::kMlp;
  static constexpr int kPsoGroupThreads = 512;
  using PsoEval = typename dev::GroupEvalSelect<F, kPsoGroupThreads, Gradient::Adjoint>::type;
  // PSO with a team of lanes per particle: the separable objectives beyond
  // four coordinates and the binned likelihood
  static constexpr int kPsoTeam = dev::pso_team_size<F, D>();
  static constexpr bool kPsoMany = F::id == obj::kLogLikelihood;
  static constexpr int kPsoPpb = kMfmaPso        ? dev::kPsoTile
                                 : kGroupPso     ? dev::kPsoGroupPpb
                                 : kPsoTeam != 0 ? 256 / (kPsoTeam != 0 ? kPsoTeam : 1)
                                                 : 256;

  static hipError_t pso(const dev::PsoArgs& a, int nb, hipStream_t s)
  {
    if (fault_take_launch())
      return hipErrorLaunchFailure;
    if constexpr (kMfmaPso)
      dev::pso_gaussian_mfma_kernel<D><<<nb, dev::kPsoTileThreads, 0, s>>>(a);
    else if constexpr (kGroupPso)
      dev::pso_group_kernel<F, D, kPsoGroupThreads, kPsoPpb, PsoEval, dev::BuiltinProvider>
        <<<nb, kPsoGroupThreads, 0, s>>>(a, {});
    else if constexpr (kPsoTeam != 0) {
      if constexpr (kPsoMany)
        if (a.ts == dev::kPsoManyTeam) {
          dev::pso_team_kernel<F, D, dev::kPsoManyTeam, dev::BuiltinProvider>
            <<<nb, 256, 0, s>>>(a, {});
          return hipGetLastError();
        }
      dev::pso_team_kernel<F, D, kPsoTeam, dev::BuiltinProvider><<<nb, 256, 0, s>>>(a, {});
    }
    else
      dev::pso_lane_kernel<F, D, dev::BuiltinProvider><<<nb, 256, 0, s>>>(a, {});
    return hipGetLastError();
  }

  // gBest after each problem's last iteration (one workgroup per problem)
  static hipError_t pso_final(const dev::PsoArgs& a, int n_probs, hipStream_t s)
  {
    if (fault_take_launch())
      return hipErrorLaunchFailure;
    dev::pso_final_kernel<256, D><<<n_probs, 256, 0, s>>>(a);
    return hipGetLastError();
  }

  static hipError_t bfgs_thread(const dev::ClassArgs& a, int gradient, hipStream_t s)
  {
    if constexpr (!kThreadOk) {
      return hipErrorInvalidConfiguration;
    } else {
      if (fault_take_launch())
        return hipErrorLaunchFailure;
      const int nb = int((a.total_starts + 255) / 256);
      if (gradient == 1)
        dev::bfgs_thread_kernel<F, D, Gradient::Dual, dev::BuiltinProvider>
          <<<nb, 256, 0, s>>>(a, {});
      else
        dev::bfgs_thread_kernel<F, D, Gradient::Adjoint, dev::BuiltinProvider>
          <<<nb, 256, 0, s>>>(a, {});
      return hipGetLastError();
    }
  }

  template <int NT>
  static constexpr bool kHReg = dev::RowChunk<D, NT>::kPerThread <= 50;

  // A large Gaussian's workgroup of 512 threads with the adjoint gradient keeps
  // the matrix in registers (bfgs_solo.hpp).
  template <int NT>
  static constexpr bool kSolo = F::id == obj::kGaussian && D > 64 && D <= 160 && NT == 512;

  template <int NT, Gradient G>
  static auto group_kernel()
  {
    if constexpr (kSolo<NT> && G == Gradient::Adjoint)
      return &dev::bfgs_solo_kernel<F, D, NT, dev::BuiltinProvider>;
    else
      return &dev::bfgs_group_kernel<F, D, NT, G, kHReg<NT>, dev::BuiltinProvider>;
  }

  template <int NT>
  static hipError_t group_nt(const dev::ClassArgs& a, int gradient, int grid, hipStream_t s)
  {
    if (gradient == 1)
      group_kernel<NT, Gradient::Dual>()<<<grid, NT, 0, s>>>(a, {});
    else
      group_kernel<NT, Gradient::Adjoint>()<<<grid, NT, 0, s>>>(a, {});
    return hipGetLastError();
  }

  // team form: separable built-in objectives whose H rows fit a lane
  static constexpr bool kTeamObj = F::id == obj::kRosenbrock || F::id == obj::kRastrigin ||
                                   F::id == obj::kAckley || F::id == obj::kSphere;
  template <int TS>
  static constexpr bool kTeamOk = kTeamObj && dev::team_fits<D, TS>();

  template <int TS, Gradient G>
  static auto team_kernel()
  {
    return &dev::bfgs_team_kernel<F, D, TS, G, dev::BuiltinProvider>;
  }
  template <int TS>
  static hipError_t team_ts(const dev::ClassArgs& a, int gradient, int grid, hipStream_t s)
  {
    if constexpr (!kTeamOk<TS>) {
      return hipErrorInvalidConfiguration;
    } else {
      if (gradient == 1)
        team_kernel<TS, Gradient::Dual>()<<<grid, dev::kTeamThreads, 0, s>>>(a, {});
      else
        team_kernel<TS, Gradient::Adjoint>()<<<grid, dev::kTeamThreads, 0, s>>>(a, {});
      return hipGetLastError();
    }
  }
  static hipError_t bfgs_team(const dev::ClassArgs& a, int gradient, int ts, int grid,
                              hipStream_t s)
  {
    if (fault_take_launch())
      return hipErrorLaunchFailure;
    if (ts == 4)
      return team_ts<4>(a, gradient, grid, s);
    if (ts == 8)
      return team_ts<8>(a, gradient, grid, s);
    if (ts == 16)
      return team_ts<16>(a, gradient, grid, s);
    return hipErrorInvalidConfiguration;
  }
  template <int TS>
  static int team_occ(int gradient)
  {
    if constexpr (!kTeamOk<TS>) {
      return 1;
    } else {
      static int cached[2] = {0, 0}; // per gradient; queried once per process
      int& c = cached[gradient == 1];
      if (c == 0) {
        int n = 0;
        const hipError_t e =
          gradient == 1
            ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, reinterpret_cast<const void*>(team_kernel<TS, Gradient::Dual>()),
                dev::kTeamThreads, 0)
            : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, reinterpret_cast<const void*>(team_kernel<TS, Gradient::Adjoint>()),
                dev::kTeamThreads, 0);
        c = (e == hipSuccess && n > 0) ? n : 1;
      }
      return c;
    }
  }
  static int team_blocks_per_cu(int gradient, int ts)
  {
    return ts == 4 ? team_occ<4>(gradient) : ts == 8 ? team_occ<8>(gradient) : team_occ<16>(gradient);
  }

  static hipError_t bfgs_group(const dev::ClassArgs& a, int gradient, int nt, int grid,
                               hipStream_t s)
  {
    if (fault_take_launch())
      return hipErrorLaunchFailure;
    if (nt == nt_at(0))
      return group_nt<nt_at(0)>(a, gradient, grid, s);
    if constexpr (kNGroup > 1)
      if (nt == nt_at(1))
        return group_nt<nt_at(1)>(a, gradient, grid, s);
    if constexpr (kNGroup > 2)
      if (nt == nt_at(2))
        return group_nt<nt_at(2)>(a, gradient, grid, s);
    return hipErrorInvalidConfiguration;
  }

  template <int NT>
  static int occ(int gradient)
  {
    static int cached[2] = {0, 0}; // per gradient; queried once per process
    int& c = cached[gradient == 1];
    if (c == 0)
      c = occ_query<NT>(gradient);
    return c;
  }
  template <int NT>
  static int occ_query(int gradient)
  {
    int n = 0;
    hipError_t e;
    if (gradient == 1)
      e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, reinterpret_cast<const void*>(group_kernel<NT, Gradient::Dual>()), NT, 0);
    else
      e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, reinterpret_cast<const void*>(group_kernel<NT, Gradient::Adjoint>()), NT, 0);
    return (e == hipSuccess && n > 0) ? n : 1;
  }

  static int group_blocks_per_cu(int gradient, int nt)
  {
    if (nt == nt_at(0))
      return occ<nt_at(0)>(gradient);
    if constexpr (kNGroup > 1)
      if (nt == nt_at(1))
        return occ<nt_at(1)>(gradient);
    if constexpr (kNGroup > 2)
      if (nt == nt_at(2))
        return occ<nt_at(2)>(gradient);
    return 1;
  }

  template <int NT>
  static constexpr int64_t slab_doubles()
  {
    constexpr int64_t n = dev::group_slab_doubles<D, NT, kHReg<NT>>();
    if constexpr (kSolo<NT>)
      return std::max(n, dev::SoloShape<D, NT>::kSlabDoubles);
    else
      return n;
  }
  static int64_t group_slab_per_block(int nt)
  {
    if (nt == nt_at(0))
      return slab_doubles<nt_at(0)>();
    if constexpr (kNGroup > 1)
      if (nt == nt_at(1))
        return slab_doubles<nt_at(1)>();
    if constexpr (kNGroup > 2)
      if (nt == nt_at(2))
        return slab_doubles<nt_at(2)>();
    return 0;
  }

  // tile form (bfgs_tile.hpp)
  static hipError_t bfgs_tile(const dev::TileArgs& a, int grid, hipStream_t s)
  {
    if constexpr (!kTileOk) {
      return hipErrorInvalidConfiguration;
    } else {
      if (fault_take_launch())
        return hipErrorLaunchFailure;
      dev::bfgs_tile_kernel<D><<<grid, dev::kTileThreads, 0, s>>>(a);
      return hipGetLastError();
    }
  }
  static int tile_blocks_per_cu()
  {
    if constexpr (!kTileOk) {
      return 1;
    } else {
      static int cached = 0;
      if (cached == 0) {
        int n = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &n, reinterpret_cast<const void*>(&dev::bfgs_tile_kernel<D>), dev::kTileThreads, 0);
        cached = (e == hipSuccess && n > 0) ? n : 1;
      }
      return cached;
    }
  }

  static hipError_t eval(const dev::ProblemDesc& P, const double* x, int64_t n, double* f,
                         double* g, int gradient, hipStream_t s)
  {
    if (fault_take_launch())
      return hipErrorLaunchFailure;
    const int nb = int((n + 127) / 128);
    if (nb == 0)
      return hipSuccess;
    if constexpr (F::id == obj::kLogLikelihood) {
      const int grid = int(std::min<int64_t>((n + kEvalTeams - 1) / kEvalTeams, 1 << 20));
      if (gradient == 1)
        eval_bins_kernel<Gradient::Dual><<<grid, 256, 0, s>>>(P, x, n, f, g);
      else
        eval_bins_kernel<Gradient::Adjoint><<<grid, 256, 0, s>>>(P, x, n, f, g);
      return hipGetLastError();
    } else {
      if (gradient == 1)
        eval_kernel<F, D, Gradient::Dual><<<nb, 128, 0, s>>>(P, x, n, f, g);
      else
        eval_kernel<F, D, Gradient::Adjoint><<<nb, 128, 0, s>>>(P, x, n, f, g);
      return hipGetLastError();
    }
  }

  static const ClassOps* table()
  {
    static const ClassOps t = [] {
      ClassOps o;
      o.objective = F::id;
      o.dim = D;
      o.pso_ppb = kPsoPpb;
      o.pso_team = kPsoTeam != 0;
      o.pso_many_ts = kPsoMany ? dev::kPsoManyTeam : 0;
      o.pso = &pso;
      o.pso_final = &pso_final;
      o.thread_ok = kThreadOk;
      o.bfgs_thread = &bfgs_thread;
      o.thread_slab_per_start = D <= dev::kThreadRegMaxD ? 0 : int64_t(D) * (D + 1) / 2;
      o.n_group = kNGroup;
      for (int k = 0; k < o.n_group; ++k)
        o.group_nt[k] = nt_at(k);
      o.bfgs_group = &bfgs_group;
      o.group_blocks_per_cu = &group_blocks_per_cu;
      o.group_slab_per_block = &group_slab_per_block;
      o.eval = &eval;
      if constexpr (kTeamOk<4>)
        o.team_ts[o.n_team++] = 4;
      if constexpr (kTeamOk<8>)
        o.team_ts[o.n_team++] = 8;
      if constexpr (kTeamOk<16>)
        o.team_ts[o.n_team++] = 16;
      o.bfgs_team = &bfgs_team;
      o.team_blocks_per_cu = &team_blocks_per_cu;
      o.tile_ok = kTileOk;
      if constexpr (kSolo<512>)
        o.solo_threads = 512;
      o.bfgs_tile = &bfgs_tile;
      o.tile_blocks_per_cu = &tile_blocks_per_cu;
      o.tile_slot_doubles = kTileOk ? dev::TileShape<D>::kSlotDoubles : 0;
      return o;
    }();
    return &t;
  }
};

} // namespace zeus::rt
