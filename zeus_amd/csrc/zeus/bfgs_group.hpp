// bfgs_group.hpp -- per-workgroup BFGS: one workgroup owns one start at a
// time and walks a strided list of starts (persistent grid).
//
// Restates the reference's tile form (include/bfgs_parallel.cuh:67-285) and
// keeps its per-start semantics, but every lane works, not only lane 0:
//   * H lives in the row-chunk layout of block.hpp, in registers when it
//     fits, in a per-workgroup global slab up to 256 dimensions and as a list
//     of rank-2 pairs beyond (PairMatrix);
//   * one read-modify-write pass over H per iteration: the rank-2 update of
//     iteration k is applied lazily inside iteration k+1's product
//     v = H' g_new, and since H is symmetric, u = H y = v + p and the next
//     direction p' = -H' g follow from v, u and two dot products;
//   * the objective is evaluated cooperatively (GroupEval below), the
//     gradient by a hand-written adjoint or by D dual passes spread over
//     the lanes (the reference's grad_ad_tile method, bfgs_parallel.cuh:17-54).
// Sums are workgroup reductions in a fixed order: results are deterministic
// but not bit-identical to the serial oracle (parity is to tolerance).
#pragma once

#include "batch.hpp"
#include "block.hpp"
#include "cs_product.hpp"
#include "lane_ops.hpp"
#include "philox.hpp"
#include "prng.hpp"
#include "trig.hpp"

namespace zeus::dev {

// LDS scratch handed to the evaluators.
struct GroupScratch {
  double* part;   // CH * D
  double* stash;  // D
  double* scalar; // 4
};

// ---------------------------------------------------------------------------
// Default evaluator: one lane evaluates (works for any functor); gradient by
// the functor's adjoint on one lane, or by dual passes spread over lanes.
template <class F, int D, int NT, Gradient G>
struct GroupEvalLane {
  GroupScratch sc;
  int par = 0;
  ZEUS_D void bind(const F&, const ProblemDesc&) {}
  ZEUS_D double value(const F& f, const double* x, Block<NT>&)
  {
    double* b = sc.scalar + par;
    par ^= 1;
    if (threadIdx.x == 0)
      *b = lane_value<F, D>(f, x);
    __syncthreads();
    return *b;
  }
  ZEUS_D void gradient(const F& f, const double* x, double* g, bool, Block<NT>&)
  {
    if constexpr (G == Gradient::Adjoint && HasAdjoint<F>) {
      if (threadIdx.x == 0)
        (void)f.value_and_gradient(x, g);
    } else {
      for (int i = threadIdx.x; i < D; i += NT)
        g[i] = lane_dual_pass<F, D>(f, x, i);
    }
  }
};

// Dual gradient shared by the cooperative evaluators: pass i on lane i.
template <class F, int D, int NT>
ZEUS_D ZEUS_FI void
group_dual_gradient(const F& f, const double* x, double* g)
{
  for (int i = threadIdx.x; i < D; i += NT)
    g[i] = lane_dual_pass<F, D>(f, x, i);
}

// ---------------------------------------------------------------------------
// Gaussian: Cs = (C + C^T) / 2 (prepared once per call, ProblemDesc::aux)
// held in the row-chunk layout; f = 0.5 x.(Cs x); g = Cs x is the
// by-product of the value, so an accepted line-search trial already carries
// the gradient.
template <int D, int NT, Gradient G>
struct GroupEvalGaussian {
  using F = obj::Gaussian<D>;
  using Lay = RowChunk<D, NT>;
  static constexpr bool kReg = Lay::kPerThread <= 50;
  DistMatrix<D, NT, kReg> C;
  const double* Cs = nullptr;
  GroupScratch sc;

  ZEUS_D void bind(const F&, const ProblemDesc& P)
  {
    Cs = P.aux;
    if constexpr (kReg)
      C.load(Cs);
  }
  // part <- chunk partials of Cs x
  ZEUS_D ZEUS_FI void partials(const double* x)
  {
    if constexpr (kReg) {
      C.pass(x, nullptr, nullptr, false, sc.part);
    } else {
      const int c = threadIdx.x % Lay::CH, r0 = threadIdx.x / Lay::CH;
      for (int k = 0; k < Lay::R; ++k) {
        const int row = r0 + k * Lay::RPP;
        if (row < D) {
          double acc = 0.0;
          for (int l = 0; l < Lay::L; ++l) {
            const int col = c * Lay::L + l;
            if (col < D) // Cs symmetric: read column-wise, lanes coalesce
              acc = ::fma(Cs[col * D + row], x[col], acc);
          }
          sc.part[c * D + row] = acc;
        }
      }
    }
  }
  ZEUS_D double value(const F&, const double* x, Block<NT>& blk)
  {
    partials(x);
    __syncthreads();
    double t = 0.0;
    for (int row = threadIdx.x; row < D; row += NT) {
      const double v = chunk_total<D, NT>(sc.part, row);
      sc.stash[row] = v;
      t = ::fma(x[row], v, t);
    }
    return 0.5 * blk.sum1(t);
  }
  ZEUS_D void gradient(const F& f, const double* x, double* g, bool at_last_value,
                       Block<NT>& blk)
  {
    if constexpr (G == Gradient::Dual) {
      group_dual_gradient<F, D, NT>(f, x, g);
    } else {
      if (!at_last_value) {
        partials(x);
        __syncthreads();
        for (int row = threadIdx.x; row < D; row += NT)
          sc.stash[row] = chunk_total<D, NT>(sc.part, row);
      }
      for (int row = threadIdx.x; row < D; row += NT)
        g[row] = sc.stash[row];
    }
    (void)blk;
  }
};

// ---------------------------------------------------------------------------
// Separable sums over the coordinates (Rosenbrock, Rastrigin, Ackley,
// sphere): lane i evaluates term i, the workgroup sums.
template <class F, int D, int NT, Gradient G>
struct GroupEvalSeparable {
  GroupScratch sc;
  ZEUS_D void bind(const F&, const ProblemDesc&) {}

  ZEUS_D double value(const F&, const double* x, Block<NT>& blk)
  {
    if constexpr (F::id == obj::kAckley) {
      double v[2] = {0.0, 0.0};
      for (int i = threadIdx.x; i < D; i += NT) {
        v[0] = ::fma(x[i], x[i], v[0]);
        v[1] += ::cos(2.0 * obj::kPi * x[i]);
      }
      blk.template sum<2>(v);
      return finish(v[0], v[1]);
    } else {
      double t = 0.0;
      for (int i = threadIdx.x; i < D; i += NT)
        t += term(x, i);
      return finish(blk.sum1(t), 0.0);
    }
  }
  ZEUS_D ZEUS_FI double term(const double* x, int i) const
  {
    if constexpr (F::id == obj::kRosenbrock) {
      if (i >= D - 1)
        return 0.0;
      const double t1 = 1.0 - x[i];
      const double t2 = x[i + 1] - x[i] * x[i];
      return t1 * t1 + 100.0 * t2 * t2;
    } else if constexpr (F::id == obj::kRastrigin) {
      return x[i] * x[i] - 10.0 * ::cos(2.0 * obj::kPi * x[i]);
    } else {
      return x[i] * x[i];
    }
  }
  // Line-search trials without a trip through LDS: the values at x + alpha p,
  // alpha = a0, a0 / 2, ... for kTrials trials side by side.  A lane holds its
  // coordinates of x and p (and the next coordinate's for Rosenbrock's
  // coupling) during the search; each trial's terms and sum are value()'s.
  static constexpr int kTrials = 4;
  // One wavefront with no more than half a wavefront of coordinates: kPack
  // trials share it, kLane lanes each (whole rows, so each sum keeps its bits:
  // the rows left out added 0.0).  A search is bound by the instructions of its
  // trials, and at 20 coordinates 44 of 64 lanes had none: Rastrigin-20 (2048
  // starts) 0.81 -> 0.63 ms a call, Ackley-10 (1000) 0.167 -> 0.153.
  static constexpr int kPack = NT != kWave || D <= 4 || D > 32 ? 1 : D <= 16 ? 4 : 2;
  static constexpr int kLane = NT / kPack;
  static constexpr int KC = (D + kLane - 1) / kLane;
  static_assert(kPack == 1 || KC == 1, "a trial's coordinates in one pass");
  static constexpr bool kNext = F::id == obj::kRosenbrock;
  // Rastrigin and Ackley: the lane's angles of the search are small
  static constexpr bool kAngles = F::id == obj::kRastrigin || F::id == obj::kAckley;
  double tx[KC], tp[KC], nx[kNext ? KC : 1], np[kNext ? KC : 1];
  bool small = !kAngles;

  ZEUS_D ZEUS_FI void trials_begin(const double* x, const double* p)
  {
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      const int i = int(threadIdx.x) % kLane + k * NT;
      tx[k] = i < D ? x[i] : 0.0;
      tp[k] = i < D ? p[i] : 0.0;
      if constexpr (kNext) {
        nx[k] = i < D - 1 ? x[i + 1] : 0.0;
        np[k] = i < D - 1 ? p[i + 1] : 0.0;
      }
    }
    if constexpr (kAngles) {
      small = true;
#pragma unroll
      for (int k = 0; k < KC; ++k)
        small = small && ::fabs(tx[k]) + ::fabs(tp[k]) < kSmallCoordinate;
    }
  }
  // One trial per lane, for dimensions whose value is a few operations: lane t
  // takes x + 2^-t p by itself, with the terms added in the pairs of the
  // wavefront's sum, so the whole search is one evaluation.
  static constexpr bool kLaneTrials = D <= 4 && NT == kWave;
  ZEUS_D ZEUS_FI double lane_trial(double alpha, const double* x, const double* p) const
  {
    double y[D + 1], u[4] = {0.0, 0.0, 0.0, 0.0}, c[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < D; ++i)
      y[i] = ::fma(alpha, p[i], x[i]);
    y[D] = 0.0;
#pragma unroll
    for (int i = 0; i < D && i < 4; ++i) {
      if constexpr (F::id == obj::kAckley) {
        u[i] = ::fma(y[i], y[i], u[i]);
        c[i] += ::cos(2.0 * obj::kPi * y[i]);
      } else {
        u[i] += term(y, i);
      }
    }
    const double v = (u[0] + u[1]) + (u[2] + u[3]);
    return finish(v, (c[0] + c[1]) + (c[2] + c[3]));
  }
  // the value from the sum(s) of the terms
  ZEUS_D ZEUS_FI static double finish(double v, double c)
  {
    if constexpr (F::id == obj::kAckley) {
      const double term1 = -20.0 * ::exp(-0.2 * ::sqrt(v / int(D)));
      const double term2 = -::exp(c / int(D));
      return term1 + term2 + 20.0 + ::exp(1.0);
    } else if constexpr (F::id == obj::kRastrigin) {
      return 10.0 * D + v;
    } else {
      return v;
    }
  }

  // the lane's terms of the trials at a0, a0 2^-kPack, ... (K of them)
  template <int K, bool Small, int KA>
  ZEUS_D ZEUS_FI void trial_terms(double a0, double (&v)[K], double (&c)[KA]) const
  {
#pragma unroll
    for (int t = 0; t < K; ++t) {
      const double alpha = a0 * (1.0 / double(1 << (t * kPack)));
      v[t] = 0.0;
      if constexpr (F::id == obj::kAckley)
        c[t] = 0.0;
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        const int i = int(threadIdx.x) % kLane + k * NT;
        const double xi = ::fma(alpha, tp[k], tx[k]);
        if constexpr (F::id == obj::kRosenbrock) {
          const double xn = ::fma(alpha, np[k], nx[k]);
          const double t1 = 1.0 - xi;
          const double t2 = xn - xi * xi;
          if (i < D - 1)
            v[t] += t1 * t1 + 100.0 * t2 * t2;
        } else if constexpr (F::id == obj::kRastrigin) {
          if (i < D)
            v[t] += xi * xi - 10.0 * angle_cos<Small>(2.0 * obj::kPi * xi);
        } else if constexpr (F::id == obj::kAckley) {
          if (i < D) {
            v[t] = ::fma(xi, xi, v[t]);
            c[t] += angle_cos<Small>(2.0 * obj::kPi * xi);
          }
        } else if (i < D) {
          v[t] += xi * xi;
        }
      }
    }
  }
  // the sum over a trial's lanes, as the wavefront's sum has it
  ZEUS_D ZEUS_FI static double pack_sum(double v)
  {
    v = row_sum(v);
    if constexpr (kPack == 2) {
      const double lo = readlane_f64(v, 0) + readlane_f64(v, 16);
      const double hi = readlane_f64(v, 32) + readlane_f64(v, 48);
      v = threadIdx.x < 32 ? lo : hi;
    }
    return 0.0 + v;
  }
  // K batches of kPack trials: the lane's are at a0, a0 2^-kPack, ...
  template <int K>
  ZEUS_D ZEUS_FI void pack_trials(double a0, double (&v)[K])
  {
    double c[F::id == obj::kAckley ? K : 1] = {};
    by_angle(small, [&](auto sm) { trial_terms<K, sm()>(a0, v, c); });
#pragma unroll
    for (int t = 0; t < K; ++t)
      if constexpr (F::id == obj::kAckley)
        v[t] = finish(pack_sum(v[t]), pack_sum(c[t]));
      else
        v[t] = finish(pack_sum(v[t]), 0.0);
  }
  template <int K>
  ZEUS_D ZEUS_FI void trials(double a0, double (&v)[K], Block<NT>& blk)
  {
    double c[F::id == obj::kAckley ? K : 1] = {};
    by_angle(small, [&](auto sm) { trial_terms<K, sm()>(a0, v, c); });
    blk.template sum<K>(v);
    if constexpr (F::id == obj::kAckley)
      blk.template sum<K>(c);
#pragma unroll
    for (int t = 0; t < K; ++t)
      v[t] = finish(v[t], c[F::id == obj::kAckley ? t : 0]);
  }
  ZEUS_D void gradient(const F& f, const double* x, double* g, bool, Block<NT>& blk)
  {
    if constexpr (G == Gradient::Dual) {
      group_dual_gradient<F, D, NT>(f, x, g);
    } else if constexpr (F::id == obj::kRosenbrock) {
      for (int i = threadIdx.x; i < D; i += NT) {
        double gi = 0.0;
        if (i < D - 1) {
          const double t1 = 1.0 - x[i];
          const double t2 = x[i + 1] - x[i] * x[i];
          gi = -2.0 * t1 - (2.0 * x[i]) * (200.0 * t2);
        }
        if (i > 0) {
          const double t2p = x[i] - x[i - 1] * x[i - 1];
          gi += 200.0 * t2p;
        }
        g[i] = gi;
      }
    } else if constexpr (F::id == obj::kRastrigin) {
      const double k = 10.0 * (2.0 * obj::kPi);
      for (int i = threadIdx.x; i < D; i += NT)
        g[i] = 2.0 * x[i] + k * ::sin(2.0 * obj::kPi * x[i]);
    } else if constexpr (F::id == obj::kAckley) {
      double v[2] = {0.0, 0.0};
      for (int i = threadIdx.x; i < D; i += NT) {
        v[0] = ::fma(x[i], x[i], v[0]);
        v[1] += ::cos(2.0 * obj::kPi * x[i]);
      }
      blk.template sum<2>(v);
      const double r = ::sqrt(v[0] / int(D));
      const double e1 = ::exp(-0.2 * r);
      const double e2 = ::exp(v[1] / int(D));
      const double q = (4.0 * e1) / (double(int(D)) * r);
      const double c = (2.0 * obj::kPi / int(D)) * e2;
      for (int i = threadIdx.x; i < D; i += NT)
        g[i] = q * x[i] + c * ::sin(2.0 * obj::kPi * x[i]);
    } else {
      for (int i = threadIdx.x; i < D; i += NT)
        g[i] = 2.0 * x[i];
    }
  }
};

// ---------------------------------------------------------------------------
// Poisson NLL: bins spread over the lanes.  The first kKeep bins stay in LDS
// from problem to problem, and their means at the last value, from which the
// gradient there follows without evaluating the powers again; every lane reads
// back only what it wrote.  The dual gradient makes its four forward passes
// bin by bin on the bin's lane and adds them in bin order.
template <int NT, Gradient G>
struct GroupEvalLogLik {
  using F = obj::LogLikelihood;
  static constexpr bool kOneSite = true;
  static constexpr int kKeep = 128;
  static constexpr int kFields = 5; // x, k, lgamma(k + 1), ln x, ln(1 - x)
  struct Lds {
    double bin[kFields][kKeep];
    double mean[kKeep], ratio[kKeep];
    double dual[G == Gradient::Dual ? 4 : 1][G == Gradient::Dual ? NT : 1];
  };
  GroupScratch sc;
  Lds* L;

  // the bins are the functor's: a caller's own functor (zeus.hpp) has none in P
  ZEUS_D void bind(const F& f, const ProblemDesc&)
  {
    __shared__ Lds lds;
    L = &lds;
    for (int i = threadIdx.x; i < f.n && i < kKeep; i += NT) {
      const F::Bin b = f.bin(i);
      const double v[kFields] = {b.x, b.k, b.lgk, b.t.lx, b.t.l1};
#pragma unroll
      for (int e = 0; e < kFields; ++e)
        L->bin[e][i] = v[e];
    }
  }
  ZEUS_D ZEUS_FI F::Bin bin(const F& f, int i) const
  {
    if (i >= kKeep)
      return f.bin(i);
    return {L->bin[0][i], L->bin[1][i], L->bin[2][i], {L->bin[3][i], 0.0, L->bin[4][i], 0.0}};
  }
  ZEUS_D double value(const F& f, const double* th, Block<NT>& blk)
  {
    const double a = th[0], b = th[1], c = th[2], d = th[3];
    double t = 0.0;
#pragma unroll 1
    for (int i = threadIdx.x; i < f.n; i += NT) {
      const F::Bin e = bin(f, i);
      const BinPow m = bin_pow(a, b, c, d, e.x, e.t);
      if (i < kKeep) {
        L->mean[i] = m.mean;
        L->ratio[i] = m.ratio;
      }
      t += F::pow_term(e, m);
    }
    return blk.sum1(t);
  }
  // the gradient at the point of the last value
  ZEUS_D void gradient(const F& f, const double* th, double* g, bool, Block<NT>& blk)
  {
    if constexpr (G == Gradient::Dual) {
      double t = 0.0; // lane k < 4: derivative k
#pragma unroll 1
      for (int c0 = 0; c0 < f.n; c0 += NT) {
        const int i = c0 + int(threadIdx.x);
        if (i < f.n)
#pragma unroll 1
          for (int k = 0; k < 4; ++k)
            L->dual[k][threadIdx.x] = f.bin_dual(obj::SeededView{th, k}, i).dual;
        __syncthreads();
        if (threadIdx.x < 4) {
          const int n = f.n - c0 < NT ? f.n - c0 : NT;
#pragma unroll 8
          for (int j = 0; j < n; ++j)
            t = t - L->dual[threadIdx.x][j];
        }
        __syncthreads();
      }
      if (threadIdx.x < 4)
        g[threadIdx.x] = t;
    } else {
      const double a = th[0], b = th[1], c = th[2], d = th[3];
      double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
      for (int i = threadIdx.x; i < f.n; i += NT) {
        const F::Bin e = bin(f, i);
        const BinPow m = i < kKeep ? BinPow{L->mean[i], L->ratio[i]}
                                   : bin_pow(a, b, c, d, e.x, e.t);
        F::pow_gradient(e, m, v);
      }
      blk.template sum<4>(v);
      if (threadIdx.x < 4)
        g[threadIdx.x] = v[threadIdx.x];
    }
  }
};

// ---------------------------------------------------------------------------
// MLP (1-16-16-1 tanh, least squares over m points), a wavefront taking 16
// points at a time in the operand layout of the FP64 MFMA: lane l works for
// point l % 16 and, in every layer, for the neurons 4 q + l / 16 (q < 4).  The
// first layer's activations are then the B operand of the product with the
// hidden weights, whose result has the second layer's neurons in the same lanes
// and registers, and its deltas are again the B operand of the product with
// the transposed weights.  Only the weights' own gradient d2 h1^T contracts over
// the points and turns both 16 x 16 blocks round through LDS.  The 65
// per-neuron gradient terms add up in registers and are summed over a row of
// lanes once per gradient; the wavefronts' shares are added in order.
//
// The 32 hyperbolic tangents of a point bound it (VALU issue).  With a lane per
// point, every weight was an LDS broadcast to every wavefront, which cost as
// much again, and the sums over points were 65 wavefront reductions and a serial
// product (18 us a value and 41 us a gradient).  A lane's activations of its
// first kKeep groups stay in registers from the value to the gradient at the
// same point.  The dual gradient keeps the reference's D forward passes spread
// over the lanes.
template <int NT, Gradient G>
struct GroupEvalMlp {
  using F = obj::Mlp;
  static constexpr bool kOneSite = true;
  static constexpr int H = F::H, W2 = F::W2, W3 = F::W3, D = int(F::arity);
  static constexpr int NW = NT / kWave;
  static constexpr int kPoints = 16;            // points of a group
  static constexpr int kKeep = 256 / (kPoints * NW); // groups kept per wavefront
  static constexpr int Q = 4;                   // neurons per lane and layer
  GroupScratch sc;
  struct Point { // a lane's share of its point
    double h1[Q], h2[Q], res;
  };
  Point kept[kKeep];
  ZEUS_D void bind(const F&, const ProblemDesc&) {}

  // the weights a lane needs of the forward pass
  struct Weights {
    double w1[Q], b1[Q], a2[Q], b2[Q], w3[Q], b3;
    ZEUS_D ZEUS_FI explicit Weights(const double* th)
    {
      const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int n = 4 * q + lk;
        w1[q] = th[2 * n];
        b1[q] = th[2 * n + 1];
        a2[q] = th[W2 + li * (H + 1) + n];
        b2[q] = th[W2 + n * (H + 1) + H];
        w3[q] = th[W3 + n];
      }
      b3 = th[W3 + H];
    }
  };
  // forward pass of the point; all lanes of the wavefront
  ZEUS_D ZEUS_FI static void forward(const Weights& w, double x, double y, Point& o)
  {
#pragma unroll
    for (int q = 0; q < Q; ++q)
      o.h1[q] = tanh_unit(::fma(w.w1[q], x, w.b1[q]));
    mfma_acc_t z = {w.b2[0], w.b2[1], w.b2[2], w.b2[3]};
#pragma unroll
    for (int q = 0; q < Q; ++q)
      z = __builtin_amdgcn_mfma_f64_16x16x4f64(w.a2[q], o.h1[q], z, 0, 0, 0);
    double out = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      o.h2[q] = tanh_unit(z[q]);
      out = ::fma(o.h2[q], w.w3[q], out);
    }
    o.res = (xor_sum<32>(xor_sum<16>(out)) + w.b3) - y;
  }
  // fn(group's index in the wavefront, its point (any valid one past the end),
  // whether it exists) over the wavefront's groups
  template <class Fn>
  ZEUS_D ZEUS_FI static void groups(const F& f, Fn&& fn)
  {
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
#pragma unroll
    for (int j = 0; j < kKeep; ++j) {
      const int p = (w + j * NW) * kPoints + (int(threadIdx.x) & 15);
      if ((w + j * NW) * kPoints < f.m)
        fn(j, p < f.m ? p : f.m - 1, p < f.m);
    }
#pragma unroll 1
    for (int j = kKeep; (w + j * NW) * kPoints < f.m; ++j) {
      const int p = (w + j * NW) * kPoints + (int(threadIdx.x) & 15);
      fn(j, p < f.m ? p : f.m - 1, p < f.m);
    }
  }

  ZEUS_D double value(const F& f, const double* th, Block<NT>& blk)
  {
    const Weights wt(th);
    const bool counts = (threadIdx.x & 63) < 16; // one of a point's four lanes
    double t = 0.0;
    groups(f, [&](auto j, int p, bool live) {
      Point o;
      forward(wt, f.P[p], f.P[f.m + p], o);
      if (counts && live)
        t = ::fma(o.res, o.res, t);
      if (j < kKeep)
        kept[j < kKeep ? j : 0] = o;
    });
    return blk.sum1(t) / double(f.m);
  }

  // the gradient at the point of the last value
  ZEUS_D void gradient(const F& f, const double* th, double* g, bool, Block<NT>&)
  {
    if constexpr (G == Gradient::Dual) {
      group_dual_gradient<F, D, NT>(f, th, g);
    } else {
      __shared__ double turn[NW][2][H][H + 1];
      const int tid = threadIdx.x, w = tid / kWave, lane = tid % kWave;
      const int li = lane & 15, lk = lane >> 4;
      const double scale = 2.0 / double(f.m);
      auto& A = turn[w][0];
      auto& B = turn[w][1];
      double a2t[Q], w3[Q]; // transposed hidden weights, output weights
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        a2t[q] = th[W2 + (4 * q + lk) * (H + 1) + li];
        w3[q] = th[W3 + 4 * q + lk];
      }
      mfma_acc_t acc = {0.0, 0.0, 0.0, 0.0}; // weights (4 q + lk, li)
      double sw1[Q] = {}, sb1[Q] = {}, sb2[Q] = {}, sw3[Q] = {}, sb3 = 0.0;
      groups(f, [&](auto j, int p, bool live) {
        Point o;
        const double x = f.P[p];
        if (j < kKeep)
          o = kept[j < kKeep ? j : 0];
        else
          forward(Weights(th), x, f.P[f.m + p], o);
        const double dy = live ? scale * o.res : 0.0;
        double d2[Q];
        mfma_acc_t d1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          d2[q] = (dy * w3[q]) * ::fma(-o.h2[q], o.h2[q], 1.0);
          sb2[q] += d2[q];
          sw3[q] = ::fma(dy, o.h2[q], sw3[q]);
          A[4 * q + lk][li] = d2[q];
          B[4 * q + lk][li] = o.h1[q];
        }
        sb3 += dy;
#pragma unroll
        for (int q = 0; q < Q; ++q)
          d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a2t[q], d2[q], d1, 0, 0, 0);
        team_exchange();
#pragma unroll
        for (int q = 0; q < Q; ++q)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[li][4 * q + lk], B[li][4 * q + lk], acc, 0,
                                                     0, 0);
        team_exchange();
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const double d = d1[q] * ::fma(-o.h1[q], o.h1[q], 1.0);
          sb1[q] += d;
          sw1[q] = ::fma(d, x, sw1[q]);
        }
      });
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        sw1[q] = row_sum(sw1[q]);
        sb1[q] = row_sum(sb1[q]);
        sb2[q] = row_sum(sb2[q]);
        sw3[q] = row_sum(sw3[q]);
      }
      sb3 = row_sum(sb3);
      // the wavefronts' shares (kParts at a time), then their sum
      constexpr int kParts = pair_parts<D, NT>();
#pragma unroll 1
      for (int t = 0; t < NW / kParts; ++t) {
        if (w / kParts == t) {
          double* part = sc.part + (w % kParts) * D;
          auto put = [&](int i, double v) { part[i] = t == 0 ? v : part[i] + v; };
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            const int n = 4 * q + lk;
            put(W2 + n * (H + 1) + li, acc[q]);
            if (li == 0) {
              put(2 * n, sw1[q]);
              put(2 * n + 1, sb1[q]);
              put(W2 + n * (H + 1) + H, sb2[q]);
              put(W3 + n, sw3[q]);
            }
          }
          if (lane == 0)
            put(W3 + H, sb3);
        }
        __syncthreads();
      }
      for (int i = tid; i < D; i += NT) {
        double t = sc.part[i];
#pragma unroll
        for (int v = 1; v < kParts; ++v)
          t += sc.part[v * D + i];
        g[i] = t;
      }
    }
  }
};

// Evaluator per objective type.  Specialisations key on the objective type
// alone (its dimension parameter is a std::size_t; deducing it through an
// int parameter would fail and silently select the one-lane fallback).
template <class F, int NT, Gradient G>
struct GroupEvalSelect {
  using type = GroupEvalLane<F, int(F::arity), NT, G>;
};
template <std::size_t D, int NT, Gradient G>
struct GroupEvalSelect<obj::Gaussian<D>, NT, G> {
  using type = GroupEvalGaussian<int(D), NT, G>;
};
template <std::size_t D, int NT, Gradient G>
struct GroupEvalSelect<obj::Rosenbrock<D>, NT, G> {
  using type = GroupEvalSeparable<obj::Rosenbrock<D>, int(D), NT, G>;
};
template <std::size_t D, int NT, Gradient G>
struct GroupEvalSelect<obj::Rastrigin<D>, NT, G> {
  using type = GroupEvalSeparable<obj::Rastrigin<D>, int(D), NT, G>;
};
template <std::size_t D, int NT, Gradient G>
struct GroupEvalSelect<obj::Ackley<D>, NT, G> {
  using type = GroupEvalSeparable<obj::Ackley<D>, int(D), NT, G>;
};
template <std::size_t D, int NT, Gradient G>
struct GroupEvalSelect<obj::Sphere<D>, NT, G> {
  using type = GroupEvalSeparable<obj::Sphere<D>, int(D), NT, G>;
};
template <int NT, Gradient G>
struct GroupEvalSelect<obj::LogLikelihood, NT, G> {
  using type = GroupEvalLogLik<NT, G>;
};
template <int NT, Gradient G>
struct GroupEvalSelect<obj::Mlp, NT, G> {
  using type = GroupEvalMlp<NT, G>;
};

// Whether an evaluator takes line-search trials together: 0 one by one through
// LDS, 1 several side by side (kTrials, a divisor of the 20 after the full
// step), 2 one per lane.
template <class Eval>
constexpr int
group_batches_trials()
{
  if constexpr (requires { Eval::kTrials; }) {
    static_assert(kLineSearchTrials % Eval::kTrials == 0, "whole batches");
    return Eval::kLaneTrials ? 2 : 1;
  } else {
    return 0;
  }
}

// Whether the kernel evaluates starting points and trials at one place in its
// code (the binned likelihood's four power functions per pair of bins).
template <class Eval>
constexpr bool
group_one_site()
{
  return requires { Eval::kOneSite; };
}

// ---------------------------------------------------------------------------
// LDS vectors of one workgroup.
template <int D, int NT, bool PAIRS>
struct GroupVectors {
  double x[D], g[D], p[D], xt[D], gn[D], v[D];
  double s0[D], a0[D]; // current rank-2 pair
  double s1[PAIRS ? 1 : D], a1[PAIRS ? 1 : D]; // pending one (none with a pair list)
  double part[PAIRS ? pair_parts<D, NT>() * D : RowChunk<D, NT>::CH * D];
  double stash[D];
  double red[8 * (NT / kWave)];
  double scalar[4];
  int flag;
};

template <class F, int D, int NT, Gradient G, bool HREG, class Eval>
ZEUS_D void
group_bfgs(const F& f, GroupVectors<D, NT, kPairForm<D, NT, HREG>>& L,
           GroupH<D, NT, HREG>& H, Eval& ev,
           Block<NT>& blk, const ProblemDesc& P, Control* ctl, int64_t s,
           const double* starts, const StartOut& out)
{
  const int tid = threadIdx.x;
  const int64_t sl = s - P.start0;
  constexpr bool kPairs = kPairForm<D, NT, HREG>;
  double* sc = L.s0; // s of this iteration
  double* ac = L.a0;
  double* sp = L.s1; // pending pair from the previous iteration
  double* ap = L.a1;
  bool pending = false;

  H.set_identity();
  for (int d = tid; d < D; d += NT) {
    if (starts)
      L.x[d] = starts[s * D + d];
    else if (P.x0)
      L.x[d] = P.x0[sl * D + d];
    else
      L.x[d] = start_uniform_in(P, uint64_t(sl), d);
  }
  __syncthreads();
  double bestVal = 0.0, fval = 333777.0, gnorm = 69.0;
  int grads = 0, ls_evals = 0;
  int status = kStatusUnset;
  bool done = false;
  const bool stoppable = may_stop(P);
  // One evaluation site for the starting point and every trial (kOneSite: the
  // first pass of the loop evaluates the starting point) keeps one copy of a
  // large objective's code and constants in the kernel.
  constexpr bool kOneSite = group_one_site<Eval>();
  int iter = kOneSite ? -1 : 0;
  if constexpr (!kOneSite) {
    bestVal = ev.value(f, L.x, blk);
    ev.gradient(f, L.x, L.g, true, blk);
    ++grads;
    __syncthreads();
    for (int i = tid; i < D; i += NT)
      L.p[i] = -L.g[i];
  }

  for (; iter < P.max_iter; ++iter) {
    const bool first = kOneSite && iter < 0;
    int64_t to = -1;
    double ddir = 0.0;
    if (!first) {
      // trajectory step (bfgs_parallel.cuh:155-166); uniform per workgroup
      to = traj_slot(P.traj, sl, iter);
      if (to >= 0) {
        double gg = 0.0;
        for (int i = tid; i < D; i += NT)
          gg = ::fma(L.g[i], L.g[i], gg);
        const double nrm = ::sqrt(blk.sum1(gg));
        for (int d = tid; d < D; d += NT)
          P.traj.coords[(int64_t(iter) * D + d) * P.traj.starts + sl] = L.x[d];
        if (tid == 0) {
          P.traj.fval[to] = bestVal;
          P.traj.grad[to] = nrm;
          P.traj.status[to] = int8_t(kStatusUnset);
        }
      }
      bool stop = false; // uniform per workgroup
      if (stoppable) {
        if (tid == 0)
          L.flag = load_flag(&ctl->stop_flag);
        __syncthreads();
        stop = L.flag != 0;
      }
      if (stop) {
        status = kStatusStopped;
        fval = bestVal;
        double gg = 0.0;
        for (int i = tid; i < D; i += NT)
          gg = ::fma(L.g[i], L.g[i], gg);
        gnorm = ::sqrt(blk.sum1(gg));
        done = true;
        break;
      }
      double dd = 0.0;
      for (int i = tid; i < D; i += NT)
        dd = ::fma(L.g[i], L.p[i], dd);
      ddir = blk.sum1(dd);
    }

    // trials t < 20 at alpha = 2^-t; the point at 2^-20 is taken as it is
    double alpha = 1.0, fnew = 0.0;
    auto accepts = [&](int t, double a, double v) {
      return t == kLineSearchTrials ||
             (v <= ::fma(kArmijoC1 * a, ddir, bestVal) && v < bestVal);
    };
    if constexpr (group_batches_trials<Eval>() == 2) {
      // every trial at once, the first accepted one counts
      const int t = tid < kLineSearchTrials ? tid : kLineSearchTrials;
      const double a = ::ldexp(1.0, -t);
      const double v = ev.lane_trial(a, L.x, L.p);
      const int pick = __builtin_ctzll(__ballot(accepts(t, a, v)));
      alpha = ::ldexp(1.0, -pick);
      fnew = readlane_f64(v, pick);
      ls_evals += pick + 1;
    } else if constexpr (group_batches_trials<Eval>() == 1) {
      ev.trials_begin(L.x, L.p);
      if constexpr (Eval::kPack > 1) {
        // kPack trials at a time, side by side in the wavefront: one batch,
        // then two of them interleaved
        constexpr int kP = Eval::kPack;
        const int q = tid / Eval::kLane;
        double a0 = 1.0 / double(1 << q); // the lane's trial of the batch
        int t0 = q;
        bool found = false;
        auto batch = [&](auto n) {
          constexpr int S = n();
          double v[S];
          ev.template pack_trials<S>(a0, v);
#pragma unroll
          for (int t = 0; t < S; ++t)
            if (!found) {
              const double a = a0 * (1.0 / double(1 << (t * kP)));
              const uint64_t m = __ballot(accepts(t0 + t * kP, a, v[t]));
              found = m != 0;
              if (found) {
                const int l = __builtin_ctzll(m);
                alpha = readlane_f64(a, l);
                fnew = readlane_f64(v[t], l);
                ls_evals += l / Eval::kLane + 1;
              } else {
                ls_evals += kP;
              }
            }
          a0 *= 1.0 / double(1 << (S * kP));
          t0 += S * kP;
        };
        batch(std::integral_constant<int, 1>{});
#pragma unroll 1
        while (!found)
          batch(std::integral_constant<int, 2>{});
      } else {
        // the full step alone, then four trials at a time (1-4, ... 17-20)
        double v1[1];
        ev.template trials<1>(1.0, v1, blk);
        fnew = v1[0];
        ++ls_evals;
        bool found = accepts(0, 1.0, fnew);
#pragma unroll 1
        for (int t0 = 1; !found; t0 += Eval::kTrials) {
          double v[Eval::kTrials];
          const double a0 = alpha * 0.5;
          ev.template trials<Eval::kTrials>(a0, v, blk);
#pragma unroll
          for (int t = 0; t < Eval::kTrials; ++t)
            if (!found) {
              alpha = a0 * (1.0 / double(1 << t));
              fnew = v[t];
              ++ls_evals;
              found = accepts(t0 + t, alpha, fnew);
            }
        }
      }
    }
    if constexpr (group_batches_trials<Eval>() != 0) {
      for (int j = tid; j < D; j += NT)
        L.xt[j] = ::fma(alpha, L.p[j], L.x[j]);
      __syncthreads();
    } else if constexpr (kOneSite) {
      for (int t = 0;; ++t) {
        for (int j = tid; j < D; j += NT)
          L.xt[j] = first ? L.x[j] : ::fma(alpha, L.p[j], L.x[j]);
        __syncthreads();
        fnew = ev.value(f, L.xt, blk);
        if (first)
          break;
        ++ls_evals;
        if (accepts(t, alpha, fnew))
          break;
        alpha *= 0.5;
      }
    } else {
      bool accepted = false;
      for (int t = 0; t < kLineSearchTrials; ++t) {
        for (int j = tid; j < D; j += NT)
          L.xt[j] = ::fma(alpha, L.p[j], L.x[j]);
        __syncthreads();
        fnew = ev.value(f, L.xt, blk);
        ++ls_evals;
        if (accepts(t, alpha, fnew)) {
          accepted = true;
          break;
        }
        alpha *= 0.5;
      }
      if (!accepted) {
        for (int j = tid; j < D; j += NT)
          L.xt[j] = ::fma(alpha, L.p[j], L.x[j]);
        __syncthreads();
        fnew = ev.value(f, L.xt, blk);
        ++ls_evals;
      }
    }
    if (tid == 0 && to >= 0 && P.traj.alpha) // bfgs_parallel.cuh:182-184
      P.traj.alpha[to] = alpha;
    ev.gradient(f, L.xt, L.gn, true, blk);
    ++grads;
    __syncthreads();
    if (first) {
      bestVal = fnew;
      for (int i = tid; i < D; i += NT) {
        L.g[i] = L.gn[i];
        L.p[i] = -L.gn[i];
      }
      continue;
    }

    // v = H' g_new: from the pairs, or while applying the pending update (one
    // pass over H)
    if constexpr (kPairs) {
      H.apply(L.gn, L.part);
    } else {
      H.pass(L.gn, sp, ap, pending, L.part);
      __syncthreads();
    }
    double st[2] = {0.0, 0.0};
    for (int i = tid; i < D; i += NT) {
      double v;
      if constexpr (kPairs)
        v = H.total(L.part, L.gn, i);
      else
        v = chunk_total<D, NT>(L.part, i);
      L.v[i] = v;
      const double si = L.xt[i] - L.x[i];
      const double yi = L.gn[i] - L.g[i];
      sc[i] = si;
      st[0] = ::fma(si, yi, st[0]);
      st[1] = ::fma(yi, v + L.p[i], st[1]); // u = H y = v + p
    }
    blk.template sum<2>(st);
    const double sTy = st[0];
    const bool upd = !(::fabs(sTy) < kCurvatureSkip);
    const bool acc = fnew < bestVal;
    if (upd) {
      const double rho = 1.0 / sTy;
      const double beta = ::fma(rho * rho, st[1], rho);
      const double hb = 0.5 * beta;
      double q[2] = {0.0, 0.0};
      for (int i = tid; i < D; i += NT) {
        const double u = L.v[i] + L.p[i];
        const double ai = ::fma(hb, sc[i], -(rho * u));
        ac[i] = ai;
        const double ga = acc ? L.gn[i] : L.g[i];
        q[0] = ::fma(ai, ga, q[0]);
        q[1] = ::fma(sc[i], ga, q[1]);
      }
      blk.template sum<2>(q);
      for (int i = tid; i < D; i += NT) {
        const double hg = acc ? L.v[i] : -L.p[i];
        L.p[i] = -::fma(ac[i], q[1], ::fma(sc[i], q[0], hg));
      }
      if constexpr (kPairs)
        H.append(sc, ac);
    } else {
      for (int i = tid; i < D; i += NT)
        L.p[i] = acc ? -L.v[i] : L.p[i];
    }
    if (acc) {
      bestVal = fnew;
      for (int i = tid; i < D; i += NT) {
        L.x[i] = L.xt[i];
        L.g[i] = L.gn[i];
      }
    }
    double gg = 0.0;
    for (int i = tid; i < D; i += NT)
      gg = ::fma(L.g[i], L.g[i], gg);
    const double nrm = ::sqrt(blk.sum1(gg));
    if constexpr (!kPairs) { // the new pair becomes pending for the next pass
      pending = upd;
      double* t0 = sp;
      double* t1 = ap;
      sp = sc;
      ap = ac;
      sc = t0;
      ac = t1;
    }

    if (!::isfinite(nrm) || !::isfinite(fnew)) {
      status = kStatusNonFinite;
      fval = fnew;
      gnorm = nrm;
      done = true;
      break;
    }
    if (nrm < P.tol) {
      if (tid == 0)
        count_converged(ctl, P.required);
      status = kStatusConverged;
      fval = bestVal;
      gnorm = nrm;
      done = true;
      break;
    }
  }
  if (!done) {
    status = kStatusSurrendered;
    fval = bestVal;
    double gg = 0.0;
    for (int i = tid; i < D; i += NT)
      gg = ::fma(L.g[i], L.g[i], gg);
    gnorm = ::sqrt(blk.sum1(gg));
  }
  double e2 = 0.0;
  if (status == kStatusConverged) {
    double t = 0.0;
    for (int d = tid; d < D; d += NT) {
      const double df = L.x[d] - known_min(P.min_kind, d);
      t = ::fma(df, df, t);
    }
    e2 = blk.sum1(t);
  }
  if (tid == 0) {
    traj_final_status(P.traj, sl, status, iter, P.max_iter);
    out.status[s] = status;
    out.iter[s] = iter;
    out.fval[s] = fval;
    out.gnorm[s] = gnorm;
    out.ls_evals[s] = ls_evals;
    out.grads[s] = grads;
    out.near[s] = status == kStatusConverged && ::sqrt(e2) < 0.5;
  }
  for (int d = tid; d < D; d += NT)
    out.x[s * D + d] = L.x[d];
  __syncthreads();
}

// Wavefronts per SIMD the kernel is compiled for.  The binned likelihood (one
// wavefront per start, bound by the issue of its power functions and by their
// chains): 64 fits of 256 starts took 1.66 ms at four, 1.80 at three and 1.85
// at two.  The MLP with the adjoint gradient keeps 256 registers per lane (one
// workgroup of eight wavefronts per CU): 512 starts x 24 iterations took 1.95
// ms so, 2.34 ms at three wavefronts per SIMD and 2.45 ms at four, which spill.
template <class F, Gradient G>
constexpr int group_min_waves()
{
  if constexpr (requires { F::id; }) // built-in objectives
    return F::id == obj::kLogLikelihood                   ? 4
           : F::id == obj::kMlp && G == Gradient::Adjoint ? 2
                                                          : 1;
  else
    return 1;
}

template <class F, int D, int NT, Gradient G, bool HREG, class Prov>
__global__ __launch_bounds__(NT, (group_min_waves<F, G>())) void
bfgs_group_kernel(ClassArgs a, Prov prov)
{
  __shared__ GroupVectors<D, NT, kPairForm<D, NT, HREG>> L;
  Block<NT> blk{L.red};
  using Eval = typename GroupEvalSelect<F, NT, G>::type;
  static_assert(int(F::arity) == D, "objective arity and kernel dimension differ");
  Eval ev;
  ev.sc = GroupScratch{L.part, L.stash, L.scalar};
  GroupH<D, NT, HREG> H;
  if constexpr (!HREG)
    H.slab = a.h_slab + int64_t(blockIdx.x) * a.h_slab_stride;
  int bound = -1;
  for (int64_t s = blockIdx.x; s < a.total_starts; s += gridDim.x) {
    const int pi = find_problem(a.probs, a.n_probs, s);
    const ProblemDesc P = a.probs[pi];
    decltype(auto) f = prov.template get<F>(P);
    if (pi != bound) {
      ev.bind(f, P);
      bound = pi;
    }
    group_bfgs<F, D, NT, G, HREG>(f, L, H, ev, blk, P, a.ctl + pi, s, a.starts, a.out);
  }
}

} // namespace zeus::dev
