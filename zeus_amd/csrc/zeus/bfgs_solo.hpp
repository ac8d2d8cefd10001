// bfgs_solo.hpp -- Gaussian BFGS with a workgroup per start and the matrix in
// registers: the per-workgroup form of large Gaussians with the adjoint
// gradient.
//
// f = 0.5 x^T Cs x needs one product Cs x per point, which is the gradient
// there.  A thread keeps a block of Cs (rows rg + kRg r, columns lc + kLc j)
// for all starts of a problem, and its columns of x and p, so a line-search
// trial is: the trial's columns, the block's products, a sum over the kLc lanes
// of a row (DPP), and one barrier over which the wavefronts' partial values and
// the gradient's rows go through LDS.  Every wavefront sums the partial values
// in the same order and decides alike.
//
// The inverse Hessian is the tile form's, H = B + W M W^T (bfgs_tile.hpp):
// directions and a tridiagonal matrix, here with W in LDS and the vectors spread
// over the wavefronts; wavefront 0 then makes the update.  A full list is folded
// into an explicit B in global memory.  Sums run in a fixed order, another one
// than the serial oracle's: parity is to tolerance.
//
// What bounds it: the chain of one start.  A tile of 16 starts shares its rounds
// between starts at different points of their iterations; with fewer starts than
// CUs the chip has a CU for every start instead.
#pragma once

#include "batch.hpp"
#include "bfgs_tile.hpp"
#include "block.hpp"
#include "cs_product.hpp"
#include "philox.hpp"
#include "prng.hpp"

namespace zeus::dev {

template <int D, int NT>
struct SoloShape {
  static constexpr int NW = NT / kWave;
  static constexpr int kLc = 16; // lanes of a row of Cs
  static constexpr int kRg = NT / kLc;
  static constexpr int RB = (D + kRg - 1) / kRg, CB = (D + kLc - 1) / kLc;
  static constexpr int EL = (D + kWave - 1) / kWave; // rows per lane of a vector
  static constexpr int kHist = 64;                   // vectors before folding into B
  static_assert(RB <= kLc, "one lane per row of the block stores its sum");
  static_assert(EL <= NW && kHist <= kWave, "H g: a wavefront per 64 rows, a lane per vector");
  static constexpr int kParts = (NW + EL - 1) / EL; // of H g's vectors
  static constexpr int64_t kSlabDoubles = int64_t(D) * D;
};

template <int D, int NT>
struct SoloLds {
  using S = SoloShape<D, NT>;
  double w[S::kHist][D];
  double y[2][D];        // Cs x at the last two points
  double fp[2][S::NW];   // x . Cs x, per wavefront
  double vp[S::kParts][D]; // H g, per part of the vectors
  double x[D], g[D], p[D];
  double d[S::kHist];    // w_j . g
  double2 ml[S::kHist];  // M's diagonal and the link to the next vector
  double ddir;
  int k, base, status, stop;
};

template <int D, int NT>
ZEUS_D void
solo_start(SoloLds<D, NT>& L, const double (&c)[SoloShape<D, NT>::RB][SoloShape<D, NT>::CB],
           double* B, const ProblemDesc& P, Control* ctl, const int64_t s, const ClassArgs& a)
{
  using S = SoloShape<D, NT>;
  constexpr int NW = S::NW, RB = S::RB, CB = S::CB, EL = S::EL, kLc = S::kLc, kRg = S::kRg;
  int tid = threadIdx.x; // opaque: what follows from it is not held across starts
  asm volatile("" : "+v"(tid));
  const int lane = tid % kWave;
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lc = tid % kLc, rg = tid / kLc;
  const int64_t sl = s - P.start0;
  const StartOut& out = a.out;
  const bool stoppable = may_stop(P);
  // a vector's elements lane + 64 e
  auto in = [&](int e) { return (e + 1) * kWave <= D || lane + e * kWave < D; };
  auto load = [&](const double* v, double (&r)[EL]) {
#pragma unroll
    for (int e = 0; e < EL; ++e)
      r[e] = in(e) ? v[lane + e * kWave] : 0.0;
  };
  auto store = [&](double* v, const double (&r)[EL]) {
#pragma unroll
    for (int e = 0; e < EL; ++e)
      if (in(e))
        v[lane + e * kWave] = r[e];
  };

  for (int d = tid; d < D; d += NT)
    L.x[d] = a.starts ? a.starts[s * D + d]
             : P.x0   ? P.x0[sl * D + d]
                      : start_uniform_in(P, uint64_t(sl), d);
  __syncthreads();
  // x and p: the block's columns, and the lane's own row (of its row block's)
  double xc[CB], pc[CB], xm, pm;
  const int own = lc < RB ? rg + kRg * lc : D;
  auto reload = [&](const double* v, double (&vc)[CB], double& vm) {
#pragma unroll
    for (int j = 0; j < CB; ++j)
      vc[j] = kLc * (j + 1) <= D || lc + kLc * j < D ? v[lc + kLc * j] : 0.0;
    vm = own < D ? v[own] : 0.0;
  };
  reload(L.x, xc, xm);
#pragma unroll
  for (int j = 0; j < CB; ++j)
    pc[j] = 0.0;
  pm = 0.0;

  int par = 1; // of the last point evaluated: its gradient is L.y[par]
  // f at x + alpha p
  auto eval = [&](double alpha) {
    par ^= 1;
    double y[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r)
      y[r] = 0.0;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const double xt = ::fma(alpha, pc[j], xc[j]);
#pragma unroll
      for (int r = 0; r < RB; ++r)
        y[r] = ::fma(c[r][j], xt, y[r]);
    }
#pragma unroll
    for (int r = 0; r < RB; ++r)
      y[r] = row_sum(y[r]);
    double mine = y[0];
#pragma unroll
    for (int r = 1; r < RB; ++r)
      mine = lc == r ? y[r] : mine;
    if (own < D)
      L.y[par][own] = mine;
    const double f = wave_sum(::fma(alpha, pm, xm) * mine); // own = D: times 0
    if (lane == 0)
      L.fp[par][w] = f;
    __syncthreads();
    double t = L.fp[par][0];
#pragma unroll
    for (int i = 1; i < NW; ++i)
      t += L.fp[par][i];
    return 0.5 * t;
  };

  double best = eval(0.0);
  int ls_evals = 0, grads = 1, iter = 0;
  if (w == 0) {
    double t = 0.0, g[EL], p[EL];
    load(L.y[par], g);
#pragma unroll
    for (int e = 0; e < EL; ++e) {
      p[e] = -g[e];
      t = ::fma(g[e], p[e], t);
    }
    t = wave_sum(t);
    store(L.g, g);
    store(L.p, p);
    store(L.w[0], p);
    if (lane == 0) {
      L.ml[0] = double2{0.0, 0.0};
      L.ddir = t;
      L.k = 1;
      L.base = 0;
      L.status = kStatusUnset;
      L.stop = stoppable ? load_flag(&ctl->stop_flag) : 0;
    }
  }
  __syncthreads();
  reload(L.p, pc, pm);

  int status = kStatusUnset;
  double fval = 0.0;
  double gg = 0.0; // |g|^2 after the iteration (wavefront 0)
  if (w == 0) {
    double t = 0.0, g[EL];
    load(L.g, g);
#pragma unroll
    for (int e = 0; e < EL; ++e)
      t = ::fma(g[e], g[e], t);
    gg = wave_sum(t);
  }
  for (;; ++iter) {
    if (iter >= P.max_iter) {
      status = kStatusSurrendered;
      fval = best;
      break;
    }
    const int64_t to = traj_slot(P.traj, sl, iter);
    if (to >= 0 && w == 0) {
#pragma unroll
      for (int e = 0; e < EL; ++e)
        if (in(e))
          P.traj.coords[(int64_t(iter) * D + lane + e * kWave) * P.traj.starts + sl] = L.x[lane + e * kWave];
      if (lane == 0) {
        P.traj.fval[to] = best;
        P.traj.grad[to] = ::sqrt(gg);
        P.traj.status[to] = int8_t(kStatusUnset);
      }
    }
    if (L.stop != 0) {
      status = kStatusStopped;
      fval = best;
      break;
    }
    const double ddir = L.ddir;
    // trials t < 20 at alpha = 2^-t; the point at 2^-20 is taken as it is
    double alpha = 1.0, fnew;
#pragma unroll 1
    for (int t = 0;; ++t) {
      fnew = eval(alpha);
      ++ls_evals;
      if (t == kLineSearchTrials ||
          (fnew <= ::fma(kArmijoC1 * alpha, ddir, best) && fnew < best))
        break;
      alpha *= 0.5;
    }
    ++grads;
    const bool acc = fnew < best;
    if (tid == 0 && to >= 0 && P.traj.alpha)
      P.traj.alpha[to] = alpha;

    int k = __builtin_amdgcn_readfirstlane(L.k);
    if (k + 2 > S::kHist) { // fold the list into B, restart at the last direction
      const bool base = L.base != 0;
#pragma unroll 1
      for (int e = tid; e < D * D; e += NT) {
        const int row = e % D, col = e / D;
        double b = base ? B[e] : row == col ? 1.0 : 0.0;
        double wp = 0.0, lp = 0.0, wc = L.w[0][col];
#pragma unroll 1
        for (int j = 0; j < k; ++j) {
          const double2 m = L.ml[j];
          const double wn = j + 1 < k ? L.w[j + 1][col] : 0.0;
          b = ::fma(L.w[j][row], ::fma(m.y, wn, ::fma(m.x, wc, lp * wp)), b);
          wp = wc;
          wc = wn;
          lp = m.y;
        }
        B[e] = b;
      }
      __syncthreads();
      for (int d = tid; d < D; d += NT)
        L.w[0][d] = L.w[k - 1][d];
      if (tid == 0) {
        L.ml[0] = double2{0.0, 0.0};
        L.k = 1;
        L.base = 1;
      }
      __syncthreads(); // (also the fold's writes of B before the reads below)
      k = 1;
    }
    // w_j . g, a row of kLc lanes per vector
    {
      double gc[CB];
#pragma unroll
      for (int j = 0; j < CB; ++j)
        gc[j] = kLc * (j + 1) <= D || lc + kLc * j < D ? L.y[par][lc + kLc * j] : 0.0;
#pragma unroll 1
      for (int j = rg; j < k; j += kRg) {
        double t = 0.0;
#pragma unroll
        for (int c = 0; c < CB; ++c)
          if (kLc * (c + 1) <= D || lc + kLc * c < D)
            t = ::fma(L.w[j][lc + kLc * c], gc[c], t);
        t = row_sum(t);
        if (lc == 0)
          L.d[j] = t;
      }
    }
    __syncthreads();
    // v = H g: wavefront w takes 64 rows and one of the parts of the vectors; lane
    // j has vector j's coefficient
    {
      double cj = 0.0;
      if (lane < k) {
        cj = L.ml[lane].x * L.d[lane];
        if (lane > 0)
          cj = ::fma(L.ml[lane - 1].y, L.d[lane - 1], cj);
        if (lane + 1 < k)
          cj = ::fma(L.ml[lane].y, L.d[lane + 1], cj);
      }
      const int e = w % EL, q = w / EL, nq = (NW - e + EL - 1) / EL;
      const int row = lane + e * kWave < D ? lane + e * kWave : 0;
      double t = 0.0;
      if (L.base)
#pragma unroll 4
        for (int col = q; col < D; col += nq)
          t = ::fma(B[col * D + row], L.y[par][col], t);
#pragma unroll 4
      for (int j = q; j < k; j += nq)
        t = ::fma(L.w[j][row], readlane_f64(cj, j), t);
      if (lane + e * kWave < D)
        L.vp[q][row] = t;
    }
    __syncthreads();

    if (w == 0) { // the update (the tile form's, bfgs_tile.hpp)
      const bool base = L.base != 0;
      double gn[EL], v[EL], g[EL], p[EL];
      load(L.y[par], gn);
      load(L.g, g);
      load(L.p, p);
#pragma unroll
      for (int e = 0; e < EL; ++e) {
        double t = base ? 0.0 : gn[e];
        if (in(e))
#pragma unroll
          for (int q = 0; q < (NW - e + EL - 1) / EL; ++q)
            t += L.vp[q][lane + e * kWave];
        v[e] = t;
      }
      double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0, t4 = 0.0;
#pragma unroll
      for (int e = 0; e < EL; ++e) {
        const double se = alpha * p[e], ye = gn[e] - g[e], u = v[e] + p[e];
        const double ga = acc ? gn[e] : g[e];
        t0 = ::fma(se, ye, t0);
        t1 = ::fma(ye, u, t1);
        t2 = ::fma(ga, ga, t2);
        t3 = ::fma(se, ga, t3);
        t4 = ::fma(u, ga, t4);
      }
      const double sTy = wave_sum(t0), yu = wave_sum(t1), sg = wave_sum(t3), ug = wave_sum(t4);
      gg = wave_sum(t2);
      const bool upd = !(::fabs(sTy) < kCurvatureSkip);
      int kn = k; // place of the new direction
      if (upd || acc) {
        if (!upd && (k == 1 || L.ml[k - 2].y == 0.0))
          kn = k - 1;
        double2 mk = {0.0, 0.0};
        if (upd) {
          const double rho = 1.0 / sTy;
          const double hb = 0.5 * ::fma(rho * rho, yu, rho);
          const double q0 = ::fma(hb, sg, -(rho * ug));
          const double sd = alpha * ddir; // s.g
          double ae[EL];
#pragma unroll
          for (int e = 0; e < EL; ++e) {
            const double se = alpha * p[e];
            ae[e] = ::fma(hb, se, -(rho * (v[e] + p[e])));
            v[e] = -::fma(ae[e], sg, ::fma(se, q0, acc ? v[e] : -p[e]));
          }
          if (acc && ::fabs(rho * sd) >= kSpanMin) {
            const double r = -1.0 / sd;
            const double A = r * ::fma(0.5, ::fma(rho, yu, 1.0), q0);
            mk = double2{2.0 * alpha * ::fma(A, alpha, -r), alpha * r};
          } else {
            store(L.w[kn], ae);
            L.ml[kn++] = double2{0.0, 0.0};
            mk.y = alpha;
          }
        } else {
#pragma unroll
          for (int e = 0; e < EL; ++e)
            v[e] = -v[e];
        }
        L.ml[k - 1] = mk;
        L.ml[kn] = double2{0.0, 0.0};
        store(L.w[kn], v);
        kn = kn + 1;
      } else {
#pragma unroll
        for (int e = 0; e < EL; ++e)
          v[e] = p[e];
      }
      double dd = 0.0;
#pragma unroll
      for (int e = 0; e < EL; ++e) {
        if (in(e)) {
          const int i = lane + e * kWave;
          if (acc) {
            L.x[i] = ::fma(alpha, p[e], L.x[i]);
            L.g[i] = gn[e];
          }
          L.p[i] = v[e];
        }
        dd = ::fma(acc ? gn[e] : g[e], v[e], dd);
      }
      dd = wave_sum(dd);
      const double nrm = ::sqrt(gg);
      if (lane == 0) {
        L.k = kn;
        L.ddir = dd;
        if (!::isfinite(nrm) || !::isfinite(fnew)) {
          L.status = kStatusNonFinite;
        } else if (nrm < P.tol) {
          count_converged(ctl, P.required);
          L.status = kStatusConverged;
        }
        if (stoppable)
          L.stop = load_flag(&ctl->stop_flag);
      }
    }
    __syncthreads();
    status = L.status;
    if (acc) {
      best = fnew;
#pragma unroll
      for (int j = 0; j < CB; ++j)
        xc[j] = ::fma(alpha, pc[j], xc[j]);
      xm = ::fma(alpha, pm, xm);
    }
    if (status != kStatusUnset) {
      fval = status == kStatusNonFinite ? fnew : best;
      break;
    }
    reload(L.p, pc, pm);
  }

  if (w == 0) {
    double e2 = 0.0;
    if (status == kStatusConverged) {
      double t = 0.0;
#pragma unroll
      for (int e = 0; e < EL; ++e) {
        const double df = in(e) ? L.x[lane + e * kWave] - known_min(P.min_kind, lane + e * kWave) : 0.0;
        t = ::fma(df, df, t);
      }
      e2 = wave_sum(t);
    }
    if (lane == 0) {
      traj_final_status(P.traj, sl, status, iter, P.max_iter);
      out.status[s] = status;
      out.iter[s] = iter;
      out.fval[s] = fval;
      out.gnorm[s] = ::sqrt(gg);
      out.ls_evals[s] = ls_evals;
      out.grads[s] = grads;
      out.near[s] = status == kStatusConverged && ::sqrt(e2) < 0.5;
    }
#pragma unroll
    for (int e = 0; e < EL; ++e)
      if (in(e))
        out.x[s * D + lane + e * kWave] = L.x[lane + e * kWave];
  }
  __syncthreads(); // LDS reuse by the next start
}

template <class F, int D, int NT, class Prov>
__global__ __launch_bounds__(NT) void
bfgs_solo_kernel(ClassArgs a, Prov)
{
  using S = SoloShape<D, NT>;
  __shared__ SoloLds<D, NT> L;
  double* B = a.h_slab + int64_t(blockIdx.x) * a.h_slab_stride;
  double c[S::RB][S::CB];
  int loaded = -1; // problem whose matrix c holds
  for (int64_t s = blockIdx.x; s < a.total_starts; s += gridDim.x) {
    const int pi = wave_uniform(find_problem(a.probs, a.n_probs, s));
    const ProblemDesc& P = a.probs[pi];
    if (pi != loaded) {
      const gdouble_ptr Cs = as_global(P.aux);
      // an opaque index: the addresses are formed here, not held (or spilled)
      // across the starts
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const int lc = tid % S::kLc, rg = tid / S::kLc;
#pragma unroll
      for (int r = 0; r < S::RB; ++r)
#pragma unroll
        for (int j = 0; j < S::CB; ++j) {
          const int row = rg + S::kRg * r, col = lc + S::kLc * j;
          c[r][j] = row < D && col < D ? Cs[row * D + col] : 0.0;
        }
      loaded = pi;
    }
    solo_start<D, NT>(L, c, B, P, a.ctl + pi, s, a);
  }
}

} // namespace zeus::dev
