// bfgs_tile.hpp -- tile form of the BFGS for the Gaussian objective: one
// 1024-thread workgroup advances a tile of 16 starts of one problem in
// lock-step rounds.
//
// Round structure.  Every start of the tile submits one point per round (its
// first point, a line-search trial x + alpha p, or the unconditional point
// after 20 rejected trials).  The 16 points Xt (D x 16, LDS) are evaluated
// together: G = Cs Xt on FP64 MFMA (v_mfma_f64_16x16x4f64), Cs = (C + C^T)/2
// as A operands, f_j = 0.5 Xt_j . G_j, and G_j is the adjoint gradient of
// start j at its point.  The product's MB x KB steps are cut into 16
// balanced segments, one per wavefront (cs_product.hpp, CsFullSeg), whose
// Cs fragments stay in registers for the whole tile (Cs does not change);
// each segment leaves partial blocks of G in LDS, and row d of G is the sum
// of the blocks of its row block in segment order.  Wavefront w then runs
// start w's BFGS logic for the round -- line-search decision, update,
// convergence test -- with DPP wavefront reductions only, and submits its
// next point.  Two workgroup barriers per round.
//
// Method.  The reference's per-start BFGS (include/bfgs_sequential.cuh:
// 46-221, utils.cuh:245-287, 376-426) with the same line search, update
// skip rule, statuses and counters as the other forms.  The update is
// H' = H + s a^T + a s^T, a = (beta/2) s - rho u, u = H y (the reference's
// update expanded), s = alpha p, and the next direction is p' = -H' g'.  For
// an accepted step (g' is the gradient the update used, H g' = u - p) the two
// give, with q0 = a.g' and the reciprocal r = -1 / (alpha p.g),
//   a = (A alpha - r) p + r p',   A = r ((1 + rho y.u) / 2 + q0):
// a lies in the span of the old and the new direction.  So the inverse Hessian
// is kept as H = B + W M W^T, W the directions taken so far and M tridiagonal
// (diagonal m, links l to the next vector): H g is one dot product and one
// axpy per step, half of the reads, sums and axpys that the (s, a) pairs take.
// A step that was not accepted, or whose 1 - rho s.g' = -rho alpha p.g is
// small (below kSpanMin, where the formula would lose digits), appends a
// itself.  B = I until the list is full, then the list is folded into an
// explicit B (global memory) and restarts at the last direction.  Sums run in
// a fixed order (results are deterministic), but in another order than the
// serial oracle: parity is to tolerance.
#pragma once

#include "batch.hpp"
#include "block.hpp"
#include "cs_product.hpp"
#include "philox.hpp"
#include "prng.hpp"

namespace zeus::dev {

constexpr int kTileStarts = kCsTile; // starts per tile = MFMA N dimension
// Workgroup size of the tile form: 16 wavefronts, one per start of the
// tile (a 128-register budget per lane).
constexpr int kTileThreads = 1024;
constexpr int kTileWaves = kTileThreads / kWave;
static_assert(kTileStarts % kTileWaves == 0, "whole slots per wavefront");

template <int D>
struct TileShape : CsShape<D> {
  static constexpr int EL = (D + kWave - 1) / kWave; // rows per lane in start logic
  static constexpr int kHist = 64; // vectors kept before folding into B
  static constexpr int64_t kSlotDoubles = int64_t(kHist) * D + int64_t(D) * D;
};

struct TileArgs {
  const ProblemDesc* probs;
  const int32_t* tile_problem; // tile -> problem (tiles of a problem are consecutive)
  int64_t n_tiles;
  Control* ctl;
  StartOut out;
  double* slot_mem; // per (workgroup, start slot): kHist vectors, then B (D x D)
};

// Per-start state of a slot (LDS; read and written by its wavefront only).
struct TileSlot {
  int64_t s;   // global start index
  int phase;   // 0 idle, 1 first point, 2 trial, 3 unconditional point
  int trial, iter, grads, ls_evals;
  int k;       // vectors in the list; the last one is the current direction
  int base;    // explicit B in use
  double best, alpha, ddir;
};

// The product's segments: 16, one per wavefront, every fragment of a
// segment held in registers across the rounds of a tile (kTileKeep >= the
// longest segment; 24 fragments = 48 VGPRs per lane at D = 150).
constexpr int kTileKeep = 64;
constexpr int kHgChunk = 3; // vectors read together in H g (2: 3 % slower; 4 spills)
constexpr double kSpanMin = 0x1p-10;
template <int D>
using TileSeg = CsFullSeg<D, kTileWaves, kTileKeep>;

template <int D>
struct TileLds {
  using S = TileShape<D>;
  using Seg = TileSeg<D>;
  double xt[S::KP * S::XS]; // submitted points, [row][slot]
  double gpart[Seg::NP * Seg::kSlot]; // partial blocks of Cs Xt, [part][row % 16][slot]
  double fpart[Seg::NP * kTileStarts];
  double x[kTileStarts * D], g[kTileStarts * D], p[kTileStarts * D];
  // one byte per slot, so that a wavefront reads all 16 flags in one access
  alignas(16) uint8_t live[kTileStarts];
  alignas(16) uint8_t newconv[kTileStarts]; // slot converged in the last round, not yet counted
  // the problem's converged count as read in a round (the reading
  // wavefronts' counters summed), by round parity: one is summed while the
  // other, last read in the round before, is cleared
  int conv_sum[2];
  TileSlot slot[kTileStarts];
  double2 ml[kTileStarts][S::kHist]; // M's diagonal and the link to the next vector
  ProblemDesc prob; // the tile's problem
};

// Row d of G for slot j: the partial blocks of the segments covering d's row
// block (consecutive parts), added in segment order.  Every part is read at
// once (past the block's count the first part again, not added).
template <int D>
ZEUS_D ZEUS_FI double
tile_grad(const TileLds<D>& L, int d, int j)
{
  using Seg = TileSeg<D>;
  using S = TileShape<D>;
  const int mb = (d >> 4) < S::MB - 1 ? (d >> 4) : S::MB - 1;
  const int p0 = int((Seg::kFirstBits >> (6 * mb)) & 63);
  const int n = int((Seg::kCountBits >> (4 * mb)) & 15);
  const double* gp = L.gpart + p0 * Seg::kSlot + (d & 15) * S::XS + j;
  double v[Seg::kCover];
#pragma unroll
  for (int c = 0; c < Seg::kCover; ++c)
    v[c] = gp[(c < n ? c : 0) * Seg::kSlot];
  double g = v[0];
#pragma unroll
  for (int c = 1; c < Seg::kCover; ++c)
    if (c < n)
      g += v[c];
  return g;
}

template <int EL>
ZEUS_D ZEUS_FI double
tile_dot(const double (&a)[EL], const double (&b)[EL])
{
  double t = 0.0;
#pragma unroll
  for (int e = 0; e < EL; ++e)
    t = ::fma(a[e], b[e], t);
  return wave_sum(t);
}

// Submits slot w's next point x + alpha p into the product's operand Xt.
// Every row is read before the first store (the compiler cannot tell the LDS
// rows apart); full rows need no mask (lane < 64).
template <int D>
ZEUS_D ZEUS_FI void
tile_submit(TileLds<D>& L, const int w, int lane, const double alpha)
{
  using S = TileShape<D>;
  constexpr int EL = S::EL;
  // opaque lane: the row addresses are recomputed here, not held (or
  // spilled) across the round loop
  asm volatile("" : "+v"(lane));
  const double* X = L.x + w * D;
  const double* Pd = L.p + w * D;
  double x[EL], p[EL];
#pragma unroll
  for (int e = 0; e < EL; ++e)
    if ((e + 1) * kWave <= D || lane + e * kWave < D) {
      x[e] = X[lane + e * kWave];
      p[e] = Pd[lane + e * kWave];
    }
#pragma unroll
  for (int e = 0; e < EL; ++e)
    if ((e + 1) * kWave <= D || lane + e * kWave < D)
      L.xt[(lane + e * kWave) * S::XS + w] = ::fma(alpha, p[e], x[e]);
}

// Armijo acceptance of a line-search trial with value f at step alpha
// (reference utils.cuh:376-426).
ZEUS_D ZEUS_FI bool
tile_accepts(double f, double alpha, double ddir, double best)
{
  return f <= ::fma(kArmijoC1 * alpha, ddir, best) && f < best;
}

// Logic of start slot w for one round, run by one wavefront; `f` is the
// value at the slot's submitted point, `stop` the problem's early stop as
// seen this round.
template <int D>
ZEUS_D void
tile_slot_step(TileLds<D>& L, TileSlot& st, const int w, const ProblemDesc& P,
               const StartOut& out, double* mem, double f, const bool stop)
{
  using S = TileShape<D>;
  constexpr int EL = S::EL;
  // the lane index is made opaque here, so that the per-lane addresses below
  // are recomputed each round instead of being held (or spilled) across the
  // whole round loop
  int lane = threadIdx.x % kWave;
  asm volatile("" : "+v"(lane));
  double* X = L.x + w * D;
  double* G = L.g + w * D;
  double* Pd = L.p + w * D;
  double* hist = mem;
  double* B = mem + int64_t(S::kHist) * D;
  double2* ml = L.ml[w];
  int row[EL];
  bool ok[EL];
#pragma unroll
  for (int e = 0; e < EL; ++e) {
    row[e] = lane + e * kWave;
    ok[e] = row[e] < D;
  }
  // rows every lane has (d < 64 (e + 1) <= D) need no mask; the lane index
  // is opaque to the compiler, so it cannot tell by itself
  auto okr = [&](int e) { return (e + 1) * kWave <= D || ok[e]; };
  auto load = [&](const double* v, double (&r)[EL]) {
#pragma unroll
    for (int e = 0; e < EL; ++e)
      r[e] = okr(e) ? v[row[e]] : 0.0;
  };
  auto load_grad = [&](double (&r)[EL]) { // G column from its partial blocks
#pragma unroll
    for (int e = 0; e < EL; ++e)
      r[e] = okr(e) ? tile_grad<D>(L, row[e], w) : 0.0;
  };
  auto submit = [&](int phase) {
    tile_submit<D>(L, w, lane, st.alpha);
    st.phase = phase;
  };
  auto finish = [&](int status, double fval, double gnorm) {
    double e2 = 0.0;
    if (status == kStatusConverged) {
      double x[EL], d[EL];
      load(X, x);
#pragma unroll
      for (int e = 0; e < EL; ++e)
        d[e] = ok[e] ? x[e] - known_min(P.min_kind, row[e]) : 0.0;
      e2 = tile_dot<EL>(d, d);
    }
    if (lane == 0) {
      out.status[st.s] = status;
      out.iter[st.s] = st.iter;
      out.fval[st.s] = fval;
      out.gnorm[st.s] = gnorm;
      out.ls_evals[st.s] = st.ls_evals;
      out.grads[st.s] = st.grads;
      out.near[st.s] = status == kStatusConverged && ::sqrt(e2) < 0.5;
    }
#pragma unroll
    for (int e = 0; e < EL; ++e)
      if (ok[e])
        out.x[st.s * D + row[e]] = X[row[e]];
    st.phase = 0;
  };
  auto gnorm_now = [&]() {
    double g[EL];
    load(G, g);
    return ::sqrt(tile_dot<EL>(g, g));
  };
  // top of a BFGS iteration: MAX_ITER, stop flag, first trial
  auto begin_iteration = [&]() {
    if (st.iter >= P.max_iter) {
      finish(kStatusSurrendered, st.best, gnorm_now());
      return;
    }
    if (stop) {
      finish(kStatusStopped, st.best, gnorm_now());
      return;
    }
    double g[EL], p[EL];
    load(G, g);
    load(Pd, p);
    st.ddir = tile_dot<EL>(g, p);
    st.alpha = 1.0;
    st.trial = 0;
    submit(2);
  };

  if (st.phase == 1) { // first point: value and gradient
    double g[EL];
    load_grad(g);
#pragma unroll
    for (int e = 0; e < EL; ++e)
      if (ok[e]) {
        G[row[e]] = g[e];
        Pd[row[e]] = -g[e];
        hist[row[e]] = -g[e];
      }
    ml[0] = double2{0.0, 0.0};
    st.k = 1;
    st.best = f;
    st.grads = 1;
    begin_iteration();
    return;
  }
  if (st.phase == 2) {
    ++st.ls_evals;
    const bool accept = tile_accepts(f, st.alpha, st.ddir, st.best);
    if (!accept) {
      st.alpha *= 0.5;
      if (++st.trial == kLineSearchTrials)
        submit(3);
      else
        submit(2);
      return;
    }
  } else { // phase 3: point after the last rejected trial
    ++st.ls_evals;
  }

  // ---- end of the iteration: gradient at the new point and the update ----
  // (short live ranges: vectors are re-read from LDS where they are needed)
  const double fnew = f;
  ++st.grads;
  const bool acc = fnew < st.best;
  double gn[EL], v[EL];
  load_grad(gn);
  // v = H gn, H = B + W M W^T
  if (st.base) {
#pragma unroll
    for (int e = 0; e < EL; ++e)
      v[e] = 0.0;
#pragma unroll 1
    for (int c = 0; c < D; ++c) {
      const double gc = tile_grad<D>(L, c, w);
#pragma unroll
      for (int e = 0; e < EL; ++e)
        if (ok[e])
          v[e] = ::fma(B[int64_t(c) * D + row[e]], gc, v[e]);
    }
  } else {
#pragma unroll
    for (int e = 0; e < EL; ++e)
      v[e] = gn[e];
  }
  // vectors in chunks of kHgChunk: every load of a chunk is issued before its
  // dot products (one memory latency per chunk; the vectors of the whole chip
  // are read in the same rounds, mostly beyond the L2) and the chunk's
  // wavefront sums run side by side.  Vector j's coefficient is m_j d_j +
  // l_{j-1} d_{j-1} + l_j d_{j+1}, so v takes vector j once d_{j+1} is there:
  // the last vector of a chunk is carried into the next.
  constexpr int kC = kHgChunk;
  // no LDS access is moved across the loop (the values it would keep live
  // through the loop cost registers the chunk needs)
  asm volatile("" ::: "memory");
  {
    double h[EL], ch = 0.0, dh = 0.0, lh = 0.0; // carried vector: coefficient, dot, link
#pragma unroll
    for (int e = 0; e < EL; ++e)
      h[e] = 0.0;
    const int k = __builtin_amdgcn_readfirstlane(st.k);
#pragma unroll 1
    for (int j0 = 0; j0 < k; j0 += kC) {
      double wj[kC][EL], d[kC];
#pragma unroll
      for (int c = 0; c < kC; ++c) {
        // past the list's end the last vector is loaded again; its terms are
        // not used.  Rows past D read the next vector of the slot (in bounds:
        // the explicit B follows the list) and are zeroed after the load, so
        // the loads are unconditional, addressed by a uniform base and the lane.
        const int j = j0 + c < k ? j0 + c : k - 1;
        const gdouble_ptr pj = as_global(hist) + int64_t(j) * D + lane;
#pragma unroll
        for (int e = 0; e < EL; ++e)
          wj[c][e] = pj[e * kWave];
      }
#pragma unroll
      for (int c = 0; c < kC; ++c) {
        double t = 0.0;
#pragma unroll
        for (int e = 0; e < EL; ++e) {
          wj[c][e] = okr(e) ? wj[c][e] : 0.0;
          t = ::fma(wj[c][e], gn[e], t);
        }
        d[c] = t;
      }
#pragma unroll
      for (int c = 0; c < kC; ++c)
        d[c] = wave_sum(d[c]);
#pragma unroll
      for (int c = 0; c < kC; ++c)
        if (j0 + c < k) {
          const double2 mc = ml[j0 + c];
          const double c0 = ::fma(lh, d[c], ch);
          ch = ::fma(mc.x, d[c], lh * dh);
          dh = d[c];
          lh = mc.y;
#pragma unroll
          for (int e = 0; e < EL; ++e) {
            v[e] = ::fma(h[e], c0, v[e]);
            h[e] = wj[c][e];
          }
        }
    }
#pragma unroll
    for (int e = 0; e < EL; ++e)
      v[e] = ::fma(h[e], ch, v[e]);
  }
  asm volatile("" ::: "memory");
  // s = alpha p, y = gn - g, u = H y = H gn - H g = v + p; g' the gradient
  // after the iteration (gn if accepted, else g)
  double pv[EL], gv[EL];
  load(Pd, pv);
  load(G, gv);
  double sTy, yu, gg, sg, ug;
  {
    double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0, t4 = 0.0;
#pragma unroll
    for (int e = 0; e < EL; ++e) {
      const double se = st.alpha * pv[e], y = gn[e] - gv[e], u = v[e] + pv[e];
      const double ga = acc ? gn[e] : gv[e];
      t0 = ::fma(se, y, t0);
      t1 = ::fma(y, u, t1);
      t2 = ::fma(ga, ga, t2);
      t3 = ::fma(se, ga, t3);
      t4 = ::fma(u, ga, t4);
    }
    sTy = wave_sum(t0);
    yu = wave_sum(t1);
    gg = wave_sum(t2);
    sg = wave_sum(t3);
    ug = wave_sum(t4);
  }
  double dd = 0.0; // g'.p' (the next iteration's directional derivative), in row order
  const bool upd = !(::fabs(sTy) < kCurvatureSkip);
  if (upd || acc) { // a new direction
    if (st.k + 2 > S::kHist) { // fold the list into B first
#pragma unroll 1
      for (int c = 0; c < D; ++c) {
        double bc[EL];
#pragma unroll
        for (int e = 0; e < EL; ++e)
          bc[e] = st.base ? (ok[e] ? B[int64_t(c) * D + row[e]] : 0.0)
                          : (row[e] == c ? 1.0 : 0.0);
        double wp = 0.0, lp = 0.0, wc = hist[c]; // column c of the last and this vector
#pragma unroll 1
        for (int j = 0; j < st.k; ++j) {
          const double* wj = hist + int64_t(j) * D;
          const double2 mc = ml[j];
          const double wn = j + 1 < st.k ? wj[D + c] : 0.0;
          const double cj = ::fma(mc.y, wn, ::fma(mc.x, wc, lp * wp));
#pragma unroll
          for (int e = 0; e < EL; ++e)
            if (ok[e])
              bc[e] = ::fma(wj[row[e]], cj, bc[e]);
          wp = wc;
          wc = wn;
          lp = mc.y;
        }
#pragma unroll
        for (int e = 0; e < EL; ++e)
          if (ok[e])
            B[int64_t(c) * D + row[e]] = bc[e];
      }
#pragma unroll
      for (int e = 0; e < EL; ++e)
        if (okr(e))
          hist[row[e]] = pv[e];
      st.base = 1;
      st.k = 1;
    }
    // the new direction's place; without an update it replaces a direction
    // that no link reaches
    int k = !upd && (st.k == 1 || ml[st.k - 2].y == 0.0) ? st.k - 1 : st.k;
    double2 mk = {0.0, 0.0}; // row st.k - 1 of M
    if (upd) {
      const double al = st.alpha;
      const double rho = 1.0 / sTy;
      const double hb = 0.5 * ::fma(rho * rho, yu, rho);
      const double q0 = ::fma(hb, sg, -(rho * ug));
      const double sd = al * st.ddir; // s.g
      const bool span = acc && ::fabs(rho * sd) >= kSpanMin;
      // p' = -H' g' = -(H g' + s (a.g') + a (s.g')), H g' = v (accepted) or -p
      double a[EL];
#pragma unroll
      for (int e = 0; e < EL; ++e) {
        const double se = al * pv[e];
        a[e] = ::fma(hb, se, -(rho * (v[e] + pv[e])));
        v[e] = -::fma(a[e], sg, ::fma(se, q0, acc ? v[e] : -pv[e]));
      }
      if (span) {
        const double r = -1.0 / sd;
        const double A = r * ::fma(0.5, ::fma(rho, yu, 1.0), q0);
        mk = double2{2.0 * al * ::fma(A, al, -r), al * r};
      } else {
        double* wk = hist + int64_t(k) * D;
#pragma unroll
        for (int e = 0; e < EL; ++e)
          if (okr(e))
            wk[row[e]] = a[e];
        ml[k++] = double2{0.0, 0.0};
        mk.y = al;
      }
    } else {
#pragma unroll
      for (int e = 0; e < EL; ++e)
        v[e] = -v[e];
    }
    ml[st.k - 1] = mk;
    ml[k] = double2{0.0, 0.0};
    double* wk = hist + int64_t(k) * D;
#pragma unroll
    for (int e = 0; e < EL; ++e)
      if (okr(e)) {
        Pd[row[e]] = v[e];
        wk[row[e]] = v[e];
        dd = ::fma(acc ? gn[e] : gv[e], v[e], dd);
      }
    st.k = k + 1;
  } else {
#pragma unroll
    for (int e = 0; e < EL; ++e)
      dd = ::fma(gv[e], pv[e], dd);
  }
  if (acc) {
    st.best = fnew;
#pragma unroll
    for (int e = 0; e < EL; ++e)
      if (okr(e)) {
        X[row[e]] = L.xt[row[e] * S::XS + w];
        G[row[e]] = gn[e];
      }
  }
  const double nrm = ::sqrt(gg);
  const double ddir = wave_sum(dd);
  if (!::isfinite(nrm) || !::isfinite(fnew)) {
    finish(kStatusNonFinite, fnew, nrm);
    return;
  }
  if (nrm < P.tol) {
    if (lane == 0)
      L.newconv[w] = 1; // counted for the tile at the top of the next round
    finish(kStatusConverged, st.best, nrm);
    return;
  }
  // top of the next iteration (begin_iteration with the norm and the
  // directional derivative already at hand)
  ++st.iter;
  if (st.iter >= P.max_iter) {
    finish(kStatusSurrendered, st.best, nrm);
    return;
  }
  if (stop) {
    finish(kStatusStopped, st.best, nrm);
    return;
  }
  st.ddir = ddir;
  st.alpha = 1.0;
  st.trial = 0;
  submit(2);
}

constexpr int kStopReader = kTileThreads - kWave; // thread that adds the tile's count

// Adds the slots flagged in newconv to the workgroup's counter of the
// problem's converged count (one relaxed atomic, none when no slot
// converged) and clears the flags.
template <int D>
ZEUS_D ZEUS_FI void
tile_count_converged(TileLds<D>& L, Control* ctl)
{
  static_assert(kTileStarts == 16, "the flags are one 16-byte word");
  uint4* fl = reinterpret_cast<uint4*>(L.newconv);
  const uint4 v = *fl;
  *fl = uint4{0u, 0u, 0u, 0u};
  // bytes are 0 or 1: the byte sum of the four words' sum is the count
  const unsigned b = v.x + v.y + v.z + v.w;
  const int n = int((b * 0x01010101u) >> 24);
  if (n > 0)
    (void)__hip_atomic_fetch_add(&ctl->conv_lines[(blockIdx.x % kConvLines) * kConvStride], n,
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int D>
__global__ __launch_bounds__(kTileThreads) void
bfgs_tile_kernel(TileArgs a)
{
  using S = TileShape<D>;
  __shared__ TileLds<D> L;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int li0 = lane & 15, lk0 = lane >> 4;
  auto slot_mem = [&](int j) {
    return a.slot_mem + (int64_t(blockIdx.x) * kTileStarts + j) * S::kSlotDoubles;
  };

  using Seg = TileSeg<D>;
  for (int e = tid; e < S::KP * S::XS; e += kTileThreads)
    L.xt[e] = 0.0; // padding rows stay zero
  Seg seg;

  for (int64_t tile = blockIdx.x; tile < a.n_tiles; tile += gridDim.x) {
    const int pi = wave_uniform(a.tile_problem[tile]);
    if (tid == 0)
      L.prob = a.probs[pi];
    __syncthreads();
    const ProblemDesc& P = L.prob;
    const double* Cf = P.aux_frag;
    // slots w, w + kTileWaves, ...: every lane of the wavefront writes the
    // same values.  A problem's tiles are consecutive from
    // ProblemDesc::block0 (its PSO workgroups, which hold the same starts).
    for (int j = w; j < kTileStarts; j += kTileWaves) {
      TileSlot& st = L.slot[j];
      st = TileSlot{-1, 0, 0, 0, 0, 0, 0, 0, 0.0, 1.0, 0.0};
      L.newconv[j] = 0;
      const int64_t sl = (tile - P.block0) * kTileStarts + j; // local start
      if (sl < P.n_starts) {
        st.s = P.start0 + sl;
        double* X = L.x + j * D;
        for (int d = lane; d < D; d += kWave) {
          const double v =
            P.x0 ? P.x0[sl * D + d]
                 : start_uniform_in(P, uint64_t(sl), d);
          X[d] = v;
          L.xt[d * S::XS + j] = v;
        }
        st.phase = 1;
      }
    }
    Control* ctl = a.ctl + pi;
    if constexpr (Seg::kKeep > 0) // this problem's fragments kept across rounds
      seg.load(w, Cf, li0, lk0, 0, Seg::kKeep);
    if (tid < 2)
      L.conv_sum[tid] = 0;
    __syncthreads();

    int par = 0; // this round's conv_sum (the same in every wavefront)
    for (;; par ^= 1) {
      // Early stop (reference bfgs_common.cuh:170-208): the problem stops
      // once `required` starts have converged; a start sees it at the top of
      // its next iteration, as in the other forms.
      // per-lane indices made opaque each round: addresses derived from them
      // are recomputed here rather than held across the round loop
      int li = li0, lk = lk0;
      asm volatile("" : "+v"(li), "+v"(lk));
      // The starts that converged in the last round are added to one of the
      // problem's eight counters here, one atomic per tile and round (one
      // per start, all on one address, had queued up behind each other in
      // the rounds where most starts of the chip converge together).
      // Wavefronts 8-15 each read one counter a third of the way through
      // their product, when the other tiles' sums of the last round have
      // been added (the load's latency hides behind the rest of the
      // product), and add it to this round's LDS sum.
      if (tid == kStopReader) {
        tile_count_converged(L, ctl);
        L.conv_sum[par ^ 1] = 0; // last read in the round before
      }
      constexpr int kReader0 = kTileWaves - kConvLines;
      int conv = 0;
      auto read_count = [&]() {
        if (w >= kReader0)
          conv = __hip_atomic_load(&ctl->conv_lines[(w - kReader0) * kConvStride],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      // ---- G = Cs Xt in balanced segments, partial blocks and values ----
      if constexpr (Seg::kKeep < Seg::LMAX)
        seg.load(w, Cf, li, lk, Seg::kKeep, Seg::LMAX);
      __builtin_amdgcn_sched_barrier(0);
      seg.mma(w, L.xt, L.gpart, L.fpart, li, lk, read_count);
      if (w >= kReader0 && lane == 0)
        (void)__hip_atomic_fetch_add(&L.conv_sum[par], conv, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
      __syncthreads();
      // ---- start logic: wavefront w runs its slots one after the other ----
      for (int j = w; j < kTileStarts; j += kTileWaves) {
        TileSlot& sl = L.slot[j];
        // what a rejected line-search trial needs, read together with the
        // value's partials: most rounds end that way, and then the slot
        // takes the backtracking step here (tile_slot_step's, the same
        // arithmetic) instead of re-reading its state step by step
        const int ph = sl.phase, tr = sl.trial, le = sl.ls_evals;
        const double al = sl.alpha, dd = sl.ddir, bs = sl.best;
        // f = 0.5 sum_p fpart[p]: lane p holds part p's partial, one
        // fixed-order wavefront sum
        static_assert(Seg::NP <= kWave, "one part per lane");
        const double fu = lane < Seg::NP ? L.fpart[lane * kTileStarts + j] : 0.0;
        if (ph != 0) {
          const double f = 0.5 * wave_sum(fu);
          if (ph == 2 && !tile_accepts(f, al, dd, bs)) {
            sl.ls_evals = le + 1;
            sl.alpha = al * 0.5;
            sl.trial = tr + 1;
            sl.phase = tr + 1 == kLineSearchTrials ? 3 : 2;
            tile_submit<D>(L, j, lane, al * 0.5);
          } else {
            const bool stop = P.required > 0 && L.conv_sum[par] >= P.required;
            tile_slot_step<D>(L, sl, j, P, a.out, slot_mem(j), f, stop);
          }
        }
        if (lane == 0)
          L.live[j] = sl.phase != 0;
      }
      __syncthreads();
      const uint4 lv = *reinterpret_cast<const uint4*>(L.live);
      if ((lv.x | lv.y | lv.z | lv.w) == 0u)
        break;
    }
    if (tid == kStopReader)
      tile_count_converged(L, ctl);
    __syncthreads(); // LDS reuse by the next tile
  }
}

} // namespace zeus::dev
