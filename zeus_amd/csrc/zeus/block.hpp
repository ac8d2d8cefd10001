// block.hpp -- workgroup-level primitives for the per-workgroup BFGS.
#pragma once

#include "config.hpp"

#include <type_traits>

namespace zeus::dev {

// One DPP lane exchange of a double (two 32-bit moves).  Every pattern used
// here reads an active lane of the same row, so no lane reads out of range.
template <int kCtrl>
ZEUS_D ZEUS_FI double
dpp_f64(double v)
{
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(b)), kCtrl, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), kCtrl, 0xF, 0xF, false);
  return __builtin_bit_cast(double, (uint64_t(uint32_t(hi)) << 32) | uint32_t(lo));
}

ZEUS_D ZEUS_FI double
readlane_f64(double v, int lane)
{
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane(int(uint32_t(b)), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(int(uint32_t(b >> 32)), lane);
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

// One DPP lane exchange of any 64-bit value (two 32-bit moves).
template <int kCtrl, class T>
ZEUS_D ZEUS_FI T
dpp_b64(T v)
{
  static_assert(sizeof(T) == 8, "64-bit values");
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(b)), kCtrl, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), kCtrl, 0xF, 0xF, false);
  return __builtin_bit_cast(T, (uint64_t(uint32_t(hi)) << 32) | uint32_t(lo));
}

// The gfx950 row swaps of a 64-bit value with itself (kXor = 16:
// v_permlane16_swap, odd rows of the first operand with even rows of the
// second; kXor = 32: v_permlane32_swap, upper half with lower half).  Lane
// by lane, {first, second} hold v and v[lane ^ kXor] in some order.  All
// lanes must be active.
template <int kXor, class T>
ZEUS_D ZEUS_FI void
row_swap_b64(T v, T& first, T& second)
{
  static_assert(sizeof(T) == 8, "64-bit values");
  static_assert(kXor == 16 || kXor == 32, "row swaps only");
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const unsigned lo = unsigned(b), hi = unsigned(b >> 32);
  auto swap = [](unsigned x) {
    if constexpr (kXor == 16)
      return __builtin_amdgcn_permlane16_swap(x, x, false, false);
    else
      return __builtin_amdgcn_permlane32_swap(x, x, false, false);
  };
  const auto l = swap(lo);
  const auto h = swap(hi);
  first = __builtin_bit_cast(T, (uint64_t(h[0]) << 32) | l[0]);
  second = __builtin_bit_cast(T, (uint64_t(h[1]) << 32) | l[1]);
}

// v + v[lane ^ kXor] in every lane, kXor = 16 or 32, by the gfx950 lane
// swaps (v_permlane16_swap: odd rows of the first operand with even rows of
// the second; v_permlane32_swap: upper half with lower half): register moves,
// no LDS.  With both operands v, the two results hold, lane by lane, v and
// its partner's v in some order; IEEE addition is commutative, so every lane
// gets the bits of v + v[lane ^ kXor].  All lanes must be active.
template <int kXor>
ZEUS_D ZEUS_FI double
xor_sum(double v)
{
  double a, c;
  row_swap_b64<kXor>(v, a, c);
  return a + c;
}

// Sum of a 64-bit integer over the 64 lanes, every lane gets it (integer
// sums are exact in any order): DPP exchanges inside each row, then the row
// swaps.  All lanes must be active.
ZEUS_D ZEUS_FI int64_t
wave_sum_i64(int64_t v)
{
  v += dpp_b64<0xB1>(v);  // quad_perm [1,0,3,2]
  v += dpp_b64<0x4E>(v);  // quad_perm [2,3,0,1]
  v += dpp_b64<0x141>(v); // row_half_mirror
  v += dpp_b64<0x140>(v); // row_mirror
  int64_t a, c;
  row_swap_b64<16>(v, a, c);
  v = a + c;
  row_swap_b64<32>(v, a, c);
  return a + c;
}

// Sum over the 16 lanes of a row, the same bits in every lane of the row.
ZEUS_D ZEUS_FI double
row_sum(double v)
{
  v += dpp_f64<0xB1>(v);  // quad_perm [1,0,3,2]
  v += dpp_f64<0x4E>(v);  // quad_perm [2,3,0,1]
  v += dpp_f64<0x141>(v); // row_half_mirror
  v += dpp_f64<0x140>(v); // row_mirror
  return v;
}

// A value every lane of the wavefront holds identically, re-read from the
// first active lane so that the compiler treats it as wave-uniform (scalar
// registers) instead of one copy per lane.
template <class T>
ZEUS_D ZEUS_FI T
wave_uniform(const T& v)
{
  static_assert(sizeof(T) % 4 == 0, "whole 32-bit words");
  struct Words {
    uint32_t w[sizeof(T) / 4];
  };
  Words b = __builtin_bit_cast(Words, v);
#pragma unroll
  for (unsigned i = 0; i < sizeof(T) / 4; ++i)
    b.w[i] = __builtin_amdgcn_readfirstlane(int(b.w[i]));
  return __builtin_bit_cast(T, b);
}

// Sum over the 64 lanes of a wavefront, the same bits in every lane (a
// wave-uniform value).  Within each 16-lane row: DPP exchanges with lane
// xor 1, xor 2 (quad_perm), then the half-row and row mirrors; each step
// adds the same two operands in both lanes, so the row sum is bitwise equal
// across the row.  The four row sums are then combined in the fixed order
// (r0 + r1) + (r2 + r3).  All lanes of the wavefront must be active.
ZEUS_D ZEUS_FI double
wave_sum(double v)
{
  v += dpp_f64<0xB1>(v);  // quad_perm [1,0,3,2]
  v += dpp_f64<0x4E>(v);  // quad_perm [2,3,0,1]
  v += dpp_f64<0x141>(v); // row_half_mirror
  v += dpp_f64<0x140>(v); // row_mirror
  return (readlane_f64(v, 0) + readlane_f64(v, 16)) +
         (readlane_f64(v, 32) + readlane_f64(v, 48));
}

// LDS writes read back by other lanes of the same wavefront: the wavefront's
// LDS operations complete in order; these fences keep the compiler from moving
// accesses across the exchange.
ZEUS_D ZEUS_FI void
team_exchange()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Deterministic workgroup sums of K values at a time.  Two LDS slots are
// used alternately so that back-to-back reductions need one barrier each.
template <int NT>
struct Block {
  static constexpr int kWaves = NT / kWave;
  static_assert(NT % kWave == 0, "workgroup must be whole wavefronts");
  double* red;   // LDS, 2 * 4 * kWaves doubles
  int parity = 0;

  template <int K>
  ZEUS_D ZEUS_FI void sum(double (&v)[K])
  {
    static_assert(K <= 4, "at most 4 values per reduction");
#pragma unroll
    for (int k = 0; k < K; ++k)
      v[k] = wave_sum(v[k]);
    if constexpr (kWaves == 1) {
      // every lane has the wavefront's sum already: no trip through LDS (0.0 +
      // as the fold below starts).  The wavefront's LDS operations complete in
      // order; the fences keep the compiler from moving a caller's LDS accesses
      // across, as the barrier does for more wavefronts.
#pragma unroll
      for (int k = 0; k < K; ++k)
        v[k] = 0.0 + v[k];
      team_exchange();
      return;
    }
    double* r = red + parity * (4 * kWaves);
    parity ^= 1;
    const int w = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
#pragma unroll
      for (int k = 0; k < K; ++k)
        r[k * kWaves + w] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      double t = 0.0;
#pragma unroll
      for (int i = 0; i < kWaves; ++i)
        t += r[k * kWaves + i];
      v[k] = t;
    }
  }
  ZEUS_D ZEUS_FI double sum1(double v)
  {
    double a[1] = {v};
    sum<1>(a);
    return a[0];
  }
};

// Row-chunk layout of a D x D matrix over NT threads: thread t owns chunk
// c = t % CH of the rows r0 + k * RPP (r0 = t / CH, k < R); a chunk is L
// consecutive columns.  Matrix-vector products reduce the CH chunk partial
// sums of a row in a fixed order, so results do not depend on timing.
template <int D, int NT>
struct RowChunk {
  static constexpr int CH = (NT / D) >= 1 ? (NT / D) : 1;
  static constexpr int L = (D + CH - 1) / CH;
  static constexpr int RPP = NT / CH;
  static constexpr int R = (D + RPP - 1) / RPP;
  static constexpr int kPerThread = R * L;
};

// A D x D matrix distributed over the workgroup in the row-chunk layout,
// resident in registers (REG) or in a per-workgroup global slab whose
// element e of thread t sits at slab[e * NT + t] (coalesced).
template <int D, int NT, bool REG>
struct DistMatrix {
  static constexpr bool kPairs = false;
  using Lay = RowChunk<D, NT>;
  double m[REG ? Lay::kPerThread : 1];
  double* slab = nullptr;

  ZEUS_D ZEUS_FI double& at(int e)
  {
    if constexpr (REG)
      return m[e];
    else
      return slab[int64_t(e) * NT + threadIdx.x];
  }

  ZEUS_D ZEUS_FI void set_identity()
  {
    const int c = threadIdx.x % Lay::CH, r0 = threadIdx.x / Lay::CH;
#pragma unroll(REG ? 64 : 1)
    for (int k = 0; k < Lay::R; ++k) {
      const int row = r0 + k * Lay::RPP;
#pragma unroll(REG ? 64 : 1)
      for (int l = 0; l < Lay::L; ++l) {
        const int col = c * Lay::L + l;
        at(k * Lay::L + l) = (row == col && row < D) ? 1.0 : 0.0;
      }
    }
  }

  // Load a row-major D x D matrix.
  ZEUS_D ZEUS_FI void load(const double* src)
  {
    const int c = threadIdx.x % Lay::CH, r0 = threadIdx.x / Lay::CH;
#pragma unroll(REG ? 64 : 1)
    for (int k = 0; k < Lay::R; ++k) {
      const int row = r0 + k * Lay::RPP;
#pragma unroll(REG ? 64 : 1)
      for (int l = 0; l < Lay::L; ++l) {
        const int col = c * Lay::L + l;
        at(k * Lay::L + l) = (row < D && col < D) ? src[row * D + col] : 0.0;
      }
    }
  }

  // part[c * D + row] = sum over the chunk of M[row][col] * x[col].
  // With `pending`, first applies M += s a^T + a s^T (formed as
  // s_r a_c + a_r s_c, which is symmetric bit for bit) and stores it back:
  // one read-modify-write pass per BFGS iteration.
  ZEUS_D ZEUS_FI void pass(const double* x, const double* s, const double* a,
                           bool pending, double* part)
  {
    const int c = threadIdx.x % Lay::CH, r0 = threadIdx.x / Lay::CH;
#pragma unroll(REG ? 64 : 1)
    for (int k = 0; k < Lay::R; ++k) {
      const int row = r0 + k * Lay::RPP;
      if (row < D) {
        const double sr = pending ? s[row] : 0.0;
        const double ar = pending ? a[row] : 0.0;
        double acc = 0.0;
#pragma unroll(REG ? 64 : 1)
        for (int l = 0; l < Lay::L; ++l) {
          const int col = c * Lay::L + l;
          if (col < D) {
            double h = at(k * Lay::L + l);
            if (pending) {
              h = h + (sr * a[col] + ar * s[col]);
              at(k * Lay::L + l) = h;
            }
            acc = ::fma(h, x[col], acc);
          }
        }
        part[c * D + row] = acc;
      }
    }
  }
};

// v[row] = sum_c part[c * D + row], rows owned i = tid, tid + NT, ...
template <int D, int NT>
ZEUS_D ZEUS_FI double
chunk_total(const double* part, int row)
{
  using Lay = RowChunk<D, NT>;
  double t = 0.0;
#pragma unroll
  for (int c = 0; c < Lay::CH; ++c)
    t += part[c * D + row];
  return t;
}

// The inverse Hessian of a start as H = B + sum_j (s_j a_j^T + a_j s_j^T) in
// global memory, for dimensions whose D x D matrix neither fits the registers
// nor is worth streaming: the rank-2 pairs of the updates, B = I until the
// list is full, then the pairs are folded into an explicit B and the list
// restarts.  A product reads 2 k D doubles for k pairs, where a pass over an
// explicit H reads and writes D^2 (at D = 321 they meet at k = 321 pairs); with
// B, D^2 read and the pairs since the fold.  The list is kFirst = D / 2 pairs
// long (at most 160) before the first fold and kLater after it: a fold costs
// two passes over B and kLater / 2 pairs are read per product in between.
//
// pair_parts: partial products kept apart in LDS (the others are added in
// rounds).
template <int D, int NT>
constexpr int
pair_parts()
{
  return D > 512 ? 1 : (NT / kWave < 4 ? NT / kWave : 4);
}
template <int D, int NT>
struct PairMatrix {
  static constexpr bool kPairs = true;
  static constexpr int NW = NT / kWave, EL = (D + kWave - 1) / kWave;
  static constexpr int kFirst = D / 2 < 160 ? D / 2 : 160, kLater = 32;
  static_assert(kLater <= kFirst, "one list for both");
  static constexpr int kParts = pair_parts<D, NT>();
  static constexpr int kRounds = NW / kParts;
  static constexpr int64_t kSlabDoubles = int64_t(kFirst) * 2 * D + int64_t(D) * D;
  double* slab = nullptr;
  int k = 0;         // pairs in the list (the same in every thread)
  bool base = false; // explicit B in use

  ZEUS_D ZEUS_FI void set_identity()
  {
    k = 0;
    base = false;
  }
  ZEUS_D ZEUS_FI double* explicit_b() const { return slab + int64_t(kFirst) * 2 * D; }

  // part[q * D + i], q < kParts: the wavefronts' shares of (H - I) g, or of H g
  // with an explicit B; wavefront w takes the pairs (and rows of B) w, w + NW,
  // ..., two (four) in flight.  Ends with a barrier.
  ZEUS_D void apply(const double* g, double* part) const
  {
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int lane = threadIdx.x % kWave;
    double gr[EL], v[EL];
#pragma unroll
    for (int e = 0; e < EL; ++e) {
      const int i = lane + e * kWave;
      gr[e] = i < D ? g[i] : 0.0;
      v[e] = 0.0;
    }
    auto row = [&](const double* p, double (&r)[EL]) { // lanes past D read 0
#pragma unroll
      for (int e = 0; e < EL; ++e) {
        const int i = lane + e * kWave;
        r[e] = ((e + 1) * kWave <= D || i < D) ? p[i] : 0.0;
      }
    };
    constexpr int kC = 2;
#pragma unroll 1
    for (int j0 = w; j0 < k; j0 += kC * NW) {
      double s[kC][EL], a[kC][EL], c[kC], d[kC];
#pragma unroll
      for (int q = 0; q < kC; ++q) {
        const int j = j0 + q * NW < k ? j0 + q * NW : j0; // past the end: not used
        row(slab + int64_t(j) * 2 * D, s[q]);
        row(slab + int64_t(j) * 2 * D + D, a[q]);
      }
#pragma unroll
      for (int q = 0; q < kC; ++q) {
        c[q] = d[q] = 0.0;
#pragma unroll
        for (int e = 0; e < EL; ++e) {
          c[q] = ::fma(a[q][e], gr[e], c[q]);
          d[q] = ::fma(s[q][e], gr[e], d[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < kC; ++q) {
        c[q] = wave_sum(c[q]);
        d[q] = wave_sum(d[q]);
      }
#pragma unroll
      for (int q = 0; q < kC; ++q)
        if (j0 + q * NW < k)
#pragma unroll
          for (int e = 0; e < EL; ++e)
            v[e] = ::fma(s[q][e], c[q], ::fma(a[q][e], d[q], v[e]));
    }
    if (base) {
      const double* B = explicit_b();
      constexpr int kR = 4;
#pragma unroll 1
      for (int c0 = w; c0 < D; c0 += kR * NW) {
        double b[kR][EL];
#pragma unroll
        for (int q = 0; q < kR; ++q)
          row(B + int64_t(c0 + q * NW < D ? c0 + q * NW : c0) * D, b[q]);
#pragma unroll
        for (int q = 0; q < kR; ++q) {
          const double gc = c0 + q * NW < D ? g[c0 + q * NW] : 0.0;
#pragma unroll
          for (int e = 0; e < EL; ++e)
            v[e] = ::fma(b[q][e], gc, v[e]);
        }
      }
    }
#pragma unroll 1
    for (int t = 0; t < kRounds; ++t) {
      if (w / kParts == t) {
        double* p = part + (w % kParts) * D;
#pragma unroll
        for (int e = 0; e < EL; ++e) {
          const int i = lane + e * kWave;
          if (i < D)
            p[i] = t == 0 ? v[e] : p[i] + v[e];
        }
      }
      __syncthreads();
    }
  }
  // row i of H g from the parts
  ZEUS_D ZEUS_FI double total(const double* part, const double* g, int i) const
  {
    double t = base ? 0.0 : g[i];
#pragma unroll
    for (int q = 0; q < kParts; ++q)
      t += part[q * D + i];
    return t;
  }

  // Appends the pair (s, a) (LDS; element i read by the thread that wrote it);
  // the next product is behind a barrier of the caller.
  ZEUS_D void append(const double* s, const double* a)
  {
    double* p = slab + int64_t(k) * 2 * D;
    for (int i = threadIdx.x; i < D; i += NT) {
      p[i] = s[i];
      p[D + i] = a[i];
    }
    ++k;
    if (k == (base ? kLater : kFirst))
      fold();
  }

  // B += the pairs, kF rows at a time per wavefront.
  ZEUS_D void fold()
  {
    constexpr int kF = 4;
    __syncthreads(); // the last pair is stored
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int lane = threadIdx.x % kWave;
    double* B = explicit_b();
#pragma unroll 1
    for (int c0 = kF * w; c0 < D; c0 += kF * NW) {
      double b[kF][EL];
#pragma unroll
      for (int q = 0; q < kF; ++q)
#pragma unroll
        for (int e = 0; e < EL; ++e) {
          const int i = lane + e * kWave, c = c0 + q;
          b[q][e] = !(i < D && c < D) ? 0.0 : base ? B[int64_t(c) * D + i] : i == c ? 1.0 : 0.0;
        }
#pragma unroll 1
      for (int j = 0; j < k; ++j) {
        const double* s = slab + int64_t(j) * 2 * D;
        const double* a = s + D;
        double sc[kF], ac[kF];
#pragma unroll
        for (int q = 0; q < kF; ++q) {
          const int c = c0 + q < D ? c0 + q : D - 1;
          sc[q] = s[c];
          ac[q] = a[c];
        }
#pragma unroll
        for (int e = 0; e < EL; ++e) {
          const int i = lane + e * kWave;
          const double si = i < D ? s[i] : 0.0, ai = i < D ? a[i] : 0.0;
#pragma unroll
          for (int q = 0; q < kF; ++q)
            b[q][e] = b[q][e] + (si * ac[q] + ai * sc[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < kF; ++q)
#pragma unroll
        for (int e = 0; e < EL; ++e) {
          const int i = lane + e * kWave;
          if (i < D && c0 + q < D)
            B[int64_t(c0 + q) * D + i] = b[q][e];
        }
    }
    __syncthreads(); // before the list is overwritten and B is read
    k = 0;
    base = true;
  }
};

// Storage of a start's inverse Hessian in the per-workgroup form: registers,
// a streamed slab (up to 256 dimensions), or the pair list.
template <int D, int NT, bool REG>
constexpr bool kPairForm = !REG && (D > 256);
template <int D, int NT, bool REG>
using GroupH = std::conditional_t<kPairForm<D, NT, REG>, PairMatrix<D, NT>, DistMatrix<D, NT, REG>>;
// its doubles of global memory per workgroup
template <int D, int NT, bool REG>
constexpr int64_t
group_slab_doubles()
{
  if constexpr (REG)
    return 0;
  else if constexpr (kPairForm<D, NT, REG>)
    return PairMatrix<D, NT>::kSlabDoubles;
  else
    return int64_t(RowChunk<D, NT>::kPerThread) * NT;
}

} // namespace zeus::dev
