// Host-side plan of one compact operator along one direction.
//
// The reference assembles a global band per direction (compact_basetype.f90:
// 124-148), factors it whole (a bordered cyclic LU for periodic lines,
// pentadiagonal.f90:64-131, or a plain banded LU, :18-39) and sweeps each line
// sequentially. On the GPU a line is split into P chunks of at most CHUNK
// rows, one thread per chunk, its rows in registers. A solve is a forward and
// a backward second-order recurrence
//     x_k = r_k - l1_k x_{k-1} - l2_k x_{k-2}
//     y_k = g_k x_k - v1_k y_{k+1} - v2_k y_{k+2}
// (y times 1/c is the solution). A chunk runs each recurrence from a zero
// state to get its exit state e; its true entry state follows from the chunks
// before it (after it, backward) as E <- H_q E + e_q, with H_q the 2x2 matrix
// that takes chunk q's entry to its exit, and it re-runs the recurrence from
// there. Products of the H decay geometrically (the schemes' recurrences are
// strongly damped), so the sum starts W chunks away, where they fall below
// CARRY_TOL; around a cyclic line of fewer chunks it makes one turn and the
// remaining turns are a matrix (I - H...H)^-1.
//
// Periodic lines have a circulant LHS, which factors exactly as
//     A = c Q^T Q,   Q = I + p1 S + p2 S^2   ((S x)_i = x_{i-1}, cyclic)
// with both roots of 1 + p1 z + p2 z^2 outside the unit circle: the
// coefficients are constants (l = v = p, g = 1) and the carry wraps around.
// Bounded lines take the LU factors of the assembled band row by row; away
// from the lower end (and before the last four rows) they converge to the same
// constants, and chunks whose rows have all converged use those.
//
// RHS rows: interior rows use the interior weights; the four rows at each end
// of a bounded line use rows of their own, in the difference form
// sum_l c_l (v_{i+l} - v_i) + (sum_l c_l) v_i that the reference's forms
// amount to (compact_d1.f90:113-207, compact_r3.f90:97-157,
// compact_r4.f90:106-207); columns outside the line have no weight.
#pragma once

#include <algorithm>
#include <array>
#include <cmath>
#include <complex>
#include <stdexcept>
#include <string>
#include <vector>

#include "pyr_weights.hpp"

namespace pyr {

// Rows per thread. 16 keeps an FP64 chunk with its halo in 75-110 VGPRs (five
// waves per SIMD); measured at 256^3 on gfx950, FP64 d1 y: 54 us at 16 rows,
// 57 at 32, 79 at 8 (a copy of the field: 50 us).
constexpr int CHUNK = 16;
constexpr int PMAX = 64;    // chunks per line -> N <= 1024
constexpr int NB = 4;       // boundary rows per side with their own RHS forms
constexpr int WBROW = 10;   // a boundary row: weights at offsets -4..4, their sum

enum Kind { K_D1 = 0, K_R3 = 1, K_R4 = 2 };

inline int op_kind(int op) { return op == OP_D1 ? K_D1 : (op == OP_D2 ? K_R3 : K_R4); }
inline int kind_halo(int kind) { return kind == K_R4 ? 4 : 3; }

struct OpPlan {
  int op = 0, kind = 0, N = 0, P = 0, periodic = 0, implicit = 0, addv = 0;
  int null_op = 0, null_option = 0, R = 3;
  int mb = 0, mx = 0;         // chunk p has mb + (p < mx) rows
  double scale = 1.0;         // metric (times 1/c of an implicit operator)
  double w[4] = {};           // D1, explicit R4: weights at +1, +2, ...; R3/R4: their tail sums (rhs_interior)
  std::vector<double> wb;     // 2*NB x WBROW boundary rows of a bounded line
  double p1 = 0, p2 = 0;      // limit coefficients
  int W = 0;                  // chunks that enter a carry
  double hf[2][4] = {}, hb[2][4] = {};  // H of constant chunks of mb + 1 and mb rows
  int turns = 0;              // turns of a cyclic line beyond the first matter
  double tf[4] = {0, 0, 0, 0}, tb[4] = {0, 0, 0, 0};  // their sum (forward, backward)
  // bounded lines, for T slots (the chunks p < tlo, constant chunks of mb + 1
  // and mb rows, the last chunk): CHUNK x T x (l1, l2), CHUNK x T x (v1, v2),
  // CHUNK x T g, T x 8 H (forward, backward)
  int tlo = 0, T = 0;
  std::vector<double> tab;
};

// Propagation below this is left out of the carries. Relative to the state it
// multiplies, and so to the largest value of the line, that is under a
// thousandth of an FP64 rounding; a point W chunks away from values 1e16 times
// its own no longer gets their decayed share, which could have been its size.
constexpr long double CARRY_TOL = 1e-19L;

namespace detail {

using ld = long double;

// Spectral factor of the symmetric pentadiagonal symbol
//   b/z^2 + a/z + d + a z + b z^2 = c (1 + p1 z + p2 z^2)(1 + p1/z + p2/z^2)
// with the roots of 1 + p1 z + p2 z^2 outside the unit circle. With w = z + 1/z
// the quartic becomes b w^2 + a w + (d - 2b) = 0; each w gives the pair
// z, 1/z, of which the root inside the unit circle is kept. False if the
// symbol vanishes on the unit circle or b = 0.
inline bool spectral_factor(ld b, ld a, ld d, ld& p1, ld& p2, ld& c) {
  using cx = std::complex<ld>;
  if (b == 0.0L) return false;
  const cx disc = std::sqrt(cx(a * a - 4.0L * b * (d - 2.0L * b), 0.0L));
  const cx w[2] = {(cx(-a, 0.0L) + disc) / (2.0L * b), (cx(-a, 0.0L) - disc) / (2.0L * b)};
  cx r[2];
  for (int i = 0; i < 2; ++i) {
    const cx sq = std::sqrt(w[i] * w[i] - cx(4.0L, 0.0L));
    const cx z1 = (w[i] + sq) / 2.0L, z2 = (w[i] - sq) / 2.0L;
    r[i] = std::abs(z1) < std::abs(z2) ? z1 : z2;
    if (!(std::abs(r[i]) < 1.0L - 1e-9L)) return false;
  }
  const cx s1 = -(r[0] + r[1]), s2 = r[0] * r[1];
  if (std::fabs(s1.imag()) > 1e-15L || std::fabs(s2.imag()) > 1e-15L) return false;
  p1 = s1.real();
  p2 = s2.real();
  c = b / p2;
  const ld ed = c * (1.0L + p1 * p1 + p2 * p2) - d, ea = c * p1 * (1.0L + p2) - a;
  const ld scale = std::fabs(d) + 2.0L * std::fabs(a) + 2.0L * std::fabs(b);
  return std::fabs(ed) <= 1e-14L * scale && std::fabs(ea) <= 1e-14L * scale;
}

using M2 = std::array<ld, 4>;  // 2x2, row-major

inline M2 mul(const M2& x, const M2& y) {
  return {x[0] * y[0] + x[1] * y[2], x[0] * y[1] + x[1] * y[3], x[2] * y[0] + x[3] * y[2], x[2] * y[1] + x[3] * y[3]};
}
inline ld norm(const M2& x) {
  return std::max(std::max(std::fabs(x[0]), std::fabs(x[1])), std::max(std::fabs(x[2]), std::fabs(x[3])));
}

// Chunks that enter the carries of one direction (step -1: chunk p takes from
// p-1, p-2, ...; +1: from p+1, ...): the most, over p, whose propagation to p
// is above CARRY_TOL.
inline int carry_terms(const std::vector<M2>& H, int step, bool cyclic) {
  const int P = (int)H.size();
  int W = 0;
  for (int p = 0; p < P; ++p) {
    M2 acc = {1, 0, 0, 1};
    for (int j = 1;; ++j) {
      const int q = p + step * j;
      if (!cyclic && (q < 0 || q >= P)) break;
      if (norm(acc) < CARRY_TOL) break;
      W = std::max(W, j);
      acc = mul(acc, H[((q % P) + P) % P]);
    }
  }
  return W;
}

// (I - H around a whole cyclic line)^-1 for the entry of a chunk
inline M2 turns(const std::vector<M2>& H, int step) {
  const int P = (int)H.size();
  M2 acc = {1, 0, 0, 1};
  for (int j = 1; j <= P; ++j) acc = mul(acc, H[(((step * j) % P) + P) % P]);
  const ld a = 1 - acc[0], b = -acc[1], c = -acc[2], d = 1 - acc[3], det = a * d - b * c;
  return {d / det, -b / det, -c / det, a / det};
}

// Chunks of a line of n rows along direction dir. x lines: one wave takes G
// whole lines, so P is the most chunks that still leaves room for as many
// lines as the fewest possible chunks would (n = 300: 19 chunks needed, 3
// lines per wave, 21 chunks each). y/z lines: an even count, so that waves of
// 32 lines hold two chunks each. Every chunk has at least 8 rows (n >= 8).
inline int chunk_count(int n, int dir) {
  const int need = (n + CHUNK - 1) / CHUNK;
  if (n == need * CHUNK) return need;
  if (dir == 0) return 64 / (64 / need);
  return need > 2 ? need + (need & 1) : need;
}

}  // namespace detail

// Build the plan. v1/v2 are the boundary variants (0 NONE, +1 SYMM, -1 its
// antisymmetric member).
inline OpPlan build_plan(int op, int n, int dir, int periodic, int v1, int v2, double metric) {
  using detail::ld;
  using detail::M2;
  OpPlan pl;
  const Scheme sc = make_scheme(op);
  pl.op = op;
  pl.kind = op_kind(op);
  pl.N = n;
  pl.periodic = periodic;
  pl.implicit = sc.implicit;
  pl.addv = (sc.null_option == 1);
  pl.null_option = sc.null_option;
  pl.R = kind_halo(pl.kind);
  pl.null_op = (n < 4);  // compact_basetype.f90:86-90
  pl.scale = (op == OP_D1) ? 1.0 / metric : (op == OP_D2 ? 1.0 / (metric * metric) : 1.0);
  const int hr = sc.ncr / 2;
  if (pl.kind == K_D1 || !sc.implicit) {
    for (int l = 1; l <= pl.R; ++l) pl.w[l - 1] = sc.ari[hr + l];
  } else {
    // symmetric rows of zero sum: sum_l w_l (v_{i+l} - v_i) = sum_m c_m
    // (d_{i+m-1} - d_{i-m}) with d_j = v_{j+1} - v_j and c_m = w_m + w_{m+1} + ...
    ld c = 0.0L;
    for (int l = pl.R; l >= 1; --l) {
      c += (ld)sc.ari[hr + l];
      pl.w[l - 1] = (double)c;
    }
  }
  if (pl.null_op) return pl;
  // the reference's boundary forms read up to row 8 of a line (compact_r4.f90:
  // 117-120); shorter lines are outside what the schemes define
  if (n < 8) throw std::runtime_error("line length " + std::to_string(n) + " is below 8 (supported: 1-3 or 8-1024)");
  if (n > CHUNK * PMAX)
    throw std::runtime_error("line length " + std::to_string(n) + " exceeds " + std::to_string(CHUNK * PMAX));
  const int P = detail::chunk_count(n, dir);
  pl.P = P;
  pl.mb = n / P;
  pl.mx = n % P;
  auto start = [&](int p) { return p * pl.mb + std::min(p, pl.mx); };

  // boundary rows of a bounded line (compact_basetype.f90:124-133)
  if (!periodic) {
    pl.wb.assign(2 * NB * WBROW, 0.0);
    for (int j = 0; j < 2 * NB; ++j) {
      const bool lo = j < NB;
      const double* row = lo ? sc.arb1[v1 + 1][j] : sc.arb2[v2 + 1][j - NB];
      double* o = &pl.wb[j * WBROW];
      ld sum = 0.0L;
      for (int l = -hr; l <= hr; ++l) {
        if (std::abs(l) > 4) continue;
        const int col = (lo ? j : n - 2 * NB + j) + l;
        if (col < 0 || col >= n) continue;  // ghost columns read 0
        sum += (ld)row[l + hr];
        if (l != 0 || !sc.implicit) o[l + 4] = row[l + hr];
      }
      // rows of the NONE and SYMM variants have zero sum
      if ((lo ? v1 : v2) == -1) o[WBROW - 1] = (double)sum;
    }
  }
  if (!sc.implicit) return pl;

  ld p1, p2, cc;
  if (sc.ncl != 5 || sc.ali[0] != sc.ali[4] || sc.ali[1] != sc.ali[3] ||
      !detail::spectral_factor(sc.ali[0], sc.ali[1], sc.ali[2], p1, p2, cc))
    throw std::runtime_error("the scheme's left-hand side has no spectral factor");
  pl.p1 = (double)p1;
  pl.p2 = (double)p2;
  pl.scale = (double)((ld)pl.scale / cc);
  if (!periodic && op == OP_D2) {
    // The recurrences solve for c times the result, c = 1e4, which next to a
    // bounded end reaches eight times the largest right-hand side before the
    // scale takes c back. This factor changes no bit and keeps it below the
    // largest number wherever the right-hand sides are.
    for (double& w : pl.w) w *= 0.125;
    for (double& w : pl.wb) w *= 0.125;
    pl.scale *= 8.0;
  }

  // per-row factors (constants for a periodic line)
  std::vector<ld> l1(n, p1), l2(n, p2), u1(n, p1), u2(n, p2), g(n, 1.0L);
  if (!periodic) {
    std::vector<std::array<ld, 5>> A(n);
    for (int i = 0; i < n; ++i)
      for (int c = 0; c < 5; ++c) A[i][c] = (ld)sc.ali[c];
    for (int j = 0; j < NB; ++j)
      for (int c = 0; c < 5; ++c) {
        A[j][c] = (ld)sc.alb1[v1 + 1][j][c];
        A[n - NB + j][c] = (ld)sc.alb2[v2 + 1][j][c];
      }
    std::vector<ld> U0(n), U1(n), U2(n);
    for (int i = 0; i < n; ++i) {
      ld a0 = i >= 2 ? A[i][0] : 0.0L, a1 = i >= 1 ? A[i][1] : 0.0L, d = A[i][2];
      ld b1 = i + 1 < n ? A[i][3] : 0.0L, b2 = i + 2 < n ? A[i][4] : 0.0L;
      l1[i] = l2[i] = 0.0L;
      if (i >= 2) {
        l2[i] = a0 / U0[i - 2];
        a1 -= l2[i] * U1[i - 2];
        d -= l2[i] * U2[i - 2];
      }
      if (i >= 1) {
        l1[i] = a1 / U0[i - 1];
        d -= l1[i] * U1[i - 1];
        b1 -= l1[i] * U2[i - 1];
      }
      if (d == 0.0L) throw std::runtime_error("zero pivot in the line factorization");
      U0[i] = d; U1[i] = b1; U2[i] = b2;
      u1[i] = b1 / d;
      u2[i] = b2 / d;
      g[i] = cc / d;
    }
    // rows that have converged take the limit exactly: a chunk of such rows
    // then gives the same bits through the tables and through the constants
    auto near = [](ld x, ld y) { return std::fabs(x - y) <= 1.2e-16L * std::fabs(y); };
    std::vector<char> conv(n, 0);
    for (int i = 0; i < n; ++i)
      if (near(l1[i], p1) && near(l2[i], p2) && near(u1[i], p1) && near(u2[i], p2) && near(g[i], 1.0L)) {
        conv[i] = 1;
        l1[i] = u1[i] = p1;
        l2[i] = u2[i] = p2;
        g[i] = 1.0L;
      }
    for (int p = 0; p < P - 1; ++p)
      for (int i = start(p); i < start(p + 1); ++i)
        if (!conv[i]) pl.tlo = p + 1;
  }

  // entry-to-exit matrices and carries
  std::vector<M2> Hf(P), Hb(P);
  for (int p = 0; p < P; ++p)
    for (int j = 0; j < 2; ++j) {
      ld xm2 = j == 0, xm1 = j == 1;  // forward state (x[k-2], x[k-1])
      for (int i = start(p); i < start(p + 1); ++i) {
        const ld x = -l1[i] * xm1 - l2[i] * xm2;
        xm2 = xm1;
        xm1 = x;
      }
      Hf[p][j] = xm2;
      Hf[p][2 + j] = xm1;
      ld b1 = j == 0, b2 = j == 1;  // backward state (y[k+1], y[k+2])
      for (int i = start(p + 1) - 1; i >= start(p); --i) {
        const ld y = -u1[i] * b1 - u2[i] * b2;
        b2 = b1;
        b1 = y;
      }
      Hb[p][j] = b1;
      Hb[p][2 + j] = b2;
    }
  const int need = std::max(detail::carry_terms(Hf, -1, periodic), detail::carry_terms(Hb, 1, periodic));
  pl.W = std::min(need, periodic ? P : P - 1);
  if (need > pl.W && periodic) {
    // every H is a power of one matrix, so the sum is the same for each chunk
    pl.turns = 1;
    const M2 f = detail::turns(Hf, -1), b = detail::turns(Hb, 1);
    for (int i = 0; i < 4; ++i) {
      pl.tf[i] = (double)f[i];
      pl.tb[i] = (double)b[i];
    }
  }
  // constant chunks, from the limit coefficients
  for (int w = 0; w < 2; ++w)
    for (int j = 0; j < 2; ++j) {
      ld a0 = j == 0, a1 = j == 1, b1 = j == 0, b2 = j == 1;
      for (int k = 0; k < pl.mb + 1 - w; ++k) {
        const ld x = -p1 * a1 - p2 * a0, y = -p1 * b1 - p2 * b2;
        a0 = a1; a1 = x;
        b2 = b1; b1 = y;
      }
      pl.hf[w][j] = (double)a0; pl.hf[w][2 + j] = (double)a1;
      pl.hb[w][j] = (double)b1; pl.hb[w][2 + j] = (double)b2;
    }
  if (periodic) return pl;
  const int T = pl.T = pl.tlo + 3;
  pl.tab.assign((size_t)CHUNK * T * 5 + 8 * T, 0.0);
  double* tf = pl.tab.data();
  double* tb = tf + 2 * CHUNK * T;
  double* tg = tb + 2 * CHUNK * T;
  double* th = tg + CHUNK * T;
  for (int t = 0; t < T; ++t) {
    const bool chunk = t < pl.tlo || t == T - 1;  // else a constant slot
    const int p = t == T - 1 ? P - 1 : t;
    for (int k = 0; k < CHUNK; ++k) {
      const int i = start(p) + k;
      const bool own = chunk && i < start(p + 1);
      const size_t e = (size_t)k * T + t;
      tf[2 * e] = (double)(own ? l1[i] : p1); tf[2 * e + 1] = (double)(own ? l2[i] : p2);
      tb[2 * e] = (double)(own ? u1[i] : p1); tb[2 * e + 1] = (double)(own ? u2[i] : p2);
      tg[e] = own ? (double)g[i] : 1.0;
    }
    for (int i = 0; i < 4; ++i) {
      th[8 * t + i] = chunk ? (double)Hf[p][i] : pl.hf[t - pl.tlo][i];
      th[8 * t + 4 + i] = chunk ? (double)Hb[p][i] : pl.hb[t - pl.tlo][i];
    }
  }
  return pl;
}

}  // namespace pyr
