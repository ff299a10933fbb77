// Refined FP32 solve of bounded lines: plan and per-thread arithmetic.
//
// FP32 fields whose lines are bounded (and whose context keeps the default
// PYR_R32_SOLVE_REFINED arithmetic) are solved in FP32 and refined once with an
// FP64 residual. The line is split into chunks of at most 32 rows, one thread
// each: a thread solves its chunk's own banded block, the four values next to
// the chunk come from rows of the inverse of a small reduced system, and a
// spike correction couples them in; the same again for the correction. The
// order of every operation is part of the result (an FP32 field is reproduced
// to the bit by the same input), so it is kept apart from the FP64 recurrences
// that every other line takes (pyr_line.hpp).
//
// Interior rows of the left-hand side are the same everywhere, so all interior
// chunks of one length share their block's factors and spikes to the bit: four
// tables (first chunk, interior with mb + 1 and mb rows, last chunk) replace
// tables over the whole line and fit LDS at any line length.
#pragma once

#include <cstring>

#include "pyr_line.hpp"

namespace pyr {

constexpr int RCHUNK = 32;  // rows per thread
constexpr int MAXT = 10;    // terms per boundary row
constexpr int ENDS = 16;    // rows the terms name: slot i < 8 is row i, i < 16 row N - 16 + i, 16 reads 0
constexpr int NCLS = 4;     // first, interior (mb + 1 rows), interior (mb), last
constexpr int CROW = 12;    // floats per table row: 4 spikes | 1/u, u1, u2, 0 | l2, l1, 0, 0

struct RefPlan {
  int N = 0, P = 0, mb = 0, mx = 0;
  int Wg = 0;               // chunks on each side that the reduced rows reach
  double scale = 1.0;
  double w[9] = {};         // interior weights at offsets -R..R
  double bd[5] = {};        // interior row of the left-hand side
  std::vector<float> cls;   // NCLS x RCHUNK x CROW
  std::vector<float> g;     // P x (2 Wg + 1) x 4 x 4: reduced-system rows of the four neighbour values,
                            // for the chunks within reach (0 beyond the line's ends)
  std::vector<double> be;   // 2*NB x 5: left-hand rows at the ends
  std::vector<double> bcoef;  // 2*NB x MAXT terms coef * (v[a] - v[b])
  std::vector<int> bidx;      // 2*NB x MAXT x 2: slots of a and b among the line's end rows
};

// class of chunk p (the first one also where it is the last)
PYR_HD int ref_class(int p, int P, int mx) { return p == 0 ? 0 : (p == P - 1 ? 3 : (p < mx ? 1 : 2)); }

namespace detail {

struct TermRow {
  std::vector<double> c;
  std::vector<int> a, b;
  void add(double coef, int ia, int ib) {
    if (coef == 0.0) return;
    c.push_back(coef); a.push_back(ia); b.push_back(ib);
  }
};

// Boundary-row RHS forms of a bounded line, 0-based rows; ar(l,i) is the
// reference's (1-based l, 1-based i) weight. Ghost columns read 0.
inline void boundary_terms(int kind, int n, int v1, int v2,
                           const std::vector<std::vector<double>>& ar,
                           TermRow lo[NB], TermRow hi[NB]) {
  auto AR = [&](int l, int i1) { return ar[i1 - 1][l - 1]; };
  auto sumr = [&](int i1, int nr) { double s = 0; for (int l = 1; l <= nr; ++l) s += AR(l, i1); return s; };
  if (kind == K_D1) {
    if (v1 == -1) {
      for (int l = 4; l <= 7; ++l) lo[0].add(AR(l, 1), l - 4, -1);
      for (int l = 3; l <= 7; ++l) lo[1].add(AR(l, 2), l - 3, -1);
      for (int l = 2; l <= 7; ++l) lo[2].add(AR(l, 3), l - 2, -1);
    } else {
      for (int l = 5; l <= 7; ++l) lo[0].add(AR(l, 1), l - 4, 0);
      for (int l = 4; l <= 7; ++l) lo[1].add(AR(l, 2), l - 3, 0);
      lo[2].add(AR(5, 3), 3, 1); lo[2].add(AR(6, 3), 4, 0); lo[2].add(AR(7, 3), 5, 0);
    }
    // row 4 (1-based): interior antisymmetric form with its own weights
    lo[3].add(AR(5, 4), 4, 2); lo[3].add(AR(6, 4), 5, 1); lo[3].add(AR(7, 4), 6, 0);
    // row n-3 (1-based)
    hi[0].add(AR(5, n - 3), n - 3, n - 5); hi[0].add(AR(6, n - 3), n - 2, n - 6);
    hi[0].add(AR(7, n - 3), n - 1, n - 7);
    if (v2 == -1) {
      for (int l = 1; l <= 6; ++l) hi[1].add(AR(l, n - 2), n - 7 + l, -1);
      for (int l = 1; l <= 5; ++l) hi[2].add(AR(l, n - 1), n - 6 + l, -1);
      for (int l = 1; l <= 4; ++l) hi[3].add(AR(l, n), n - 5 + l, -1);
    } else {
      hi[1].add(AR(1, n - 2), n - 6, n - 1); hi[1].add(AR(2, n - 2), n - 5, n - 1);
      hi[1].add(AR(3, n - 2), n - 4, n - 2);
      for (int l = 1; l <= 4; ++l) hi[2].add(AR(l, n - 1), n - 6 + l, n - 1);
      for (int l = 1; l <= 3; ++l) hi[3].add(AR(l, n), n - 5 + l, n - 1);
    }
  } else if (kind == K_R3) {
    // ghosts are zero on a bounded end (compact_r3.f90:84-99)
    for (int l = 1; l <= 3; ++l) lo[0].add(AR(l, 1), -1, 0);
    for (int l = 4; l <= 7; ++l) lo[0].add(AR(l, 1), l - 4, 0);
    for (int l = 1; l <= 2; ++l) lo[1].add(AR(l, 2), -1, 1);
    for (int l = 3; l <= 7; ++l) lo[1].add(AR(l, 2), l - 3, 1);
    lo[2].add(AR(1, 3), -1, 2);
    for (int l = 2; l <= 7; ++l) lo[2].add(AR(l, 3), l - 2, 2);
    for (int l = 1; l <= 7; ++l) lo[3].add(AR(l, 4), l - 1, 3);
    if (v1 == -1)
      for (int r = 0; r < 3; ++r) lo[r].add(sumr(r + 1, 7), r, -1);
    for (int l = 1; l <= 7; ++l) hi[0].add(AR(l, n - 3), n - 8 + l, n - 4);
    for (int l = 1; l <= 6; ++l) hi[1].add(AR(l, n - 2), n - 7 + l, n - 3);
    hi[1].add(AR(7, n - 2), -1, n - 3);
    for (int l = 1; l <= 5; ++l) hi[2].add(AR(l, n - 1), n - 6 + l, n - 2);
    for (int l = 6; l <= 7; ++l) hi[2].add(AR(l, n - 1), -1, n - 2);
    for (int l = 1; l <= 4; ++l) hi[3].add(AR(l, n), n - 5 + l, n - 1);
    for (int l = 5; l <= 7; ++l) hi[3].add(AR(l, n), -1, n - 1);
    if (v2 == -1)
      for (int r = 1; r < 4; ++r) hi[r].add(sumr(n - 3 + r, 7), n - 4 + r, -1);
  } else {
    if (v1 == -1) {
      for (int l = 5; l <= 9; ++l) lo[0].add(AR(l, 1), l - 5, -1);
      for (int l = 4; l <= 9; ++l) lo[1].add(AR(l, 2), l - 4, -1);
      for (int l = 3; l <= 9; ++l) lo[2].add(AR(l, 3), l - 3, -1);
      for (int l = 2; l <= 9; ++l) lo[3].add(AR(l, 4), l - 2, -1);
    } else {
      for (int l = 6; l <= 9; ++l) lo[0].add(AR(l, 1), l - 5, 0);
      for (int l = 5; l <= 9; ++l) lo[1].add(AR(l, 2), l - 4, 0);
      for (int l = 4; l <= 9; ++l) lo[2].add(AR(l, 3), l - 3, 0);
      for (int l = 3; l <= 9; ++l) lo[3].add(AR(l, 4), l - 2, 0);
    }
    if (v2 == -1) {
      for (int l = 1; l <= 8; ++l) hi[0].add(AR(l, n - 3), n - 9 + l, -1);
      for (int l = 1; l <= 7; ++l) hi[1].add(AR(l, n - 2), n - 8 + l, -1);
      for (int l = 1; l <= 6; ++l) hi[2].add(AR(l, n - 1), n - 7 + l, -1);
      for (int l = 1; l <= 5; ++l) hi[3].add(AR(l, n), n - 6 + l, -1);
    } else {
      for (int l = 1; l <= 7; ++l) hi[0].add(AR(l, n - 3), n - 9 + l, n - 1);
      for (int l = 1; l <= 6; ++l) hi[1].add(AR(l, n - 2), n - 8 + l, n - 1);
      for (int l = 1; l <= 5; ++l) hi[2].add(AR(l, n - 1), n - 7 + l, n - 1);
      for (int l = 1; l <= 4; ++l) hi[3].add(AR(l, n), n - 6 + l, n - 1);
    }
  }
}

// Gauss-Jordan inverse with partial pivoting (small dense, long double)
inline void invert(std::vector<ld>& a, int n) {
  std::vector<ld> inv(size_t(n) * n, 0.0L);
  for (int i = 0; i < n; ++i) inv[size_t(i) * n + i] = 1.0L;
  for (int c = 0; c < n; ++c) {
    int piv = c;
    for (int r = c + 1; r < n; ++r)
      if (std::fabs(a[size_t(r) * n + c]) > std::fabs(a[size_t(piv) * n + c])) piv = r;
    if (a[size_t(piv) * n + c] == 0.0L) throw std::runtime_error("singular reduced system");
    if (piv != c)
      for (int k = 0; k < n; ++k) {
        std::swap(a[size_t(c) * n + k], a[size_t(piv) * n + k]);
        std::swap(inv[size_t(c) * n + k], inv[size_t(piv) * n + k]);
      }
    const ld d = 1.0L / a[size_t(c) * n + c];
    for (int k = 0; k < n; ++k) { a[size_t(c) * n + k] *= d; inv[size_t(c) * n + k] *= d; }
    for (int r = 0; r < n; ++r) {
      if (r == c) continue;
      const ld f = a[size_t(r) * n + c];
      if (f == 0.0L) continue;
      for (int k = 0; k < n; ++k) {
        a[size_t(r) * n + k] -= f * a[size_t(c) * n + k];
        inv[size_t(r) * n + k] -= f * inv[size_t(c) * n + k];
      }
    }
  }
  a.swap(inv);
}

}  // namespace detail

inline RefPlan build_ref_plan(int op, int n, int v1, int v2, double metric) {
  using detail::ld;
  RefPlan pl;
  const Scheme sc = make_scheme(op);
  const int kind = op_kind(op), R = kind_halo(kind);
  pl.N = n;
  pl.scale = (op == OP_D1) ? 1.0 / metric : (op == OP_D2 ? 1.0 / (metric * metric) : 1.0);
  const int hr = sc.ncr / 2;
  for (int l = -R; l <= R; ++l) pl.w[l + R] = sc.ari[l + hr];
  for (int c = 0; c < 5; ++c) pl.bd[c] = sc.ali[c];
  // assembled rows (compact_basetype.f90:124-133), 0-based
  std::vector<std::vector<double>> gal(n, std::vector<double>(5, 0.0));
  std::vector<std::vector<double>> gar(n, std::vector<double>(9, 0.0));
  for (int i = 0; i < n; ++i) {
    for (int c = 0; c < sc.ncl; ++c) gal[i][c] = sc.ali[c];
    for (int l = 0; l < sc.ncr; ++l) gar[i][l] = sc.ari[l];
  }
  {
    for (int j = 0; j < 4; ++j) {
      for (int c = 0; c < sc.ncl; ++c) {
        gal[j][c] = sc.alb1[v1 + 1][j][c];
        gal[n - 4 + j][c] = sc.alb2[v2 + 1][j][c];
      }
      for (int l = 0; l < sc.ncr; ++l) {
        gar[j][l] = sc.arb1[v1 + 1][j][l];
        gar[n - 4 + j][l] = sc.arb2[v2 + 1][j][l];
      }
    }
  }
  pl.be.resize(2 * NB * 5);
  for (int j = 0; j < 2 * NB; ++j)
    for (int c = 0; c < 5; ++c) pl.be[j * 5 + c] = gal[j < NB ? j : n - 2 * NB + j][c];
  pl.bcoef.assign(2 * NB * MAXT, 0.0);
  pl.bidx.assign(2 * NB * MAXT * 2, ENDS);
  {
    auto end_slot = [&](int i) {
      if (i < 0) return ENDS;
      if (i < ENDS / 2) return i;
      if (i < n - ENDS / 2) throw std::runtime_error("boundary term outside the line's ends");
      return i - n + ENDS;
    };
    detail::TermRow lo[NB], hi[NB];
    detail::boundary_terms(kind, n, v1, v2, gar, lo, hi);
    for (int r = 0; r < 2 * NB; ++r) {
      const detail::TermRow& t = r < NB ? lo[r] : hi[r - NB];
      if ((int)t.c.size() > MAXT) throw std::runtime_error("boundary row has too many terms");
      for (size_t q = 0; q < t.c.size(); ++q) {
        if (t.a[q] < -1 || t.a[q] >= n || t.b[q] < -1 || t.b[q] >= n)
          throw std::runtime_error("boundary term outside the line");
        pl.bcoef[r * MAXT + q] = t.c[q];
        pl.bidx[(r * MAXT + q) * 2 + 0] = end_slot(t.a[q]);
        pl.bidx[(r * MAXT + q) * 2 + 1] = end_slot(t.b[q]);
      }
    }
  }

  // chunk partition: balanced lengths (all >= 8)
  const int P = (n + RCHUNK - 1) / RCHUNK;
  pl.P = P;
  pl.mb = n / P;
  pl.mx = n % P;
  std::vector<int> cstart(P + 1);
  for (int p = 0; p <= P; ++p) cstart[p] = p * pl.mb + std::min(p, pl.mx);
  pl.cls.assign(NCLS * RCHUNK * CROW, 0.0f);
  bool have[NCLS] = {};
  auto Aent = [&](int i, int col) -> double {  // A[i][col], col may wrap
    const int off = col - i;
    if (off < -2 || off > 2 || col < 0 || col >= n) return 0.0;
    return gal[i][off + 2];
  };

  std::vector<ld> S(size_t(4 * P) * 4 * P, 0.0L);
  for (int p = 0; p < P; ++p) {
    const int s = cstart[p], e = cstart[p + 1], m = e - s;
    const int cl = ref_class(p, P, pl.mx);
    std::vector<float> tab(RCHUNK * CROW, 0.0f);
    // dense block, no pivoting LU (SPD-like blocks of the compact LHS)
    std::vector<ld> blk(size_t(m) * m, 0.0L);
    for (int i = 0; i < m; ++i)
      for (int j = std::max(0, i - 2); j <= std::min(m - 1, i + 2); ++j)
        blk[size_t(i) * m + j] = (ld)gal[s + i][j - i + 2];
    std::vector<ld> L(size_t(m) * 3, 0.0L);  // multipliers for i-2, i-1
    for (int k = 0; k < m; ++k) {
      const ld piv = blk[size_t(k) * m + k];
      if (piv == 0.0L) throw std::runtime_error("zero pivot in chunk LU");
      for (int i = k + 1; i <= std::min(m - 1, k + 2); ++i) {
        const ld f = blk[size_t(i) * m + k] / piv;
        L[size_t(i) * 3 + (i - k == 2 ? 0 : 1)] = f;
        for (int j = k; j <= std::min(m - 1, k + 2); ++j) blk[size_t(i) * m + j] -= f * blk[size_t(k) * m + j];
      }
    }
    for (int i = 0; i < m; ++i) {
      const double c[5] = {(double)L[size_t(i) * 3 + 0], (double)L[size_t(i) * 3 + 1],
                           (double)(1.0L / blk[size_t(i) * m + i]),
                           (i + 1 < m) ? (double)blk[size_t(i) * m + i + 1] : 0.0,
                           (i + 2 < m) ? (double)blk[size_t(i) * m + i + 2] : 0.0};
      const int at[5] = {8, 9, 4, 5, 6};
      for (int q = 0; q < 5; ++q) tab[i * CROW + at[q]] = (float)c[q];
    }
    // solve with the long-double factors for the spike columns
    auto solve = [&](std::vector<ld>& r) {
      for (int i = 0; i < m; ++i) {
        if (i >= 1) r[i] -= L[size_t(i) * 3 + 1] * r[i - 1];
        if (i >= 2) r[i] -= L[size_t(i) * 3 + 0] * r[i - 2];
      }
      for (int i = m - 1; i >= 0; --i) {
        ld v = r[i];
        if (i + 1 < m) v -= blk[size_t(i) * m + i + 1] * r[i + 1];
        if (i + 2 < m) v -= blk[size_t(i) * m + i + 2] * r[i + 2];
        r[i] = v / blk[size_t(i) * m + i];
      }
    };
    std::vector<ld> w0(m, 0.0L), w1(m, 0.0L), wm2(m, 0.0L), wm1(m, 0.0L);
    w0[0] = 1; w1[1] = 1; wm2[m - 2] = 1; wm1[m - 1] = 1;
    solve(w0); solve(w1); solve(wm2); solve(wm1);
    const bool has_lo = p > 0, has_hi = p < P - 1;
    // couplings to the previous chunk's last two unknowns (y[s-2], y[s-1])
    const ld a_s_m2 = has_lo ? (ld)Aent(s, s - 2) : 0.0L;
    const ld a_s_m1 = has_lo ? (ld)Aent(s, s - 1) : 0.0L;
    const ld a_s1_m1 = has_lo ? (ld)Aent(s + 1, s - 1) : 0.0L;
    // couplings to the next chunk's first two unknowns (y[e], y[e+1])
    const ld a_e2_e = has_hi ? (ld)Aent(e - 2, e) : 0.0L;
    const ld a_e1_e = has_hi ? (ld)Aent(e - 1, e) : 0.0L;
    const ld a_e1_e1 = has_hi ? (ld)Aent(e - 1, e + 1) : 0.0L;
    std::vector<ld> r0(m), r1(m), r2(m), r3(m);
    for (int i = 0; i < m; ++i) {
      r0[i] = a_s_m2 * w0[i];
      r1[i] = a_s_m1 * w0[i] + a_s1_m1 * w1[i];
      r2[i] = a_e2_e * wm2[i] + a_e1_e * wm1[i];
      r3[i] = a_e1_e1 * wm1[i];
      const ld r[4] = {r0[i], r1[i], r2[i], r3[i]};
      for (int q = 0; q < 4; ++q) tab[i * CROW + q] = (float)(double)r[q];
    }
    float* have_tab = &pl.cls[cl * RCHUNK * CROW];
    if (!have[cl]) std::memcpy(have_tab, tab.data(), tab.size() * sizeof(float));
    else if (std::memcmp(have_tab, tab.data(), tab.size() * sizeof(float)) != 0)
      throw std::runtime_error("interior chunks of one length differ");
    have[cl] = true;
    // reduced-system rows for this chunk's four edge unknowns
    const int pm = (p - 1 + P) % P, pp = (p + 1) % P;
    const int edge[4] = {0, 1, m - 2, m - 1};
    for (int q = 0; q < 4; ++q) {
      const int row = 4 * p + q, li = edge[q];
      S[size_t(row) * 4 * P + row] += 1.0L;
      if (has_lo) {
        S[size_t(row) * 4 * P + 4 * pm + 2] += r0[li];
        S[size_t(row) * 4 * P + 4 * pm + 3] += r1[li];
      }
      if (has_hi) {
        S[size_t(row) * 4 * P + 4 * pp + 0] += r2[li];
        S[size_t(row) * 4 * P + 4 * pp + 1] += r3[li];
      }
    }
  }
  detail::invert(S, 4 * P);
  auto row_of = [&](int p, int q, int c) -> double {
    const int rows[4] = {4 * (p - 1) + 2, 4 * (p - 1) + 3, 4 * (p + 1) + 0, 4 * (p + 1) + 1};
    if (q < 2 ? p == 0 : p == P - 1) return 0.0;
    return (double)S[size_t(rows[q]) * 4 * P + c];
  };
  for (int p = 0; p < P; ++p)
    for (int c = 0; c < 4 * P; ++c)
      for (int q = 0; q < 4; ++q)
        // (as CARRY_TOL: 1e-10 of an FP32 rounding of the values they multiply)
        if (std::fabs(row_of(p, q, c)) > 1e-17) pl.Wg = std::max(pl.Wg, std::abs(c / 4 - p));
  const int K = 2 * pl.Wg + 1;
  pl.g.assign((size_t)P * K * 16, 0.0f);
  for (int p = 0; p < P; ++p)
    for (int j = 0; j < K; ++j) {
      const int qc = p - pl.Wg + j;
      if (qc < 0 || qc >= P) continue;
      for (int i = 0; i < 4; ++i)
        for (int q = 0; q < 4; ++q) pl.g[(((size_t)p * K + j) * 4 + i) * 4 + q] = (float)row_of(p, q, 4 * qc + i);
    }
  return pl;
}

struct RefArgs {
  int N, P, mb, mx, nlines, nbytes;
  long long A, B, stride;
  int lines;
  int addv, epi;
  double scale, epi_c;
  double w[9];
  double bd[5];
  int Wg, vec;
  const float* cls;
  const float* g;
  const double* be;
  const double* bcoef;
  const int* bidx;
};

// A chunk has mb or mb + 1 rows, mb the same in all chunks of a line, so a
// group of four rows is skipped or taken as a whole by a wave-uniform test.
// Past a chunk's end the solve starts from zeros, and the zeros of its tables
// keep the rows there at 0 and out of the others.
constexpr int RGROUP = 4;

// --- right-hand side ------------------------------------------------------
// win[w] holds v[s - R + w]; rows of skipped groups get 0.
template <int KIND, typename TW>
PYR_HD void ref_rhs_interior(const RefArgs& a, const TW* win, double* rhs) {
  constexpr int R = Halo<KIND>::R;
#pragma unroll
  for (int g = 0; g < RCHUNK; g += RGROUP) {
    if (g <= a.mb) {
#pragma unroll
      for (int k = g; k < g + RGROUP; ++k) {
        double acc;
        if (KIND == K_D1) {
          // antisymmetric pairs (compact_d1.f90:156)
          acc = a.w[4] * ((double)win[k + R + 1] - (double)win[k + R - 1]) +
                a.w[5] * ((double)win[k + R + 2] - (double)win[k + R - 2]) +
                a.w[6] * ((double)win[k + R + 3] - (double)win[k + R - 3]);
        } else {
          // difference form sum_l w_l (v_{i+l} - v_i) (compact_r3.f90:124-132,
          // compact_r4.f90:144-156)
          const double vc = (double)win[k + R];
          acc = 0.0;
#pragma unroll
          for (int l = -R; l <= R; ++l)
            if (l != 0) acc += ((double)win[k + R + l] - vc) * a.w[l + R];
        }
        rhs[k] = acc;
      }
    } else {
#pragma unroll
      for (int k = g; k < g + RGROUP; ++k) rhs[k] = 0.0;
    }
  }
}

// One boundary row from its term list; rd(slot) returns the value of an end
// slot of this line. All MAXT terms are read (unused ones have no weight and
// read 0), so that their loads are independent of each other.
template <typename Reader>
PYR_HD double ref_boundary_row(const RefArgs& a, int slot, Reader rd) {
  double s = 0.0;
#pragma unroll
  for (int t = 0; t < MAXT; ++t) {
    const double c = a.bcoef[slot * MAXT + t];
    const double va = (double)rd(a.bidx[(slot * MAXT + t) * 2 + 0]);
    const double vb = (double)rd(a.bidx[(slot * MAXT + t) * 2 + 1]);
    s += c * (va - vb);
  }
  return s;
}

// Row of an end slot, and the slot's value given the line's rows.
template <typename Row>
PYR_HD float end_value(int slot, int N, Row row) {
  const int i = slot < ENDS / 2 ? slot : (slot < ENDS ? N - ENDS + slot : 0);
  const float v = row(i);
  return slot < ENDS ? v : 0.0f;
}

struct alignas(16) F4 { float x, y, z, w; };
struct alignas(8) F2 { float x, y; };

// Replace the rows of the line's ends by their own right-hand sides.
template <typename Reader>
PYR_HD void ref_rhs_boundary(const RefArgs& a, int p, double* rhs, Reader rd) {
  if (p == 0) {
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      PYR_ROW_FENCE(k, 1);
      rhs[k] = ref_boundary_row(a, k, rd);
    }
  }
  if (p == a.P - 1) {
    double g[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      PYR_ROW_FENCE(j, 1);
      g[j] = ref_boundary_row(a, NB + j, rd);
    }
    const double g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3];
#pragma unroll
    for (int k = NB; k < RCHUNK; ++k) {
      const int j = k - (a.mb - NB);  // the last chunk has mb rows in every line
      if (j >= 0 && j < NB) rhs[k] = (j == 0) ? g0 : (j == 1) ? g1 : (j == 2) ? g2 : g3;
    }
  }
}

// --- chunk solve ------------------------------------------------------------
// t: the table of this chunk's class; r: the right-hand sides, whose rows past
// the chunk's end (longer: it has mb + 1) are sums over part of their points and
// can overflow FP32 where no whole row does (constant fields above 5e36)
template <typename T>
PYR_HD void ref_local_solve(const RefArgs& a, bool longer, const float* t, const T* r, float* x) {
#pragma unroll
  for (int g = 0; g < RCHUNK; g += RGROUP) {
#pragma unroll
    for (int k = g; k < g + RGROUP; ++k) x[k] = g <= a.mb ? (float)r[k] : 0.0f;
    if (g <= a.mb) {
      if (a.mb < g + RGROUP) {
#pragma unroll
        for (int k = g; k < g + RGROUP; ++k) x[k] = k < a.mb || (k == a.mb && longer) ? x[k] : 0.0f;
      }
      PYR_ROW_FENCE(g, RGROUP);
#pragma unroll
      for (int k = g; k < g + RGROUP; ++k) {
        const F2 l = *reinterpret_cast<const F2*>(t + k * CROW + 8);
        float v = x[k];
        if (k >= 1) v -= l.y * x[k - 1];
        if (k >= 2) v -= l.x * x[k - 2];
        x[k] = v;
      }
    }
  }
#pragma unroll
  for (int g = RCHUNK - RGROUP; g >= 0; g -= RGROUP) {
    if (g <= a.mb) {
      PYR_ROW_FENCE(g, RGROUP);
#pragma unroll
      for (int k = g + RGROUP - 1; k >= g; --k) {
        const F4 u = *reinterpret_cast<const F4*>(t + k * CROW + 4);
        float v = x[k];
        if (k + 1 < RCHUNK) v -= u.y * x[k + 1];
        if (k + 2 < RCHUNK) v -= u.z * x[k + 2];
        x[k] = v * u.x;
      }
    }
  }
}

// The chunk's first two and last two values (longer: it has mb + 1 rows).
PYR_HD F4 ref_edges(const RefArgs& a, bool longer, const float* x) {
  float l0 = 0, l1 = 0, l2 = 0;  // rows mb - 2, mb - 1, mb
#pragma unroll
  for (int k = 2 * NB - 2; k < RCHUNK; ++k) {
    if (k == a.mb - 2) l0 = x[k];
    if (k == a.mb - 1) l1 = x[k];
    if (k == a.mb) l2 = x[k];
  }
  return F4{x[0], x[1], longer ? l1 : l0, longer ? l2 : l1};
}

// z = the four values next to chunk p: rows g of the reduced inverse times the
// edge values of the chunks within reach; yr(q) returns those of chunk q
template <typename YR>
PYR_HD void ref_neighbours(const RefArgs& a, const float* g, int p, YR yr, float* z) {
  const int K = 2 * a.Wg + 1;
  const F4* c = reinterpret_cast<const F4*>(g) + (size_t)p * K * 4;
  float z0 = 0, z1 = 0, z2 = 0, z3 = 0;
#pragma unroll 3
  for (int j = 0; j < K; ++j) {
    const int q = p - a.Wg + j;
    const F4 e = yr(q < 0 ? 0 : (q >= a.P ? a.P - 1 : q));
    const float y[4] = {e.x, e.y, e.z, e.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const F4 r = c[4 * j + i];
      z0 += r.x * y[i];
      z1 += r.y * y[i];
      z2 += r.z * y[i];
      z3 += r.w * y[i];
    }
  }
  z[0] = z0; z[1] = z1; z[2] = z2; z[3] = z3;
}

PYR_HD void ref_spike(const RefArgs& a, const float* t, const float* z, float* x) {
#pragma unroll
  for (int g = 0; g < RCHUNK; g += RGROUP) {
    if (g <= a.mb) {
      PYR_ROW_FENCE(g, RGROUP);
#pragma unroll
      for (int k = g; k < g + RGROUP; ++k) {
        const F4 r = *reinterpret_cast<const F4*>(t + k * CROW);
        x[k] -= r.x * z[0] + r.y * z[1] + r.z * z[2] + r.w * z[3];
      }
    }
  }
}

// d = the FP32 rounding of the FP64 residual rhs - A y of every row, with
// z = (y[s-2], y[s-1], y[e], y[e+1]) the values of y outside the chunk. The
// solve that follows drops what lands past the chunk's end.
PYR_HD void ref_residual(const RefArgs& a, int p, bool longer, const double* rhs, const float* y, const float* z,
                         float* d) {
  // rows m and m + 1 of y are the next chunk's
  const float z0 = z[0], z1 = z[1], z2 = z[2], z3 = z[3];
  const float n1 = longer ? z2 : z3;  // row mb + 1
  float ye[RCHUNK + 2];
#pragma unroll
  for (int k = 0; k < RCHUNK + 2; ++k) {
    const float v = k < RCHUNK ? y[k] : 0.0f;
    const float v0 = longer ? v : z2, v2 = longer ? z3 : v;
    ye[k] = k == a.mb ? v0 : (k == a.mb + 1 ? n1 : (k == a.mb + 2 ? v2 : v));
  }
  auto row = [&](const double* b, int k) {
    const double y0 = k >= 2 ? (double)ye[k >= 2 ? k - 2 : 0] : (k == 0 ? (double)z0 : (double)z1);
    const double y1 = k >= 1 ? (double)ye[k >= 1 ? k - 1 : 0] : (double)z1;
    return (float)(rhs[k] - (b[0] * y0 + b[1] * y1 + b[2] * (double)ye[k] + b[3] * (double)ye[k + 1] +
                             b[4] * (double)ye[k + 2]));
  };
#pragma unroll
  for (int g = 0; g < RCHUNK; g += RGROUP) {
    if (g <= a.mb) {
#pragma unroll
      for (int k = g; k < g + RGROUP; ++k) d[k] = row(a.bd, k);
    } else {
#pragma unroll
      for (int k = g; k < g + RGROUP; ++k) d[k] = 0.0f;
    }
  }
  if (p == 0) {
#pragma unroll
    for (int k = 0; k < NB; ++k) d[k] = row(a.be + 5 * k, k);
  }
  if (p == a.P - 1) {
#pragma unroll
    for (int k = NB; k < RCHUNK; ++k) {
      const int j = k - (a.mb - NB);
      if (j >= 0 && j < NB) d[k] = row(a.be + 5 * (NB + j), k);
    }
  }
}

}  // namespace pyr
