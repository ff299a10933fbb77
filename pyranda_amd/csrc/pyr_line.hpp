// Per-thread arithmetic of the line-operator kernels, written once for the
// device and for the host emulation used by CPU tests.
//
// A thread owns one chunk (rows s..s+m-1, m <= CHUNK) of one line:
//   A  right-hand side of its rows from the register window; forward
//      recurrence from a zero state, whose exit state goes to the other chunks;
//   B  entry state from the exits of the chunks before it, the recurrence
//      proper, and the exit state of the backward one;
//   C  entry state from the chunks after it and the backward recurrence,
//      whose rows go straight to the epilogue.
// All array indices are compile-time after unrolling, so the chunk lives in
// VGPRs. Periodic lines of FP32 fields, and bounded ones in the FP64 solve mode,
// are solved in FP64 as well: an FP64 FMA issues at the rate of an FP32 one on
// CDNA3/4, and one FP64 solve is less work than an FP32 solve refined with an
// FP64 residual (256^3 d8 y: 65 -> 33 us) and closer to exact. Bounded FP32 lines
// in the default mode take that refined solve (pyr_refined.hpp).
#pragma once

#include "pyr_plan.hpp"

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define PYR_HD __host__ __device__ __forceinline__
#else
#define PYR_HD inline
#endif

// Keeps the table reads of one group of rows from being hoisted over the rows
// before it: with a whole chunk's factors in flight the kernels that read them
// spill (bounded FP64 y lines: 180 bytes a lane).
#if defined(__HIP_DEVICE_COMPILE__)
#define PYR_ROW_FENCE(k, every) \
  do {                          \
    if ((k) % (every) == 0) asm volatile("" ::: "memory"); \
  } while (0)
#else
#define PYR_ROW_FENCE(k, every) (void)0
#endif

namespace pyr {

enum Epi { EPI_STORE = 0, EPI_ADD = 1, EPI_ABS = 2, EPI_MAXABS = 3 };
PYR_HD bool reads_out(int epi) { return epi == EPI_ADD || epi == EPI_MAXABS; }

// Everything a kernel needs about one operator/direction, passed by value.
struct LineArgs {
  int N, P, mb, mx;        // rows, chunks; chunk p has mb + (p < mx) rows
  int nlines, periodic;
  int nbytes;              // bytes of one field (buffer range of the y/z kernels)
  long long A, B, stride;  // y/z: line L starts at (L % A) + B*(L / A), rows `stride` apart
  int lines;               // lines per workgroup (y/z: a power of two)
  int addv, epi;
  double scale, epi_c;
  double w[4];             // interior right-hand side (rhs_interior, rhs_explicit)
  double p1, p2;           // recurrence constants
  int W;                   // chunks that enter a carry
  double hf[2][4], hb[2][4];  // H of constant chunks of mb + 1 and mb rows
  int turns;               // cyclic lines: the turns beyond the first matter
  double tf[4], tb[4];     // their sum, (I - H of the line)^-1, forward and backward
  // bounded lines: the tables of T slots (OpPlan::tab), then the boundary rows
  const double* tab;
  int tlo, T, ntab;
  int vec;                 // x lines: the pointers allow 16-byte accesses
  // FP64 sweeps with the store epilogue: when set, every stored value is also
  // written here rounded to FP32 (same element index as the output); with
  // only32 the FP64 result itself is not stored
  float* out32;
  int only32;
};

PYR_HD int chunk_start(const LineArgs& a, int p) { return p * a.mb + (p < a.mx ? p : a.mx); }

template <int KIND> struct Halo { static constexpr int R = (KIND == K_R4) ? 4 : 3; };

// --- right-hand side ------------------------------------------------------
// win[w] holds v[s - R + w].
template <int KIND, typename TW>
PYR_HD void rhs_interior(const LineArgs& a, const TW* win, double* rhs) {
  constexpr int R = Halo<KIND>::R;
  if constexpr (KIND == K_D1) {
    // antisymmetric pairs (compact_d1.f90:156)
#pragma unroll
    for (int k = 0; k < CHUNK; ++k)
      rhs[k] = a.w[0] * ((double)win[k + R + 1] - (double)win[k + R - 1]) +
               a.w[1] * ((double)win[k + R + 2] - (double)win[k + R - 2]) +
               a.w[2] * ((double)win[k + R + 3] - (double)win[k + R - 3]);
  } else {
    // sum_l w_l (v_{i+l} - v_i) (compact_r3.f90:124-132, compact_r4.f90:
    // 144-156) of a symmetric row through first differences, which
    // neighbouring rows share: 2R + 1 operations a row instead of 4R
    double d[2 * R];  // d[q]: v_{i-R+q+1} - v_{i-R+q}
#pragma unroll
    for (int q = 0; q < 2 * R - 1; ++q) d[q + 1] = (double)win[q + 1] - (double)win[q];
#pragma unroll
    for (int k = 0; k < CHUNK; ++k) {
#pragma unroll
      for (int q = 0; q < 2 * R - 1; ++q) d[q] = d[q + 1];
      d[2 * R - 1] = (double)win[k + 2 * R] - (double)win[k + 2 * R - 1];
      double acc = a.w[R - 1] * (d[2 * R - 1] - d[0]);
#pragma unroll
      for (int q = R - 2; q >= 0; --q) acc += a.w[q] * (d[R + q] - d[R - 1 - q]);
      rhs[k] = acc;
    }
  }
}

// The explicit filter's rows, sum_l w_l (v_{i+l} - v_i) as it stands: first
// differences of an infinity hold both signs of it and give NaN for neighbours
// whose value is that infinity. Those are fewer operations (y sweep of 256^3 in
// FP32 25.9 us against 26.4, bounded x sweep of 1000x301x53 35.3 against 39.0,
// with the end rows below), but a second look at rows that are not finite costs
// more than it saves (29.6 us for the first).
template <typename TW>
PYR_HD void rhs_explicit(const LineArgs& a, const TW* win, double* rhs) {
  constexpr int R = Halo<K_R4>::R;
#pragma unroll
  for (int k = 0; k < CHUNK; ++k) {
    const double vc = (double)win[k + R];
    double acc = 0.0;
#pragma unroll
    for (int l = -R; l <= R; ++l)
      if (l != 0) acc += a.w[(l < 0 ? -l : l) - 1] * ((double)win[k + R + l] - vc);
    rhs[k] = acc;
  }
}

// One boundary row: c points at its weights, v at the row itself in the window.
template <int KIND, typename TW>
PYR_HD double boundary_row(const double* c, const TW* v) {
  constexpr int R = Halo<KIND>::R;
  const double vc = (double)v[0];
  double acc = c[WBROW - 1] * vc;
#pragma unroll
  for (int l = -R; l <= R; ++l)
    if (l != 0) acc += c[l + 4] * ((double)v[l] - vc);
  return acc;
}

// ... of the explicit filter, `in` rows from the line's end, which lies at
// offset -in (SIDE -1) or in (+1) and has the value e: sum_l c_l (v_{i+l} - e),
// or sum_l c_l v_{i+l} where the last weight is not 0 (compact_r4.f90:106-207).
// Points that are not in the sum are left out and not multiplied by 0: e may be
// infinite.
template <int SIDE, typename TW>
PYR_HD double explicit_row(const double* c, const TW* v, int in, double e) {
  constexpr int R = Halo<K_R4>::R;
  const bool plain = c[WBROW - 1] != 0.0;
  if (plain) e = 0.0;
  double acc = 0.0;
#pragma unroll
  for (int l = -R; l <= R; ++l) {
    const int to_end = SIDE * l;  // rows towards the end
    if (to_end > NB - 1) continue;
    const double t = (double)v[l] - e;
    if (to_end < 0) acc += c[l + 4] * t;
    else acc += c[l + 4] * (to_end < in || (to_end == in && plain) ? t : 0.0);
  }
  return acc;
}

struct B4 { double a, b, c, d; };  // four values, never indexed at run time

// The right-hand sides of a bounded line's end rows: into lo by the first
// chunk, into hi by the last one (p: this chunk; every chunk has at least 2*NB
// rows, the last one mb of them in every line). Taken before the interior rows,
// while the window is all that is in registers.
template <int KIND, bool EXPLICIT, bool FULL, typename TW>
PYR_HD void boundary_rows(const LineArgs& a, const double* wb, int p, const TW* win, B4& lo, B4& hi) {
  constexpr int R = Halo<KIND>::R;
  if (p == 0) {
    [[maybe_unused]] const double e = (double)win[R];
    auto row = [&](int k) {
      PYR_ROW_FENCE(0, 1);
      if constexpr (EXPLICIT) return explicit_row<-1>(wb + k * WBROW, win + k + R, k, e);
      else return boundary_row<KIND>(wb + k * WBROW, win + k + R);
    };
    lo.a = row(0);
    lo.b = row(1);
    lo.c = row(2);
    lo.d = row(3);
  }
  if (p == a.P - 1) {
    [[maybe_unused]] double e = (double)win[CHUNK - 1 + R];
    if (EXPLICIT && !FULL) {
#pragma unroll
      for (int k = 2 * NB - 1; k < CHUNK; ++k) e = k == a.mb - 1 ? (double)win[k + R] : e;
    }
#pragma unroll
    for (int k = FULL ? CHUNK - NB : NB; k < CHUNK; ++k) {
      const int j = k - ((FULL ? CHUNK : a.mb) - NB);
      if (j >= 0 && j < NB) {
        PYR_ROW_FENCE(k, 1);
        double v;
        if constexpr (EXPLICIT) v = explicit_row<1>(wb + (NB + j) * WBROW, win + k + R, NB - 1 - j, e);
        else v = boundary_row<KIND>(wb + (NB + j) * WBROW, win + k + R);
        hi.a = j == 0 ? v : hi.a;
        hi.b = j == 1 ? v : hi.b;
        hi.c = j == 2 ? v : hi.c;
        hi.d = j == 3 ? v : hi.d;
      }
    }
  }
}
// ... and into their rows of the chunk
template <bool FULL>
PYR_HD void put_boundary_rows(const LineArgs& a, int p, const B4& lo, const B4& hi, double* rhs) {
  rhs[0] = p == 0 ? lo.a : rhs[0];
  rhs[1] = p == 0 ? lo.b : rhs[1];
  rhs[2] = p == 0 ? lo.c : rhs[2];
  rhs[3] = p == 0 ? lo.d : rhs[3];
  const double h0 = hi.a, h1 = hi.b, h2 = hi.c, h3 = hi.d;
#pragma unroll
  for (int k = FULL ? CHUNK - NB : NB; k < CHUNK; ++k) {
    const int j = k - ((FULL ? CHUNK : a.mb) - NB);
    if (j >= 0 && j < NB) {
      const double v = j == 0 ? h0 : j == 1 ? h1 : j == 2 ? h2 : h3;
      rhs[k] = p == a.P - 1 ? v : rhs[k];
    }
  }
}

// --- recurrences ------------------------------------------------------------
// Coefficients of row k of the chunk: the constants, or the line's own factors.
struct ConstRows {
  double p1, p2;
  PYR_HD static void fence(int) {}
  PYR_HD void fwd(int, double& c1, double& c2) const { c1 = p1; c2 = p2; }
  PYR_HD void bwd(int, double& c1, double& c2) const { c1 = p1; c2 = p2; }
  PYR_HD double diag(int, double x) const { return x; }
};

// Where the parts of a bounded line's tables sit (in LDS on the device).
struct Tables {
  const double *tf, *tb, *tg, *th, *wb;
  PYR_HD Tables(const double* t, int T)
      : tf(t), tb(t + 2 * CHUNK * T), tg(t + 4 * CHUNK * T), th(t + 5 * CHUNK * T), wb(t + 5 * CHUNK * T + 8 * T) {}
};
// table slot of chunk p
PYR_HD int slot_of(const LineArgs& a, int p) {
  if (p == a.P - 1) return a.T - 1;
  return p < a.tlo ? p : a.tlo + (p < a.mx ? 0 : 1);
}
struct TableRows {
  Tables t;
  int T, slot;
  PYR_HD static void fence([[maybe_unused]] int k) { PYR_ROW_FENCE(k, 4); }
  PYR_HD void fwd(int k, double& c1, double& c2) const {
    const double* e = t.tf + 2 * (k * T + slot);
    c1 = e[0]; c2 = e[1];
  }
  PYR_HD void bwd(int k, double& c1, double& c2) const {
    const double* e = t.tb + 2 * (k * T + slot);
    c1 = e[0]; c2 = e[1];
  }
  PYR_HD double diag(int k, double x) const { return x * t.tg[k * T + slot]; }
};

// Which rows a chunk has: mb of them, the same in every chunk of the line (so
// the test is wave-uniform), and one more where `longer`. Every chunk has at
// least 2*NB rows.
struct ChunkRows {
  int mb;
  bool longer;
  template <typename F>
  PYR_HD void row(int k, F f) const {
    if (k < 2 * NB || k < mb) f();
    else if (k == mb && longer) f();
  }
};
struct AllRows {
  template <typename F>
  PYR_HD void row(int, F f) const { f(); }
};

// Forward recurrence entered with (x_{-2}, x_{-1}) = (e0, e1), which becomes
// the exit state; STORE keeps the rows. The older state is subtracted first,
// so one FMA per row is on the dependent chain.
template <bool STORE, typename Have, typename Rows>
PYR_HD void fwd_pass(const Have& have, const Rows& rows, double* x, double& e0, double& e1) {
#pragma unroll
  for (int k = 0; k < CHUNK; ++k) {
    have.row(k, [&] {
      double c1, c2;
      rows.fence(k);
      rows.fwd(k, c1, c2);
      const double t = x[k] - c2 * e0;
      const double v = t - c1 * e1;
      if (STORE) x[k] = v;
      e0 = e1;
      e1 = v;
    });
  }
}

// Diagonal and exit state of the backward recurrence entered with zeros; the
// rows are scaled by the diagonal in place.
template <typename Have, typename Rows>
PYR_HD void bwd_exit(const Have& have, const Rows& rows, double* x, double& b1, double& b2) {
#pragma unroll
  for (int k = CHUNK - 1; k >= 0; --k) {
    have.row(k, [&] {
      double c1, c2;
      rows.fence(k);
      rows.bwd(k, c1, c2);
      x[k] = rows.diag(k, x[k]);
      const double t = x[k] - c2 * b2;
      const double v = t - c1 * b1;
      b2 = b1;
      b1 = v;
    });
  }
}

// Backward recurrence entered with (y_m, y_{m+1}) = (b1, b2); row k goes to
// sink(k, y_k).
template <typename Have, typename Rows, typename Sink>
PYR_HD void bwd_sink(const Have& have, const Rows& rows, const double* x, double b1, double b2, Sink sink) {
#pragma unroll
  for (int k = CHUNK - 1; k >= 0; --k) {
    have.row(k, [&] {
      double c1, c2;
      rows.fence(k);
      rows.bwd(k, c1, c2);
      const double t = x[k] - c2 * b2;
      const double v = t - c1 * b1;
      b2 = b1;
      b1 = v;
      sink(k, v);
    });
  }
}

// Entry state of chunk p from the exits of the W chunks on its near side
// (STEP -1: forward, from p-W up to p-1; +1: backward, from p+W down to p+1):
// E <- H_q E + e_q. exit_of(q, u0, u1) reads chunk q's exit, h(q) its matrix.
// Beyond the ends of a bounded line nothing enters.
template <bool CYCLIC, int STEP, typename H, typename ExitOf>
PYR_HD void carry_in(const LineArgs& a, int p, H h, ExitOf exit_of, double& e0, double& e1) {
  e0 = e1 = 0.0;
  int q = p + STEP * a.W;
  if (CYCLIC) q = q < 0 ? q + a.P : (q >= a.P ? q - a.P : q);
#pragma unroll 2
  for (int j = 0; j < a.W; ++j) {
    const bool in = CYCLIC || (q >= 0 && q < a.P);
    const int qq = in ? q : p;
    double u0, u1;
    exit_of(qq, u0, u1);
    const double* m = h(qq);
    const double s0 = (in ? u0 : 0.0) + m[1] * e1;
    const double s1 = (in ? u1 : 0.0) + m[3] * e1;
    e1 = s1 + m[2] * e0;
    e0 = s0 + m[0] * e0;
    q -= STEP;
    if (CYCLIC) q = q < 0 ? a.P - 1 : (q >= a.P ? 0 : q);
  }
  if (CYCLIC && a.turns) {
    const double* m = STEP > 0 ? a.tb : a.tf;
    const double t0 = m[0] * e0 + m[1] * e1;
    e1 = m[2] * e0 + m[3] * e1;
    e0 = t0;
  }
}

template <typename TS>
PYR_HD TS epilogue(int epi, double c, double val, TS old) {
  switch (epi) {
    case EPI_ADD: return (TS)((double)old + val);
    case EPI_ABS: return (TS)(fabs(val) * c);
    case EPI_MAXABS: {
      const double t = fabs(val) * c;
      const double o = (double)old;
      return (TS)(o > t ? o : t);
    }
    default: return (TS)val;
  }
}

}  // namespace pyr
