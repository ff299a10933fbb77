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
// VGPRs. FP32 fields are solved in FP64 as well: an FP64 FMA issues at the rate
// of an FP32 one on CDNA3/4, and one FP64 solve is less work than an FP32 solve
// refined with an FP64 residual (256^3 d8 y: 65 -> 33 us) and closer to exact.
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

// Everything a kernel needs about one operator/direction, passed by value.
struct LineArgs {
  int N, P, mb, mx;        // rows, chunks; chunk p has mb + (p < mx) rows
  int nlines, periodic;
  int nbytes;              // bytes of one field (buffer range of the y/z kernels)
  long long A, B, stride;  // y/z: line L starts at (L % A) + B*(L / A), rows `stride` apart
  int lines;               // lines per workgroup (y/z: a power of two)
  int addv, epi;
  double scale, epi_c;
  double w[4];             // interior right-hand side (rhs_interior)
  const double* wb;        // boundary rows of a bounded line
  double p1, p2;           // recurrence constants
  int W, kp;               // carry terms; carry matrices per term (1 or P)
  const double* kf;
  const double* kb;
  // bounded lines: row factors of the chunks p < tlo and p = P - 1
  const double* tf;
  const double* tb;
  const double* tg;
  int tlo;
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

// Replace the rows of a bounded line's ends by their own right-hand sides
// (p: this chunk; every chunk has at least 2*NB rows).
template <int KIND, bool FULL, typename TW>
PYR_HD void rhs_boundary(const LineArgs& a, const double* wb, int p, const TW* win, double* rhs) {
  constexpr int R = Halo<KIND>::R;
  if (p == 0) {
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      PYR_ROW_FENCE(k, 1);
      rhs[k] = boundary_row<KIND>(wb + k * WBROW, win + k + R);
    }
  }
  if (p == a.P - 1) {
    if constexpr (FULL) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        PYR_ROW_FENCE(j, 1);
        rhs[CHUNK - NB + j] = boundary_row<KIND>(wb + (NB + j) * WBROW, win + CHUNK - NB + j + R);
      }
    } else {
      // the last chunk has mb rows in every line: the row is wave-uniform
#pragma unroll
      for (int k = NB; k < CHUNK; ++k) {
        const int j = k - (a.mb - NB);
        if (j >= 0 && j < NB) rhs[k] = boundary_row<KIND>(wb + (NB + j) * WBROW, win + k + R);
      }
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
struct TableRows {
  const double* tf;
  const double* tb;
  const double* tg;
  int P, p;
  PYR_HD static void fence([[maybe_unused]] int k) { PYR_ROW_FENCE(k, 4); }
  struct alignas(16) D2 { double x, y; };
  // row k of chunk p as a uniform row address plus the chunk's 32-bit offset
  template <typename T>
  PYR_HD T row(const double* t, int k) const {
    const char* base = reinterpret_cast<const char*>(t) + (size_t)(unsigned)(k * P) * sizeof(T);
    return *reinterpret_cast<const T*>(base + (unsigned)p * (unsigned)sizeof(T));
  }
  PYR_HD void fwd(int k, double& c1, double& c2) const {
    const D2 t = row<D2>(tf, k);
    c1 = t.x; c2 = t.y;
  }
  PYR_HD void bwd(int k, double& c1, double& c2) const {
    const D2 t = row<D2>(tb, k);
    c1 = t.x; c2 = t.y;
  }
  PYR_HD double diag(int k, double x) const { return x * row<double>(tg, k); }
};

// Forward recurrence entered with (x_{-2}, x_{-1}) = (e0, e1), which becomes
// the exit state; STORE keeps the rows. The older state is subtracted first,
// so one FMA per row is on the dependent chain.
template <bool FULL, bool STORE, typename Rows>
PYR_HD void fwd_pass(const Rows& rows, double* x, int m, double& e0, double& e1) {
#pragma unroll
  for (int k = 0; k < CHUNK; ++k) {
    if (FULL || k < m) {
      double c1, c2;
      rows.fence(k);
      rows.fwd(k, c1, c2);
      const double t = x[k] - c2 * e0;
      const double v = t - c1 * e1;
      if (STORE) x[k] = v;
      e0 = e1;
      e1 = v;
    }
  }
}

// Diagonal and exit state of the backward recurrence entered with zeros; the
// rows are scaled by the diagonal in place.
template <bool FULL, typename Rows>
PYR_HD void bwd_exit(const Rows& rows, double* x, int m, double& b1, double& b2) {
#pragma unroll
  for (int k = CHUNK - 1; k >= 0; --k) {
    if (FULL || k < m) {
      double c1, c2;
      rows.fence(k);
      rows.bwd(k, c1, c2);
      x[k] = rows.diag(k, x[k]);
      const double t = x[k] - c2 * b2;
      const double v = t - c1 * b1;
      b2 = b1;
      b1 = v;
    }
  }
}

// Backward recurrence entered with (y_m, y_{m+1}) = (b1, b2); row k goes to
// sink(k, y_k).
template <bool FULL, typename Rows, typename Sink>
PYR_HD void bwd_sink(const Rows& rows, const double* x, int m, double b1, double b2, Sink sink) {
#pragma unroll
  for (int k = CHUNK - 1; k >= 0; --k) {
    if (FULL || k < m) {
      double c1, c2;
      rows.fence(k);
      rows.bwd(k, c1, c2);
      const double t = x[k] - c2 * b2;
      const double v = t - c1 * b1;
      b2 = b1;
      b1 = v;
      sink(k, v);
    }
  }
}

// Add one chunk's exit (u0, u1) to an entry state through its carry matrix.
PYR_HD void carry_add(const double* K, double u0, double u1, double& e0, double& e1) {
  e0 += K[0] * u0 + K[1] * u1;
  e1 += K[2] * u0 + K[3] * u1;
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
