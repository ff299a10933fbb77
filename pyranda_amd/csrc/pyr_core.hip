// MI355X (gfx950) kernels and C-ABI of the compact finite-difference core.
//
// One launch applies one compact operator along one direction to a whole
// (nx,ny,nz) field. Each thread owns one chunk of one line (pyr_plan.hpp):
//   y/z lines: lanes of a wave are adjacent lines, i.e. adjacent x, so every
//     row load/store of a wave is made of 128-512 B segments; the chunks of a
//     line are in one workgroup and exchange their carries through LDS;
//   x lines:   a wave owns a few whole lines, moves them through its own LDS
//     tile with 16-byte accesses, and needs no workgroup barrier at all.
// Every field element is read once and written once from HBM.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/pyranda_amd.h"
#include "pyr_line.hpp"
#include "pyr_refined.hpp"

using namespace pyr;

// ---------------------------------------------------------------------------
// error reporting
// ---------------------------------------------------------------------------
// The file compiles as several translation units that build in parallel:
// PYR_PART 0 holds the host code and the C-ABI, the others the line kernels
// (1, 2: periodic lines of FP64 and FP32 fields; 3, 4: bounded lines and the
// explicit filter; 5, 6: grouped launches; 7: the refined FP32 solve) through
// explicit instantiations of the launch functions.
#ifndef PYR_PART
#define PYR_PART 0
#endif
#if PYR_PART == 0
static thread_local std::string g_err;
static int fail(const std::string& m) {
  g_err = m;
  return 1;
}
namespace pyr {
// errors of the other translation units (pyr_mlp.hip, the kernel parts) go
// to pyr_last_error too
int report_error(const std::string& m) { return fail(m); }
}  // namespace pyr
#else
namespace pyr {
int report_error(const std::string& m);
}  // namespace pyr
static int fail(const std::string& m) { return pyr::report_error(m); }
#endif
#define HIPCHECK(x)                                                              \
  do {                                                                           \
    hipError_t e_ = (x);                                                         \
    if (e_ != hipSuccess) return fail(std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
enum Solve { SOLVE_NONE = 0, SOLVE_BND = 1, SOLVE_CIRC = 2 };

template <int KIND, int SOLVE, typename TW>
PYR_HD void right_hand_side(const LineArgs& a, const TW* win, double* rhs) {
  if constexpr (SOLVE == SOLVE_NONE) rhs_explicit(a, win, rhs);
  else rhs_interior<KIND>(a, win, rhs);
}

// What a y/z row's epilogue does and needs besides the solution, in registers
// before the backward pass so that no store waits on a load: store it
// (PRE_NONE), add the input back and store (PRE_V, filters), or join the
// current output (PRE_OLD: the maximum for the r4 kind's ring, the sum for the
// others). These are the composites' own sweeps, with nothing to decide per
// row: the branches over the epilogue and the FP32 copy, taken for each of the
// 16 rows, had cut the backward pass and its stores into pieces (256^3 FP64
// gradient 165 -> 155 us, filter 145 -> 137, FP32 ring 102 -> 98; bounded
// Laplacian on 192^3 118 -> 112). PRE_ANY takes every other epilogue and the
// FP32 copy, read from the arguments row by row.
enum Pre { PRE_NONE = 0, PRE_V = 1, PRE_OLD = 2, PRE_ANY = 3 };
constexpr int joined_epi(int kind) { return kind == K_R4 ? EPI_MAXABS : EPI_ADD; }
static int pre_of(int kind, bool addv, int epi, bool out32) {
  if (epi == EPI_STORE && !out32) return addv ? PRE_V : PRE_NONE;
  return !addv && epi == joined_epi(kind) ? PRE_OLD : PRE_ANY;
}

constexpr int WG_MAX = 1024;

// Raw buffer access to one field: the lane part of an address sits in a VGPR
// and the row part (uniform across the wave) in an SGPR, so no per-row 64-bit
// address is formed, and an access at OOB reads 0 or stores nothing without a
// branch. Fields are below 2 GiB (at most 512^3 FP64). dword3 0x00020000:
// 32-bit data format, the raw (untyped) configuration of gfx9-family buffer
// descriptors.
constexpr int BUF_DWORD3 = 0x00020000;
constexpr int OOB = (int)0x80000000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* p, int nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, nbytes, BUF_DWORD3);
}
__device__ __forceinline__ double buf_load(double, __amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ float buf_load(float, __amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ void buf_store(double v, __amdgpu_buffer_rsrc_t r, int voff, int soff) {
  using U2 = unsigned int __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, voff, soff, 0);
}
__device__ __forceinline__ void buf_store(float v, __amdgpu_buffer_rsrc_t r, int voff, int soff) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, voff, soff, 0);
}

// A pair of FP64 values moved as one 16-byte LDS or global access.
using D2 = double __attribute__((ext_vector_type(2)));

// The chunks of one wave that need the line's own factors (the wave then
// takes them for all of its chunks: converged rows give the same bits).
__device__ __forceinline__ bool wave_needs_tables(const LineArgs& a, int p) {
  return __ballot(p < a.tlo || p == a.P - 1) != 0;
}

template <bool FULL>
__device__ __forceinline__ auto rows_of_chunk(const LineArgs& a, int p) {
  if constexpr (FULL) return AllRows{};
  else return ChunkRows{a.mb, p < a.mx};
}

// The passes of one chunk around its two exchanges. `rows` are ConstRows or
// TableRows; the bounded solve picks one per wave.
template <int SOLVE, typename F>
__device__ __forceinline__ void with_rows(const LineArgs& a, bool tab, const Tables& t, int slot, F f) {
  if (SOLVE == SOLVE_BND && tab) f(TableRows{t, a.T, slot});
  else f(ConstRows{a.p1, a.p2});
}

// Carry of chunk p. Periodic lines: constant matrices from the kernel
// arguments (FULL lines have chunks of one length); bounded lines: the table's.
template <int SOLVE, bool FULL, int STEP, typename ExitOf>
__device__ __forceinline__ void carry_of(const LineArgs& a, const Tables& t, int p, ExitOf exit_of, double& e0,
                                         double& e1) {
  auto read = [&](int q, double& u0, double& u1) {
    const D2 u = exit_of(q);
    u0 = u.x;
    u1 = u.y;
  };
  if constexpr (SOLVE == SOLVE_BND) {
    carry_in<false, STEP>(a, p, [&](int q) { return t.th + 8 * slot_of(a, q) + (STEP > 0 ? 4 : 0); }, read, e0, e1);
  } else {
    const double(*h)[4] = STEP < 0 ? a.hf : a.hb;
    if constexpr (FULL) {
      carry_in<true, STEP>(a, p, [&](int) { return h[1]; }, read, e0, e1);
    } else {
      double m[4];
      carry_in<true, STEP>(a, p, [&](int q) {
        const bool longer = q < a.mx;
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = longer ? h[0][i] : h[1][i];
        return (const double*)m;
      }, read, e0, e1);
    }
  }
}

// The work item of this workgroup when neighbouring items share cache lines:
// consecutive workgroups start on the 8 XCDs in turn, each with an L2 of its
// own, so each XCD takes a run of consecutive items. A refined y/z group of
// 256 threads is 8 lines of 32 chunks, 32-byte rows of the same 128-byte lines
// as three neighbours': in an ensemble of 24 members (3.7M points) d1 30.2 ->
// 27.2 us, the filter 44.3 -> 35.4, the ring's maximum 40.2 -> 34.2.
// The explicit filter's groups along a line share halo rows, of which each XCD
// fetched its own copy (20% more bytes at 256^3 in FP64): y sweep 47.0 -> 44.8
// us, 1000x301x53 in FP32 94.3 -> 89.5 us for the three sweeps.
__device__ __forceinline__ int xcd_order() {
  const int n = (int)gridDim.x, b = (int)blockIdx.x, x = b & 7, q = n >> 3, r = n & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// First element of y/z line L (the last line for L past it): 32-bit division,
// the lines and elements of a field are fewer than 2^28.
template <typename Args>
__device__ __forceinline__ int line_offset(const Args& a, int L) {
  const unsigned l = (unsigned)(L < a.nlines ? L : a.nlines - 1), n = (unsigned)a.A;
  const unsigned q = l / n;
  return (int)(l - q * n + (unsigned)a.B * q);
}

// The tables of a bounded line into LDS: they are read row by row in the
// solves' passes, each read a latency on the critical path of a workgroup
// (from memory, the 2-D and ragged bounded sweeps took 28-36 us for fields
// of a few MB).
__device__ __forceinline__ void stage_tables(const LineArgs& a, double* tab) {
  for (int e = threadIdx.x; e < a.ntab / 2; e += blockDim.x)
    reinterpret_cast<D2*>(tab)[e] = reinterpret_cast<const D2*>(a.tab)[e];
}

// y/z lines. Thread (lane, p): line blk * lines + lane, chunk p; a.lines
// (a power of two) adjacent lines per workgroup. Bound by HBM: 16 rows a
// thread keep the kernel at 75-110 VGPRs, so that the load, solve and store
// phases of two or more workgroups overlap on a CU.
// FULL: every chunk has CHUNK rows (N a multiple of CHUNK), so the row
// predicates vanish at compile time.
// GRP: a workgroup shaped for other members of a grouped launch; threads
// without a chunk only take the barriers.
// The body takes the workgroup's line-group index `blk` (blockIdx.x for one
// field, the member-local index for a grouped launch over several fields).
template <typename TS, int KIND, int SOLVE, bool FULL, int PRE, bool GRP = false>
__device__ __forceinline__ void line_yz_body(const LineArgs& a, int blk, const TS* __restrict__ in,
                                             TS* __restrict__ out) {
  constexpr int R = Halo<KIND>::R;
  extern __shared__ __align__(16) unsigned char smem[];
  const int LY = a.lines;
  const int lane = threadIdx.x & (LY - 1);
  int p = (int)threadIdx.x >> __builtin_ctz(LY);
  if constexpr (SOLVE == SOLVE_NONE) {
    // chunks of the explicit filter are independent: a workgroup takes some of
    // a line group's chunks
    const int per = (int)blockDim.x >> __builtin_ctz(LY), groups = (a.P + per - 1) / per;
    p += (int)((unsigned)blk % (unsigned)groups) * per;
    blk = (int)((unsigned)blk / (unsigned)groups);
  }
  const bool act = (!GRP && SOLVE != SOLVE_NONE) || p < a.P;
  const int L = blk * LY + lane;
  const bool valid = act && L < a.nlines;
  const int lane_off = line_offset(a, L) * (int)sizeof(TS);
  const int rb = (int)(a.stride * (long long)sizeof(TS));
  const int s = FULL ? p * CHUNK : chunk_start(a, p);
  const int m = FULL ? CHUNK : a.mb + (p < a.mx ? 1 : 0);
  const auto have = rows_of_chunk<FULL>(a, p);
  const bool last = p == a.P - 1;
  const bool wrap = SOLVE == SOLVE_CIRC || (SOLVE == SOLVE_NONE && a.periodic);
  const bool bounded = SOLVE == SOLVE_BND || (SOLVE == SOLVE_NONE && !a.periodic);
  // LDS: two exchange buffers, a flag per line, the tables of a bounded line
  const int nex = SOLVE == SOLVE_NONE ? 0 : (GRP ? (int)blockDim.x : a.P * LY);
  D2* X0 = reinterpret_cast<D2*>(smem);
  D2* X1 = X0 + nex;
  double* tab = reinterpret_cast<double*>(X1 + nex);
  int* bad = reinterpret_cast<int*>(tab + (bounded ? a.ntab : 0));
  const Tables tabs(tab, a.T);
  if (bounded) stage_tables(a, tab);
  const __amdgpu_buffer_rsrc_t rin = buf_rsrc(in, a.nbytes), rout = buf_rsrc(out, a.nbytes);
  // the FP32 copy of an FP64 result (LineArgs::out32), half the bytes per element
  [[maybe_unused]] const __amdgpu_buffer_rsrc_t rout32 = buf_rsrc(a.out32, a.nbytes / 2);
  // rows s .. s+m-1; the halo rows wrap around a periodic line and are 0
  // beyond the ends of a bounded one
  const int vmid = act ? lane_off + s * rb : OOB;
  const int vlo = !act ? OOB : (p > 0 ? vmid - R * rb : (wrap ? lane_off + (a.N - R) * rb : OOB));
  const int vhi = !act ? OOB : (!last ? vmid + CHUNK * rb : (wrap ? lane_off : OOB));  // FULL only
  auto row_off = [&](int k) { return (int)((unsigned)vmid + (unsigned)k * (unsigned)rb); };
  TS pre[PRE == PRE_OLD ? CHUNK : 1];
  TS win[CHUNK + 2 * R];
#pragma unroll
  for (int w = 0; w < CHUNK + 2 * R; ++w) {
    const int k = w - R;
    if (w < R) {
      win[w] = buf_load(TS(), rin, vlo, w * rb);
    } else if (FULL) {
      win[w] = k < CHUNK ? buf_load(TS(), rin, vmid, k * rb)
                         : buf_load(TS(), rin, vhi, (k - CHUNK) * rb);
    } else if (k < 2 * NB) {  // every chunk has 2 NB rows
      win[w] = buf_load(TS(), rin, vmid, k * rb);
    } else {
      const bool over = s + k >= a.N;
      int off = over ? (wrap ? lane_off + (s + k - a.N) * rb : OOB) : row_off(k);
      if (!act || k >= m + R) off = OOB;
      win[w] = buf_load(TS(), rin, off, 0);
    }
  }
  double x[CHUNK];
  B4 lo = {}, hi = {};
  if (bounded) {
    __syncthreads();  // tables visible
    if (act) boundary_rows<KIND, SOLVE == SOLVE_NONE, FULL>(a, tabs.wb, p, win, lo, hi);
  }
  right_hand_side<KIND, SOLVE>(a, win, x);
  if (bounded) put_boundary_rows<FULL>(a, p, lo, hi, x);

  // row k of the result: metric scale, filters add v back, fused epilogue, store
  auto emit = [&](int k, double y) {
    double val = y * a.scale;
    if constexpr (PRE == PRE_V) val += (double)win[k + R];
    const int off = FULL ? vmid : row_off(k);
    const int soff = FULL ? k * rb : 0;
    if constexpr (PRE == PRE_ANY) {
      if (KIND == K_R4 && a.addv) val += (double)win[k + R];
      const TS old = reads_out(a.epi) ? buf_load(TS(), rout, off, soff) : (TS)0;
      const TS r = epilogue<TS>(a.epi, a.epi_c, val, old);
      if (sizeof(TS) != 8 || GRP || !a.only32) buf_store(r, rout, off, soff);
      if constexpr (sizeof(TS) == 8 && !GRP)
        if (a.out32) buf_store((float)r, rout32, off / 2, soff / 2);
    } else if constexpr (PRE == PRE_OLD) {
      buf_store(epilogue<TS>(joined_epi(KIND), a.epi_c, val, pre[k]), rout, off, soff);
    } else {
      buf_store((TS)val, rout, off, soff);
    }
  };
  if constexpr (SOLVE == SOLVE_NONE) {
    if (!valid) return;
#pragma unroll
    for (int k = 0; k < CHUNK; ++k) have.row(k, [&] { emit(k, x[k]); });
  } else {
    const bool own = SOLVE == SOLVE_BND && wave_needs_tables(a, p);
    const int slot = SOLVE == SOLVE_BND ? slot_of(a, p) : 0;
    if (p == 0) bad[lane] = 0;
    double e0 = 0.0, e1 = 0.0;
    if (act) {
      with_rows<SOLVE>(a, own, tabs, slot, [&](auto rows) { fwd_pass<false>(have, rows, x, e0, e1); });
      X0[p * LY + lane] = D2{e0, e1};
    }
    __syncthreads();
    // the current output, on its way while the recurrences run (the window's
    // registers are free by now)
    if constexpr (PRE == PRE_OLD) {
#pragma unroll
      for (int k = 0; k < CHUNK; ++k)
        if (FULL || k <= a.mb)
          pre[k] = FULL ? buf_load(TS(), rout, vmid, k * rb) : buf_load(TS(), rout, k < m ? row_off(k) : OOB, 0);
    }
    double b0 = 0.0, b1 = 0.0;
    if (act) {
      carry_of<SOLVE, FULL, -1>(a, tabs, p, [&](int q) { return X0[q * LY + lane]; }, e0, e1);
      with_rows<SOLVE>(a, own, tabs, slot, [&](auto rows) {
        fwd_pass<true>(have, rows, x, e0, e1);
        bwd_exit(have, rows, x, b0, b1);
      });
      X1[p * LY + lane] = D2{b0, b1};
      // a NaN or infinity anywhere in a line spreads to all of it, as it does
      // through a whole-line sweep; the truncated carries alone would not
      // take it further than W chunks
      if (!__builtin_isfinite(b0) || !__builtin_isfinite(b1)) bad[lane] = 1;
    }
    __syncthreads();
    if (!act) return;
    carry_of<SOLVE, FULL, 1>(a, tabs, p, [&](int q) { return X1[q * LY + lane]; }, b0, b1);
    if (bad[lane]) b0 = b1 = __builtin_nan("");
    if (!valid) return;
    with_rows<SOLVE>(a, own, tabs, slot, [&](auto rows) { bwd_sink(have, rows, x, b0, b1, emit); });
  }
}

template <typename TS, int KIND, int SOLVE, bool FULL, int PRE>
__global__ void __launch_bounds__(WG_MAX) k_line_yz(LineArgs a, const TS* __restrict__ in, TS* __restrict__ out) {
  line_yz_body<TS, KIND, SOLVE, FULL, PRE>(a, SOLVE == SOLVE_NONE ? xcd_order() : (int)blockIdx.x, in, out);
}

// 16-byte vector of the storage type
template <typename TS> struct Vec16;
template <> struct Vec16<double> { using type = double __attribute__((ext_vector_type(2))); static constexpr int W = 2; };
template <> struct Vec16<float> { using type = float __attribute__((ext_vector_type(4))); static constexpr int W = 4; };

// Orders the LDS accesses of one wave: its own reads and writes reach LDS in
// program order, so only the compiler has to be held back.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Moves the lines of one wave between HBM and its LDS tile. `end` elements
// from src on (element 0 is the first of the 16-byte vector that holds the
// lines' first element, `sh` the offset of that element in it); CH rows per
// chunk, at most 64 chunks. One extra vector after every CH elements of the
// tile spreads the lanes' reads, a chunk apart, over the banks (without it 16
// lanes share one bank; gbar on 1000-point FP32 lines 53 -> 41 us). Elements
// from -CH on may be addressed and, past the lines, 2 CH more: a window can be
// read whole where part of it is not used.
template <typename TS, int CH>
struct XTile {
  using V = typename Vec16<TS>::type;
  static constexpr int VW = Vec16<TS>::W;
  static constexpr int CP = CH + VW;                 // tile elements per chunk
  static constexpr int ORIGIN = CP;
  static constexpr int SIZE = 64 * CP + 4 * CP;
  static __device__ __forceinline__ int at(int i) { return i + (i >= 0 ? i / CH : -1) * VW; }

  // Positions of elements i0, i0 + 1, ... for compile-time steps w < 2 CH: a
  // run of CH elements crosses one boundary, which a comparison finds.
  struct Run {
    int b0, f;
    __device__ __forceinline__ explicit Run(int i0) {
      const int c = i0 >= 0 ? i0 / CH : -1;
      b0 = i0 + c * VW;
      f = i0 - c * CH;
    }
    __device__ __forceinline__ int operator()(int w) const {
      return b0 + w + (f >= CH - w ? VW : 0) + (w > CH && f >= 2 * CH - w ? VW : 0);
    }
  };

  // avail: elements from src to the end of the field
  // WHOLE: the lines are whole vectors from an aligned start, CH elements a lane
  template <bool WHOLE>
  static __device__ __forceinline__ void load(TS* tile, const TS* src, int end, long long avail, int vec, int lane) {
    constexpr int NV = CH / VW + (WHOLE ? 0 : 1);  // vectors per lane
    if (!vec) {
      for (int e = lane; e < end; e += 64) tile[at(e)] = src[e];
      return;
    }
    // whole vectors that lie inside the field, then the rest one by one
    int nv = (end + VW - 1) / VW;
    if (!WHOLE && (long long)nv * VW > avail) --nv;
    V t[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = lane + 64 * j;
      t[j] = reinterpret_cast<const V*>(src)[e < nv ? e : 0];
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = lane + 64 * j;
      if (e < nv) *reinterpret_cast<V*>(tile + at(e * VW)) = t[j];
    }
    if (!WHOLE && nv * VW + lane < end) tile[at(nv * VW + lane)] = src[nv * VW + lane];
  }

  // the results, with the epilogue; dst as src, o32 (if not null) the FP32
  // copy of FP64 results, only32 instead of them
  template <bool WHOLE>
  static __device__ __forceinline__ void store(const TS* tile, TS* dst, int sh, int end, int vec, int lane, int epi,
                                               double epi_c, float* o32, int only32) {
    constexpr int NV = CH / VW + (WHOLE ? 0 : 1);
    const bool need_old = reads_out(epi);
    auto put = [&](int e) {
      TS r = tile[at(e)];
      if (epi != EPI_STORE) r = epilogue<TS>(epi, epi_c, (double)r, need_old ? dst[e] : (TS)0);
      if (sizeof(TS) != 8 || !only32) dst[e] = r;
      if constexpr (sizeof(TS) == 8)
        if (o32) o32[e] = (float)r;
    };
    if (!vec) {
      for (int e = sh + lane; e < end; e += 64) put(e);
      return;
    }
    // whole vectors of these lines; the elements of shared vectors one by one
    const int v0 = (sh + VW - 1) / VW, v1 = end / VW;
    V* dv = reinterpret_cast<V*>(dst);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int e = lane + 64 * j;
      if (e >= v0 && e < v1) {
        V r = *reinterpret_cast<const V*>(tile + at(e * VW));
        if (epi != EPI_STORE) {
          const V o = need_old ? dv[e] : V{};
#pragma unroll
          for (int i = 0; i < VW; ++i) r[i] = epilogue<TS>(epi, epi_c, (double)r[i], o[i]);
        }
        if (sizeof(TS) != 8 || !only32) dv[e] = r;
        if constexpr (sizeof(TS) == 8) {
          using F2 = float __attribute__((ext_vector_type(2)));
          if (o32) reinterpret_cast<F2*>(o32)[e] = F2{(float)r[0], (float)r[1]};
        }
      }
    }
    if constexpr (!WHOLE) {
      if (lane >= sh && lane < v0 * VW && lane < end) put(lane);
      const int tail = v1 * VW + lane;
      if (lane < VW && tail >= v0 * VW && tail < end) put(tail);
    }
  }
};

// The lanes of line l of a wave whose lines have P lanes each.
__device__ __forceinline__ unsigned long long line_lanes(int l, int P) {
  return (P >= 64 ? ~0ull : (1ull << P) - 1) << ((l * P) & 63);
}

// x lines. A workgroup is one wave, which owns a.lines whole lines (64 / P):
// their elements are contiguous, come in and leave as 16-byte vectors through
// the wave's own LDS tile, and lane l * P + p solves chunk p of line l. The
// chunks of a line are lanes of one wave, so the carries need no barrier and
// the waves of a CU run independently: 14-20 of them fit its LDS, enough
// loads and stores in flight to reach the rate of a plain copy. Measured at
// 256^3 (64-thread workgroups with 8 lines and 32-row chunks before): FP64
// fbar 84 -> 53 us, d1 79 -> 50 us, FP32 d1 47 -> 33 us; a copy takes 50 and
// 25 us. A persistent variant that fetches its next lines into registers
// while it solves measured slower (512^3 d1 408 us against 373).
// Waves per workgroup: the waves of a bounded sweep share the line's tables.
template <int SOLVE> struct XWaves { static constexpr int v = SOLVE == SOLVE_BND ? 4 : 1; };

// PRE_NONE and PRE_V as for the y/z rows. Every other epilogue is applied as the
// vectors leave, to rows that add the input back (PRE_ANY) or not (PRE_OLD). A
// row with neither a test for the filter nor one for an idle lane: FP32 ring on
// 256^3 98 -> 97 us, bounded Laplacian on 192^3 112 -> 109, divergence on
// 180x130x75 43.7 -> 41.9, filter on 1024x512 17.4 -> 16.6; refined FP32 lines
// 225 -> 218 (ragged bounded gradient).
template <typename TS, int KIND, int SOLVE, bool FULL, int PRE, bool GRP = false>
__device__ __forceinline__ void line_x_body(const LineArgs& a, long long blk, const TS* __restrict__ in,
                                            TS* __restrict__ out) {
  constexpr int R = Halo<KIND>::R;
  using T = XTile<TS, CHUNK>;
  constexpr int CP = T::CP;
  constexpr int NW = XWaves<SOLVE>::v;
  __shared__ __align__(16) TS tiles[NW][T::SIZE];
  __shared__ __align__(16) D2 exits[NW][64];
  extern __shared__ __align__(16) unsigned char smem[];
  double* tab = reinterpret_cast<double*>(smem);
  const Tables tabs(tab, a.T);
  const bool bounded = SOLVE == SOLVE_BND || (SOLVE == SOLVE_NONE && !a.periodic);
  if (bounded) {
    stage_tables(a, tab);
    __syncthreads();
  }
  const int N = a.N, P = a.P;
  const int lane = threadIdx.x & 63;
  const int wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  TS* tile = tiles[wave] + T::ORIGIN;
  [[maybe_unused]] D2* ex = exits[wave];
  const long long L0 = (blk * NW + wave) * a.lines;
  const long long rem = (long long)a.nlines - L0;
  if (NW > 1 && rem <= 0) return;
  const int nval = (int)(rem < a.lines ? rem : a.lines);
  const long long E0 = L0 * N;
  const int sh = (!FULL && a.vec) ? (int)(E0 & (T::VW - 1)) : 0;
  const int end = sh + nval * N;
  T::template load<FULL>(tile, in + (E0 - sh), end, (long long)a.nlines * N - (E0 - sh), a.vec, lane);
  wave_fence();
  const int l = lane / P, p = lane - l * P;
  const bool act = l < nval;
  const int s = FULL ? p * CHUNK : chunk_start(a, p);
  const int m = FULL ? CHUNK : a.mb + (p < a.mx ? 1 : 0);
  const auto have = rows_of_chunk<FULL>(a, p);
  const bool last = p == P - 1;
  const bool wrap = SOLVE == SOLVE_CIRC || (SOLVE == SOLVE_NONE && a.periodic);
  const int i0 = sh + (act ? l : 0) * N;  // the line's first element in the tile
  const typename T::Run run(i0 + s - R);
  auto own = [&](int k) -> TS& { return tile[FULL ? (i0 / CHUNK + p) * CP + k : run(k + R)]; };
  TS win[CHUNK + 2 * R];
  if constexpr (FULL) {
    const TS* row0 = tile + i0 / CHUNK * CP;
    const TS* lo = row0 + (p == 0 ? P - 1 : p - 1) * CP;
    const TS* hi = row0 + (last ? 0 : p + 1) * CP;
#pragma unroll
    for (int w = 0; w < CHUNK + 2 * R; ++w) {
      if (w < R) win[w] = lo[CHUNK - R + w];
      else if (w < CHUNK + R) win[w] = own(w - R);
      else win[w] = hi[w - CHUNK - R];
    }
    if (!wrap) {
#pragma unroll
      for (int w = 0; w < R; ++w) {
        if (p == 0) win[w] = (TS)0;
        if (last) win[CHUNK + R + w] = (TS)0;
      }
    }
  } else {
    // the rows as they lie in the tile, then the halos beyond the line's ends
    // (the last chunk has mb rows); what is read past a chunk's own halo is
    // not used
#pragma unroll
    for (int w = 0; w < CHUNK + 2 * R; ++w) win[w] = tile[run(w)];
    if (p == 0) {
#pragma unroll
      for (int w = 0; w < R; ++w) win[w] = wrap ? tile[T::at(i0 + N - R + w)] : (TS)0;
    }
    if (last) {
#pragma unroll
      for (int w = 2 * NB + R; w < CHUNK + 2 * R; ++w) {
        const int j = w - R - a.mb;
        if (j >= 0 && j < R) win[w] = wrap ? tile[T::at(i0 + j)] : (TS)0;
      }
    }
  }
  double x[CHUNK];
  B4 lo = {}, hi = {};
  if (bounded) boundary_rows<KIND, SOLVE == SOLVE_NONE, FULL>(a, tabs.wb, p, win, lo, hi);
  right_hand_side<KIND, SOLVE>(a, win, x);
  if (bounded) put_boundary_rows<FULL>(a, p, lo, hi, x);
  // filters add v back here, read from the tile before the result takes its place
  auto emit = [&](int k, double y) {
    double val = y * a.scale;
    TS& o = own(k);
    if constexpr (PRE == PRE_V || PRE == PRE_ANY) val += (double)o;
    o = (TS)val;
  };
  if constexpr (SOLVE == SOLVE_NONE) {
    wave_fence();  // every window is in registers
    if (act) {
#pragma unroll
      for (int k = 0; k < CHUNK; ++k) have.row(k, [&] { emit(k, x[k]); });
    }
  } else {
    // lanes past the last whole line read some exit and drop the result
    auto exit_of = [&](int q) { return ex[l * P + q < 64 ? l * P + q : 0]; };
    const int slot = SOLVE == SOLVE_BND ? slot_of(a, p) : 0;
    double e0 = 0.0, e1 = 0.0, b0 = 0.0, b1 = 0.0;
    with_rows<SOLVE>(a, true, tabs, slot, [&](auto rows) { fwd_pass<false>(have, rows, x, e0, e1); });
    ex[lane] = D2{e0, e1};
    wave_fence();
    carry_of<SOLVE, FULL, -1>(a, tabs, p, exit_of, e0, e1);
    with_rows<SOLVE>(a, true, tabs, slot, [&](auto rows) {
      fwd_pass<true>(have, rows, x, e0, e1);
      bwd_exit(have, rows, x, b0, b1);
    });
    // as in line_yz_body: a NaN or infinity spreads to the whole line
    const unsigned long long bad = __ballot(act && (!__builtin_isfinite(b0) || !__builtin_isfinite(b1)));
    wave_fence();
    ex[lane] = D2{b0, b1};
    wave_fence();
    carry_of<SOLVE, FULL, 1>(a, tabs, p, exit_of, b0, b1);
    if (bad & line_lanes(l, P)) b0 = b1 = __builtin_nan("");
    if (act) with_rows<SOLVE>(a, true, tabs, slot, [&](auto rows) { bwd_sink(have, rows, x, b0, b1, emit); });
  }
  wave_fence();
  if constexpr (PRE == PRE_ANY || PRE == PRE_OLD) {
    float* o32 = nullptr;
    if constexpr (sizeof(TS) == 8 && !GRP) o32 = a.out32 ? a.out32 + (E0 - sh) : nullptr;
    T::template store<FULL>(tile, out + (E0 - sh), sh, end, a.vec, lane, a.epi, a.epi_c, o32, GRP ? 0 : a.only32);
  } else {
    T::template store<FULL>(tile, out + (E0 - sh), sh, end, a.vec, lane, EPI_STORE, 0.0, nullptr, 0);
  }
}

template <typename TS, int KIND, int SOLVE, bool FULL, int PRE>
__global__ void __launch_bounds__(64 * XWaves<SOLVE>::v) k_line_x(LineArgs a, const TS* __restrict__ in, TS* __restrict__ out) {
  line_x_body<TS, KIND, SOLVE, FULL, PRE>(a, blockIdx.x, in, out);
}

// Grouped launches: one launch applies the same operator to the fields of
// several simulations (an ensemble's members, each at `off` elements into
// one allocation), with lines of any lengths. Entry j covers workgroups
// [blk0_j, blk0_{j+1}); a workgroup reads its member from a map (one load; a
// binary search over blk0 is a chain of them) and runs the single-field body with that member's line
// arguments: every member has its own lines per workgroup (x: 64 / P, y/z: as
// many as P chunk threads each leave room for), so one launch serves all
// line lengths.
struct GrpEntry {
  LineArgs a;
  long long off;
  long long blk0;
};

template <typename TS, int KIND, int SOLVE, int PRE>
__global__ void __launch_bounds__(64 * XWaves<SOLVE>::v) k_line_x_grp(const GrpEntry* __restrict__ g,
                                                                      const int* __restrict__ member,
                                                                      const TS* __restrict__ in,
                                                                      TS* __restrict__ out) {
  const int j = member[blockIdx.x];
  const LineArgs a = g[j].a;
  const long long off = g[j].off, b0 = g[j].blk0;
  line_x_body<TS, KIND, SOLVE, false, PRE, true>(a, (long long)blockIdx.x - b0, in + off, out + off);
}
template <typename TS, int KIND, int SOLVE, int PRE>
__global__ void __launch_bounds__(WG_MAX) k_line_yz_grp(const GrpEntry* __restrict__ g, const int* __restrict__ member,
                                                        const TS* __restrict__ in, TS* __restrict__ out) {
  const int blk = SOLVE == SOLVE_NONE ? xcd_order() : (int)blockIdx.x;
  const int j = member[blk];
  const LineArgs a = g[j].a;
  const long long off = g[j].off, b0 = g[j].blk0;
  line_yz_body<TS, KIND, SOLVE, false, PRE, true>(a, (int)(blk - b0), in + off, out + off);
}

// --- refined FP32 solve of bounded lines (pyr_refined.hpp) -------------------
// Threads are shaped as in the FP64 kernels above, with up to 32 rows each (two
// waves per SIMD by registers) and workgroups of 256: as many lines as fit, any
// number of them, so that few threads idle and an ensemble's sweep fits the
// chip in one go (24 members, 3.7M points: 489 workgroups for 512 places; 512
// threads and a power of two of lines gave 319 for 256). x: two waves, each
// with its own lines and tile. What bounds these kernels is the latency of one
// workgroup: the class tables and the reduced rows of the chunks within reach
// are staged in LDS, and the boundary rows' terms are independent reads.
constexpr int REF_THREADS = 256;
constexpr int REF_X_WAVES = 2;

// class tables and reduced rows into LDS
__device__ __forceinline__ void ref_stage(const RefArgs& a, float* tab, float* g) {
  for (int e = threadIdx.x; e < NCLS * RCHUNK * CROW / 4; e += blockDim.x)
    reinterpret_cast<F4*>(tab)[e] = reinterpret_cast<const F4*>(a.cls)[e];
  for (int e = threadIdx.x; e < a.P * (2 * a.Wg + 1) * 4; e += blockDim.x)
    reinterpret_cast<F4*>(g)[e] = reinterpret_cast<const F4*>(a.g)[e];
}

template <int KIND, int PRE>
__device__ __forceinline__ void ref_yz_body(const RefArgs& a, int blk, const float* __restrict__ in,
                                            float* __restrict__ out) {
  constexpr int R = Halo<KIND>::R;
  __shared__ __align__(16) float tab[NCLS * RCHUNK * CROW];
  __shared__ __align__(16) F4 Y0[REF_THREADS], Y1[REF_THREADS];
  __shared__ float ends[2 * (ENDS + 1) * 64];
  __shared__ int bad[64];
  extern __shared__ __align__(16) unsigned char smem[];
  float* g = reinterpret_cast<float*>(smem);
  const int LY = a.lines;
  const int p = (int)((unsigned)threadIdx.x / (unsigned)LY);
  const int lane = (int)threadIdx.x - p * LY;
  if (p == 0) bad[lane] = 0;
  const bool act = p < a.P;
  const int L = blk * LY + lane;
  const int lane_off = line_offset(a, L) * (int)sizeof(float);
  const int rb = (int)(a.stride * (long long)sizeof(float));
  const int s = p * a.mb + (p < a.mx ? p : a.mx);
  const int m = a.mb + (p < a.mx ? 1 : 0);
  const __amdgpu_buffer_rsrc_t rin = buf_rsrc(in, a.nbytes), rout = buf_rsrc(out, a.nbytes);
  auto off_of = [&](int row) { return (int)((unsigned)lane_off + (unsigned)row * (unsigned)rb); };
  // rows beyond the ends read 0
  float win[RCHUNK + 2 * R];
#pragma unroll
  for (int w = 0; w < RCHUNK + 2 * R; ++w) {
    const int row = s - R + w;
    win[w] = 0.0f;
    if (w <= a.mb + 2 * R)
      win[w] = buf_load(0.0f, rin, act && w < m + 2 * R && row >= 0 && row < a.N ? off_of(row) : OOB, 0);
  }
  ref_stage(a, tab, g);  // behind the window's loads
  double rhs[RCHUNK];
  ref_rhs_interior<KIND>(a, win, rhs);
  if (act && (p == 0 || p == a.P - 1)) {
    // the boundary rows name any of the eight rows at their end: this thread's
    // copy of them in LDS, indexed at run time (no other thread reads it)
    float* mine = ends + (p == 0 ? 0 : ENDS + 1) * 64 + lane;
    mine[ENDS * 64] = 0.0f;
    if (p == 0) {
#pragma unroll
      for (int k = 0; k < ENDS / 2; ++k) mine[k * 64] = win[k + R];
    }
    if (p == a.P - 1) {
#pragma unroll
      for (int k = 0; k < RCHUNK; ++k) {
        const int j = k - (a.mb - ENDS / 2);
        if (j >= 0 && j < ENDS / 2) mine[(ENDS / 2 + j) * 64] = win[k + R];
      }
    }
    ref_rhs_boundary(a, p, rhs, [&](int slot) { return mine[slot * 64]; });
  }
  __syncthreads();  // class tables visible
  const float* t = tab + ref_class(p, a.P, a.mx) * (RCHUNK * CROW);
  float x[RCHUNK], d[RCHUNK], z[4];
  const bool longer = p < a.mx;
  if (act) {
    ref_local_solve(a, longer, t, rhs, x);
    const F4 e = ref_edges(a, longer, x);
    Y0[p * LY + lane] = e;
    // as in line_yz_body: a NaN or infinity spreads to the whole line
    if (!__builtin_isfinite(e.x) || !__builtin_isfinite(e.y)) bad[lane] = 1;
  }
  __syncthreads();
  if (act) {
    ref_neighbours(a, g, p, [&](int q) { return Y0[q * LY + lane]; }, z);
    if (bad[lane]) z[0] = z[1] = z[2] = z[3] = __builtin_nanf("");
    ref_spike(a, t, z, x);
    ref_residual(a, p, longer, rhs, x, z, d);
  }
  // the filter's input or the current output, on its way while the correction
  // is solved (the right-hand sides' registers are free by now)
  float pre[PRE == PRE_NONE ? 1 : RCHUNK];
  if constexpr (PRE != PRE_NONE) {
    const bool v = PRE == PRE_V || (PRE == PRE_ANY && a.addv);
#pragma unroll
    for (int k = 0; k < RCHUNK; ++k)
      if (k <= a.mb) pre[k] = buf_load(0.0f, v ? rin : rout, act && k < m ? off_of(s + k) : OOB, 0);
  }
  if (act) {
    ref_local_solve(a, longer, t, d, d);
    Y1[p * LY + lane] = ref_edges(a, longer, d);
  }
  __syncthreads();
  if (!act || L >= a.nlines) return;
  ref_neighbours(a, g, p, [&](int q) { return Y1[q * LY + lane]; }, z);
  ref_spike(a, t, z, d);
#pragma unroll
  for (int k = 0; k < RCHUNK; ++k) {
    if (k <= a.mb) {
      double val = ((double)x[k] + (double)d[k]) * a.scale;
      const int off = k < m ? off_of(s + k) : OOB;
      if constexpr (PRE == PRE_V) val += (double)pre[k];
      if constexpr (PRE == PRE_ANY) {
        float old = pre[k];
        if (a.addv) {
          val += (double)pre[k];
          if (reads_out(a.epi)) old = buf_load(0.0f, rout, off, 0);
        }
        buf_store(epilogue<float>(a.epi, a.epi_c, val, old), rout, off, 0);
      } else if constexpr (PRE == PRE_OLD) {
        buf_store(epilogue<float>(joined_epi(KIND), a.epi_c, val, pre[k]), rout, off, 0);
      } else {
        buf_store((float)val, rout, off, 0);
      }
    }
  }
}

template <int KIND, int PRE>
__device__ __forceinline__ void ref_x_body(const RefArgs& a, long long blk, const float* __restrict__ in,
                                           float* __restrict__ out) {
  constexpr int R = Halo<KIND>::R;
  constexpr int NW = REF_X_WAVES;
  using T = XTile<float, RCHUNK>;
  __shared__ __align__(16) float tab[NCLS * RCHUNK * CROW];
  __shared__ __align__(16) float tiles[NW][T::SIZE];
  __shared__ __align__(16) F4 ex[NW][64];
  extern __shared__ __align__(16) unsigned char smem[];
  float* g = reinterpret_cast<float*>(smem);
  ref_stage(a, tab, g);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  float* tile = tiles[wave] + T::ORIGIN;
  const int N = a.N, P = a.P;
  const long long L0 = (blk * NW + wave) * a.lines;
  const long long rem = (long long)a.nlines - L0;
  if (rem <= 0) return;
  const int nval = (int)(rem < a.lines ? rem : a.lines);
  const long long E0 = L0 * N;
  const int sh = a.vec ? (int)(E0 & (T::VW - 1)) : 0;
  const int end = sh + nval * N;
  T::load<false>(tile, in + (E0 - sh), end, (long long)a.nlines * N - (E0 - sh), a.vec, lane);
  wave_fence();
  const int l = lane / P, p = lane - l * P;
  const bool act = l < nval;
  const int s = p * a.mb + (p < a.mx ? p : a.mx);
  const int m = a.mb + (p < a.mx ? 1 : 0);
  const int i0 = sh + (act ? l : 0) * N;
  const T::Run run(i0 + s - R);
  // the rows as they lie in the tile; beyond the line's ends 0
  float win[RCHUNK + 2 * R];
#pragma unroll
  for (int w = 0; w < RCHUNK + 2 * R; ++w) win[w] = w < m + 2 * R ? tile[run(w)] : 0.0f;
  if (p == 0) {
#pragma unroll
    for (int w = 0; w < R; ++w) win[w] = 0.0f;
  }
  if (p == P - 1) {
#pragma unroll
    for (int w = 2 * NB + R; w < RCHUNK + 2 * R; ++w)
      if (w >= a.mb + R) win[w] = 0.0f;
  }
  double rhs[RCHUNK];
  ref_rhs_interior<KIND>(a, win, rhs);
  ref_rhs_boundary(a, p, rhs, [&](int slot) { return end_value(slot, N, [&](int i) { return tile[T::at(i0 + i)]; }); });
  const float* t = tab + ref_class(p, P, a.mx) * (RCHUNK * CROW);
  float x[RCHUNK], d[RCHUNK], z[4];
  const bool longer = p < a.mx;
  auto edges_of = [&](int q) { return ex[wave][l * P + q < 64 ? l * P + q : 0]; };
  ref_local_solve(a, longer, t, rhs, x);
  const F4 e = ref_edges(a, longer, x);
  ex[wave][lane] = e;
  const unsigned long long bad = __ballot(act && (!__builtin_isfinite(e.x) || !__builtin_isfinite(e.y)));
  wave_fence();
  ref_neighbours(a, g, p, edges_of, z);
  if (bad & line_lanes(l, P)) z[0] = z[1] = z[2] = z[3] = __builtin_nanf("");
  ref_spike(a, t, z, x);
  ref_residual(a, p, longer, rhs, x, z, d);
  ref_local_solve(a, longer, t, d, d);
  const F4 ed = ref_edges(a, longer, d);
  wave_fence();
  ex[wave][lane] = ed;
  wave_fence();
  ref_neighbours(a, g, p, edges_of, z);
  ref_spike(a, t, z, d);
  if (act) {
#pragma unroll
    for (int k = 0; k < RCHUNK; ++k) {
      double val = ((double)x[k] + (double)d[k]) * a.scale;
      // (rows below mb are every chunk's: a test of the wave, not of the lane)
      if (k < a.mb || k < m) {
        float& o = tile[run(k + R)];
        if constexpr (PRE == PRE_V || PRE == PRE_ANY) val += (double)o;
        o = (float)val;
      }
    }
  }
  wave_fence();
  constexpr bool ST = PRE == PRE_NONE || PRE == PRE_V;
  T::store<false>(tile, out + (E0 - sh), sh, end, a.vec, lane, ST ? EPI_STORE : a.epi, a.epi_c, nullptr, 0);
}

struct RefEntry {
  RefArgs a;
  long long off;
  long long blk0;
};

template <int KIND, int PRE>
__global__ void __launch_bounds__(REF_THREADS) k_ref_yz(RefArgs a, const float* __restrict__ in,
                                                        float* __restrict__ out) {
  ref_yz_body<KIND, PRE>(a, xcd_order(), in, out);
}
template <int KIND, int PRE>
__global__ void __launch_bounds__(64 * REF_X_WAVES) __attribute__((amdgpu_waves_per_eu(2, 8))) k_ref_x(RefArgs a, const float* __restrict__ in,
                                                            float* __restrict__ out) {
  ref_x_body<KIND, PRE>(a, blockIdx.x, in, out);
}
template <int KIND, int PRE>
__global__ void __launch_bounds__(REF_THREADS) k_ref_yz_grp(const RefEntry* __restrict__ g, const int* __restrict__ member,
                                                            const float* __restrict__ in, float* __restrict__ out) {
  const int blk = xcd_order();
  const int j = member[blk];
  const RefArgs a = g[j].a;
  const long long off = g[j].off, b0 = g[j].blk0;
  ref_yz_body<KIND, PRE>(a, (int)(blk - b0), in + off, out + off);
}
template <int KIND, int PRE>
__global__ void __launch_bounds__(64 * REF_X_WAVES) __attribute__((amdgpu_waves_per_eu(2, 8))) k_ref_x_grp(const RefEntry* __restrict__ g, const int* __restrict__ member,
                                                                const float* __restrict__ in,
                                                                float* __restrict__ out) {
  const int j = member[blockIdx.x];
  const RefArgs a = g[j].a;
  const long long off = g[j].off, b0 = g[j].blk0;
  ref_x_body<KIND, PRE>(a, (long long)blockIdx.x - b0, in + off, out + off);
}

// null operator of a direction with fewer than 4 points (zero or copy)
template <typename TS>
__global__ void k_null(long long n, int copy, int epi, double c, const TS* __restrict__ in,
                       TS* __restrict__ out, float* __restrict__ out32) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double val = copy ? (double)in[i] : 0.0;
  const TS old = reads_out(epi) ? out[i] : (TS)0;
  const TS r = epilogue<TS>(epi, c, val, old);
  if (out) out[i] = r;
  if (out32) out32[i] = (float)r;
}

// RK4 stage update (pyranda.py:800-804), one pass over F, PHI and U. With
// A == 0 (the first stage) A*PHI is zero and PHI is not read, so it needs no
// clearing before the step. dtp (if not null) holds dt in device memory: one
// value, or with mid (the member index of every point of an ensemble's
// fields) one value per member.
template <typename TF, typename TS>
__global__ void k_rk_update(long long n, const TF* __restrict__ F, double* __restrict__ PHI,
                            const TS* __restrict__ Uin, TS* __restrict__ Uout,
                            double* __restrict__ U64, const double* __restrict__ dtp,
                            const int* __restrict__ mid, double dt, double A, double B) {
  if (dtp && !mid) dt = *dtp;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double dti = mid ? dtp[mid[i]] : dt;
    const double tmp1 = A == 0.0 ? 0.0 : A * PHI[i];
    // explicit FMAs: the generated kernels that fuse a right-hand side into
    // this update round the same way
    const double phi = fma(dti, (double)F[i], tmp1);
    PHI[i] = phi;
    if (U64) {
      const double u = fma(B, phi, U64[i]);
      U64[i] = u;
      if (Uout) Uout[i] = (TS)u;
    } else {
      Uout[i] = (TS)fma(B, phi, (double)Uin[i]);
    }
  }
}

// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------
// Device addresses of a plan's tables, all inside the context's one table
// allocation (pyr_ctx::tables).
struct DevPlan {
  const double* tab = nullptr;  // row tables with the boundary rows
};

struct DevRefPlan {
  const float *cls = nullptr, *g = nullptr;
  const double *be = nullptr, *bcoef = nullptr;
  const int* bidx = nullptr;
};

struct pyr_ctx {
  int n[3] = {1, 1, 1};
  int bc[6] = {PYR_BC_NONE, PYR_BC_NONE, PYR_BC_NONE, PYR_BC_NONE, PYR_BC_NONE, PYR_BC_NONE};
  double x1[3] = {0, 0, 0};
  double dpatch[3] = {1, 1, 1};  // patch dx (metric of derivatives)
  double dmesh[3] = {1, 1, 1};   // mesh d1..d3 (ring length scales)
  double gridlen = 1.0;
  bool device = false;
  hipStream_t stream = nullptr;
  OpPlan plan[NOPS][3];
  DevPlan dplan[NOPS][3];
  // second member of the symmetric/antisymmetric pair (compact.f90:78-84):
  // variant -1 at each SYMM end of a direction that has one
  bool has_anti[3] = {false, false, false};
  OpPlan plan_a[NOPS][3];
  DevPlan dplan_a[NOPS][3];
  // refined FP32 solve of the bounded implicit lines (N > 0), both members
  RefPlan rplan[NOPS][3], rplan_a[NOPS][3];
  DevRefPlan drplan[NOPS][3], drplan_a[NOPS][3];
  void* tables = nullptr;  // the tables of every plan
  void* field_tmp[2] = {nullptr, nullptr};  // one field-sized temp per precision
  int periodic_solver = PYR_PSOLVE_CIRCULANT;
  int r32_solve = PYR_R32_SOLVE_REFINED;
  // launch knobs (pyr_set_tuning): lines per y/z workgroup (0: the rule of
  // yz_lines), and the y/z kernel with runtime row counts; per operator,
  // direction and field width (0 FP64, 1 FP32), -1 / 0 = the default
  int yz_lines = 0;
  int tune_ly[NOPS][3][2];
  int tune_rt[NOPS][3][2] = {};
  // FP32 solve mode per operator and direction (-1 = r32_solve; r32_mode)
  int tune_solve[NOPS][3];
  // settings that change no launch, kept as group members have to agree on
  // them: the x-line LDS budget and the periodic solver (above)
  int x_lds_kb = 40;
  pyr_ctx() {
    for (int o = 0; o < NOPS; ++o)
      for (int d = 0; d < 3; ++d) {
        tune_solve[o][d] = -1;
        for (int w = 0; w < 2; ++w) tune_ly[o][d][w] = -1;
      }
  }
  int ncu = 256;                             // compute units of the device
  void* noalloc_tmp = nullptr;               // this device's copy of `scratch` (pyr_sfilter_noalloc)
  float* out32 = nullptr;                    // FP32 copy of the next FP64 sweep's output
  int only32 = 0;                            // ... and no FP64 store
  size_t npts() const { return (size_t)n[0] * n[1] * n[2]; }
};

// what a bounded sweep stages: the row tables, then the boundary rows
static std::vector<double> with_boundary_rows(const OpPlan& pl) {
  std::vector<double> t = pl.tab;
  t.insert(t.end(), pl.wb.begin(), pl.wb.end());
  return t;
}

// The tables of all plans of a context back to back, 256-byte aligned: added
// one by one, then uploaded in one piece.
struct TableImage {
  std::vector<unsigned char> host;
  template <typename T>
  size_t add(const std::vector<T>& t) {
    const size_t at = host.size();
    host.resize((at + t.size() * sizeof(T) + 255) & ~(size_t)255, 0);
    if (!t.empty()) std::memcpy(host.data() + at, t.data(), t.size() * sizeof(T));
    return at;
  }
};

// adds the tables of a plan to the image; the addresses are offsets until
// rebase() is called with the image's device address
static void add_plan(TableImage& im, const OpPlan& pl, DevPlan& d) {
  d.tab = reinterpret_cast<const double*>(im.add(with_boundary_rows(pl)));
}
static void add_plan(TableImage& im, const RefPlan& pl, DevRefPlan& d) {
  if (pl.N == 0) return;
  d.cls = reinterpret_cast<const float*>(im.add(pl.cls));
  d.g = reinterpret_cast<const float*>(im.add(pl.g));
  d.be = reinterpret_cast<const double*>(im.add(pl.be));
  d.bcoef = reinterpret_cast<const double*>(im.add(pl.bcoef));
  d.bidx = reinterpret_cast<const int*>(im.add(pl.bidx));
}
template <typename T>
static void rebase(const T*& p, const unsigned char* base) {
  p = reinterpret_cast<const T*>(base + reinterpret_cast<size_t>(p));
}
static void rebase(DevPlan& d, const unsigned char* base) {
  rebase(d.tab, base);
}
static void rebase(DevRefPlan& d, const unsigned char* base) {
  rebase(d.cls, base);
  rebase(d.g, base);
  rebase(d.be, base);
  rebase(d.bcoef, base);
  rebase(d.bidx, base);
}

// every plan's tables onto the device: one allocation and one copy
static int upload_plans(pyr_ctx* c) {
  TableImage im;
  auto each = [&](auto f) {
    for (int op = 0; op < NOPS; ++op)
      for (int d = 0; d < 3; ++d) {
        f(c->plan[op][d], c->dplan[op][d]);
        f(c->rplan[op][d], c->drplan[op][d]);
        if (!c->has_anti[d]) continue;
        f(c->plan_a[op][d], c->dplan_a[op][d]);
        f(c->rplan_a[op][d], c->drplan_a[op][d]);
      }
  };
  each([&](const auto& pl, auto& d) { add_plan(im, pl, d); });
  if (im.host.empty()) return 0;
  HIPCHECK(hipMalloc(&c->tables, im.host.size()));
  HIPCHECK(hipMemcpy(c->tables, im.host.data(), im.host.size(), hipMemcpyHostToDevice));
  each([&](const auto&, auto& d) { rebase(d, static_cast<const unsigned char*>(c->tables)); });
  return 0;
}

// host pointers of the same tables (host emulation)
static void host_ref_tables(const RefPlan& pl, DevRefPlan& d) {
  d.cls = pl.cls.data();
  d.g = pl.g.data();
  d.be = pl.be.data();
  d.bcoef = pl.bcoef.data();
  d.bidx = pl.bidx.data();
}
static LineArgs make_args(const pyr_ctx* c, const OpPlan& pl, const DevPlan& d, int dir, int epi,
                          double ec, int prec) {
  LineArgs a;
  std::memset(&a, 0, sizeof(a));
  const long long nx = c->n[0], ny = c->n[1], nz = c->n[2];
  a.N = pl.N;
  a.P = pl.P;
  a.periodic = pl.periodic;
  if (dir == 0) {
    a.nlines = (int)(ny * nz);
    a.A = 1; a.B = nx; a.stride = 1;
  } else if (dir == 1) {
    a.nlines = (int)(nx * nz);
    a.A = nx; a.B = nx * ny; a.stride = nx;
  } else {
    a.nlines = (int)(nx * ny);
    a.A = nx * ny; a.B = 0; a.stride = nx * ny;
  }
  a.nbytes = (int)(c->npts() * (prec == PYR_F64 ? sizeof(double) : sizeof(float)));
  a.addv = pl.addv;
  a.epi = epi;
  a.scale = pl.scale;
  a.epi_c = ec;
  a.mb = pl.mb;
  a.mx = pl.mx;
  for (int i = 0; i < 4; ++i) a.w[i] = pl.w[i];
  a.p1 = pl.p1;
  a.p2 = pl.p2;
  a.W = pl.W;
  std::memcpy(a.hf, pl.hf, sizeof a.hf);
  std::memcpy(a.hb, pl.hb, sizeof a.hb);
  a.turns = pl.turns;
  std::memcpy(a.tf, pl.tf, sizeof a.tf);
  std::memcpy(a.tb, pl.tb, sizeof a.tb);
  a.tab = d.tab;
  a.tlo = pl.tlo;
  a.T = pl.T;
  a.ntab = (int)(pl.tab.size() + pl.wb.size());
  return a;
}

// line arguments of the refined solve, from those of the same operator
static RefArgs make_ref_args(const LineArgs& l, const RefPlan& pl, const DevRefPlan& d) {
  RefArgs a;
  std::memset(&a, 0, sizeof(a));
  a.N = pl.N; a.P = pl.P; a.mb = pl.mb; a.mx = pl.mx;
  a.nlines = l.nlines; a.nbytes = l.nbytes;
  a.A = l.A; a.B = l.B; a.stride = l.stride;
  a.addv = l.addv; a.epi = l.epi; a.epi_c = l.epi_c;
  a.scale = pl.scale;
  for (int i = 0; i < 9; ++i) a.w[i] = pl.w[i];
  for (int i = 0; i < 5; ++i) a.bd[i] = pl.bd[i];
  a.Wg = pl.Wg;
  a.cls = d.cls; a.g = d.g; a.be = d.be; a.bcoef = d.bcoef; a.bidx = d.bidx;
  return a;
}

// solve used for a plan: explicit, bounded lines, or periodic lines
static int plan_solve(const OpPlan& pl) {
  if (!pl.implicit) return SOLVE_NONE;
  return pl.periodic ? SOLVE_CIRC : SOLVE_BND;
}

// ---------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------
// LDS of a y/z workgroup of nthr chunk threads: two exchange buffers, one flag
// per line, the tables of a bounded line.
static size_t yz_lds(int solve, int nthr, int lines, int ntab) {
  return (solve == SOLVE_NONE ? 0 : 2 * (size_t)nthr * sizeof(D2)) + (size_t)lines * sizeof(int) +
         (size_t)ntab * sizeof(double);
}

// Workgroups of the explicit filter per line group: its chunks need no
// exchange, so a workgroup is 64 lines by as many chunks as 256 threads hold.
constexpr int NONE_THREADS = 256;
static int explicit_groups(int P, int nthr, int lines) { return (P + nthr / lines - 1) / (nthr / lines); }

// Lines per y/z workgroup (forced: the tuned value, 0 = none). At 256^3 32
// lines measured fastest for FP64 fields (d1 y 54 us; 16 lines 58, 64 lines
// 64: one workgroup of 16 waves fills a CU alone) and for FP32 y lines (33
// us); FP32 z lines, whose rows are a plane apart, gain from 256-byte rows (64
// lines 36 us, 32 lines 41). Lines of more than 32 chunks leave room for 16
// in a workgroup. Fields too small to give every CU a workgroup take 16.
static int yz_lines(int P, int nlines, int dir, int elem, int forced, int ncu) {
  int ly = forced > 0 ? forced : (elem == 4 && dir == 2 ? 64 : 32);
  while (ly > 16 && ly * P > WG_MAX) ly /= 2;
  if (forced <= 0)
    while (ly > 16 && nlines < ly * ncu) ly /= 2;
  return ly;
}

template <typename TS, int KIND, int SOLVE, bool FULL>
static auto x_kernel(int pre, bool addv) {
  // filters only exist for the r4 kind, the explicit operator is one
  if constexpr (KIND == K_R4) {
    if (pre == PRE_V) return k_line_x<TS, KIND, SOLVE, FULL, PRE_V>;
    if (SOLVE == SOLVE_NONE || addv) return k_line_x<TS, KIND, SOLVE, FULL, PRE_ANY>;
  }
  if constexpr (SOLVE != SOLVE_NONE) {
    return pre == PRE_NONE ? k_line_x<TS, KIND, SOLVE, FULL, PRE_NONE> : k_line_x<TS, KIND, SOLVE, FULL, PRE_OLD>;
  }
}

template <typename TS, int KIND, int SOLVE, bool FULL>
static int launch_typed(pyr_ctx* c, int dir, int forced, LineArgs a, const TS* in, TS* out) {
  const int pre = pre_of(KIND, a.addv, a.epi, a.out32 != nullptr);
  if (dir == 0) {
    a.vec = ((uintptr_t)in % 16 == 0) && ((uintptr_t)out % 16 == 0) && ((uintptr_t)a.out32 % 8 == 0);
    a.lines = 64 / a.P;
    const int per = a.lines * XWaves<SOLVE>::v;
    const dim3 grid((unsigned)((a.nlines + per - 1) / per)), block(64 * XWaves<SOLVE>::v);
    const auto k = x_kernel<TS, KIND, SOLVE, FULL>(pre, a.addv);
    hipLaunchKernelGGL(k, grid, block, (size_t)a.ntab * sizeof(double), c->stream, a, in, out);
  } else {
    a.lines = SOLVE == SOLVE_NONE && forced <= 0 ? 64 : yz_lines(a.P, a.nlines, dir, (int)sizeof(TS), forced, c->ncu);
    unsigned nblk = (unsigned)((a.nlines + a.lines - 1) / a.lines);
    int nthr = a.lines * a.P;
    if (SOLVE == SOLVE_NONE) {
      nthr = std::min(nthr, NONE_THREADS);
      nblk *= (unsigned)explicit_groups(a.P, nthr, a.lines);
    }
    const dim3 grid(nblk), block(nthr);
    const size_t shm = yz_lds(SOLVE, nthr, a.lines, a.ntab);
    auto k = k_line_yz<TS, KIND, SOLVE, FULL, PRE_ANY>;
    // filters only exist for the r4 kind, the explicit operator is one
    if constexpr (KIND == K_R4) {
      if (pre == PRE_V) k = k_line_yz<TS, KIND, SOLVE, FULL, PRE_V>;
    }
    if constexpr (SOLVE != SOLVE_NONE) {
      if (pre == PRE_NONE) k = k_line_yz<TS, KIND, SOLVE, FULL, PRE_NONE>;
      if (pre == PRE_OLD) k = k_line_yz<TS, KIND, SOLVE, FULL, PRE_OLD>;
    }
    hipLaunchKernelGGL(k, grid, block, shm, c->stream, a, in, out);
  }
  HIPCHECK(hipGetLastError());
  return 0;
}

// CIRC: the periodic solve; otherwise bounded lines and the explicit filter
template <typename TS, bool CIRC>
int launch_kind(pyr_ctx* c, int dir, int kind, int sv, bool full, int forced, const LineArgs& a, const TS* in, TS* out) {
  constexpr int SV = CIRC ? SOLVE_CIRC : SOLVE_BND;
  switch (kind) {
    case K_D1:
      return full ? launch_typed<TS, K_D1, SV, true>(c, dir, forced, a, in, out)
                  : launch_typed<TS, K_D1, SV, false>(c, dir, forced, a, in, out);
    case K_R3:
      return full ? launch_typed<TS, K_R3, SV, true>(c, dir, forced, a, in, out)
                  : launch_typed<TS, K_R3, SV, false>(c, dir, forced, a, in, out);
    default:
      if constexpr (!CIRC) {
        if (sv == SOLVE_NONE)
          return full ? launch_typed<TS, K_R4, SOLVE_NONE, true>(c, dir, forced, a, in, out)
                      : launch_typed<TS, K_R4, SOLVE_NONE, false>(c, dir, forced, a, in, out);
      }
      return full ? launch_typed<TS, K_R4, SV, true>(c, dir, forced, a, in, out)
                  : launch_typed<TS, K_R4, SV, false>(c, dir, forced, a, in, out);
  }
}

#define PYR_LAUNCH_KIND(TS, CIRC) \
  template int launch_kind<TS, CIRC>(pyr_ctx*, int, int, int, bool, int, const LineArgs&, const TS*, TS*);
#if PYR_PART == 1
PYR_LAUNCH_KIND(double, true)
#elif PYR_PART == 2
PYR_LAUNCH_KIND(float, true)
#elif PYR_PART == 3
PYR_LAUNCH_KIND(double, false)
#elif PYR_PART == 4
PYR_LAUNCH_KIND(float, false)
#elif PYR_PART == 0
extern PYR_LAUNCH_KIND(double, true)
extern PYR_LAUNCH_KIND(float, true)
extern PYR_LAUNCH_KIND(double, false)
extern PYR_LAUNCH_KIND(float, false)
#endif
#undef PYR_LAUNCH_KIND

// lines per workgroup of P chunk threads: as many as fit, at most 64; LDS of
// the reduced rows
static int ref_lines(int P) { return std::min(64, REF_THREADS / P); }
static size_t ref_lds(const RefArgs& a) { return (size_t)a.P * (2 * a.Wg + 1) * 16 * sizeof(float); }

#if PYR_PART == 7
template <int KIND>
static auto ref_x_kernel(int pre, bool addv) {
  if constexpr (KIND == K_R4) {
    if (addv) return pre == PRE_V ? k_ref_x<KIND, PRE_V> : k_ref_x<KIND, PRE_ANY>;
  }
  return pre == PRE_NONE ? k_ref_x<KIND, PRE_NONE> : k_ref_x<KIND, PRE_OLD>;
}
template <int KIND>
static int launch_ref_kind(hipStream_t stream, int dir, RefArgs a, const float* in, float* out) {
  const int pre = pre_of(KIND, a.addv, a.epi, false);
  if (dir == 0) {
    a.vec = ((uintptr_t)in % 16 == 0) && ((uintptr_t)out % 16 == 0);
    a.lines = 64 / a.P;
    const int per = a.lines * REF_X_WAVES;
    hipLaunchKernelGGL((ref_x_kernel<KIND>(pre, a.addv)), dim3((unsigned)((a.nlines + per - 1) / per)), dim3(64 * REF_X_WAVES),
                       ref_lds(a), stream, a, in, out);
  } else {
    a.lines = ref_lines(a.P);
    auto k = k_ref_yz<KIND, PRE_ANY>;
    if constexpr (KIND == K_R4) {
      if (pre == PRE_V) k = k_ref_yz<KIND, PRE_V>;
    }
    if (pre == PRE_NONE) k = k_ref_yz<KIND, PRE_NONE>;
    if (pre == PRE_OLD) k = k_ref_yz<KIND, PRE_OLD>;
    hipLaunchKernelGGL(k, dim3((unsigned)((a.nlines + a.lines - 1) / a.lines)), dim3(a.lines * a.P), ref_lds(a),
                       stream, a, in, out);
  }
  HIPCHECK(hipGetLastError());
  return 0;
}
int launch_ref(hipStream_t stream, int dir, int kind, const RefArgs& a, const float* in, float* out) {
  if (kind == K_D1) return launch_ref_kind<K_D1>(stream, dir, a, in, out);
  if (kind == K_R3) return launch_ref_kind<K_R3>(stream, dir, a, in, out);
  return launch_ref_kind<K_R4>(stream, dir, a, in, out);
}
#else
int launch_ref(hipStream_t stream, int dir, int kind, const RefArgs& a, const float* in, float* out);
#endif

#if PYR_PART == 0

// FP32 solve setting of one operator and direction: its tuned choice, else the
// context's
static int r32_mode(const pyr_ctx* c, int op, int dir) {
  return c->tune_solve[op][dir] >= 0 ? c->tune_solve[op][dir] : c->r32_solve;
}

// bounded FP32 lines of a context in the refined mode keep the refined FP32
// arithmetic; the FP64 recurrences serve every other line (periodic FP32 lines
// in either mode: a refined solve of them rounds to another last bit at about 1
// point in 30 000)
static bool use_refined(const pyr_ctx* c, int op, int dir) {
  return c->rplan[op][dir].N > 0 && r32_mode(c, op, dir) == PYR_R32_SOLVE_REFINED;
}

template <typename TS>
static int launch_op(pyr_ctx* c, int op, int dir, const TS* in, TS* out, int epi, double ec, bool anti) {
  // anti: the antisymmetric member where the direction has a SYMM end, as
  // d1x/d8x(v, dv, bc=-1) select it (compact_operators.f90:300-303)
  const bool ua = anti && c->has_anti[dir];
  const OpPlan& pl = ua ? c->plan_a[op][dir] : c->plan[op][dir];
  if (pl.null_op) {
    const long long n = (long long)c->npts();
    float* o32 = sizeof(TS) == 8 ? c->out32 : nullptr;
    hipLaunchKernelGGL((k_null<TS>), dim3((n + 255) / 256), dim3(256), 0, c->stream, n,
                       pl.null_option == 1 ? 1 : 0, epi, ec, in, (o32 && c->only32) ? nullptr : out, o32);
    HIPCHECK(hipGetLastError());
    return 0;
  }
  LineArgs a = make_args(c, pl, ua ? c->dplan_a[op][dir] : c->dplan[op][dir], dir, epi, ec,
                         sizeof(TS) == 8 ? PYR_F64 : PYR_R32);
  if (c->out32) {
    // the plain kernels of FP64 fields with the store epilogue write the
    // rounded copy
    if (sizeof(TS) != 8 || epi != EPI_STORE) return fail("an FP32 copy of the output needs an FP64 sweep that stores");
    a.out32 = c->out32;
    a.only32 = c->only32;
  }
  if constexpr (sizeof(TS) == 4) {
    if (use_refined(c, op, dir))
      return launch_ref(c->stream, dir, pl.kind,
                        make_ref_args(a, ua ? c->rplan_a[op][dir] : c->rplan[op][dir],
                                      ua ? c->drplan_a[op][dir] : c->drplan[op][dir]), in, out);
  }
  const int sv = plan_solve(pl);
  const int wd = sizeof(TS) == 8 ? 0 : 1;
  const int forced = c->tune_ly[op][dir][wd] >= 0 ? c->tune_ly[op][dir][wd] : c->yz_lines;
  const bool full = pl.N == pl.P * CHUNK && !(dir != 0 && c->tune_rt[op][dir][wd]);
  return sv == SOLVE_CIRC ? launch_kind<TS, true>(c, dir, pl.kind, sv, full, forced, a, in, out)
                          : launch_kind<TS, false>(c, dir, pl.kind, sv, full, forced, a, in, out);
}

static int check_ctx(pyr_ctx* c) {
  if (!c) return fail("null context");
  if (!c->device) return fail("context was set up host-only (pyr_setup_host)");
  return 0;
}

// one input and one output field of a sweep: what every entry point refuses
static int check_fields(const void* in, const void* out) {
  if (!in || !out) return fail("null field pointer");
  if (in == out) return fail("input and output must not alias");
  return 0;
}

static int apply_any(pyr_ctx* c, int op, int dir, int prec, const void* in, void* out, int epi,
                     double ec, bool anti = false) {
  if (check_ctx(c)) return 1;
  if (op < 0 || op >= NOPS || dir < 0 || dir > 2) return fail("bad operator or direction");
  // (an FP64 sweep that stores only the FP32 rounding has no FP64 output)
  const bool only32 = c->out32 && c->only32;
  if (!in || (!out && !only32)) return fail("null field pointer");
  if (in == out || (void*)in == (void*)c->out32) return fail("input and output must not alias");
  if (only32 && prec != PYR_F64) return fail("an FP32-only result needs an FP64 sweep");
  if (prec == PYR_F64)
    return launch_op<double>(c, op, dir, (const double*)in, (double*)out, epi, ec, anti);
  if (prec == PYR_R32)
    return launch_op<float>(c, op, dir, (const float*)in, (float*)out, epi, ec, anti);
  return fail("bad precision");
}

static int field_temp(pyr_ctx* c, int prec, void** p) {
  const size_t bytes = c->npts() * (prec == PYR_F64 ? sizeof(double) : sizeof(float));
  if (!c->field_tmp[prec]) HIPCHECK(hipMalloc(&c->field_tmp[prec], bytes));
  *p = c->field_tmp[prec];
  return 0;
}

// The directions in which an operator is more than the null operator of a
// short direction (fewer than 4 points). On 2-D and 1-D grids the composites
// below sweep these alone: the identity (filters) or the zero (derivatives) of
// a null direction was a pass over the field of its own, 4.8 us of the 23.4 us
// of the FP64 filter on 1024x512 points (18.7 us without it). A grid with fewer
// than `least` live directions keeps all passes: none live, or one where the
// last pass also stores a rounded copy (which may lie in the input's memory, as
// it may where the sweep before has read the input).
struct Live {
  int n = 0;
  int d[3] = {0, 0, 0};
};
static Live live_dirs(const pyr_ctx* c, int op, int least = 1) {
  Live l;
  for (int d = 0; d < 3; ++d)
    if (!c->plan[op][d].null_op) l.d[l.n++] = d;
  if (l.n < least) {
    l.n = 3;
    for (int d = 0; d < 3; ++d) l.d[d] = d;
  }
  return l;
}

// filter x -> y -> z (operators.f90:847-875); `tmp` is a field temp where more
// than one direction is swept. o32 (if not null) receives the FP32 rounding of
// the result from the last sweep.
static int filter3_with(pyr_ctx* c, int op, int prec, const void* in, void* out, void* tmp, float* o32 = nullptr) {
  if (check_fields(in, out)) return 1;
  const Live l = live_dirs(c, op, o32 ? 2 : 1);
  // the sweeps alternate between tmp and out so that the last one writes out
  const void* src = in;
  for (int i = 0; i < l.n; ++i) {
    const bool last = i == l.n - 1;
    void* dst = (l.n - 1 - i) % 2 ? tmp : out;
    if (last) c->out32 = o32;
    const int r = apply_any(c, op, l.d[i], prec, src, dst, EPI_STORE, 0.0);
    c->out32 = nullptr;
    if (r) return 1;
    src = dst;
  }
  return 0;
}

// filter x -> y -> z (operators.f90:847-875)
static int filter3(pyr_ctx* c, int op, int prec, const void* in, void* out, float* o32 = nullptr) {
  void* tmp = nullptr;
  if (check_ctx(c)) return 1;
  if (live_dirs(c, op, o32 ? 2 : 1).n > 1 && field_temp(c, prec, &tmp)) return 1;
  return filter3_with(c, op, prec, in, out, tmp, o32);
}

// ring L=2 (operators.f90:615-643): max_d |d8_d f| * d_d^2, fused into the
// stores. Every direction keeps its pass: the maximum with a null direction's
// zero clears a NaN, which an epilogue of the last live sweep could only do
// with one more case for every row (ring on 256^3 in FP32 102.9 -> 105.0 us,
// the Laplacian on 192^3 118.4 -> 121.5 us).
static int ring(pyr_ctx* c, int prec, const void* in, void* out) {
  for (int d = 0; d < 3; ++d) {
    const double s = c->dmesh[d] * c->dmesh[d];
    if (apply_any(c, OP_D8, d, prec, in, out, d == 0 ? EPI_ABS : EPI_MAXABS, s)) return 1;
  }
  return 0;
}

// sum over directions of op_d(f_d); anti: each f_d is the normal component of
// direction d and takes the antisymmetric member at SYMM ends (divV,
// operators.f90:38-53)
static int sum3(pyr_ctx* c, int op, int prec, const void* f0, const void* f1, const void* f2,
                void* out, bool anti = false) {
  const void* f[3] = {f0, f1, f2};
  if (check_ctx(c)) return 1;
  for (int d = 0; d < 3; ++d)
    if (check_fields(f[d], out)) return 1;
  const Live l = live_dirs(c, op);
  for (int i = 0; i < l.n; ++i)
    if (apply_any(c, op, l.d[i], prec, f[l.d[i]], out, i == 0 ? EPI_STORE : EPI_ADD, 0.0, anti)) return 1;
  return 0;
}

// ---------------------------------------------------------------------------
// device memory of the entry point that allocates nothing
// ---------------------------------------------------------------------------
// pyr_sfilter_noalloc keeps the field temporary of the x -> y -> z filter in
// this file-scope array (one copy per GPU, resident until the process ends)
// instead of allocating it. Host code never passes `scratch` itself to a
// kernel: its device address on each GPU comes from hipGetSymbolAddress at
// the first pyr_setup on that GPU (noalloc_init) and is kept per device.
constexpr size_t PYR_NOALLOC_BYTES = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[PYR_NOALLOC_BYTES];
constexpr int PYR_MAX_DEVICES = 64;
static std::mutex g_noalloc_mu;
static void* g_noalloc_ptr[PYR_MAX_DEVICES] = {};

static int noalloc_init(int dev, void** ptr) {
  if (dev < 0 || dev >= PYR_MAX_DEVICES) return fail("device ordinal out of range for the filter scratch");
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_noalloc_ptr[dev] = p;
  }
  *ptr = g_noalloc_ptr[dev];
  return 0;
}

// ---------------------------------------------------------------------------
// setup
// ---------------------------------------------------------------------------
static int setup_common(pyr_ctx** out, int nx, int ny, int nz, double x1, double xn, double y1,
                        double yn, double z1, double zn, const int* bc6, bool device) {
  if (!out) return fail("null output handle");
  *out = nullptr;
  if (nx < 1 || ny < 1 || nz < 1) return fail("grid sizes must be >= 1");
  // the y/z kernels address a field through a 32-bit buffer range
  if ((double)nx * ny * nz * sizeof(double) > 2147483647.0) return fail("field exceeds 2 GiB");
  if (!bc6) return fail("null bc array");
  std::unique_ptr<pyr_ctx> c(new pyr_ctx);
  c->n[0] = nx; c->n[1] = ny; c->n[2] = nz;
  if (const char* e = std::getenv("PYRANDA_AMD_X_LDS_KB")) {
    const int kb = std::atoi(e);
    if (kb >= 8 && kb <= 160) c->x_lds_kb = kb;
  }
  for (int i = 0; i < 6; ++i) {
    if (bc6[i] < PYR_BC_PERI || bc6[i] > PYR_BC_SYMM) return fail("bad boundary code");
    c->bc[i] = bc6[i];
  }
  const double lo[3] = {x1, y1, z1}, hi[3] = {xn, yn, zn};
  for (int d = 0; d < 3; ++d) {
    // faces from nodes (parcop.f90:46-56), patch spacing (patch.f90:83-85)
    const double du = (hi[d] - lo[d]) / (double)(c->n[d] - 1 > 1 ? c->n[d] - 1 : 1);
    const double f1 = lo[d] - du / 2.0, fn = hi[d] + du / 2.0;
    c->x1[d] = f1;
    c->dpatch[d] = (fn - f1) / (double)c->n[d];
  }
  // mesh length scales (mesh.f90:190-211)
  c->dmesh[0] = nx == 1 ? std::fmax(c->dpatch[1], c->dpatch[2]) : c->dpatch[0];
  c->dmesh[1] = ny == 1 ? std::fmax(c->dpatch[0], c->dpatch[2]) : c->dpatch[1];
  c->dmesh[2] = nz == 1 ? std::fmax(c->dpatch[0], c->dpatch[1]) : c->dpatch[2];
  c->gridlen = std::fmin(c->dmesh[0], std::fmin(c->dmesh[1], c->dmesh[2]));
  try {
    for (int d = 0; d < 3; ++d) {
      const int periodic = c->bc[2 * d] == PYR_BC_PERI;
      const int v1 = c->bc[2 * d] == PYR_BC_SYMM ? 1 : 0;
      const int v2 = c->bc[2 * d + 1] == PYR_BC_SYMM ? 1 : 0;
      for (int op = 0; op < NOPS; ++op) {
        c->plan[op][d] = build_plan(op, c->n[d], d, periodic, v1, v2, c->dpatch[d]);
        if (!periodic && c->plan[op][d].implicit && !c->plan[op][d].null_op)
          c->rplan[op][d] = build_ref_plan(op, c->n[d], v1, v2, c->dpatch[d]);
      }
      c->has_anti[d] = !periodic && (v1 || v2) && c->n[d] >= 4;
      if (c->has_anti[d])
        for (int op = 0; op < NOPS; ++op) {
          c->plan_a[op][d] = build_plan(op, c->n[d], d, periodic, -v1, -v2, c->dpatch[d]);
          if (c->plan_a[op][d].implicit) c->rplan_a[op][d] = build_ref_plan(op, c->n[d], -v1, -v2, c->dpatch[d]);
        }
    }
  } catch (const std::exception& e) {
    return fail(std::string("setup: ") + e.what());
  }
  if (device) {
    int dev = 0;
    HIPCHECK(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0)
      c->ncu = prop.multiProcessorCount;
    // once per GPU, with that GPU current: its copy of the scratch array
    if (noalloc_init(dev, &c->noalloc_tmp)) return 1;
    if (upload_plans(c.get())) {
      if (c->tables) (void)hipFree(c->tables);
      return 1;
    }
    c->device = true;
  }
  *out = c.release();
  return 0;
}

// ---------------------------------------------------------------------------
// host emulation of the kernels (tests only): the same per-thread arithmetic,
// chunk by chunk, with the LDS exchanges as plain arrays
// ---------------------------------------------------------------------------
template <typename TS, int KIND, int SOLVE>
static void emulate_line(const LineArgs& a, const TS* vin, long long stride, TS* vout) {
  constexpr int R = Halo<KIND>::R;
  struct St {
    TS win[CHUNK + 2 * R];
    double x[CHUNK];
    double e[2], b[2];
    int s, m;
  };
  const int P = a.P, N = a.N;
  std::vector<St> st(P);
  const Tables tabs(a.tab, a.T);
  auto rows_of = [&](int p, auto f) {
    if (SOLVE == SOLVE_BND && (p < a.tlo || p == P - 1)) f(TableRows{tabs, a.T, slot_of(a, p)});
    else f(ConstRows{a.p1, a.p2});
  };
  auto carry = [&](int p, auto step, double& e0, double& e1) {
    constexpr int STEP = decltype(step)::value;
    auto read = [&](int q, double& u0, double& u1) {
      const double* u = STEP < 0 ? st[q].e : st[q].b;
      u0 = u[0];
      u1 = u[1];
    };
    if constexpr (SOLVE == SOLVE_BND)
      carry_in<false, STEP>(a, p, [&](int q) { return tabs.th + 8 * slot_of(a, q) + (STEP > 0 ? 4 : 0); }, read, e0, e1);
    else
      carry_in<true, STEP>(a, p, [&](int q) { return (STEP < 0 ? a.hf : a.hb)[q < a.mx ? 0 : 1]; }, read, e0, e1);
  };
  for (int p = 0; p < P; ++p) {
    St& t = st[p];
    t.s = chunk_start(a, p);
    t.m = chunk_start(a, p + 1) - t.s;
    for (int w = 0; w < CHUNK + 2 * R; ++w) {
      int row = t.s - R + w;
      TS v = (TS)0;
      if (w < t.m + 2 * R && (a.periodic || (row >= 0 && row < N))) {
        row = row < 0 ? row + N : (row >= N ? row - N : row);
        v = vin[stride * row];
      }
      t.win[w] = v;
    }
    B4 lo = {}, hi = {};
    if (!a.periodic) boundary_rows<KIND, SOLVE == SOLVE_NONE, false>(a, tabs.wb, p, t.win, lo, hi);
    right_hand_side<KIND, SOLVE>(a, t.win, t.x);
    if (!a.periodic) put_boundary_rows<false>(a, p, lo, hi, t.x);
    if (SOLVE == SOLVE_NONE) continue;
    t.e[0] = t.e[1] = 0.0;
    rows_of(p, [&](auto rows) { fwd_pass<false>(ChunkRows{a.mb, p < a.mx}, rows, t.x, t.e[0], t.e[1]); });
  }
  bool bad = false;
  if (SOLVE != SOLVE_NONE)
    for (int p = 0; p < P; ++p) {
      St& t = st[p];
      double e0, e1;
      carry(p, std::integral_constant<int, -1>(), e0, e1);
      t.b[0] = t.b[1] = 0.0;
      rows_of(p, [&](auto rows) {
        fwd_pass<true>(ChunkRows{a.mb, p < a.mx}, rows, t.x, e0, e1);
        bwd_exit(ChunkRows{a.mb, p < a.mx}, rows, t.x, t.b[0], t.b[1]);
      });
      bad = bad || !std::isfinite(t.b[0]) || !std::isfinite(t.b[1]);
    }
  for (int p = 0; p < P; ++p) {
    St& t = st[p];
    auto emit = [&](int k, double y) {
      double val = y * a.scale;
      if (a.addv) val += (double)t.win[k + R];
      vout[stride * (t.s + k)] = (TS)val;
    };
    if (SOLVE == SOLVE_NONE) {
      for (int k = 0; k < t.m; ++k) emit(k, t.x[k]);
      continue;
    }
    double b0, b1;
    carry(p, std::integral_constant<int, 1>(), b0, b1);
    if (bad) b0 = b1 = std::nan("");
    rows_of(p, [&](auto rows) { bwd_sink(ChunkRows{a.mb, p < a.mx}, rows, t.x, b0, b1, emit); });
  }
}

template <int KIND>
static void emulate_ref_line(const RefArgs& a, const float* vin, long long stride, float* vout) {
  constexpr int R = Halo<KIND>::R;
  struct St {
    float win[RCHUNK + 2 * R];
    double rhs[RCHUNK];
    float x[RCHUNK], d[RCHUNK], z[4];
    const float* t;
    int s, m;
  };
  const int P = a.P, N = a.N;
  std::vector<St> st(P);
  std::vector<F4> Y(P), Yd(P);
  auto rd = [&](int i) { return vin[stride * i]; };
  bool bad = false;
  for (int p = 0; p < P; ++p) {
    St& t = st[p];
    t.s = p * a.mb + std::min(p, a.mx);
    t.m = a.mb + (p < a.mx ? 1 : 0);
    t.t = a.cls + ref_class(p, P, a.mx) * (RCHUNK * CROW);
    for (int w = 0; w < RCHUNK + 2 * R; ++w) {
      const int row = t.s - R + w;
      t.win[w] = w < t.m + 2 * R && row >= 0 && row < N ? rd(row) : 0.0f;
    }
    ref_rhs_interior<KIND>(a, t.win, t.rhs);
    ref_rhs_boundary(a, p, t.rhs, [&](int slot) { return end_value(slot, N, rd); });
    ref_local_solve(a, p < a.mx, t.t, t.rhs, t.x);
    Y[p] = ref_edges(a, p < a.mx, t.x);
    bad = bad || !std::isfinite(Y[p].x) || !std::isfinite(Y[p].y);
  }
  for (int p = 0; p < P; ++p) {
    St& t = st[p];
    ref_neighbours(a, a.g, p, [&](int q) { return Y[q]; }, t.z);
    if (bad) t.z[0] = t.z[1] = t.z[2] = t.z[3] = std::nanf("");
    ref_spike(a, t.t, t.z, t.x);
    ref_residual(a, p, p < a.mx, t.rhs, t.x, t.z, t.d);
    ref_local_solve(a, p < a.mx, t.t, t.d, t.d);
    Yd[p] = ref_edges(a, p < a.mx, t.d);
  }
  for (int p = 0; p < P; ++p) {
    St& t = st[p];
    ref_neighbours(a, a.g, p, [&](int q) { return Yd[q]; }, t.z);
    ref_spike(a, t.t, t.z, t.d);
    for (int k = 0; k < t.m; ++k) {
      double val = ((double)t.x[k] + (double)t.d[k]) * a.scale;
      if (a.addv) val += (double)t.win[k + R];
      vout[stride * (t.s + k)] = (float)val;
    }
  }
}

template <typename TS>
static int emulate(pyr_ctx* c, int op, int dir, const TS* in, TS* out, bool anti) {
  const bool ua = anti && c->has_anti[dir];
  const OpPlan& pl = ua ? c->plan_a[op][dir] : c->plan[op][dir];
  const size_t n = c->npts();
  if (pl.null_op) {
    for (size_t i = 0; i < n; ++i) out[i] = pl.null_option == 1 ? in[i] : (TS)0;
    return 0;
  }
  const std::vector<double> tab = with_boundary_rows(pl);
  DevPlan d;
  d.tab = tab.data();
  const LineArgs a = make_args(c, pl, d, dir, EPI_STORE, 0.0, sizeof(TS) == 8 ? PYR_F64 : PYR_R32);
  const int sv = plan_solve(pl);
  const bool refined = sizeof(TS) == 4 && use_refined(c, op, dir);
  RefArgs ra;
  if (refined) {
    const RefPlan& rp = ua ? c->rplan_a[op][dir] : c->rplan[op][dir];
    DevRefPlan rd;
    host_ref_tables(rp, rd);
    ra = make_ref_args(a, rp, rd);
  }
  for (long long L = 0; L < a.nlines; ++L) {
    const long long base = (dir == 0) ? L * pl.N : (L % a.A) + a.B * (L / a.A);
    const TS* vi = in + base;
    TS* vo = out + base;
    if constexpr (sizeof(TS) == 4) {
      if (refined) {
        if (pl.kind == K_D1) emulate_ref_line<K_D1>(ra, vi, a.stride, vo);
        else if (pl.kind == K_R3) emulate_ref_line<K_R3>(ra, vi, a.stride, vo);
        else emulate_ref_line<K_R4>(ra, vi, a.stride, vo);
        continue;
      }
    }
    switch (pl.kind) {
      case K_D1:
        if (sv == SOLVE_CIRC) emulate_line<TS, K_D1, SOLVE_CIRC>(a, vi, a.stride, vo);
        else emulate_line<TS, K_D1, SOLVE_BND>(a, vi, a.stride, vo);
        break;
      case K_R3:
        if (sv == SOLVE_CIRC) emulate_line<TS, K_R3, SOLVE_CIRC>(a, vi, a.stride, vo);
        else emulate_line<TS, K_R3, SOLVE_BND>(a, vi, a.stride, vo);
        break;
      default:
        if (sv == SOLVE_CIRC) emulate_line<TS, K_R4, SOLVE_CIRC>(a, vi, a.stride, vo);
        else if (sv == SOLVE_BND) emulate_line<TS, K_R4, SOLVE_BND>(a, vi, a.stride, vo);
        else emulate_line<TS, K_R4, SOLVE_NONE>(a, vi, a.stride, vo);
    }
  }
  return 0;
}

#endif  // PYR_PART == 0

// ---------------------------------------------------------------------------
// groups: one operator over the fields of several simulations
// ---------------------------------------------------------------------------
// Members of a group are contexts of any grid sizes whose fields live in one
// allocation (member m at off[m] elements). An operator along one direction
// runs as ONE grouped launch over every member, plus a k_null launch for a
// member whose direction is a null operator. The per-member line arguments of
// a launch are built once per (operator, direction, precision, epilogue) and
// kept on the device.
struct GrpLaunch {
  void* dev = nullptr;  // GrpEntry or, with refined, RefEntry per member
  bool refined = false;
  const int* member = nullptr;  // member of each workgroup, after the entries in dev
  long long nblocks = 0;
  dim3 block;
  size_t shm = 0;
  int kind = 0, solve = 0, pre = 0;
  bool x = false, addv = false;
};
struct GrpNull {
  int member;
  int copy;
  double ec;
};
struct GrpPlan {
  std::vector<GrpLaunch> launches;
  std::vector<GrpNull> nulls;
};
struct GrpKey {
  int op, dir, prec, epi, power, aligned;
  int refined;  // FP32 solve arithmetic (a part of the plan)
  double ec;
  bool operator<(const GrpKey& o) const {
    if (op != o.op) return op < o.op;
    if (dir != o.dir) return dir < o.dir;
    if (prec != o.prec) return prec < o.prec;
    if (refined != o.refined) return refined < o.refined;
    if (epi != o.epi) return epi < o.epi;
    if (power != o.power) return power < o.power;
    if (aligned != o.aligned) return aligned < o.aligned;
    return ec < o.ec;
  }
};
struct pyr_group {
  std::vector<pyr_ctx*> mem;
  std::vector<long long> off;
  hipStream_t stream = nullptr;
  std::map<GrpKey, GrpPlan> plans;
  ~pyr_group() {
    for (auto& kv : plans)
      for (auto& l : kv.second.launches)
        if (l.dev) (void)hipFree(l.dev);
  }
};

#if PYR_PART == 0
template <typename TS>
static int grp_build(pyr_group* g, const GrpKey& key, GrpPlan& gp) {
  const int M = (int)g->mem.size();
  std::vector<int> ms;
  for (int m = 0; m < M; ++m) {
    pyr_ctx* c = g->mem[m];
    const OpPlan& pl = c->plan[key.op][key.dir];
    const double ec = key.ec * std::pow(c->dmesh[key.dir], (double)key.power);
    if (pl.null_op) gp.nulls.push_back({m, pl.null_option == 1 ? 1 : 0, ec});
    else ms.push_back(m);
  }
  if (ms.empty()) return 0;
  const OpPlan& pl0 = g->mem[ms[0]]->plan[key.op][key.dir];
  const int sv = plan_solve(pl0);
  std::vector<GrpEntry> all(ms.size());
  for (size_t j = 0; j < ms.size(); ++j) {
    pyr_ctx* c = g->mem[ms[j]];
    const OpPlan& pl = c->plan[key.op][key.dir];
    if (plan_solve(pl) != sv || pl.kind != pl0.kind)
      return fail("group members differ in boundary conditions along a direction");
    const double ec = key.ec * std::pow(c->dmesh[key.dir], (double)key.power);
    all[j].a = make_args(c, pl, c->dplan[key.op][key.dir], key.dir, key.epi, ec, key.prec);
    all[j].off = g->off[ms[j]];
  }
  GrpLaunch L;
  L.kind = pl0.kind;
  L.solve = sv;
  L.x = key.dir == 0;
  std::vector<int> member;  // of each workgroup
  auto upload = [&](const void* host, size_t bytes) -> int {
    std::vector<unsigned char> image(bytes + member.size() * sizeof(int));
    std::memcpy(image.data(), host, bytes);
    std::memcpy(image.data() + bytes, member.data(), member.size() * sizeof(int));
    HIPCHECK(hipMalloc(&L.dev, image.size()));
    L.member = reinterpret_cast<const int*>(static_cast<unsigned char*>(L.dev) + bytes);
    L.nblocks = (long long)member.size();
    gp.launches.push_back(L);
    HIPCHECK(hipMemcpy(L.dev, image.data(), image.size(), hipMemcpyHostToDevice));
    return 0;
  };
  auto add_blocks = [&](size_t j, int nlines, int per, int times = 1) {
    const long long blk0 = (long long)member.size();
    member.insert(member.end(), (size_t)((nlines + per - 1) / per) * times, (int)j);
    return blk0;
  };
  const int pre = pre_of(pl0.kind, all[0].a.addv, key.epi, false);
  if (key.refined && sv == SOLVE_BND) {
    std::vector<RefEntry> ref(all.size());
    size_t lds = 0;
    for (size_t j = 0; j < all.size(); ++j) {
      pyr_ctx* c = g->mem[ms[j]];
      RefArgs& a = ref[j].a;
      a = make_ref_args(all[j].a, c->rplan[key.op][key.dir], c->drplan[key.op][key.dir]);
      a.vec = key.aligned && ((all[j].off * (long long)sizeof(float)) % 16 == 0);
      a.lines = L.x ? 64 / a.P : ref_lines(a.P);
      ref[j].off = all[j].off;
      ref[j].blk0 = add_blocks(j, a.nlines, L.x ? a.lines * REF_X_WAVES : a.lines);
      lds = std::max(lds, ref_lds(a));
    }
    L.shm = lds;
    L.refined = true;
    L.pre = pre;
    L.addv = all[0].a.addv;
    L.block = dim3(L.x ? 64 * REF_X_WAVES : REF_THREADS);
    return upload(ref.data(), ref.size() * sizeof(RefEntry));
  }
  int nthr = 64, ntab = 0;
  for (auto& e : all) ntab = std::max(ntab, e.a.ntab);
  if (L.x) {
    nthr = 64 * (sv == SOLVE_BND ? XWaves<SOLVE_BND>::v : 1);
    L.shm = (size_t)ntab * sizeof(double);
  } else {
    // 512 chunk threads a workgroup (64 lines of 8 chunks to 16 of 32), 1024
    // where a member's lines have more than 32 chunks
    int Pmax = 1;
    for (auto& e : all) Pmax = std::max(Pmax, e.a.P);
    nthr = sv == SOLVE_NONE ? NONE_THREADS : (Pmax > 32 ? WG_MAX : WG_MAX / 2);
    L.shm = yz_lds(sv, nthr, 128, ntab);
  }
  L.pre = pre;
  L.addv = all[0].a.addv;
  L.block = dim3(nthr);
  for (size_t j = 0; j < all.size(); ++j) {
    GrpEntry& e = all[j];
    if (L.x) {
      e.a.vec = key.aligned && ((e.off * (long long)sizeof(TS)) % 16 == 0);
      e.a.lines = 64 / e.a.P;
    } else {
      e.a.lines = sv == SOLVE_NONE ? 64 : 128;
      while (sv != SOLVE_NONE && e.a.lines * e.a.P > nthr) e.a.lines /= 2;
    }
    e.blk0 = add_blocks(j, e.a.nlines, L.x ? e.a.lines * (nthr / 64) : e.a.lines,
                        !L.x && sv == SOLVE_NONE ? explicit_groups(e.a.P, nthr, e.a.lines) : 1);
  }
  return upload(all.data(), all.size() * sizeof(GrpEntry));
}

#endif  // PYR_PART == 0

template <typename TS, int KIND, int SOLVE>
static int grp_launch_typed(pyr_group* g, const GrpLaunch& L, const TS* in, TS* out) {
  if (L.nblocks <= 0) return 0;
  const dim3 grid((unsigned)L.nblocks);
  auto k = L.x ? k_line_x_grp<TS, KIND, SOLVE, KIND == K_R4 ? PRE_ANY : PRE_OLD>
               : k_line_yz_grp<TS, KIND, SOLVE, PRE_ANY>;
  if constexpr (KIND == K_R4) {
    if (L.pre == PRE_V) k = L.x ? k_line_x_grp<TS, KIND, SOLVE, PRE_V> : k_line_yz_grp<TS, KIND, SOLVE, PRE_V>;
  }
  if constexpr (SOLVE != SOLVE_NONE) {
    if (L.pre == PRE_NONE) k = L.x ? k_line_x_grp<TS, KIND, SOLVE, PRE_NONE> : k_line_yz_grp<TS, KIND, SOLVE, PRE_NONE>;
    else if (L.x && !L.addv) k = k_line_x_grp<TS, KIND, SOLVE, PRE_OLD>;
    else if (L.pre == PRE_OLD) k = k_line_yz_grp<TS, KIND, SOLVE, PRE_OLD>;
  }
  hipLaunchKernelGGL(k, grid, L.block, L.shm, g->stream, (const GrpEntry*)L.dev, L.member, in, out);
  HIPCHECK(hipGetLastError());
  return 0;
}

template <typename TS>
int grp_launch(pyr_group* g, const GrpLaunch& L, const TS* in, TS* out) {
  switch (L.kind) {
    case K_D1:
      return L.solve == SOLVE_CIRC ? grp_launch_typed<TS, K_D1, SOLVE_CIRC>(g, L, in, out)
                                   : grp_launch_typed<TS, K_D1, SOLVE_BND>(g, L, in, out);
    case K_R3:
      return L.solve == SOLVE_CIRC ? grp_launch_typed<TS, K_R3, SOLVE_CIRC>(g, L, in, out)
                                   : grp_launch_typed<TS, K_R3, SOLVE_BND>(g, L, in, out);
    default:
      if (L.solve == SOLVE_CIRC) return grp_launch_typed<TS, K_R4, SOLVE_CIRC>(g, L, in, out);
      if (L.solve == SOLVE_BND) return grp_launch_typed<TS, K_R4, SOLVE_BND>(g, L, in, out);
      return grp_launch_typed<TS, K_R4, SOLVE_NONE>(g, L, in, out);
  }
}

#if PYR_PART == 7
template <int KIND>
static auto ref_x_kernel_grp(int pre, bool addv) {
  if constexpr (KIND == K_R4) {
    if (addv) return pre == PRE_V ? k_ref_x_grp<KIND, PRE_V> : k_ref_x_grp<KIND, PRE_ANY>;
  }
  return pre == PRE_NONE ? k_ref_x_grp<KIND, PRE_NONE> : k_ref_x_grp<KIND, PRE_OLD>;
}
template <int KIND>
static int grp_launch_ref_kind(hipStream_t stream, const GrpLaunch& L, const float* in, float* out) {
  if (L.nblocks <= 0) return 0;
  auto k = k_ref_yz_grp<KIND, PRE_ANY>;
  if constexpr (KIND == K_R4) {
    if (L.pre == PRE_V) k = k_ref_yz_grp<KIND, PRE_V>;
  }
  if (L.pre == PRE_NONE) k = k_ref_yz_grp<KIND, PRE_NONE>;
  if (L.pre == PRE_OLD) k = k_ref_yz_grp<KIND, PRE_OLD>;
  if (L.x) k = ref_x_kernel_grp<KIND>(L.pre, L.addv);
  hipLaunchKernelGGL(k, dim3((unsigned)L.nblocks), L.block, L.shm, stream, (const RefEntry*)L.dev, L.member, in, out);
  HIPCHECK(hipGetLastError());
  return 0;
}
int grp_launch_ref(hipStream_t stream, const GrpLaunch& L, const float* in, float* out) {
  if (L.kind == K_D1) return grp_launch_ref_kind<K_D1>(stream, L, in, out);
  if (L.kind == K_R3) return grp_launch_ref_kind<K_R3>(stream, L, in, out);
  return grp_launch_ref_kind<K_R4>(stream, L, in, out);
}
#else
int grp_launch_ref(hipStream_t stream, const GrpLaunch& L, const float* in, float* out);
#endif

#define PYR_GRP(TS) template int grp_launch<TS>(pyr_group*, const GrpLaunch&, const TS*, TS*);
#if PYR_PART == 5
PYR_GRP(double)
#elif PYR_PART == 6
PYR_GRP(float)
#elif PYR_PART == 0
extern PYR_GRP(double)
extern PYR_GRP(float)
#endif
#undef PYR_GRP

#if PYR_PART == 0
template <typename TS>
static int grp_apply(pyr_group* g, const GrpKey& key, const TS* in, TS* out) {
  auto it = g->plans.find(key);
  if (it == g->plans.end()) {
    GrpPlan gp;
    if (grp_build<TS>(g, key, gp)) {
      for (auto& l : gp.launches)
        if (l.dev) (void)hipFree(l.dev);
      return 1;
    }
    it = g->plans.emplace(key, std::move(gp)).first;
  }
  for (const GrpLaunch& L : it->second.launches) {
    if constexpr (sizeof(TS) == 4) {
      if (L.refined) {
        if (grp_launch_ref(g->stream, L, in, out)) return 1;
        continue;
      }
    }
    if (grp_launch<TS>(g, L, in, out)) return 1;
  }
  for (const GrpNull& z : it->second.nulls) {
    const long long n = (long long)g->mem[z.member]->npts();
    const long long o = g->off[z.member];
    hipLaunchKernelGGL((k_null<TS>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, g->stream, n, z.copy,
                       key.epi, z.ec, in + o, out + o, nullptr);
    HIPCHECK(hipGetLastError());
  }
  return 0;
}

// ---------------------------------------------------------------------------
// C-ABI
// ---------------------------------------------------------------------------
extern "C" {

const char* pyr_last_error(void) { return g_err.c_str(); }

int pyr_setup(pyr_ctx** ctx, int nx, int ny, int nz, double x1, double xn, double y1, double yn,
              double z1, double zn, const int* bc6) {
  return setup_common(ctx, nx, ny, nz, x1, xn, y1, yn, z1, zn, bc6, true);
}

int pyr_setup_host(pyr_ctx** ctx, int nx, int ny, int nz, double x1, double xn, double y1,
                   double yn, double z1, double zn, const int* bc6) {
  return setup_common(ctx, nx, ny, nz, x1, xn, y1, yn, z1, zn, bc6, false);
}

int pyr_destroy(pyr_ctx* c) {
  if (!c) return 0;
  if (c->device) {
    if (c->tables) (void)hipFree(c->tables);
    for (int i = 0; i < 2; ++i)
      if (c->field_tmp[i]) (void)hipFree(c->field_tmp[i]);
  }
  delete c;
  return 0;
}

int pyr_set_stream(pyr_ctx* c, void* stream) {
  if (!c) return fail("null context");
  c->stream = (hipStream_t)stream;
  return 0;
}

int pyr_set_r32_solve(pyr_ctx* c, int mode) {
  if (!c) return fail("null context");
  if (mode != PYR_R32_SOLVE_REFINED && mode != PYR_R32_SOLVE_FP64) return fail("bad r32 solve mode");
  c->r32_solve = mode;
  return 0;
}

int pyr_set_tuning(pyr_ctx* c, int op, int dir, int prec, int x_lds_kb, int yz_pipe, int yz_lines) {
  if (!c) return fail("null context");
  if (op < 0 || op >= NOPS || dir < 0 || dir > 2) return fail("bad operator or direction");
  if (x_lds_kb >= 0 && (x_lds_kb < 8 || x_lds_kb > 160)) return fail("x_lds_kb must be 8..160 (or -1)");
  if (yz_pipe > 3 || (yz_pipe == 2 && dir != 0) || (yz_pipe == 3 && dir == 0))
    return fail("yz_pipe must be 0, 1, 2 (x) or 3 (y/z) (or -1)");
  if (yz_lines >= 0 && yz_lines != 16 && yz_lines != 32 && yz_lines != 64)
    return fail("yz_lines must be 16, 32 or 64 (or -1)");
  if (prec != PYR_F64 && prec != PYR_R32) return fail("bad precision");
  const int wd = prec == PYR_F64 ? 0 : 1;
  c->tune_ly[op][dir][wd] = yz_lines < 0 ? -1 : yz_lines;
  c->tune_rt[op][dir][wd] = yz_pipe == 3;
  return 0;
}

int pyr_set_solve_tuning(pyr_ctx* c, int op, int dir, int r32_solve) {
  if (!c) return fail("null context");
  if (op < 0 || op >= NOPS || dir < 0 || dir > 2) return fail("bad operator or direction");
  if (r32_solve != -1 && r32_solve != PYR_R32_SOLVE_REFINED && r32_solve != PYR_R32_SOLVE_FP64)
    return fail("bad r32 solve mode");
  c->tune_solve[op][dir] = r32_solve;
  return 0;
}

int pyr_set_periodic_solver(pyr_ctx* c, int mode) {
  if (!c) return fail("null context");
  if (mode != PYR_PSOLVE_CIRCULANT && mode != PYR_PSOLVE_LU) return fail("bad periodic solver");
  c->periodic_solver = mode;
  return 0;
}

int pyr_axis_coords(pyr_ctx* c, int axis, double* coords) {
  if (!c || !coords || axis < 0 || axis > 2) return fail("bad arguments to pyr_axis_coords");
  // xgrid = x1f + (2i-1)*half*dx (mesh.f90:173-177)
  for (int i = 1; i <= c->n[axis]; ++i)
    coords[i - 1] = c->x1[axis] + (double)(2 * i - 1) * 0.5 * c->dpatch[axis];
  return 0;
}

int pyr_mesh_scalars(pyr_ctx* c, double* dpatch3, double* dmesh3, double* gridlen) {
  if (!c) return fail("null context");
  for (int d = 0; d < 3; ++d) {
    if (dpatch3) dpatch3[d] = c->dpatch[d];
    if (dmesh3) dmesh3[d] = c->dmesh[d];
  }
  if (gridlen) *gridlen = c->gridlen;
  return 0;
}

int pyr_apply(pyr_ctx* c, int op, int dir, int prec, const void* in, void* out, int epi,
              double epi_scale) {
  if (epi < PYR_EPI_STORE || epi > PYR_EPI_MAXABS_SCALED) return fail("bad epilogue");
  const bool anti = (op & PYR_OP_ANTISYM) != 0;
  return apply_any(c, op & ~PYR_OP_ANTISYM, dir, prec, in, out, epi, epi_scale, anti);
}

#define PYR_DIR_OP(name, op, dir)                                                     \
  int name##_f64(pyr_ctx* c, const double* v, double* o) {                           \
    return apply_any(c, op, dir, PYR_F64, v, o, EPI_STORE, 0.0);                     \
  }
PYR_DIR_OP(pyr_ddx, OP_D1, 0)
PYR_DIR_OP(pyr_ddy, OP_D1, 1)
PYR_DIR_OP(pyr_ddz, OP_D1, 2)
PYR_DIR_OP(pyr_dd8x, OP_D8, 0)
PYR_DIR_OP(pyr_dd8y, OP_D8, 1)
PYR_DIR_OP(pyr_dd8z, OP_D8, 2)
PYR_DIR_OP(pyr_d2x, OP_D2, 0)
PYR_DIR_OP(pyr_d2y, OP_D2, 1)
PYR_DIR_OP(pyr_d2z, OP_D2, 2)
#undef PYR_DIR_OP

int pyr_ddx_r32(pyr_ctx* c, const float* v, float* o) { return apply_any(c, OP_D1, 0, PYR_R32, v, o, EPI_STORE, 0.0); }
int pyr_ddy_r32(pyr_ctx* c, const float* v, float* o) { return apply_any(c, OP_D1, 1, PYR_R32, v, o, EPI_STORE, 0.0); }
int pyr_ddz_r32(pyr_ctx* c, const float* v, float* o) { return apply_any(c, OP_D1, 2, PYR_R32, v, o, EPI_STORE, 0.0); }

int pyr_plaplacian_f64(pyr_ctx* c, const double* v, double* o) { return sum3(c, OP_D2, PYR_F64, v, v, v, o); }
int pyr_plaplacian_r32(pyr_ctx* c, const float* v, float* o) { return sum3(c, OP_D2, PYR_R32, v, v, v, o); }
int pyr_pring_f64(pyr_ctx* c, const double* v, double* o) { return ring(c, PYR_F64, v, o); }
int pyr_pring_r32(pyr_ctx* c, const float* v, float* o) { return ring(c, PYR_R32, v, o); }

int pyr_pringv_f64(pyr_ctx* c, const double* vx, const double* vy, const double* vz, double* o) {
  // ringV L=1 (operators.f90:645-699): max over components and directions of |d8| * d
  const double* f[3] = {vx, vy, vz};
  bool first = true;
  for (int d = 0; d < 3; ++d)
    for (int comp = 0; comp < 3; ++comp) {
      // the normal component takes the antisymmetric member at SYMM ends
      // (ringx(f,..,isymX) etc., operators.f90:661-671)
      if (apply_any(c, OP_D8, d, PYR_F64, f[comp], o, first ? EPI_ABS : EPI_MAXABS, c ? c->dmesh[d] : 0.0,
                    comp == d))
        return 1;
      first = false;
    }
  return 0;
}

int pyr_sfilter_f64(pyr_ctx* c, const double* v, double* o) { return filter3(c, OP_SF, PYR_F64, v, o); }
int pyr_apply_rounded(pyr_ctx* c, int op, int dir, const double* in, double* out, float* o32) {
  if (check_ctx(c)) return 1;
  if (!o32 || !out) return fail("null field pointer");
  c->out32 = o32;
  const int r = apply_any(c, op, dir, PYR_F64, in, out, EPI_STORE, 0.0);
  c->out32 = nullptr;
  return r;
}
int pyr_apply_to_r32(pyr_ctx* c, int op, int dir, const double* in, float* o32) {
  if (check_ctx(c)) return 1;
  if (!o32 || !in) return fail("null field pointer");
  c->out32 = o32;
  c->only32 = 1;
  const int r = apply_any(c, op, dir, PYR_F64, in, nullptr, EPI_STORE, 0.0);
  c->out32 = nullptr;
  c->only32 = 0;
  return r;
}
int pyr_sfilter_f64_rounded(pyr_ctx* c, const double* v, double* o, float* o32) {
  if (check_ctx(c)) return 1;
  if (!o32) return fail("null field pointer");
  // (the last sweep also stores the FP32 rounding of the result)
  return filter3(c, OP_SF, PYR_F64, v, o, o32);
}
int pyr_sfilter_r32(pyr_ctx* c, const float* v, float* o) { return filter3(c, OP_SF, PYR_R32, v, o); }
int pyr_sfilter_noalloc(pyr_ctx* c, int prec, const void* v, void* o) {
  // pyr_sfilter_f64/_r32 with the field temporary in `scratch` (this device's
  // copy, from pyr_setup): no allocation; overlapping calls on one GPU race
  if (check_ctx(c)) return 1;
  if (prec != PYR_F64 && prec != PYR_R32) return fail("bad precision");
  if (!v || !o) return fail("null field pointer");
  const size_t bytes = c->npts() * (prec == PYR_F64 ? sizeof(double) : sizeof(float));
  if (bytes > PYR_NOALLOC_BYTES)
    return fail("pyr_sfilter_noalloc: the field needs " + std::to_string(bytes) +
                " bytes of temporary, above the 64 MiB scratch (use pyr_sfilter_f64/_r32)");
  if (!c->noalloc_tmp) return fail("pyr_sfilter_noalloc: no scratch address for this context's device");
  return filter3_with(c, OP_SF, prec, v, o, c->noalloc_tmp);
}
int pyr_gfilter_f64(pyr_ctx* c, const double* v, double* o) { return filter3(c, OP_GF, PYR_F64, v, o); }
int pyr_gfilter_r32(pyr_ctx* c, const float* v, float* o) { return filter3(c, OP_GF, PYR_R32, v, o); }
int pyr_gfilterdir_f64(pyr_ctx* c, const double* v, double* o, int dir) {
  if (dir < 1 || dir > 3) return fail("gfilterdir direction must be 1, 2 or 3");
  return apply_any(c, OP_GF, dir - 1, PYR_F64, v, o, EPI_STORE, 0.0);
}
int pyr_gfilterdir_r32(pyr_ctx* c, const float* v, float* o, int dir) {
  if (dir < 1 || dir > 3) return fail("gfilterdir direction must be 1, 2 or 3");
  return apply_any(c, OP_GF, dir - 1, PYR_R32, v, o, EPI_STORE, 0.0);
}
int pyr_grads_f64(pyr_ctx* c, const double* v, double* a, double* b, double* e) {
  if (apply_any(c, OP_D1, 0, PYR_F64, v, a, EPI_STORE, 0.0)) return 1;
  if (apply_any(c, OP_D1, 1, PYR_F64, v, b, EPI_STORE, 0.0)) return 1;
  return apply_any(c, OP_D1, 2, PYR_F64, v, e, EPI_STORE, 0.0);
}
int pyr_grads_r32(pyr_ctx* c, const float* v, float* a, float* b, float* e) {
  if (apply_any(c, OP_D1, 0, PYR_R32, v, a, EPI_STORE, 0.0)) return 1;
  if (apply_any(c, OP_D1, 1, PYR_R32, v, b, EPI_STORE, 0.0)) return 1;
  return apply_any(c, OP_D1, 2, PYR_R32, v, e, EPI_STORE, 0.0);
}
int pyr_divergence_f64(pyr_ctx* c, const double* fx, const double* fy, const double* fz, double* o) {
  return sum3(c, OP_D1, PYR_F64, fx, fy, fz, o, true);
}
int pyr_divergence_r32(pyr_ctx* c, const float* fx, const float* fy, const float* fz, float* o) {
  return sum3(c, OP_D1, PYR_R32, fx, fy, fz, o, true);
}

static int rk_update(hipStream_t stream, int prec, long long n, const void* F, double* PHI, const void* Uin,
                     void* Uout, double* U64, const double* dtp, const int* mid, double dt, double A,
                     double B) {
  // with an FP64 state the rounded field may be left unwritten (Uout null)
  if (!F || !PHI || (!U64 && (!Uin || !Uout))) return fail("null pointer to pyr_rk_update");
  if (n <= 0) return 0;
  long long blocks = (n + 1023) / 1024;
  if (blocks > 8192) blocks = 8192;
  if (prec == PYR_F64)
    hipLaunchKernelGGL((k_rk_update<double, double>), dim3((unsigned)blocks), dim3(256), 0, stream, n,
                       (const double*)F, PHI, (const double*)Uin, (double*)Uout, U64, dtp, mid, dt, A, B);
  else if (prec == PYR_R32)
    hipLaunchKernelGGL((k_rk_update<float, float>), dim3((unsigned)blocks), dim3(256), 0, stream, n,
                       (const float*)F, PHI, (const float*)Uin, (float*)Uout, U64, dtp, mid, dt, A, B);
  else if (prec == PYR_RK_F32_U64)
    hipLaunchKernelGGL((k_rk_update<float, double>), dim3((unsigned)blocks), dim3(256), 0, stream, n,
                       (const float*)F, PHI, (const double*)Uin, (double*)Uout, U64, dtp, mid, dt, A, B);
  else if (prec == PYR_RK_F64_U32)
    hipLaunchKernelGGL((k_rk_update<double, float>), dim3((unsigned)blocks), dim3(256), 0, stream, n,
                       (const double*)F, PHI, (const float*)Uin, (float*)Uout, U64, dtp, mid, dt, A, B);
  else
    return fail("bad precision");
  HIPCHECK(hipGetLastError());
  return 0;
}

int pyr_rk_update(pyr_ctx* c, int prec, long long n, const void* F, double* PHI, const void* Uin,
                  void* Uout, double* U64, double dt, double A, double B) {
  if (check_ctx(c)) return 1;
  return rk_update(c->stream, prec, n, F, PHI, Uin, Uout, U64, nullptr, nullptr, dt, A, B);
}

int pyr_rk_update_dt(pyr_ctx* c, int prec, long long n, const void* F, double* PHI, const void* Uin,
                     void* Uout, double* U64, const double* dt, double A, double B) {
  if (check_ctx(c)) return 1;
  if (!dt) return fail("null dt pointer to pyr_rk_update_dt");
  return rk_update(c->stream, prec, n, F, PHI, Uin, Uout, U64, dt, nullptr, 0.0, A, B);
}

int pyr_rk_update_member_dt(void* stream, int prec, long long n, const void* F, double* PHI,
                            const void* Uin, void* Uout, double* U64, const double* dt_member,
                            const int* member_of_point, double A, double B) {
  if (!dt_member || !member_of_point) return fail("null pointer to pyr_rk_update_member_dt");
  return rk_update((hipStream_t)stream, prec, n, F, PHI, Uin, Uout, U64, dt_member, member_of_point, 0.0, A, B);
}

int pyr_group_create(pyr_group** out, int M, pyr_ctx* const* members, const long long* offsets) {
  if (!out || M < 1 || !members || !offsets) return fail("bad arguments to pyr_group_create");
  std::unique_ptr<pyr_group> g(new pyr_group());
  for (int m = 0; m < M; ++m) {
    if (check_ctx(members[m])) return 1;
    if (offsets[m] < 0) return fail("negative member offset");
    g->mem.push_back(members[m]);
    g->off.push_back(offsets[m]);
  }
  *out = g.release();
  return 0;
}

int pyr_group_destroy(pyr_group* g) {
  delete g;
  return 0;
}

int pyr_group_set_stream(pyr_group* g, void* stream) {
  if (!g) return fail("null group");
  g->stream = (hipStream_t)stream;
  return 0;
}

int pyr_group_apply(pyr_group* g, int op, int dir, int prec, const void* in, void* out, int epi, double ec,
                    int mesh_power) {
  if (!g) return fail("null group");
  if (op < 0 || op >= NOPS || dir < 0 || dir > 2) return fail("bad operator or direction");
  if (!in || !out) return fail("null field pointer");
  if (in == out) return fail("input and output must not alias");
  if (mesh_power < 0 || mesh_power > 2) return fail("mesh_power must be 0, 1 or 2");
  GrpKey key;
  key.op = op;
  key.dir = dir;
  key.prec = prec;
  key.epi = epi;
  key.power = mesh_power;
  key.aligned = ((uintptr_t)in % 16 == 0) && ((uintptr_t)out % 16 == 0);
  key.ec = ec;
  for (pyr_ctx* c : g->mem)
    if (c->periodic_solver != g->mem[0]->periodic_solver || c->x_lds_kb != g->mem[0]->x_lds_kb)
      return fail("group members differ in their periodic solver or x-line LDS budget");
  key.refined = 0;
  if (prec == PYR_F64) return grp_apply<double>(g, key, (const double*)in, (double*)out);
  if (prec == PYR_R32) {
    for (pyr_ctx* c : g->mem)
      if (r32_mode(c, op, dir) != r32_mode(g->mem[0], op, dir))
        return fail("group members differ in their FP32 solve mode");
    key.refined = r32_mode(g->mem[0], op, dir) == PYR_R32_SOLVE_REFINED;
    return grp_apply<float>(g, key, (const float*)in, (float*)out);
  }
  return fail("bad precision");
}

int pyr_host_weights(int op, double* ali, double* ari, double* alb1, double* alb2, double* arb1,
                     double* arb2, int* dims6) {
  if (op < 0 || op >= NOPS) return fail("bad operator");
  const Scheme s = make_scheme(op);
  std::memcpy(ali, s.ali, sizeof s.ali);
  std::memcpy(ari, s.ari, sizeof s.ari);
  std::memcpy(alb1, s.alb1, sizeof s.alb1);
  std::memcpy(alb2, s.alb2, sizeof s.alb2);
  std::memcpy(arb1, s.arb1, sizeof s.arb1);
  std::memcpy(arb2, s.arb2, sizeof s.arb2);
  const int dims[6] = {s.nol, s.nor, s.ncl, s.ncr, s.null_option, s.implicit};
  std::memcpy(dims6, dims, sizeof dims);
  return 0;
}

int pyr_host_emulate(pyr_ctx* c, int op, int dir, int prec, const void* in, void* out) {
  if (!c) return fail("null context");
  const bool anti = (op & PYR_OP_ANTISYM) != 0;
  op &= ~PYR_OP_ANTISYM;
  if (op < 0 || op >= NOPS || dir < 0 || dir > 2) return fail("bad operator or direction");
  if (prec == PYR_F64) return emulate<double>(c, op, dir, (const double*)in, (double*)out, anti);
  if (prec == PYR_R32) return emulate<float>(c, op, dir, (const float*)in, (float*)out, anti);
  return fail("bad precision");
}

}  // extern "C"
#endif  // PYR_PART == 0
