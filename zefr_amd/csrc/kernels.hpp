// kernels.hpp -- device code of the DFR residual hot path (gfx950), shared by the
// per-shape translation units (kernels_shape.hip, one object per (nDims, order)) and the
// shape-independent kernels and C entry points (kernels.hip).
//
// Design (MI355X-first, not a translation of the reference's kernel set):
//  * Element-major storage: element e owns the contiguous block U[e][var][spt].  A
//    workgroup takes EB consecutive elements, so its global loads are one contiguous
//    chunk, staged into LDS.
//  * The reference's constant-operator GEMMs (GiMMiK, src/gimmik_gpu.cu) are replaced by
//    sum-factorised line contractions: every DFR operator on tensor-product elements is
//    a 1D operator applied along the lines of the element (oppE -> lE, oppD -> Dss + Dsf,
//    oppDiv -> the same, oppDiv_fpts -> signed Dsf).  The 1D tables are staged in LDS.
//  * Face coupling is element-centric: each element reads its partner's trace through an
//    integer map (no pointer tables), and computes the common solution / common flux for
//    its own side of the face.  Both sides evaluate the same formula on the same L/R
//    states, so the interface flux stays single-valued.
//  * With LDG beta = +-1/2 (the usual setting) only one side's gradient enters each
//    common flux and the common solution is the other side's trace, so the "owner" side
//    can finish the whole common flux right after its own gradient, and the only other-
//    side data it needs (the partner's trace at its owned points) it extrapolates from the
//    partner's U itself: gradient_flux (gradient, volume divergence, owned common fluxes)
//    -> face_correction, two launches.  No gradient trace is stored at all.
//  * Navier-Stokes with a general LDG beta runs through the same two kernels: each side writes
//    its weighted share of the common flux (both_sides_flux -> both_sides_correction).  The
//    three launches with gradient traces (extrapolate -> gradient -> divergence, whose last
//    one alone writes, and only its own elements) serve a residual over its own state.
//  * Euler: divergence alone, extrapolating the partner traces from the partner's U; a fused
//    RK update writes another buffer, or in place reads the traces that a launch or the update
//    before it wrote.
//
// All arithmetic is FP64.  Reference call sites are cited at each kernel.  Times in the
// comments: microseconds per residual, VJP, step or V-cycle by the host clock over 20 calls or
// more between two waits, the smallest of several such bursts, both forms in turn on one card;
// where a kernel is named alone, its mean in rocprofv3's trace.  Longer runs at steady clocks
// give smaller figures (V-cycle of 128^2 quads p=4: 450 in bursts, 335 in long runs).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "zefr_amd.h"
#include "common.hpp"
#include "physics.hpp"

namespace zk {

constexpr int kMaxThreads = 256;
constexpr int kMaxRkStages = 4;  // RK44; the stage tables of the RK update hold this many

template <int D, int N>
struct Shape {
  static constexpr int nS = (D == 2) ? N * N : N * N * N;
  static constexpr int nFF = (D == 2) ? N : N * N;
  static constexpr int nF = 2 * D * nFF;
  static constexpr int V = D + 2;
  static constexpr int nM = D * D + 1;
  static constexpr int FPT = (nF + nS - 1) / nS;  // flux points per thread
  static constexpr int NOPS = 2 * N + N * N + 2 * N;
  static constexpr int NOPS_PAD = (NOPS + 7) & ~7;
  static constexpr int defaultEB() { return (kMaxThreads / nS) > 0 ? kMaxThreads / nS : 1; }
  // workgroup size bound of the per-shape kernels: 256 threads, or one element's points
  // rounded up to whole waves where an element has more (hexes of order 6 to 8)
  static constexpr int kThreads = (nS > kMaxThreads) ? ((nS + 63) / 64) * 64 : kMaxThreads;
  // LDS stride of per-element blocks of x doubles.  A wave's 64-bit LDS access goes 16 lanes at
  // a time over 32 banks, so doubles a multiple of 16 apart collide; with strides that are nS
  // modulo 16, lanes of neighbouring elements continue one run of banks (where a workgroup can
  // hold two elements at all).  Blocks back to back put up to 16 lanes on one bank for quads
  // p=1: Navier-Stokes residual of 300x301 of them 42.2 us, padded 35.6; 256^2 quads p=4 114
  // / 111, V-cycle of 128^2 quads p=4 458 / 454.  (Planes of hexes p=3 padded to 19, so that
  // the face phase's line gathers hit distinct banks too, gained nothing: 64^3 1525 / 1530.)
  static constexpr int ele(int x) { return 2 * nS > kMaxThreads ? x : x + ((nS - x) % 16 + 16) % 16; }
};

// The hardware dispatches workgroup b of a grid to XCD b % 8 (each XCD has its own L2).
// xcd_block renumbers the grid so that every XCD walks one contiguous range of element
// blocks in increasing order: the partner lines an element reads from its next neighbours
// along x and y (one and one row of blocks later) then come from that XCD's L2 when the
// neighbour's own workgroup reads them.  A bijection of [0, n) for any n.
constexpr long kXcds = 8;
__device__ __forceinline__ long xcd_block(long b, long n) {
  const long q = n / kXcds, r = n % kXcds, x = b % kXcds, i = b / kXcds;
  return x * q + (x < r ? x : r) + i;
}

// Offsets of the 1D tables inside ops1d.
template <int N> __device__ __forceinline__ const double *tab_lE(const double *o, int side) { return o + side * N; }
template <int N> __device__ __forceinline__ const double *tab_Dss(const double *o, int i) { return o + 2 * N + i * N; }
template <int N> __device__ __forceinline__ const double *tab_Dsf(const double *o, int i) { return o + 2 * N + N * N + 2 * i; }

struct KArgs {
  int E, EB, viscous;
  int fix_vis;
  double gamma, prandtl, mu, rt, c_sth;
  double rus_k, ldg_b, ldg_tau;
  const double *ops;
  const double *metric;
  const double *fgeo;
  const unsigned int *nbr;
  double *Utr;
  double *Gtr;
  double *Ftr;
  // k_extrapolate: 0 = the trace at every flux point; 1 = only where the partner owns the
  // face (the one-sided LDG path reads nothing else)
  int trace_sel;
  // Epilogue of the last kernel of a residual: mode 0 none; 1 RK stage update; 2 final RK
  // combination; 3 srcw -= divF (p-multigrid source term: srcw holds the restricted
  // residual); 4 divF += src (a residual plus the source term)
  struct Rk {
    double *U;
    const double *Uini, *divF0;  // divF0: stage 0 of the [nStages][E][V][nS] residuals
    const double *src;           // p-multigrid source term added to every divF_s (modes 1, 2, 4), or null
    long total;
    double alpha, dt, beta[kMaxRkStages];
    int nStages, stage, mode;
    double *trace;  // mode 1: also write the new state's trace here (the next stage's Utr), or null
    double *Uini_out;         // modes 1, 2: a copy of Uini (read before U is written), or null
    double *corr;             // mode 2: corr = new U - corr_base, or null
    const double *corr_base;
    double *srcw;             // mode 3
    // p-multigrid transfers of each element fused after its residual or update
    // (PMGrid::restrict_pmg, prolong_err): restriction (modes 0, 4) of U and of the
    // residual with the table pmgR [pmgRn][N] into pmgUc, pmgRc ([E][V][pmgRn^D]), the U
    // read from pmgU when the kernel holds no copy of it; prolongation (mode 2 with corr)
    // pmgUf += pmgAlpha * P corr with pmgP [pmgPn][N]
    const double *pmgR, *pmgU;
    double *pmgUc, *pmgRc;
    int pmgRn, pmgPn;
    const double *pmgP;
    double pmgAlpha;
    double *pmgUf;
  } rk;
};

// One case of a multi-case launch: its kernel arguments and arrays.  A multi-case launch
// runs the same kernel over several independent solvers of one shape in one grid:
// workgroup b does block b - starts[c] of case c, where starts[c] <= b < starts[c + 1].
struct MultiCase {
  KArgs a;
  const double *U;
  double *out;
  int N;  // points per direction of the case's elements (the order of a mixed-order launch)
  int D;  // nDims of the case (a launch over quads and hexes together)
};

// The case of workgroup b: binary search over the cases' first workgroups (uniform across
// the workgroup, so the loads are scalar).
__device__ __forceinline__ int find_case(const long *__restrict__ starts, int nc, long b) {
  int lo = 0, hi = nc - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (starts[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Flux point f of the reference ordering (src/quads.cpp:86-123, src/hexas.cpp:133-194):
// normal direction, side (0: the -1 end, 1: the +1 end), first spt of the line through
// it along 'dim', and that line's spt stride.
// Selections, no branches: the points of a wave lie on several faces, and a switch makes
// every wave walk most of its cases one after the other.
template <int D, int N>
__device__ __forceinline__ void fpt_info(int f, int &dim, int &side, int &base, int &str) {
  if constexpr (D == 2) {
    // faces 0..3: dim 1, 0, 1, 0; side 0, 1, 1, 0; the last two run backwards
    const int face = f / N, j = f - face * N, odd = face & 1;
    const int jj = (face >= 2) ? N - 1 - j : j;
    dim = 1 - odd;
    side = (face + 1) >> 1 & 1;
    str = odd ? 1 : N;
    base = odd ? N * jj : jj;
  } else {
    // face pairs 0..2 along z, x, y, each - then +; the in-face index k runs backwards on
    // the + ends of z and x and on the - end of y
    constexpr int NN = N * N;
    const int face = f / NN, r = f - face * NN, j = r / N, k = r - j * N, pair = face >> 1;
    side = face & 1;
    dim = (pair == 0) ? 2 : pair - 1;
    str = (pair == 0) ? NN : ((pair == 1) ? 1 : N);
    const int kk = ((pair == 2) ? 1 - side : side) ? N - 1 - k : k;
    base = ((pair == 1) ? N * kk : kk) + ((pair == 0) ? N * j : NN * j);
  }
}

// The flux point at the 'side' end of the line through spt (a, b, c) along 'dim'.
template <int D, int N>
__device__ __forceinline__ int fpt_end(int a, int b, int c, int dim, int side) {
  if constexpr (D == 2) {
    if (dim == 0) return side ? (N + b) : (3 * N + (N - 1 - b));
    return side ? (2 * N + (N - 1 - a)) : a;
  } else {
    constexpr int NN = N * N;
    if (dim == 0) return side ? (3 * NN + c * N + (N - 1 - b)) : (2 * NN + c * N + b);
    if (dim == 1) return side ? (5 * NN + c * N + a) : (4 * NN + c * N + (N - 1 - a));
    return side ? (NN + b * N + (N - 1 - a)) : (b * N + a);
  }
}

// ---------------------------------------------------------------- pointwise physics
// primitives, conv_proj, viscous_dir, visc_proj_sub, visc_normal, common_flux and their
// reverse-mode counterparts live in physics.hpp (shared with a host build).
using namespace zphys;

// Partner map entries: ele << (B + 1) | slot << B | fpt, with B = 8 flux-point bits for
// elements of at most 256 flux points and 9 above (hexes of order 6 to 8).
template <int D, int N>
struct NbrBits {
  static constexpr int B = (Shape<D, N>::nF <= 256) ? 8 : 9;
};

template <int D, int N>
__device__ __forceinline__ void unpack_nbr(unsigned int p, long &ep, int &slot, int &fp) {
  constexpr int B = NbrBits<D, N>::B;
  ep = (long)(p >> (B + 1));
  slot = (int)((p >> B) & 1u);
  fp = (int)(p & ((1u << B) - 1u));
}

template <int D, int N>
__device__ __forceinline__ int nbr_slot(unsigned int p) {
  return (int)((p >> NbrBits<D, N>::B) & 1u);
}

// Which sides' gradients enter the LDG flux (src/faces.cpp:1520-1545).
__device__ __forceinline__ bool need_left_grad(double beta) { return beta != -0.5; }
__device__ __forceinline__ bool need_right_grad(double beta) { return beta != 0.5; }

// Stage EB consecutive elements' U blocks and the 1D tables into LDS.
// stage_U in two halves, so that a kernel can issue other loads between them: the first
// batch of loads into registers, then the LDS stores and the rest.
template <int D, int N>
struct StageRegs {
  double ro[(Shape<D, N>::NOPS + 63) / 64], ru[Shape<D, N>::V];
};

template <int D, int N>
__device__ __forceinline__ void stage_U_load(const double *__restrict__ U, const KArgs &a, long e0, long neb,
                                             StageRegs<D, N> &r) {
  using S = Shape<D, N>;
  constexpr int VS = S::V * S::nS, OB = (S::NOPS + 63) / 64, B = S::V;
  const int tid = threadIdx.x, NT = blockDim.x;
  const double *Ub = U + e0 * VS;
  const long n = neb * VS;
#pragma unroll
  for (int k = 0; k < OB; k++) {
    const int i = tid + k * NT;
    r.ro[k] = a.ops[i < S::NOPS ? i : 0];
  }
#pragma unroll
  for (int k = 0; k < B; k++) {
    const long i = tid + (long)k * NT;
    r.ru[k] = Ub[i < n ? i : 0];
  }
}

template <int D, int N>
__device__ __forceinline__ void stage_U_store(const double *__restrict__ U, const KArgs &a, double *lops,
                                              double *lU, long e0, long neb, int Ustride, const StageRegs<D, N> &r) {
  using S = Shape<D, N>;
  constexpr int VS = S::V * S::nS, OB = (S::NOPS + 63) / 64, B = S::V;
  const int tid = threadIdx.x, NT = blockDim.x;
  const double *Ub = U + e0 * VS;
  const long n = neb * VS;
#pragma unroll
  for (int k = 0; k < OB; k++) {
    const int i = tid + k * NT;
    if (i < S::NOPS) lops[i] = r.ro[k];
  }
#pragma unroll
  for (int k = 0; k < B; k++) {
    const long i = tid + (long)k * NT;
    if (i < n) {
      const long el = i / VS;
      lU[el * Ustride + (i - el * VS)] = r.ru[k];
    }
  }
  for (int i = tid + OB * NT; i < S::NOPS; i += NT) lops[i] = a.ops[i];
  for (long i = tid + (long)B * NT; i < n; i += NT) {
    const long el = i / VS;
    lU[el * Ustride + (i - el * VS)] = Ub[i];
  }
}

template <int D, int N>
__device__ __forceinline__ void stage_U(const double *__restrict__ U, const KArgs &a, double *lops, double *lU,
                                        long e0, long neb, int Ustride) {
  using S = Shape<D, N>;
  constexpr int VS = S::V * S::nS;
  // every load of the first batch (OB table values and V state values per thread: the
  // whole block when it has >= 64 threads and EB * nS of them) is issued before the
  // first LDS store, so the staging costs one memory round trip, not one per value
  constexpr int OB = (S::NOPS + 63) / 64, B = S::V;
  const int tid = threadIdx.x, NT = blockDim.x;
  const double *Ub = U + e0 * VS;
  const long n = neb * VS;
  double ro[OB], ru[B];
#pragma unroll
  for (int k = 0; k < OB; k++) {
    const int i = tid + k * NT;
    ro[k] = a.ops[i < S::NOPS ? i : 0];
  }
#pragma unroll
  for (int k = 0; k < B; k++) {
    const long i = tid + (long)k * NT;
    ru[k] = Ub[i < n ? i : 0];
  }
#pragma unroll
  for (int k = 0; k < OB; k++) {
    const int i = tid + k * NT;
    if (i < S::NOPS) lops[i] = ro[k];
  }
#pragma unroll
  for (int k = 0; k < B; k++) {
    const long i = tid + (long)k * NT;
    if (i < n) {
      const long el = i / VS;
      lU[el * Ustride + (i - el * VS)] = ru[k];
    }
  }
  // the rest, for blocks smaller than that
  for (int i = tid + OB * NT; i < S::NOPS; i += NT) lops[i] = a.ops[i];
  for (long i = tid + (long)B * NT; i < n; i += NT) {
    const long el = i / VS;
    lU[el * Ustride + (i - el * VS)] = Ub[i];
  }
}

// Value of var v along the line (base, str) of a [var][spt] block, extrapolated to one end.
template <int N>
__device__ __forceinline__ double line_extrap(const double *lE, const double *blk, int base, int str) {
  double s = 0.0;
#pragma unroll
  for (int m = 0; m < N; m++) s += lE[m] * blk[base + m * str];
  return s;
}

// The partner's trace at its flux point fp (all V variables), extrapolated from the
// partner's solution line in global memory with the 1D table (global copy of ops1d): what
// k_extrapolate writes there, for kernels that run without a trace launch before them.
template <int D, int N>
__device__ __forceinline__ void partner_trace(const double *__restrict__ U, const double *ops, long ep, int fp,
                                              double *out) {
  using S = Shape<D, N>;
  int dim, side, base, str;
  fpt_info<D, N>(fp, dim, side, base, str);
  const double *lE = tab_lE<N>(ops, side);
  const double *Up = U + ep * S::V * S::nS + base;
#pragma unroll
  for (int v = 0; v < S::V; v++) {
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < N; m++) s += lE[m] * Up[v * S::nS + m * str];
    out[v] = s;
  }
}

// Whether a fused epilogue writes the array the residual reads its state from.
inline bool rk_writes_input(const KArgs::Rk &r, const double *U) {
  if (r.mode != 1 && r.mode != 2) return false;
  return r.U == U || r.Uini_out == U || r.corr == U;
}

// partner_trace in two halves: the partner's N-point solution line through fp (V N values
// into registers, with the table row), then the extrapolation, the same sums.
template <int D, int N>
struct PartnerLine {
  double x[Shape<D, N>::V][N], l[N];
};

template <int D, int N>
__device__ __forceinline__ void partner_line_load(const double *__restrict__ U, const double *ops, long ep, int fp,
                                                  PartnerLine<D, N> &p) {
  using S = Shape<D, N>;
  int dim, side, base, str;
  fpt_info<D, N>(fp, dim, side, base, str);
  const double *lE = tab_lE<N>(ops, side);
  const double *Up = U + ep * S::V * S::nS + base;
#pragma unroll
  for (int m = 0; m < N; m++) p.l[m] = lE[m];
#pragma unroll
  for (int v = 0; v < S::V; v++)
#pragma unroll
    for (int m = 0; m < N; m++) p.x[v][m] = Up[v * S::nS + m * str];
}

template <int D, int N>
__device__ __forceinline__ void partner_line_reduce(const PartnerLine<D, N> &p, double *out) {
#pragma unroll
  for (int v = 0; v < Shape<D, N>::V; v++) {
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < N; m++) s += p.l[m] * p.x[v][m];
    out[v] = s;
  }
}

// RK update of one spt straight after its residual, in the last kernel of the residual
// (the stage update of src/solver.cpp:2897-2941 and the final combination of
// :2997-3062, with the same arithmetic as k_rk_stage / k_rk_final).  acc holds this
// stage's divF at the spt; the other stages' come from memory.  With a source term
// (src/solver.cpp:2946-2962, 3061-3073) every divF_s is replaced by divF_s + src.
// Side outputs: a copy of the starting state (Uini_out), and after a final combination
// the change against a stored state (corr: p-multigrid's coarse correction,
// src/multigrid.cpp:236-256).  Mode 3 subtracts the residual from a p-multigrid source
// term in place (src/multigrid.cpp:474-518).  pre: the spt's starting state, source term
// and detJ loaded ahead by rk_prefetch (null: loaded here).
template <int D>
struct RkPre {
  double u0[D + 2], src[D + 2], detJ;
};

template <int D>
__device__ __forceinline__ void rk_prefetch(const KArgs &a, long e, int t, int nS, RkPre<D> &p) {
  constexpr int V = D + 2, nM = D * D + 1;
  const bool upd = a.rk.mode == 1 || a.rk.mode == 2;
  const bool src = a.rk.src && (upd || a.rk.mode == 4);
  p.detJ = upd ? a.metric[(e * nM + D * D) * nS + t] : 1.0;
#pragma unroll
  for (int v = 0; v < V; v++) {
    const long i = (e * V + v) * nS + t;
    p.u0[v] = upd ? a.rk.Uini[i] : 0.0;
    p.src[v] = src ? a.rk.src[i] : 0.0;
  }
}

// BATCH: the final combination loads every other stage's residual before it consumes
// the first (one memory round trip instead of one per stage and variable; the short
// launches of the coarse p-multigrid levels are latency-bound); it holds (nStages - 1) V
// more values, which the kernels that carry it without a prefetched state (face
// correction, viscous divergence) would pay in occupancy, so they keep the plain loop.
template <int D, bool BATCH = false>
__device__ __forceinline__ void rk_epilogue(const KArgs &a, long e, int t, int nS, const double *acc,
                                            double *unew = nullptr, const RkPre<D> *pre = nullptr) {
  constexpr int V = D + 2, nM = D * D + 1;
  if (a.rk.mode == 0 || a.rk.mode == 4) return;
  if (a.rk.mode == 3) {
#pragma unroll
    for (int v = 0; v < V; v++) a.rk.srcw[(e * V + v) * nS + t] -= acc[v];
    return;
  }
  const double detJ = pre ? pre->detJ : a.metric[(e * nM + D * D) * nS + t];
  if (BATCH && a.rk.mode == 2) {
    const long i0 = e * V * nS + t;
    double u[V], sv[V], rs[kMaxRkStages][V];
#pragma unroll
    for (int v = 0; v < V; v++) {
      u[v] = pre ? pre->u0[v] : a.rk.Uini[i0 + v * nS];
      sv[v] = a.rk.src ? (pre ? pre->src[v] : a.rk.src[i0 + v * nS]) : 0.0;
    }
#pragma unroll
    for (int s = 0; s < kMaxRkStages; s++) {
      if (s < a.rk.nStages && s != a.rk.stage) {
#pragma unroll
        for (int v = 0; v < V; v++) rs[s][v] = a.rk.divF0[s * a.rk.total + i0 + v * nS];
      }
    }
    double cb[V];
    if (a.rk.corr) {
#pragma unroll
      for (int v = 0; v < V; v++) cb[v] = a.rk.corr_base[i0 + v * nS];
    }
    if (a.rk.Uini_out) {
#pragma unroll
      for (int v = 0; v < V; v++) a.rk.Uini_out[i0 + v * nS] = u[v];
    }
    // each variable's sum over the stages in order, as k_rk_final's
#pragma unroll
    for (int s = 0; s < kMaxRkStages; s++) {
      if (s < a.rk.nStages) {
#pragma unroll
        for (int v = 0; v < V; v++) {
          double r = (s == a.rk.stage) ? acc[v] : rs[s][v];
          if (a.rk.src) r += sv[v];
          u[v] -= a.rk.beta[s] * a.rk.dt / detJ * r;
        }
      }
    }
#pragma unroll
    for (int v = 0; v < V; v++) {
      const long i = i0 + v * nS;
      a.rk.U[i] = u[v];
      if (unew) unew[v] = u[v];
      if (a.rk.corr) a.rk.corr[i] = u[v] - cb[v];
    }
    return;
  }
#pragma unroll
  for (int v = 0; v < V; v++) {
    const long i = (e * V + v) * nS + t;
    const double u0 = pre ? pre->u0[v] : a.rk.Uini[i];
    double sv = a.rk.src ? (pre ? pre->src[v] : a.rk.src[i]) : 0.0;
    if (a.rk.Uini_out) a.rk.Uini_out[i] = u0;
    if (a.rk.mode == 1 && a.rk.srcw) {  // form the source term first: srcw = src - divF
      sv = sv - acc[v];
      a.rk.srcw[i] = sv;
    }
    if (a.rk.mode == 1) {
      const double r = a.rk.src ? acc[v] + sv : acc[v];
      const double u = u0 - a.rk.alpha * a.rk.dt / detJ * r;
      a.rk.U[i] = u;
      if (unew) unew[v] = u;
    } else {
      double u = u0;
      for (int s = 0; s < a.rk.nStages; s++) {
        double r = (s == a.rk.stage) ? acc[v] : a.rk.divF0[s * a.rk.total + i];
        if (a.rk.src) r += sv;
        u -= a.rk.beta[s] * a.rk.dt / detJ * r;
      }
      a.rk.U[i] = u;
      if (unew) unew[v] = u;
      if (a.rk.corr) a.rk.corr[i] = u - a.rk.corr_base[i];
    }
  }
}

// After a fused RK stage update: the trace of the new state at this element's flux points,
// written to a.rk.trace ([E][V][nF], the next stage's Utr), so that the next stage's
// extrapolation launch is skipped.  owner < 0 writes every point (k_extrapolate with
// trace_sel 0); otherwise only the points whose partner owns the face (trace_sel 1 with
// that owner slot).  The new state goes through the element's LDS block w (V * nS
// doubles), which no thread may still read; every thread of the workgroup calls this (it
// holds barriers).
template <int D, int N>
__device__ __forceinline__ void rk_trace(const KArgs &a, const double *lops, double *w, long e, int t, bool valid,
                                         const double *unew, int owner) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  __syncthreads();
  if (valid) {
#pragma unroll
    for (int v = 0; v < V; v++) w[v * nS + t] = unew[v];
  }
  __syncthreads();
  if (!valid) return;
#pragma unroll
  for (int k = 0; k < S::FPT; k++) {
    const int f = t + k * nS;
    if (f >= nF) continue;
    if (owner >= 0 && nbr_slot<D, N>(a.nbr[e * nF + f]) == owner) continue;
    int dim, side, base, str;
    fpt_info<D, N>(f, dim, side, base, str);
    const double *lE = tab_lE<N>(lops, side);
#pragma unroll
    for (int v = 0; v < V; v++) a.rk.trace[(e * V + v) * nF + f] = line_extrap<N>(lE, w + v * nS, base, str);
  }
}

// Output o (x fastest) of a tensor-product table A [no][N] (one 1D table per direction)
// applied to one [N^D] block, with k_pmg_transfer's roundings: the sums along x, then y,
// then z, each from 0.0 over increasing input index.  Every output recomputes the partial
// sums of its lines, which are the same numbers the separate passes form.  blk and A are
// in LDS.
template <int D, int N>
__device__ __forceinline__ double tp_out(const double *blk, const double *A, int no, int o) {
  const unsigned uo = o, uno = no;  // unsigned: cheaper division sequences
  const int o1 = uo % uno, o2 = (uo / uno) % uno, o3 = (D == 3) ? uo / (uno * uno) : 0;
  const double *A1 = A + o1 * N, *A2 = A + o2 * N, *A3 = A + o3 * N;
  double a1[N];
#pragma unroll
  for (int i1 = 0; i1 < N; i1++) a1[i1] = A1[i1];
  double s3 = 0.0;
#pragma unroll 1
  for (int i3 = 0; i3 < ((D == 3) ? N : 1); i3++) {
    const double *b = blk + i3 * N * N;
    double s2 = 0.0;
    auto line = [&](int i2) {
      double s1 = 0.0;
#pragma unroll
      for (int i1 = 0; i1 < N; i1++) s1 = __builtin_fma(a1[i1], b[i2 * N + i1], s1);
      s2 = __builtin_fma(A2[i2], s1, s2);
    };
    if constexpr (D == 3) {
      // kept rolled: the hex kernels that carry this epilogue hold no registers to spare
#pragma unroll 1
      for (int i2 = 0; i2 < N; i2++) line(i2);
    } else {
#pragma unroll
      for (int i2 = 0; i2 < N; i2++) line(i2);
    }
    s3 = (D == 3) ? __builtin_fma(A3[i3], s2, s3) : s2;
  }
  return s3;
}

// One element's transfer out [V][no^D] = A blk (add: out += alpha A blk) by the element's nS
// threads; each (variable, output point) pair is one work item.  A thread takes K items at
// a time and, when it adds to the output, loads all K old values before it forms the first
// (one memory round trip per K items, not one per item).  NO > 0: no == NO, a constant.
template <int D, int N, int NO>
__device__ __forceinline__ void pmg_apply(const double *blk, const double *A, int no_rt, double *out, long e, int t,
                                          double alpha, bool add) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, V = S::V, K = 4;
  const int no = NO > 0 ? NO : no_rt;
  const int noD = (D == 3) ? no * no * no : no * no;
  const int total = V * noD;
  double *oe = out + e * total;  // [V][no^D] of this element
#pragma unroll 1
  for (int k0 = t; k0 < total; k0 += K * nS) {
    double old[K];
    if (add) {
#pragma unroll
      for (int j = 0; j < K; j++) {
        const int k = k0 + j * nS;
        old[j] = (k < total) ? oe[k] : 0.0;
      }
    }
#pragma unroll
    for (int j = 0; j < K; j++) {
      const int k = k0 + j * nS;
      if (k < total) {
        const int v = (unsigned)k / (unsigned)noD, o = k - v * noD;
        const double x = tp_out<D, N>(blk + v * nS, A, no, o);
        oe[k] = add ? __builtin_fma(alpha, x, 1.0 * old[j]) : x;
      }
    }
  }
}

// The p-multigrid transfers fused at the end of a residual kernel (every thread of the
// workgroup calls this; it holds barriers).  res: this thread's residual (after the source
// term); unew: its new state (mode 2); ublk: the element's U block in LDS, or null (then U
// is read from a.rk.pmgU); w: a free per-element LDS block of at least V nS doubles; lops:
// the block's operator tables, no longer needed, which take the transfer table (the host
// fuses a transfer only where its table fits their N^2 + 4 N doubles, padded).
template <int D, int N>
__device__ __forceinline__ void pmg_epilogue(const KArgs &a, double *lops, const double *ublk, double *w, long e,
                                             int t, bool valid, const double *res, const double *unew) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, V = S::V;
  const KArgs::Rk &r = a.rk;
  auto apply = [&](const double *blk, int no, double *out, double alpha, bool add) {
    if (!valid) return;
    // the usual transfers (one order down, one up) with their output count known at compile
    // time: the work item's index splits by multiplications instead of integer divisions
    if (no == N - 1) pmg_apply<D, N, (N > 1 ? N - 1 : 0)>(blk, lops, no, out, e, t, alpha, add);
    else if (no == N + 1) pmg_apply<D, N, N + 1>(blk, lops, no, out, e, t, alpha, add);
    else pmg_apply<D, N, 0>(blk, lops, no, out, e, t, alpha, add);
  };
  const bool restr = r.pmgRc && (r.mode == 0 || r.mode == 4);
  const bool prol = r.pmgUf && r.mode == 2 && r.corr;
  if (!restr && !prol) return;
  __syncthreads();  // lops and w are consumed
  const double *A = restr ? r.pmgR : r.pmgP;
  const int nA = (restr ? r.pmgRn : r.pmgPn) * N;
  for (int i = threadIdx.x; i < nA; i += blockDim.x) lops[i] = A[i];
  if (valid) {
#pragma unroll
    for (int v = 0; v < V; v++)
      w[v * nS + t] = restr ? res[v] : unew[v] - r.corr_base[(e * V + v) * nS + t];
  }
  __syncthreads();
  if (prol) {
    apply(w, r.pmgPn, r.pmgUf, r.pmgAlpha, true);
    return;
  }
  apply(w, r.pmgRn, r.pmgRc, 1.0, false);
  if (ublk) {
    apply(ublk, r.pmgRn, r.pmgUc, 1.0, false);
  } else {
    __syncthreads();
    if (valid) {
#pragma unroll
      for (int v = 0; v < V; v++) w[v * nS + t] = r.pmgU[(e * V + v) * nS + t];
    }
    __syncthreads();
    apply(w, r.pmgRn, r.pmgUc, 1.0, false);
  }
}

// A set of faces as a list: the faces in increasing order, four bits each.
template <int D>
__device__ __forceinline__ unsigned face_list(unsigned mask) {
  unsigned list = 0u;
  int n = 0;
#pragma unroll
  for (int b = 0; b < 2 * D; b++) {
    const unsigned bit = (mask >> b) & 1u;
    list |= (bit ? (unsigned)b : 0u) << n;
    n += bit ? 4 : 0;
  }
  return list;
}

// The k-th flux point of a list of faces, its faces taken in order.
template <int D, int N>
__device__ __forceinline__ int list_fpt(unsigned list, int k) {
  using S = Shape<D, N>;
  const int q = k / S::nFF;
  return (int)((list >> (4 * q)) & 15u) * S::nFF + (k - q * S::nFF);
}

// The faces of element e that it owns (bit q = face q): all flux points of a face share its
// slot, so one partner-map entry per face tells.  Every thread of an element reads the same
// 2 D entries (a broadcast), which costs one memory round trip and no LDS.
template <int D, int N>
__device__ __forceinline__ unsigned owned_faces(const unsigned *__restrict__ nbr, int owner) {
  using S = Shape<D, N>;
  unsigned p[2 * D], mask = 0u;
#pragma unroll
  for (int q = 0; q < 2 * D; q++) p[q] = nbr[q * S::nFF];
#pragma unroll
  for (int q = 0; q < 2 * D; q++)
    if (nbr_slot<D, N>(p[q]) == owner) mask |= 1u << q;
  return mask;
}

// ---------------------------------------------------------------- kernel 1: traces
// Elements::extrapolate_U (src/elements.cpp:1337-1360): U_fpts = oppE U_spts.  With
// trace_sel = 1 only the points of faces the partner owns are written: on the one-sided
// LDG path the owner reads the other side's trace and nothing reads its own.
template <int D, int N>
__device__ __forceinline__ void extrapolate_block(const double *__restrict__ U, const KArgs &a, long bid) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  extern __shared__ double lds[];
  double *lops = lds;
  double *lU = lds + S::NOPS_PAD;
  const long e0 = bid * a.EB;
  const long neb = min((long)a.EB, (long)a.E - e0);
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  // this thread's slots, fetched before the staging barrier so the loads overlap it
  int slot[S::FPT];
#pragma unroll
  for (int k = 0; k < S::FPT; k++) {
    const int f = t + k * nS;
    slot[k] = (a.trace_sel && el < neb && f < nF) ? nbr_slot<D, N>(a.nbr[e * nF + f]) : -1;
  }
  stage_U<D, N>(U, a, lops, lU, e0, neb, S::ele(V * nS));
  __syncthreads();
  if (el >= neb) return;
  const double *u = lU + el * S::ele(V * nS);
  const int owner = (a.ldg_b == 0.5) ? 0 : 1;
#pragma unroll
  for (int k = 0; k < S::FPT; k++) {
    const int f = t + k * nS;
    if (f < nF) {
      if (a.trace_sel && slot[k] == owner) continue;
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
#pragma unroll
      for (int v = 0; v < V; v++) a.Utr[(e * V + v) * nF + f] = line_extrap<N>(lE, u + v * nS, base, str);
    }
  }
}

template <int D, int N>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_extrapolate(const double *__restrict__ U, KArgs a) {
  extrapolate_block<D, N>(U, a, xcd_block(blockIdx.x, gridDim.x));
}

// The same kernel for workgroups of one wave (see k_visc_onesided_w64).
template <int D, int N>
__global__ __launch_bounds__(64) void k_extrapolate_w64(const double *__restrict__ U, KArgs a) {
  extrapolate_block<D, N>(U, a, xcd_block(blockIdx.x, gridDim.x));
}

template <int D, int N>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_extrapolate_multi(const MultiCase *__restrict__ cs, const long *__restrict__ starts, int nc) {
  const int c = find_case(starts, nc, blockIdx.x);
  extrapolate_block<D, N>(cs[c].U, cs[c].a, (long)blockIdx.x - starts[c]);
}

// LDG common solution at this thread's flux points (src/faces.cpp:1366-1474):
// Ucomm = 1/2 (UL + UR) - beta (UL - UR), with the beta = +-1/2 one-sided branches.
template <int D, int N>
__device__ __forceinline__ void common_solution(const KArgs &a, const double *lops, const double *u, double *lC,
                                                long e, int t) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  const double beta = a.ldg_b;
#pragma unroll
  for (int k = 0; k < S::FPT; k++) {
    const int f = t + k * nS;
    if (f >= nF) continue;
    int dim, side, base, str;
    fpt_info<D, N>(f, dim, side, base, str);
    const double *lE = tab_lE<N>(lops, side);
    long ep; int sl, fp;
    unpack_nbr<D, N>(a.nbr[e * nF + f], ep, sl, fp);
#pragma unroll
    for (int v = 0; v < V; v++) {
      const double own = line_extrap<N>(lE, u + v * nS, base, str);
      const double par = a.Utr[(ep * V + v) * nF + fp];
      const double uL = sl ? par : own, uR = sl ? own : par;
      const double l = (beta == 0.5) ? 0.0 : uL;
      const double r = (beta == -0.5) ? 0.0 : uR;
      lC[v * nF + f] = 0.5 * (l + r) - beta * (l - r);
    }
  }
}

// Corrected reference-space gradient at spt t (oppD U + oppD_fpts Ucomm), mapped to
// physical space with the adjugate metric (src/elements.cpp:1393-1447, 1630-1650).
template <int D, int N>
__device__ __forceinline__ void spt_gradient(const double *lops, const double *u, const double *lC, int t,
                                             const double ij[][D], double detJ, double g[][D]) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
  double gr[D][V];
#pragma unroll
  for (int d = 0; d < D; d++) {
    const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
    const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
    const int base = t - id * str;
    const double *Dr = tab_Dss<N>(lops, id);
    const double *Df = tab_Dsf<N>(lops, id);
    const int f0 = fpt_end<D, N>(ia, ib, ic, d, 0), f1 = fpt_end<D, N>(ia, ib, ic, d, 1);
#pragma unroll
    for (int v = 0; v < V; v++) {
      double s = 0.0;
#pragma unroll
      for (int m = 0; m < N; m++) s += Dr[m] * u[v * nS + base + m * str];
      s += Df[0] * lC[v * nF + f0];
      s += Df[1] * lC[v * nF + f1];
      gr[d][v] = s;
    }
  }
  const double inv_det = 1.0 / detJ;
#pragma unroll
  for (int v = 0; v < V; v++)
#pragma unroll
    for (int d1 = 0; d1 < D; d1++) {
      double s = 0.0;
#pragma unroll
      for (int d2 = 0; d2 < D; d2++) s += gr[d2][v] * ij[d2][d1];
      g[v][d1] = s * inv_det;
    }
}

template <int D>
__device__ __forceinline__ void load_metric(const KArgs &a, long e, int t, int nS, double ij[][D], double &detJ,
                                            bool want_det) {
  constexpr int nM = D * D + 1;
  const double *m = a.metric + e * nM * nS + t;
#pragma unroll
  for (int d1 = 0; d1 < D; d1++)
#pragma unroll
    for (int d2 = 0; d2 < D; d2++) ij[d1][d2] = m[(d1 * D + d2) * nS];
  detJ = want_det ? m[D * D * nS] : 1.0;
}

// ---------------------------------------------------------------- kernel 2: gradient
// Common solution + corrected gradient + physical transform + gradient extrapolation to
// the flux points whose gradient the partner element needs.  LDS per element holds U and
// Ucomm, then (aliased) the physical gradient.
template <int D, int N>
__device__ __forceinline__ void gradient_block(const double *__restrict__ U, double *__restrict__ dU_out,
                                               const KArgs &a, long bid) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  constexpr int W = S::ele((V * nS + V * nF > D * V * nS) ? V * nS + V * nF : D * V * nS);
  extern __shared__ double lds[];
  double *lops = lds;
  double *lW = lds + S::NOPS_PAD;
  const long e0 = bid * a.EB;
  const long neb = min((long)a.EB, (long)a.E - e0);
  stage_U<D, N>(U, a, lops, lW, e0, neb, W);
  __syncthreads();
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  double *u = lW + el * W;
  double *c = u + V * nS;
  if (valid) common_solution<D, N>(a, lops, u, c, e, t);
  __syncthreads();
  double g[V][D];
  if (valid) {
    double ij[D][D], detJ;
    load_metric<D>(a, e, t, nS, ij, detJ, true);
    spt_gradient<D, N>(lops, u, c, t, ij, detJ, g);
    if (dU_out) {
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++) dU_out[((e * D + d) * V + v) * nS + t] = g[v][d];
    }
  }
  __syncthreads();  // U and Ucomm are dead: the region now holds the gradient
  if (valid) {
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int v = 0; v < V; v++) u[(d * V + v) * nS + t] = g[v][d];
  }
  __syncthreads();
  if (!valid) return;
  const double beta = a.ldg_b;
#pragma unroll
  for (int k = 0; k < S::FPT; k++) {
    const int f = t + k * nS;
    if (f >= nF) continue;
    const int sl = nbr_slot<D, N>(a.nbr[e * nF + f]);
    // the partner needs this side's gradient iff this side is L and dUL is used, or R and dUR is used
    const bool write = sl ? need_right_grad(beta) : need_left_grad(beta);
    if (!write) continue;
    int dim, side, base, str;
    fpt_info<D, N>(f, dim, side, base, str);
    const double *lE = tab_lE<N>(lops, side);
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int v = 0; v < V; v++)
        a.Gtr[((e * D + d) * V + v) * nF + f] = line_extrap<N>(lE, u + (d * V + v) * nS, base, str);
  }
}

template <int D, int N>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_gradient(const double *__restrict__ U, double *__restrict__ dU_out,
                                                          KArgs a) {
  gradient_block<D, N>(U, dU_out, a, xcd_block(blockIdx.x, gridDim.x));
}

// ---------------------------------------------------------------- kernel 3: divergence
// compute_F + compute_divF_spts + compute_common_F + compute_divF_fpts.
// Phases (viscous): U -> LDS | Ucomm -> lC | gradient -> lG | common flux -> lC |
// transformed flux -> lG | divergence.  Inviscid: U -> LDS | flux + common flux | divergence.
// SELF (Euler only): the partner traces are extrapolated here from the partner's U, so an
// Euler residual is this one launch; otherwise they are read from Utr.
// U is not __restrict__: with a fused RK update (a.rk.mode != 0) the epilogue writes a.rk.U,
// which is the same array; U is then read only while staging, before the first barrier.
// IDLE: launches of kMaxThreads threads whose tile may fill fewer (mixed multi-case launches,
// persistent plans).  The threads beyond the tile skip the Euler prologue's loads: 16 cases of
// 8x9 quads p=4, 50 of 256 threads in use, 7.6 us with their lines loaded and 5.8 without;
// 16 of 3^3 hexes p=3 9.3 and 7.0.
template <int D, int N, bool VISC, int BM, int FC, bool SELF, bool IDLE = false>
__device__ __forceinline__ void divergence_block(const double *U, double *__restrict__ divF, const KArgs &a,
                                                 long bid) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  extern __shared__ double lds[];
  const int EB = a.EB;
  double *lops = lds;
  double *lU = lops + S::NOPS_PAD;
  constexpr int WU = S::ele(V * nS), WC = S::ele(V * nF), WG = S::ele(D * V * nS);
  double *lC = lU + EB * WU;
  double *lG = lC + EB * WC;  // gradient (viscous), then the transformed flux
  const long e0 = bid * EB;
  const long neb = min((long)EB, (long)a.E - e0);
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  // Euler: everything this thread reads from global memory is loaded here, ahead of the first
  // barrier: first all that depends on nothing (the staged block, the partner entries and
  // face geometry of its flux points, its metric, the RK epilogue's inputs), then the partner
  // states.  Two dependent round trips; taken flux point by flux point, with the rest behind
  // them, they were 2 FPT + 1, and on small meshes a launch is little else.  Points beyond the
  // last and threads of a ragged last workgroup load a neighbour's data (in bounds) instead of
  // branching.  (29x31x27
  // hexes p=2, RK44 step 246 -> 232 us; 128^2 quads p=4, V-cycle 520 -> 495.)
  // Not so in hexes of order 6 to 8 (one element and 6 to 12 waves per workgroup, one flux
  // point at most per thread): there the lines held beside all the rest cost a wave of three
  // (p=6, 172 registers) or 42 spills (p=8), and whole waves have no flux point to load for.
  // They take the partner's line first and branch.  Residual, all ahead / line first: 8x7x7
  // hexes p=8 42.2 / 29.6 us, 15x13x14 252 / 172; 10x9x10 p=6 33.3 / 32.0, 19x17x18 188 / 159.
  constexpr int PF = VISC ? 1 : S::FPT;
  double pUs[PF][V], pn[PF][D], pdA[PF], pij[D][D], pdet = 1.0;
  int psl[PF];
  RkPre<D> pre;
  constexpr bool ahead = nS <= kMaxThreads;
  if constexpr (!VISC) {
    const long ec = valid ? e : e0;
    StageRegs<D, N> sr;
    unsigned nb[PF];
    auto partner = [&](int k) {
      long ep; int sl, fp;
      unpack_nbr<D, N>(nb[k], ep, sl, fp);
      psl[k] = sl;
      if constexpr (SELF) {
        partner_trace<D, N>(U, a.ops, ep, fp, pUs[k]);
      } else {
#pragma unroll
        for (int v = 0; v < V; v++) pUs[k][v] = a.Utr[(ep * V + v) * nF + fp];
      }
    };
    auto geometry = [&](int k, int f) {
      const double *fg = a.fgeo + ec * (D + 1) * nF + f;
#pragma unroll
      for (int d = 0; d < D; d++) pn[k][d] = fg[d * nF];
      pdA[k] = fg[D * nF];
    };
    if constexpr (ahead) {
      stage_U_load<D, N>(U, a, e0, neb, sr);
      if (!IDLE || el < EB) {
#pragma unroll
        for (int k = 0; k < PF; k++) nb[k] = a.nbr[ec * nF + (t + k * nS < nF ? t + k * nS : 0)];
#pragma unroll
        for (int k = 0; k < PF; k++) geometry(k, t + k * nS < nF ? t + k * nS : 0);
        load_metric<D>(a, ec, t, nS, pij, pdet, false);
        rk_prefetch<D>(a, ec, t, nS, pre);
#pragma unroll
        for (int k = 0; k < PF; k++) partner(k);
      }
      stage_U_store<D, N>(U, a, lops, lU, e0, neb, WU, sr);
    } else {
      if (valid) {
#pragma unroll
        for (int k = 0; k < PF; k++) {
          const int f = t + k * nS;
          psl[k] = 0;
          if (f >= nF) continue;
          nb[k] = a.nbr[ec * nF + f];
          partner(k);
          geometry(k, f);
        }
        load_metric<D>(a, ec, t, nS, pij, pdet, false);
        rk_prefetch<D>(a, ec, t, nS, pre);
      }
      stage_U<D, N>(U, a, lops, lU, e0, neb, WU);
    }
  } else {
    stage_U<D, N>(U, a, lops, lU, e0, neb, WU);
  }
  __syncthreads();
  const double *u = lU + el * WU;
  double *c = lC + el * WC;
  double *g_l = lG + el * WG;
  if (VISC) {
    if (valid) common_solution<D, N>(a, lops, u, c, e, t);
    __syncthreads();
    if (valid) {
      double ij[D][D], detJ, g[V][D];
      load_metric<D>(a, e, t, nS, ij, detJ, true);
      spt_gradient<D, N>(lops, u, c, t, ij, detJ, g);
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++) g_l[(d * V + v) * nS + t] = g[v][d];
    }
    __syncthreads();
  }

  // common flux at this thread's flux points -> lC (Ucomm has been consumed)
  if (!VISC && valid) {
#pragma unroll
    for (int k = 0; k < PF; k++) {
      const int f = t + k * nS;
      if (f >= nF) continue;
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
      double Uo[V], UL[V], UR[V], G1[1], G2[1], Fo[V];
#pragma unroll
      for (int v = 0; v < V; v++) Uo[v] = line_extrap<N>(lE, u + v * nS, base, str);
#pragma unroll
      for (int v = 0; v < V; v++) {
        UL[v] = psl[k] ? pUs[k][v] : Uo[v];
        UR[v] = psl[k] ? Uo[v] : pUs[k][v];
      }
      common_flux<D, false, BM, FC>(UL, UR, G1, G2, pn[k], pdA[k], a, Fo);
#pragma unroll
      for (int v = 0; v < V; v++) c[v * nF + f] = Fo[v];
    }
  }
  if (VISC && valid) {
#pragma unroll 1
    for (int k = 0; k < S::FPT; k++) {
      const int f = t + k * nS;
      if (f >= nF) continue;
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
      long ep; int sl, fp;
      unpack_nbr<D, N>(a.nbr[e * nF + f], ep, sl, fp);
      const double *fg = a.fgeo + e * (D + 1) * nF + f;
      double n[D];
#pragma unroll
      for (int d = 0; d < D; d++) n[d] = fg[d * nF];
      const double dAs = fg[D * nF];
      // own side's state / gradient from LDS, the partner's from its traces
      auto own_state = [&](double *Us) {
#pragma unroll
        for (int v = 0; v < V; v++) Us[v] = line_extrap<N>(lE, u + v * nS, base, str);
      };
      auto par_state = [&](double *Us) {
        if constexpr (SELF) {
          partner_trace<D, N>(U, a.ops, ep, fp, Us);
        } else {
#pragma unroll
          for (int v = 0; v < V; v++) Us[v] = a.Utr[(ep * V + v) * nF + fp];
        }
      };
      // viscous normal fluxes first (one side's state + gradient live at a time):
      // G1 = left (BM 0, 1) or right (BM 2) side, G2 = right side (BM 0)
      double G1[VISC ? V : 1], G2[(VISC && BM == 0) ? V : 1];
      if (VISC) {
        auto side_visc = [&](bool own, double *G) {
          double Us[V];
          if (own) {
            own_state(Us);
            visc_normal<D>(Us, [&](int j, double *dUj) {
#pragma unroll
              for (int v = 0; v < V; v++) {
                dUj[v] = line_extrap<N>(lE, g_l + (j * V + v) * nS, base, str);
                asm volatile("" : "+v"(dUj[v]) : : "memory");  // formed here, before the next line is loaded
              }
            }, n, a, G);
          } else {
            par_state(Us);
            visc_normal<D>(Us, [&](int j, double *dUj) {
#pragma unroll
              for (int v = 0; v < V; v++) dUj[v] = a.Gtr[((ep * D + j) * V + v) * nF + fp];
            }, n, a, G);
          }
        };
        if (BM == 0) {
          side_visc(sl == 0, G1);
          side_visc(sl == 1, G2);
        } else {
          side_visc((BM == 1) ? (sl == 0) : (sl == 1), G1);
        }
      }
      double UL[V], UR[V];
      if (sl) { par_state(UL); own_state(UR); } else { own_state(UL); par_state(UR); }
      double Fo[V];
      common_flux<D, VISC, BM, FC>(UL, UR, G1, G2, n, dAs, a, Fo);
#pragma unroll
      for (int v = 0; v < V; v++) c[v * nF + f] = Fo[v];
    }
  }
  if (VISC) __syncthreads();  // the gradient field in lG is consumed

  // pointwise flux at the spt, contracted with the adjugate rows (src/elements.cpp:1588-1699);
  // each thread reads and overwrites only its own spt column of lG
  if (valid) {
    double ij[D][D], detJ;
    if (VISC) {
      load_metric<D>(a, e, t, nS, ij, detJ, false);
    } else {
#pragma unroll
      for (int d1 = 0; d1 < D; d1++)
#pragma unroll
        for (int d2 = 0; d2 < D; d2++) ij[d1][d2] = pij[d1][d2];
    }
    double Us[V];
#pragma unroll
    for (int v = 0; v < V; v++) Us[v] = u[v * nS + t];
    const Prim<D> p = primitives<D>(Us, a.gamma);
    double tF[D][V];
#pragma unroll
    for (int d1 = 0; d1 < D; d1++) conv_proj<D>(Us, p, ij[d1], tF[d1]);
    if (VISC) {
      double g[V][D];
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++) g[v][d] = g_l[(d * V + v) * nS + t];
      const Visc<D> vs = viscous<D>(Us, p, g, a);
#pragma unroll
      for (int d1 = 0; d1 < D; d1++) visc_proj_sub<D>(vs, ij[d1], tF[d1]);
    }
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int v = 0; v < V; v++) g_l[(d * V + v) * nS + t] = tF[d][v];
  }
  __syncthreads();
  double unew[V], res[V];
  if (valid) {
    // divergence: oppDiv tF + oppDiv_fpts Fcomm (src/elements.cpp:1449-1501)
    const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
    double acc[V];
#pragma unroll
    for (int v = 0; v < V; v++) acc[v] = 0.0;
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
      const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
      const int base = t - id * str;
      const double *Dr = tab_Dss<N>(lops, id);
#pragma unroll
      for (int v = 0; v < V; v++) {
        double s = acc[v];
#pragma unroll
        for (int m = 0; m < N; m++) s += Dr[m] * g_l[(d * V + v) * nS + base + m * str];
        acc[v] = s;
      }
    }
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
      const double *Df = tab_Dsf<N>(lops, id);
      const int f0 = fpt_end<D, N>(ia, ib, ic, d, 0), f1 = fpt_end<D, N>(ia, ib, ic, d, 1);
#pragma unroll
      for (int v = 0; v < V; v++) {
        acc[v] += (-Df[0]) * c[v * nF + f0];
        acc[v] += Df[1] * c[v * nF + f1];
      }
    }
    if (a.rk.mode == 4) {
#pragma unroll
      for (int v = 0; v < V; v++) acc[v] += VISC ? a.rk.src[(e * V + v) * nS + t] : pre.src[v];
    }
#pragma unroll
    for (int v = 0; v < V; v++) divF[(e * V + v) * nS + t] = acc[v];
#pragma unroll
    for (int v = 0; v < V; v++) res[v] = acc[v];
    rk_epilogue<D, !VISC>(a, e, t, nS, acc, unew, VISC ? nullptr : &pre);
  }
  // the new state's full trace for the next stage, into a buffer other than the Utr this
  // launch reads; the element's U block is no longer read
  if (a.rk.mode == 1 && a.rk.trace) rk_trace<D, N>(a, lops, lU + el * WU, e, t, valid, unew, -1);
  // p-multigrid transfers (the U block is still the staged state; lG is free)
  if (a.rk.pmgRc || a.rk.pmgUf) pmg_epilogue<D, N>(a, lops, lU + el * WU, g_l, e, t, valid, res, unew);
}

// Occupancy target of the divergence kernel: the general-beta hex p=3 Rusanov kernel fits
// four waves per SIMD (it took 130 VGPRs, three waves, once it carried the p-multigrid
// transfer epilogue); other shapes keep the default allocation.
template <int D, int N, bool VISC, int FC>
struct DivWaves {
  static constexpr int value = (D == 3 && N == 4 && VISC && FC == 0) ? 4 : 1;
};

template <int D, int N, bool VISC, int BM, int FC, bool SELF = !VISC>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) __attribute__((amdgpu_waves_per_eu(DivWaves<D, N, VISC, FC>::value)))
void k_divergence(const double *U, double *__restrict__ divF, KArgs a) {
  static_assert(!(VISC && SELF), "the viscous divergence reads the gradient traces, hence the traces too");
  divergence_block<D, N, VISC, BM, FC, SELF>(U, divF, a, xcd_block(blockIdx.x, gridDim.x));
}

// The same kernel for workgroups of one wave (the small meshes of coarse p-multigrid
// levels and small cases): its barriers need no cross-wave synchronisation.
template <int D, int N, bool VISC, int BM, int FC, bool SELF = !VISC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(DivWaves<D, N, VISC, FC>::value)))
void k_divergence_w64(const double *U, double *__restrict__ divF, KArgs a) {
  divergence_block<D, N, VISC, BM, FC, SELF>(U, divF, a, xcd_block(blockIdx.x, gridDim.x));
}

template <int D, int N, int FC>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_divergence_multi(const MultiCase *__restrict__ cs, const long *__restrict__ starts, int nc) {
  const int c = find_case(starts, nc, blockIdx.x);
  divergence_block<D, N, false, 0, FC, true>(cs[c].U, cs[c].out, cs[c].a, (long)blockIdx.x - starts[c]);
}

// ---------------------------------------------------------------- one-sided LDG path
// With LDG beta = +1/2 (BM 1) the common viscous flux uses only the left (slot-0)
// side's gradient, with beta = -1/2 (BM 2) only the right side's (src/faces.cpp:1520-1545),
// and the common solution is the other side's state.  The element on that "owner" side
// therefore has everything for the complete common flux (Rusanov + LDG) right after its
// own corrected gradient: it writes the unscaled common normal flux to Ftr at its owned
// flux points, and no gradient trace is needed.  The partner's solution trace at an owned
// point is extrapolated from the partner's U inside the kernel.  A residual is then
//   k_visc_onesided (gradient, volume flux divergence, owned common fluxes)
//   -> k_face_correction (oppDiv_fpts Fcomm, both sides).
// Any other beta (BM 0) runs through the same two kernels: each side's viscous flux enters
// the common flux with its own weight, so each side writes its share of the flux at every
// flux point (5 values where a gradient trace is 15) and k_face_correction adds the two.
// The three launches it replaces (trace, gradient and its traces, divergence with the
// gradient and both sides' fluxes formed again) took 84 us per residual of 21x23x19 hexes
// p=2 and 1.94 ms of 48^2 x 49 hexes p=3.

// Register budget: three waves per SIMD for hex p=3 and 4.  At p=3 the kernel's LDS admits 15
// waves per CU, but 3.2 per SIMD are in flight on average, with the LDS pipe 70% and the VALU
// 54% busy (64^3, rocprofv3), so a fourth wave buys nothing: held to 128 VGPRs the Roe kernel
// spills 10 of them (0.37 GB written and read back per residual; 64^3 residual 1627 us), at
// 148 it spills none (1488 us).  Rusanov takes 124 either way.  At p=4 beta = +-1/2 takes 144
// by itself; a general beta would take 175, two waves, and at three spills 6 to 10 (14x12x13,
// two / three waves: Rusanov 52.0 / 49.2 us, Roe 52.6 / 49.8).  Other shapes keep the default
// allocation.
template <int D, int N>
struct OneSidedWaves {
  static constexpr int value = (D == 3 && (N == 4 || N == 5)) ? 3 : 1;
};

// SELF: extrapolate the partner traces this element needs from the partner's U (no trace
// launch before this kernel); otherwise read them from Utr at the partner's points (written
// by a trace launch or by the previous RK stage's update), which this kernel then leaves as
// it is.  A template parameter: as a run-time branch the two prologues together spill the
// hex p=3 kernel.
template <int D, int N, int BM, int FC, bool SELF>
__device__ __forceinline__ void visc_onesided_block(const double *__restrict__ U, double *__restrict__ divF,
                                                    const KArgs &a, long bid) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  constexpr int owner = (BM == 2) ? 1 : 0;  // slot that forms the convective flux (and, beta = +-1/2, whose gradient enters)
  // one LDS region per element holds the common solution, then (after a barrier) the
  // gradient, then the transformed flux
  constexpr int WU = S::ele(V * nS), W = S::ele((V * nF > D * V * nS) ? V * nF : D * V * nS);
  extern __shared__ double lds[];
  const int EB = a.EB;
  double *lops = lds;
  double *lU = lops + S::NOPS_PAD;
  double *lW = lU + EB * WU;
  const long e0 = bid * EB;
  const long neb = min((long)EB, (long)a.E - e0);
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  // Work item k of an element is its k-th owned flux point.  Quads of N >= 5 points per
  // direction own about 2 N of their 4 N <= N^2 flux points, and the items of an element on its
  // own points' lanes kept every wave busy in the longest phase with 2 / N of its lanes.  There
  // the first H = 2 N items of all the workgroup's elements are dealt to its threads in a row,
  // then the others (of elements that own more faces): a thread has one item at most, (fe, fk)
  // its element and item, and waves without any skip the phase.  Elsewhere items stay on their
  // element's lanes, nS apart: hexes have 3 / N of the lanes busy and lose as much by the second
  // element index (64^3 p=3 Roe 1530 / 1580 us, 13x11x17 p=5 71 / 77), quads p=3 gain nothing
  // (256^2 67 / 70).  In lanes / in a row: 256^2 quads p=4 112 / 105 us, with Roe 115 / 112;
  // 96x100 23.0 / 21.8; 200x201 p=5 106 / 97; 150x151 p=6 90 / 80; 24^2 p=6 11.7 / 11.7.  Not
  // where an element fills waves of its own (nS a multiple of 64: quads p=7), whose default
  // tile is one element, so that a row is its own lanes again (73x64 p=7 30.4 / 31.2, with Roe
  // 30.8 / 32.0).
  // A thread takes its item in the prologue and again in the face phase, so with SELF the
  // partner's trace there stays in its registers (a second item, nS further, is rare for
  // N >= 3; its trace is parked in Utr at the element's own point, which nothing else reads).
  // The staging loads are issued first and the partner's values before any is consumed; with
  // SELF they are its solution line through the point (no trace launch runs before this
  // kernel), otherwise its trace from Utr, which is only read: the face phase reads it there
  // again (held instead, hexes p=6 take 146 VGPRs for 126).
  constexpr bool self = SELF;
  constexpr bool kRow = BM != 0 && D == 2 && N >= 5 && nS % 64 != 0;
  constexpr int H = D * S::nFF, Q = kRow ? nF : nS;
  StageRegs<D, N> sr;
  stage_U_load<D, N>(U, a, e0, neb, sr);
  const int half = (kRow && tid >= EB * H) ? 1 : 0, ti = tid - half * EB * H;
  const int fe = kRow ? ti / H : el, fk = kRow ? ti - fe * H + half * H : t;
  const bool fvalid = kRow ? fe < neb : valid;
  const long ef = kRow ? e0 + fe : e;
  const unsigned mask = fvalid ? owned_faces<D, N>(a.nbr + ef * nF, owner) : 0u;
  const unsigned owned = face_list<D>(mask), unowned = face_list<D>(~mask);
  const int cnt = __popc(mask) * S::nFF;
  double *c = lW + el * W, *cf = lW + fe * W;
  double cp[V];
  // general beta: the items are all flux points, the owned ones first, and the partner's
  // trace is needed at each (nothing is parked: the few owned items beyond the first nS fetch
  // it again in the face phase)
  auto item_fpt = [&](int k) {
    return (BM == 0 && k >= cnt) ? list_fpt<D, N>(unowned, k - cnt) : list_fpt<D, N>(owned, k);
  };
  auto partner = [&](int f, double *x) {
    long ep; int sl, fp;
    unpack_nbr<D, N>(a.nbr[ef * nF + f], ep, sl, fp);
    if constexpr (self) {
      partner_trace<D, N>(U, a.ops, ep, fp, x);
    } else {
#pragma unroll
      for (int v = 0; v < V; v++) x[v] = a.Utr[(ep * V + v) * nF + fp];
    }
  };
  if constexpr (BM == 0) {
    unsigned nb[S::FPT];
#pragma unroll
    for (int k = 0; k < S::FPT; k++) {
      const int i = fk + k * nS;
      nb[k] = (fvalid && i < nF) ? a.nbr[ef * nF + item_fpt(i)] : 0u;
    }
    // the staged block has arrived with the entries (loads return in order): its registers
    // are free for the lines
    stage_U_store<D, N>(U, a, lops, lU, e0, neb, WU, sr);
    PartnerLine<D, N> pl[self ? S::FPT : 1];
    double x[S::FPT][V];
#pragma unroll
    for (int k = 0; k < S::FPT; k++) {
      if (!fvalid || fk + k * nS >= nF) continue;
      long ep; int sl, fp;
      unpack_nbr<D, N>(nb[k], ep, sl, fp);
      if constexpr (self) {
        partner_line_load<D, N>(U, a.ops, ep, fp, pl[k]);
      } else {
#pragma unroll
        for (int v = 0; v < V; v++) x[k][v] = a.Utr[(ep * V + v) * nF + fp];
      }
    }
#pragma unroll
    for (int k = 0; k < S::FPT; k++) {
      const int i = fk + k * nS;
      if (!fvalid || i >= nF) continue;
      if constexpr (self) partner_line_reduce<D, N>(pl[k], x[k]);
      const int f = item_fpt(i);
#pragma unroll
      for (int v = 0; v < V; v++) cf[v * nF + f] = x[k][v];
    }
#pragma unroll
    for (int v = 0; v < V; v++) cp[v] = x[0][v];
  }
  if (BM != 0 && fk < cnt && fvalid) {
    const int f = list_fpt<D, N>(owned, fk);
    long ep; int sl, fp;
    unpack_nbr<D, N>(a.nbr[ef * nF + f], ep, sl, fp);
    if constexpr (self) {
      PartnerLine<D, N> pl;
      partner_line_load<D, N>(U, a.ops, ep, fp, pl);
      partner_line_reduce<D, N>(pl, cp);
    } else {
#pragma unroll
      for (int v = 0; v < V; v++) cp[v] = a.Utr[(ep * V + v) * nF + fp];
    }
#pragma unroll
    for (int v = 0; v < V; v++) cf[v * nF + f] = cp[v];
  }
#pragma unroll 1
  for (int k = fk + Q; BM != 0 && k < cnt; k += Q) {
    const int f = list_fpt<D, N>(owned, k);
    double x[V];
    partner(f, x);
#pragma unroll
    for (int v = 0; v < V; v++) {
      cf[v * nF + f] = x[v];
      if (self) a.Utr[(ef * V + v) * nF + f] = x[v];
    }
  }
  if constexpr (BM != 0) stage_U_store<D, N>(U, a, lops, lU, e0, neb, WU, sr);
  __syncthreads();
  const double *u = lU + el * WU, *uf = lU + fe * WU;
  double *g_l = c, *gf = cf;
  // common solution: beta = +-1/2 the non-owner side's state, so this element's own trace
  // where the partner owns the face; else both sides' traces mixed
  if (BM == 0 && fvalid) {
    for (int k = fk; k < nF; k += Q) {
      const int f = item_fpt(k);
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
#pragma unroll
      for (int v = 0; v < V; v++) {
        const double own = line_extrap<N>(lE, uf + v * nS, base, str), par = cf[v * nF + f];
        const double l = (k < cnt) ? own : par, r = (k < cnt) ? par : own;
        cf[v * nF + f] = 0.5 * (l + r) - a.ldg_b * (l - r);
      }
    }
  }
  if (BM != 0 && fvalid) {
    const int rest = nF - cnt;
#pragma unroll 1
    for (int k = fk; k < rest; k += Q) {
      const int f = list_fpt<D, N>(unowned, k);
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
#pragma unroll
      for (int v = 0; v < V; v++) cf[v * nF + f] = line_extrap<N>(lE, uf + v * nS, base, str);
    }
  }
  __syncthreads();
  {
    double g[V][D];
    if (valid) {
      double ij[D][D], detJ;
      load_metric<D>(a, e, t, nS, ij, detJ, true);
      spt_gradient<D, N>(lops, u, c, t, ij, detJ, g);
    }
    __syncthreads();  // the common solution is consumed
    if (valid) {
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++) g_l[(d * V + v) * nS + t] = g[v][d];
    }
  }
  __syncthreads();
  // common normal flux (unscaled) at the owned flux points -> Ftr; general beta: this side's
  // share of it at every flux point (the convective flux and the penalty at owned ones, this
  // side's viscous flux with its weight at all)
  if (fvalid) {
#pragma unroll 1
    for (int k = fk; k < (BM == 0 ? nF : cnt); k += Q) {
      const int f = item_fpt(k);  // face-major: neighbouring lanes, neighbouring points
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
      const double *fg = a.fgeo + ef * (D + 1) * nF + f;
      double n[D];
#pragma unroll
      for (int d = 0; d < D; d++) n[d] = fg[d * nF];
      double Uo[V], Up[V];
#pragma unroll
      for (int v = 0; v < V; v++) Uo[v] = line_extrap<N>(lE, uf + v * nS, base, str);
      // the convective flux and the LDG penalty first, so that their temporaries and the
      // partner's state are dead before the gradient's lines are gathered (Roe in the other
      // order needs ~350 registers)
      double Fo[V], G[V];
#pragma unroll
      for (int v = 0; v < V; v++) Fo[v] = 0.0;
      if (BM != 0 || k < cnt) {
        if (self && k == fk) {
#pragma unroll
          for (int v = 0; v < V; v++) Up[v] = cp[v];
        } else if (BM == 0 || !self) {
          partner(f, Up);
        } else {
#pragma unroll
          for (int v = 0; v < V; v++) Up[v] = a.Utr[(ef * V + v) * nF + f];
        }
        if (owner == 0) {
          conv_common_flux<D, FC>(Uo, Up, n, a, Fo);
#pragma unroll
          for (int v = 0; v < V; v++) Fo[v] += a.ldg_tau * (Uo[v] - Up[v]);
        } else {
          conv_common_flux<D, FC>(Up, Uo, n, a, Fo);
#pragma unroll
          for (int v = 0; v < V; v++) Fo[v] += a.ldg_tau * (Up[v] - Uo[v]);
        }
      }
      asm volatile("" ::: "memory");
      // one variable's line at a time (a compiler barrier after each): all lines in flight at
      // once take some 30 VGPRs more, spilled or a wave less in the shapes that are full
      visc_normal<D>(Uo, [&](int j, double *dUj) {
#pragma unroll
        for (int v = 0; v < V; v++) {
          dUj[v] = line_extrap<N>(lE, gf + (j * V + v) * nS, base, str);
          asm volatile("" : "+v"(dUj[v]) : : "memory");  // formed here, before the next line is loaded
        }
      }, n, a, G);
      // this side's weight 1/2 +- beta: the owner's alone, 1, with beta = +-1/2
      const double wt = (BM == 0) ? ((k < cnt) ? 0.5 + a.ldg_b : 0.5 - a.ldg_b) : 1.0;
#pragma unroll
      for (int v = 0; v < V; v++) Fo[v] += wt * G[v];
#pragma unroll
      for (int v = 0; v < V; v++) __builtin_nontemporal_store(Fo[v], &a.Ftr[(ef * V + v) * nF + f]);
    }
  }
  __syncthreads();  // the gradient field is consumed
  // pointwise flux contracted with the adjugate rows, over the own spt column of lG
  if (valid) {
    double ij[D][D], detJ;
    load_metric<D>(a, e, t, nS, ij, detJ, false);
    double Us[V], g[V][D];
#pragma unroll
    for (int v = 0; v < V; v++) Us[v] = u[v * nS + t];
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int v = 0; v < V; v++) g[v][d] = g_l[(d * V + v) * nS + t];
    const Prim<D> p = primitives<D>(Us, a.gamma);
    const Visc<D> vs = viscous<D>(Us, p, g, a);
    double tF[D][V];
#pragma unroll
    for (int d1 = 0; d1 < D; d1++) {
      conv_proj<D>(Us, p, ij[d1], tF[d1]);
      visc_proj_sub<D>(vs, ij[d1], tF[d1]);
    }
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int v = 0; v < V; v++) g_l[(d * V + v) * nS + t] = tF[d][v];
  }
  __syncthreads();
  if (!valid) return;
  // volume part of the divergence: oppDiv tF (src/elements.cpp:1449-1474)
  const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
  double acc[V];
#pragma unroll
  for (int v = 0; v < V; v++) acc[v] = 0.0;
#pragma unroll
  for (int d = 0; d < D; d++) {
    const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
    const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
    const int base = t - id * str;
    const double *Dr = tab_Dss<N>(lops, id);
#pragma unroll
    for (int v = 0; v < V; v++) {
      double s = acc[v];
#pragma unroll
      for (int m = 0; m < N; m++) s += Dr[m] * g_l[(d * V + v) * nS + base + m * str];
      acc[v] = s;
    }
  }
  // streaming stores for the outputs (divF, Ftr): the next kernel reads them, this one
  // does not, and they should not displace the partner lines other workgroups are about to
  // read from L2 (-0.8% per residual, measured A/B)
#pragma unroll
  for (int v = 0; v < V; v++) __builtin_nontemporal_store(acc[v], &divF[(e * V + v) * nS + t]);
}

template <int D, int N, int BM, int FC, bool SELF>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) __attribute__((amdgpu_waves_per_eu(OneSidedWaves<D, N>::value)))
void k_visc_onesided(const double *__restrict__ U, double *__restrict__ divF, KArgs a) {
  visc_onesided_block<D, N, BM, FC, SELF>(U, divF, a, xcd_block(blockIdx.x, gridDim.x));
}

// The same kernel for workgroups of one wave (64 threads: one hex p=3 element per
// workgroup, the tile the autotuner picks there): the compiler knows the workgroup is a
// single wave, so its barriers need no cross-wave synchronisation.
template <int D, int N, int BM, int FC, bool SELF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(OneSidedWaves<D, N>::value)))
void k_visc_onesided_w64(const double *__restrict__ U, double *__restrict__ divF, KArgs a) {
  visc_onesided_block<D, N, BM, FC, SELF>(U, divF, a, xcd_block(blockIdx.x, gridDim.x));
}

template <int D, int N, int BM, int FC>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) __attribute__((amdgpu_waves_per_eu(OneSidedWaves<D, N>::value)))
void k_visc_onesided_multi(const MultiCase *__restrict__ cs, const long *__restrict__ starts, int nc) {
  const int c = find_case(starts, nc, blockIdx.x);
  visc_onesided_block<D, N, BM, FC, BM != 0>(cs[c].U, cs[c].out, cs[c].a, (long)blockIdx.x - starts[c]);
}


// divF += oppDiv_fpts Fcomm (src/elements.cpp:1476-1501) with Fcomm = Ftr(owner) * signed
// dA of this side; the owner's Ftr is this element's own or its partner's.
template <int D, int N, int BM>
__device__ __forceinline__ void face_correction_block(double *__restrict__ divF, const KArgs &a, long bid) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  constexpr int owner = (BM == 2) ? 1 : 0;
  // per-element LDS block: the common fluxes (V * nF), then the new state (V * nS) when the
  // RK update writes the next trace
  constexpr int W = S::ele(V * (nF > nS ? nF : nS));
  extern __shared__ double lds[];
  const int EB = a.EB;
  double *lops = lds;
  double *lF = lops + S::NOPS_PAD;
  const int tid = threadIdx.x, NT = blockDim.x;
  for (int i = tid; i < S::NOPS; i += NT) lops[i] = a.ops[i];
  const long e0 = bid * EB;
  const long neb = min((long)EB, (long)a.E - e0);
  const int el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  double *c = lF + el * W;
  if (valid) {
#pragma unroll
    for (int k = 0; k < S::FPT; k++) {
      const int f = t + k * nS;
      if (f >= nF) continue;
      long ep; int sl, fp;
      unpack_nbr<D, N>(a.nbr[e * nF + f], ep, sl, fp);
      const double dAs = a.fgeo[(e * (D + 1) + D) * nF + f];
      if constexpr (BM == 0) {  // both sides' shares
        const double *so = a.Ftr + e * V * nF + f, *sp = a.Ftr + ep * V * nF + fp;
#pragma unroll
        for (int v = 0; v < V; v++) c[v * nF + f] = (so[v * nF] + sp[v * nF]) * dAs;
      } else {
        const double *src = (sl == owner) ? a.Ftr + e * V * nF + f : a.Ftr + ep * V * nF + fp;
#pragma unroll
        for (int v = 0; v < V; v++) c[v * nF + f] = src[v * nF] * dAs;
      }
    }
  }
  __syncthreads();
  double unew[V], res[V];
  if (valid) {
    const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
    double acc[V];
#pragma unroll
    for (int v = 0; v < V; v++) acc[v] = divF[(e * V + v) * nS + t];
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
      const double *Df = tab_Dsf<N>(lops, id);
      const int f0 = fpt_end<D, N>(ia, ib, ic, d, 0), f1 = fpt_end<D, N>(ia, ib, ic, d, 1);
#pragma unroll
      for (int v = 0; v < V; v++) {
        acc[v] += (-Df[0]) * c[v * nF + f0];
        acc[v] += Df[1] * c[v * nF + f1];
      }
    }
    if (a.rk.mode == 4) {
#pragma unroll
      for (int v = 0; v < V; v++) acc[v] += a.rk.src[(e * V + v) * nS + t];
    }
#pragma unroll
    for (int v = 0; v < V; v++) __builtin_nontemporal_store(acc[v], &divF[(e * V + v) * nS + t]);
#pragma unroll
    for (int v = 0; v < V; v++) res[v] = acc[v];
    rk_epilogue<D>(a, e, t, nS, acc, unew);
  }
  // the new state's trace for the next stage: at partner-owned points, or (general beta) all
  if (a.rk.mode == 1 && a.rk.trace) rk_trace<D, N>(a, lops, c, e, t, valid, unew, BM == 0 ? -1 : owner);
  // p-multigrid transfers (the common fluxes in c are consumed; U comes from pmgU)
  if (a.rk.pmgRc || a.rk.pmgUf) pmg_epilogue<D, N>(a, lops, nullptr, c, e, t, valid, res, unew);
}

template <int D, int N, int BM>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_face_correction(double *__restrict__ divF, KArgs a) {
  face_correction_block<D, N, BM>(divF, a, xcd_block(blockIdx.x, gridDim.x));
}

template <int D, int N, int BM>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_face_correction_multi(const MultiCase *__restrict__ cs, const long *__restrict__ starts, int nc) {
  const int c = find_case(starts, nc, blockIdx.x);
  face_correction_block<D, N, BM>(cs[c].out, cs[c].a, (long)blockIdx.x - starts[c]);
}

// ---------------------------------------------------------------- reverse mode
#include "adjoint.hpp"

// ---------------------------------------------------------------- dispatch
// LDS budget per workgroup; kept at 64 KiB so several workgroups share a CU.  Shapes whose
// element alone needs more than 256 threads (hexes of order 6 to 8) may take up to the
// 160 KiB a gfx950 workgroup can allocate (one element per workgroup).
constexpr size_t kMaxLds = 64 * 1024;
constexpr size_t kMaxLdsBig = 160 * 1024;
template <int D, int N>
constexpr size_t max_lds() { return Shape<D, N>::nS > kMaxThreads ? kMaxLdsBig : kMaxLds; }
inline size_t max_lds_n(int D, int N) {
  int nS = N * N;
  if (D == 3) nS *= N;
  return nS > kMaxThreads ? kMaxLdsBig : kMaxLds;
}

// The default tile of a launch of its own (EB * nS threads).  The one-sided, divergence and
// main adjoint kernels (phased) are latency-bound and their phases are separated by
// barriers, so a workgroup of one wave, whose barriers cost nothing, is their best tile
// wherever its lanes are well filled; where they are not, and for the launches of one or
// two phases, the idle lanes cost more than the barriers and the tile of up to four waves
// with the fewest idle lanes is.  The line, measured on the one-sided kernel and the Euler
// divergence (one wave against the best-filled tile):
//   nS = 25, filled to 25/32: viscous 256^2 quads 85 against 74 us, Euler 51 against 46;
//   nS = 49, filled to 49/64: viscous 192^2 quads 121 against 107, Euler 68 against 60;
//   nS = 27, filled to 27/32: 40^3 hexes viscous 185 against 194, Euler 113 against 136;
//   nS = 64: 48^3 hexes viscous 545 against 669 (256 threads), Euler 455 against 557.
// The main adjoint kernels alone, one wave against the best-filled tile (3e5 points):
//   nS = 25: quads p=4 Rusanov 34.4 against 31.1, Euler 18.9 / 17.7, general beta 26.6 / 24.7;
//   nS = 27: hexes p=2 Rusanov 68 against 78, Roe 76 / 86, Euler 27 / 27, general beta 47 / 50;
//   nS = 16: quads p=3 27.0 against 29.4, 32.5 / 35.5, 15.0 / 15.7, 21.6 / 23.7;
//   nS = 64: hexes p=3 61 against 78, 69 / 93, 22.2 / 23.3, 46 / 51
// (k_adj_main_gen has no one-wave form: its fewer waves wait less for one another).
inline int default_tile(int nS, bool phased, long nEles) {
  const int one = 64 / nS;
  if (phased && one * nS * 32 >= 64 * 27) {
    // elements of one point: 64 of them to a wave leave a mesh of a few ten thousand on part of
    // the SIMDs; rather >= 1024 workgroups, of 32 elements or more (33x29x31 hexes, the
    // one-sided kernel with 64 / 30 / 16 per workgroup: Rusanov 17.9 / 16.8 / 17.0 us, Roe 19.2 /
    // 17.8 / 20.5; Euler residual of 31^3 8.9 with 64, 9.0 with 32, 10.8 with 16)
    const long wgs = (nEles + 1023) / 1024;
    return (nS == 1 && wgs < one) ? (int)(wgs < 32 ? 32 : wgs) : one;
  }
  int best = one < 1 ? 1 : one, waves = (best * nS + 63) / 64;
  for (int w = waves + 1; w <= kMaxThreads / 64; w++) {
    const int eb = 64 * w / nS;
    if (eb * waves > best * w || (!phased && eb * waves == best * w)) { best = eb; waves = w; }  // more lanes filled
  }
  // small meshes: rather >= 1024 workgroups (four per CU) than well filled ones: the
  // one-wave tile where that leaves as many, else as few elements as do, but never a wave
  // emptier than it need be (480 quads: of 9 points, 7 per workgroup 7.6 us, one 9.0; of 16
  // points, 4 per workgroup 6.6 us, one 7.6; of 36 points, one per workgroup 7.3 us, seven 8.0)
  if (nEles < 1024L * best) {
    const long eb = (nEles + 1023) / 1024;
    best = (one >= 1 && (nEles >= 1024L * one || eb < one)) ? one : (int)eb;
  }
  return best;
}

// Elements per workgroup: the requested tile or the default, limited by the thread count
// and the LDS the kernel needs per element (per_ele doubles).
// one_wave: the launch's workgroup is EB * nS threads, so that a one-wave tile runs as a
// one-wave workgroup; false for launches of kMaxThreads-thread workgroups (multi-case
// launches, persistent plans), where the threads beyond EB * nS would idle: those fill the
// 256 threads (defEB elements), or on small meshes keep >= 1024 workgroups.
inline int eles_per_block(const zfr_ele_desc_t *d, int defEB, size_t fixed, size_t per_ele, bool one_wave,
                          bool phased) {
  int eb = d->eles_per_block;
  if (eb <= 0 && one_wave) eb = default_tile(d->nSpts, phased, d->nEles);
  else if (eb <= 0) {
    const long per_cu4 = ((long)d->nEles + 1023) / 1024;
    eb = per_cu4 < defEB ? (per_cu4 < 1 ? 1 : (int)per_cu4) : defEB;
  }
  while (eb > 1 && (eb * d->nSpts > kMaxThreads || sizeof(double) * (fixed + eb * per_ele) > kMaxLds)) eb--;
  return eb < 1 ? 1 : eb;
}

inline KArgs make_args(const zfr_ele_desc_t *d, int EB) {
  KArgs a;
  a.E = d->nEles; a.EB = EB; a.viscous = d->viscous; a.fix_vis = d->fix_vis;
  a.gamma = d->gamma; a.prandtl = d->prandtl; a.mu = d->mu; a.rt = d->rt; a.c_sth = d->c_sth;
  a.rus_k = d->rus_k; a.ldg_b = d->ldg_b; a.ldg_tau = d->ldg_tau;
  a.ops = d->ops1d; a.metric = d->metric; a.fgeo = d->fgeo; a.nbr = d->nbr; a.Utr = d->Utr; a.Gtr = d->Gtr;
  a.Ftr = d->Ftr;
  a.trace_sel = 0;
  a.rk = KArgs::Rk{};
  return a;
}

enum class Op {
  Extrap, ExtrapPartner, Grad, Div, OneSided, OneSidedFromTrace, FaceCorr,
  BothSides, FaceCorrBoth,  // the one-sided pair's general-beta form
  BothSidesFromTrace,       // the same after a trace launch (multi-case launches)
  AdjPrep, AdjMain, AdjGather,  // reverse mode (Euler, LDG beta = +-1/2; AdjPrep and AdjGather also general beta)
  AdjFace, AdjMainGen           // reverse mode, general LDG beta
};

// Extra operands of the reverse-mode launches.
struct AdjPtrs {
  const double *w = nullptr;  // cotangent of divF
  double *Wtr = nullptr;      // [E][V][nF] face weights of w
  double *Xtr = nullptr;      // [E][V][nF] partner trace cotangent at owned points
  const KArgs::Rk *rk = nullptr;  // fused RK update for Div / FaceCorr
};

// LDS doubles per element of each kernel.
template <int D, int N>
size_t lds_per_element(Op op, bool viscous) {
  using S = Shape<D, N>;
  constexpr int VS = S::V * S::nS, VF = S::V * S::nF, G = D * VS;
  size_t per_ele = 0;
  switch (op) {
    case Op::Extrap:
    case Op::ExtrapPartner: per_ele = S::ele(VS); break;
    case Op::Grad: per_ele = S::ele(VS + VF > G ? VS + VF : G); break;
    case Op::Div: per_ele = S::ele(VS) + S::ele(VF) + S::ele(G); break;
    case Op::OneSided:
    case Op::OneSidedFromTrace:
    case Op::BothSides:
    case Op::BothSidesFromTrace:
      per_ele = S::ele(VS) + S::ele(VF > G ? VF : G);
      break;
    case Op::FaceCorr:
    case Op::FaceCorrBoth: per_ele = S::ele(VF > VS ? VF : VS); break;
    case Op::AdjPrep: per_ele = VS; break;
    case Op::AdjMain:
      per_ele = viscous ? (size_t)AdjLds<D, N, true>::per_ele : (size_t)AdjLds<D, N, false>::per_ele;
      break;
    case Op::AdjGather: per_ele = S::ele(VF); break;
    case Op::AdjFace: per_ele = 0; break;
    case Op::AdjMainGen: per_ele = (size_t)AdjGenLds<D, N>::per_ele; break;
  }
  return per_ele;
}

// One launch of a multi-case plan: every case of one kernel, shape and flux branch.
struct MultiGroup {
  Op op = Op::Extrap;
  int D = 0, N = 0, visc = 0, bm = 0, fc = 0;  // bm: LDG branch (0 general, 1 beta = 1/2, 2 beta = -1/2)
                                               // N = 0: cases of several orders (kernels_mixed.hip);
                                               // with D = 0 also of both nDims
  int EB = 1, nc = 0;
  unsigned nblk = 0;
  size_t lds = 0;
  MultiCase *cases = nullptr;  // device [nc]
  long *starts = nullptr;      // device [nc]
};

template <int D>
size_t lds_per_element_n(int N, Op op, bool viscous) {
  switch (N) {
    case 1: return lds_per_element<D, 1>(op, viscous);
    case 2: return lds_per_element<D, 2>(op, viscous);
    case 3: return lds_per_element<D, 3>(op, viscous);
    case 4: return lds_per_element<D, 4>(op, viscous);
    case 5: return lds_per_element<D, 5>(op, viscous);
    case 6: return lds_per_element<D, 6>(op, viscous);
    case 7: return lds_per_element<D, 7>(op, viscous);
    case 8: return lds_per_element<D, 8>(op, viscous);
    case 9: return lds_per_element<D, 9>(op, viscous);
  }
  if constexpr (D == 2) {
    if (N == 10) return lds_per_element<2, 10>(op, viscous);
  }
  return 0;
}

// Defined and explicitly instantiated per shape in kernels_shape.hip.
template <int D, int N>
int launch(Op op, const zfr_ele_desc_t *d, const double *U, double *out, hipStream_t st, const AdjPtrs &j);
template <int D, int N>
void launch_multi(const MultiGroup &g, hipStream_t st);
// Defined and explicitly instantiated in kernels_mixed.hip for D = 2, 3 and 0 (both).
template <int D>
void launch_mixed(const MultiGroup &g, hipStream_t st);
// The ops a mixed-order launch covers (the Euler divergence and the one-sided LDG pair).
inline bool mixed_op(Op op, int visc) { return (op == Op::Div && !visc) || op == Op::OneSided || op == Op::FaceCorr; }
// Orders a mixed-order launch compiles in (points per direction 1..6); quads of higher
// order get launches of their own shape.
constexpr int kMixedMaxN = 6;

// ---------------------------------------------------------------- persistent plans
// One phase of a persistent plan: an Euler divergence launch (a residual, or a fused RK
// stage / source-term / restriction epilogue around one), recorded instead of launched.
// k_persist runs every phase of a plan in one cooperative launch: its resident workgroups
// walk the phase's element blocks (block b as the single launch's workgroup b) and meet
// at a grid-wide barrier before the next phase.
struct PersistPhase {
  KArgs a;
  const double *U;
  double *out;
  long nblk;     // element blocks of the phase (the single launch's grid)
  int N, D, fc, self;  // points per direction, nDims, Roe, partner traces extrapolated from U
};
// While set on a thread, the Euler divergence launches of that thread are appended here
// and every other launch entry point fails (a plan holds nothing else).
struct PersistRecorder {
  std::vector<PersistPhase> phases;
  size_t lds = 0;  // the largest LDS of the phases
  int D = 0;
};
extern thread_local PersistRecorder *g_persist;
// 0, or a failure status naming the launch that cannot be recorded.
int refuse_while_recording(const char *what);
// Defined and instantiated in kernels_mixed.hip (D = 2, 3).
template <int D>
hipError_t launch_persist(const PersistPhase *phases, int nph, unsigned grid, size_t lds, hipStream_t st);
template <int D>
hipError_t persist_blocks_per_cu(size_t lds, int *n);

}  // namespace zk
