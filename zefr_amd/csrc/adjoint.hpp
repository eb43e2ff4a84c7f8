// adjoint.hpp -- reverse-mode kernels of the residual (included by kernels.hip, inside
// namespace zk, after the forward kernels and their helpers).
//
// Vector-Jacobian product of one residual: v = (d divF / dU)^T w at the state U, for the
// one-sided LDG path (beta = +-1/2) and for Euler (new; no reference counterpart).
// The forward path, read backwards, is
//   divF = Dss^T-lines(tF) + signed Dsf (Fcomm),  Fcomm = Ftr(owner) dA_side,
//   Ftr  = RusanovLDG(U_L, U_R, G_owner . n),   G = viscous flux of (Utr, E grad),
//   tF   = F(U, grad) . adj,  grad = adj^T (Dss U + Dsf Ucomm) / detJ,
//   Ucomm = partner trace at owned points, own trace elsewhere, Utr = E U.
// The owner side of each face (slot 0 for beta = +1/2 and Euler, slot 1 for -1/2) does all
// the face work, as in the forward path: it combines both sides' weights of its common
// flux, and hands the partner's share of the trace cotangent back through Xtr.
//   k_adj_prep   : Wtr = dA_side * (signed Dsf^T w) at every flux point;
//   k_adj_main   : forward recompute, volume and face adjoints, gradient adjoint; writes
//                  v (all of this element's own contributions) and Xtr at owned points;
//   k_adj_gather : v += E^T (partner Xtr) at the points the partner owns.
#pragma once

// k_adj_gather's BM for general LDG beta: the partner's cotangent at every flux point.
constexpr int kAdjAllPoints = 3;

// Stage EB consecutive [V][nS] blocks of x into LDS (stride V*nS).
template <int D, int N>
__device__ __forceinline__ void stage_block(const double *__restrict__ x, double *lx, long e0, long neb) {
  using S = Shape<D, N>;
  const double *xb = x + e0 * S::V * S::nS;
  for (long i = threadIdx.x; i < neb * S::V * S::nS; i += blockDim.x) lx[i] = xb[i];
}

// Transposed line operator: sum_i Dss[i][m] x[base + i*str].
template <int N>
__device__ __forceinline__ double line_T_Dss(const double *lops, int m, const double *blk, int base, int str) {
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < N; i++) s += tab_Dss<N>(lops, i)[m] * blk[base + i * str];
  return s;
}

// sum over the spts t of a line of Dsf[m_t][side] x(t)
template <int N>
__device__ __forceinline__ double line_Dsf(const double *lops, int side, const double *blk, int base, int str) {
  double s = 0.0;
#pragma unroll
  for (int m = 0; m < N; m++) s += tab_Dsf<N>(lops, m)[side] * blk[base + m * str];
  return s;
}

template <int D, int N>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_adj_prep(const double *__restrict__ w, double *__restrict__ Wtr,
                                                          KArgs a) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  extern __shared__ double lds[];
  double *lops = lds;
  double *lW = lops + S::NOPS_PAD;
  const long e0 = xcd_block(blockIdx.x, gridDim.x) * a.EB;
  const long neb = min((long)a.EB, (long)a.E - e0);
  for (int i = threadIdx.x; i < S::NOPS; i += blockDim.x) lops[i] = a.ops[i];
  stage_block<D, N>(w, lW, e0, neb);
  __syncthreads();
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  if (el >= neb) return;
  const double *wl = lW + el * V * nS;
#pragma unroll
  for (int k = 0; k < S::FPT; k++) {
    const int f = t + k * nS;
    if (f >= nF) continue;
    int dim, side, base, str;
    fpt_info<D, N>(f, dim, side, base, str);
    const double dAs = a.fgeo[(e * (D + 1) + D) * nF + f];
    const double sg = side ? dAs : -dAs;
#pragma unroll
    for (int v = 0; v < V; v++) Wtr[(e * V + v) * nF + f] = sg * line_Dsf<N>(lops, side, wl + v * nS, base, str);
  }
}

// LDS per element.  Viscous: U [V][nS]; R, which holds the common solution [V][nF], then the
// forward gradient [D][V][nS], then the gradient-trace cotangents of the owned points
// [D][V][nS slots], then the own trace cotangent [V][nF]; GB, which holds w [V][nS], then
// the gradient cotangent [D][V][nS].  Euler: U, w and the own trace cotangent.
template <int D, int N, bool VISC>
struct AdjLds {
  using S = Shape<D, N>;
  static constexpr int U = S::ele(S::V * S::nS);
  static constexpr int R = S::ele((S::V * S::nF > D * S::V * S::nS || !VISC) ? S::V * S::nF : D * S::V * S::nS);
  static constexpr int GB = S::ele(VISC ? D * S::V * S::nS : S::V * S::nS);
  static constexpr int per_ele = U + R + GB;  // doubles
};

// The partner's trace at this thread's owned flux point f: its neighbour entry, then its
// solution line.
template <int D, int N>
__device__ __forceinline__ void owned_partner_trace(const double *__restrict__ U, const KArgs &a, long e, int f,
                                                    double *out) {
  long ep; int sl, fp;
  unpack_nbr<D, N>(a.nbr[e * Shape<D, N>::nF + f], ep, sl, fp);
  PartnerLine<D, N> pl;
  partner_line_load<D, N>(U, a.ops, ep, fp, pl);
  partner_line_reduce<D, N>(pl, out);
}

// The common flux of one owned point reversed, without its viscous part: Fb = both sides'
// weights of w, Uo / Up the owner's and the partner's traces.  Adds to Uob (owner's trace)
// and Gb (the owner's viscous normal flux), writes the partner's share to Upb.
template <int D, int N, bool VISC, int BM, int FC>
__device__ __forceinline__ void owned_flux_vjp(const KArgs &a, const double *__restrict__ Wtr, long e, int f,
                                               const double *n, const double *Uo, const double *Up, double *Uob,
                                               double *Upb, double *Gb) {
  using S = Shape<D, N>;
  constexpr int nF = S::nF, V = S::V, owner = (BM == 2) ? 1 : 0;
  long ep; int sl, fp;
  unpack_nbr<D, N>(a.nbr[e * nF + f], ep, sl, fp);
  double Fb[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    Fb[v] = Wtr[(e * V + v) * nF + f] + Wtr[(ep * V + v) * nF + fp];
    Uob[v] = Upb[v] = Gb[v] = 0.0;
  }
  if (owner == 0) common_flux_vjp<D, VISC, BM, FC>(Uo, Up, n, 1.0, a, Fb, Uob, Upb, Gb, nullptr);
  else common_flux_vjp<D, VISC, BM, FC>(Up, Uo, n, 1.0, a, Fb, Upb, Uob, Gb, nullptr);
}

// Work item k of an element is its k-th owned flux point (owned faces in increasing
// order); thread t takes k = t, t + nS, ...: half of the flux points are owned on average,
// so for N >= 3 one pass covers nearly every element, and thread t's point stays its own
// from the prologue (its partner's trace) to the end (its own trace's cotangent), in
// registers.  An element's earlier passes, if it has any, park those values in global
// memory at the element's own owned points (Utr, Wtr), which no other element reads.
template <int D, int N, int BM, int FC>
__device__ __forceinline__ void adj_visc_block(const double *__restrict__ U, const double *__restrict__ w,
                                               double *__restrict__ Wtr, double *__restrict__ Xtr,
                                               double *__restrict__ vout, const KArgs &a, long bid) {
  using S = Shape<D, N>;
  using L = AdjLds<D, N, true>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V, nFF = S::nFF;
  constexpr int owner = (BM == 2) ? 1 : 0;
  // hexes with Roe: what must outlive the face adjoint waits in global memory (the partner's
  // trace in Utr at this element's own point, the volume adjoint's part in vout) instead of
  // in registers, which the Roe reverse sweep fills: left to the compiler they are spilled,
  // which costs more (VJP of 32^3 hexes p=3 431 us spilled, 419 this way)
  constexpr bool kPark = D == 3 && FC == 1;
  extern __shared__ double lds[];
  const int EB = a.EB;
  double *lops = lds;
  double *lU = lops + S::NOPS_PAD;
  double *lR = lU + EB * L::U;
  double *lGB = lR + EB * L::R;
  const long e0 = bid * EB;
  const long neb = min((long)EB, (long)a.E - e0);
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  double *u = lU + el * L::U;
  double *c = lR + el * L::R, *g_l = c, *T = c, *to = c;
  double *gb = lGB + el * L::GB;
  // 0. staging loads of U and w, the owned faces, and the partner's trace at this thread's
  //    owned point; only then are values consumed
  StageRegs<D, N> sr;
  stage_U_load<D, N>(U, a, e0, neb, sr);
  double wr[V];
#pragma unroll
  for (int v = 0; v < V; v++) wr[v] = valid ? w[(e * V + v) * nS + t] : 0.0;
  unsigned mask = valid ? owned_faces<D, N>(a.nbr + e * nF, owner) : 0u;
  unsigned owned = face_list<D>(mask), unowned = face_list<D>(~mask);
  int cnt = __popc(mask) * nFF;
  // the element's last pass starts at work item 'last' (0 unless more than nS points are owned)
  const int last = (cnt > nS) ? ((cnt - 1) / nS) * nS : 0;
  const int klast = t + last;
  const bool has_last = klast < cnt;
  double cp[V];
  if (has_last) {
    const int f = list_fpt<D, N>(owned, klast);
    owned_partner_trace<D, N>(U, a, e, f, cp);
#pragma unroll
    for (int v = 0; v < V; v++) {
      c[v * nF + f] = cp[v];
      if (kPark) a.Utr[(e * V + v) * nF + f] = cp[v];
    }
  }
#pragma unroll 1
  for (int k = t; k < last; k += nS) {
    const int f = list_fpt<D, N>(owned, k);
    double x[V];
    owned_partner_trace<D, N>(U, a, e, f, x);
#pragma unroll
    for (int v = 0; v < V; v++) {
      c[v * nF + f] = x[v];
      a.Utr[(e * V + v) * nF + f] = x[v];
    }
  }
  stage_U_store<D, N>(U, a, lops, lU, e0, neb, L::U, sr);
  if (valid) {
#pragma unroll
    for (int v = 0; v < V; v++) gb[v * nS + t] = wr[v];
  }
  __syncthreads();
  const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
  // 1. common solution: this element's own trace where the partner owns the face
  if (valid) {
#pragma unroll 1
    for (int k = t; k < nF - cnt; k += nS) {
      const int f = list_fpt<D, N>(unowned, k);
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
#pragma unroll
      for (int v = 0; v < V; v++) c[v * nF + f] = line_extrap<N>(lE, u + v * nS, base, str);
    }
  }
  __syncthreads();
  // 2. forward physical gradient at every spt, into the region of c; tFb[d1] = Dss^T w along
  //    the d1 lines
  double Ub[kPark ? 1 : V], tFb[D][V];
  {
    double ij[D][D], detJ, g[V][D];
    if (valid) {
      load_metric<D>(a, e, t, nS, ij, detJ, true);
      spt_gradient<D, N>(lops, u, c, t, ij, detJ, g);
    }
    __syncthreads();  // the common solution is consumed
    if (valid) {
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int v = 0; v < V; v++) g_l[(d * V + v) * nS + t] = g[v][d];
#pragma unroll
      for (int d = 0; d < D; d++) {
        const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
        const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
#pragma unroll
        for (int v = 0; v < V; v++) tFb[d][v] = line_T_Dss<N>(lops, id, gb + v * nS, t - id * str, str);
      }
    }
    __syncthreads();  // w is consumed
    // 3. volume adjoint: F(U, grad) reversed for the cotangent tFb
    if (valid) {
      double Us[V], Usb[V];
#pragma unroll
      for (int v = 0; v < V; v++) {
        Us[v] = u[v * nS + t];
        Usb[v] = 0.0;
      }
      const Prim<D> p = primitives<D>(Us, a.gamma);
#pragma unroll
      for (int d = 0; d < D; d++) conv_proj_vjp<D>(Us, p, ij[d], tFb[d], a.gamma, Usb);
      // tF[d1] -= T . adj[d1]: cotangent on T[v][j] is -sum_d1 tFb[d1][v] adj[d1][j]
      viscous_vjp<D>(
          Us, p,
          [&](int j, double *dUj) {
#pragma unroll
            for (int v = 0; v < V; v++) dUj[v] = g[v][j];
          },
          [&](int v, int j) {
            double s = 0.0;
#pragma unroll
            for (int d1 = 0; d1 < D; d1++) s += tFb[d1][v] * ij[d1][j];
            return -s;
          },
          [&](int j, const double *gbj) {
#pragma unroll
            for (int v = 0; v < V; v++) gb[(j * V + v) * nS + t] = gbj[v];
          },
          a, Usb);
#pragma unroll
      for (int v = 0; v < V; v++) {
        if (kPark) vout[(e * V + v) * nS + t] = Usb[v];
        else Ub[kPark ? 0 : v] = Usb[v];
      }
    }
  }
  // 4. face adjoint at the owned points.  An owned point's gradient cotangent belongs to the
  //    spts of its normal line; in the last pass it is left in T, one slot per work item,
  //    and the spts collect it (phase 5).  T takes the forward gradient's place, so earlier
  //    passes, which still need that, add to the lines themselves face by face (lines of one
  //    face never meet, so the order is fixed).
  double Uob[V];
#pragma unroll 1
  for (int k0 = 0; k0 < nF; k0 += nS) {
    const int k = k0 + t;
    const bool now = k0 <= last, has = now && k < cnt, fin = k0 == last;
    int f = 0, dim = 0, side = 0, base = 0, str = 0;
    double dGb[V][D];
    if (has) {
      f = list_fpt<D, N>(owned, k);
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
      const double *fg = a.fgeo + e * (D + 1) * nF + f;
      double n[D], Uo[V], Gb[V];
      {
        double Up[V], Upb[V];
#pragma unroll
        for (int d = 0; d < D; d++) n[d] = fg[d * nF];
#pragma unroll
        for (int v = 0; v < V; v++) {
          Uo[v] = line_extrap<N>(lE, u + v * nS, base, str);
          Up[v] = (fin && !kPark) ? cp[v] : a.Utr[(e * V + v) * nF + f];
        }
        owned_flux_vjp<D, N, true, BM, FC>(a, Wtr, e, f, n, Uo, Up, Uob, Upb, Gb);
#pragma unroll
        for (int v = 0; v < V; v++) Xtr[(e * V + v) * nF + f] = Upb[v];
      }
      asm volatile("" ::: "memory");
      // G = -T(Uo, grad_o) . n
      const Prim<D> po = primitives<D>(Uo, a.gamma);
      viscous_vjp<D>(
          Uo, po,
          [&](int j, double *dUj) {
#pragma unroll
            for (int v = 0; v < V; v++) {
              dUj[v] = line_extrap<N>(lE, g_l + (j * V + v) * nS, base, str);
              asm volatile("" : "+v"(dUj[v]) : : "memory");  // formed here, before the next line is loaded
            }
          },
          [&](int v, int j) { return -Gb[v] * n[j]; },
          [&](int j, const double *gbj) {
#pragma unroll
            for (int v = 0; v < V; v++) dGb[v][j] = gbj[v];
          },
          a, Uob);
    }
    // a pass that is not the last of some element (the same for every thread)
    const bool more = __syncthreads_or(k0 < last);
    if (now && fin && has) {  // the forward gradient of this element is consumed
#pragma unroll
      for (int j = 0; j < D; j++)
#pragma unroll
        for (int v = 0; v < V; v++) T[(j * V + v) * nS + t] = dGb[v][j];
    }
    if (!more) break;
    const int face = (has && !fin) ? f / nFF : -1;
    if (face >= 0) {
#pragma unroll
      for (int v = 0; v < V; v++) Wtr[(e * V + v) * nF + f] = Uob[v];
    }
#pragma unroll 1
    for (int q = 0; q < 2 * D; q++) {
      __syncthreads();
      if (face == q) {
        const double *lE = tab_lE<N>(lops, side);
#pragma unroll 1
        for (int m = 0; m < N; m++)
#pragma unroll
          for (int j = 0; j < D; j++)
#pragma unroll
            for (int v = 0; v < V; v++) gb[(j * V + v) * nS + base + m * str] += lE[m] * dGb[v][j];
      }
    }
  }
  __syncthreads();
  if (kPark) {  // formed again rather than held (or spilled) across the face adjoint
    asm volatile("" : "+v"(mask));
    owned = face_list<D>(mask);
    unowned = face_list<D>(~mask);
    cnt = __popc(mask) * nFF;
  }
  // 5. each spt collects the gradient-trace cotangents of the owned ends of its lines, then
  //    reference-space gradient cotangent: grb[d2][v] = sum_d1 adj[d2][d1] gb[v][d1] / detJ
  //    (the metric read again here: held across the face adjoint it takes registers the
  //    Roe reverse sweep needs)
  if (valid) {
    asm volatile("" ::: "memory");
    double ij[D][D], detJ;
    load_metric<D>(a, e, t, nS, ij, detJ, true);
    double gv[V][D];
#pragma unroll
    for (int j = 0; j < D; j++)
#pragma unroll
      for (int v = 0; v < V; v++) gv[v][j] = gb[(j * V + v) * nS + t];
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
#pragma unroll
      for (int sd = 0; sd < 2; sd++) {
        const int f = fpt_end<D, N>(ia, ib, ic, d, sd);
        const int q = f / nFF;  // the same face for every spt: its end of direction d
        const int k = __popc(mask & ((1u << q) - 1u)) * nFF + (f - q * nFF);
        if (((mask >> q) & 1u) && k >= last) {
          const double l = tab_lE<N>(lops, sd)[id];
          const double *Tk = T + (k - last);
#pragma unroll
          for (int j = 0; j < D; j++)
#pragma unroll
            for (int v = 0; v < V; v++) gv[v][j] += l * Tk[(j * V + v) * nS];
        }
      }
    }
    const double inv_det = 1.0 / detJ;
#pragma unroll
    for (int d2 = 0; d2 < D; d2++)
#pragma unroll
      for (int v = 0; v < V; v++) {
        double s = 0.0;
#pragma unroll
        for (int d1 = 0; d1 < D; d1++) s += ij[d2][d1] * gv[v][d1];
        gb[(d2 * V + v) * nS + t] = s * inv_det;
      }
  }
  __syncthreads();
  // 6. Dss^T into U, Dsf^T into the common solution's cotangent: the partner's trace at
  //    owned points (Xtr), this element's trace elsewhere
  double vb[V];
  if (valid) {
#pragma unroll
    for (int v = 0; v < V; v++) vb[v] = kPark ? vout[(e * V + v) * nS + t] : Ub[kPark ? 0 : v];
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
      const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
#pragma unroll
      for (int v = 0; v < V; v++) vb[v] += line_T_Dss<N>(lops, id, gb + (d * V + v) * nS, t - id * str, str);
    }
    auto dsf = [&](int f, double *cb) {
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
#pragma unroll
      for (int v = 0; v < V; v++) cb[v] = line_Dsf<N>(lops, side, gb + (dim * V + v) * nS, base, str);
    };
    double cb[V];
    if (has_last) {
      const int f = list_fpt<D, N>(owned, klast);
      dsf(f, cb);
#pragma unroll
      for (int v = 0; v < V; v++) {
        Xtr[(e * V + v) * nF + f] += cb[v];
        to[v * nF + f] = Uob[v];
      }
    }
#pragma unroll 1
    for (int k = t; k < last; k += nS) {
      const int f = list_fpt<D, N>(owned, k);
      dsf(f, cb);
#pragma unroll
      for (int v = 0; v < V; v++) {
        Xtr[(e * V + v) * nF + f] += cb[v];
        to[v * nF + f] = Wtr[(e * V + v) * nF + f];
      }
    }
#pragma unroll 1
    for (int k = t; k < nF - cnt; k += nS) {
      const int f = list_fpt<D, N>(unowned, k);
      dsf(f, cb);
#pragma unroll
      for (int v = 0; v < V; v++) to[v * nF + f] = cb[v];
    }
  }
  __syncthreads();
  if (!valid) return;
  // 7. own trace cotangent E^T into v
#pragma unroll
  for (int d = 0; d < D; d++) {
    const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
    const double l0 = tab_lE<N>(lops, 0)[id], l1 = tab_lE<N>(lops, 1)[id];
    const int f0 = fpt_end<D, N>(ia, ib, ic, d, 0), f1 = fpt_end<D, N>(ia, ib, ic, d, 1);
#pragma unroll
    for (int v = 0; v < V; v++) vb[v] += l0 * to[v * nF + f0] + l1 * to[v * nF + f1];
  }
#pragma unroll
  for (int v = 0; v < V; v++) vout[(e * V + v) * nS + t] = vb[v];
}

// Euler: the volume adjoint, the face adjoint at the owned points (slot 0), and E^T.
template <int D, int N, int FC>
__device__ __forceinline__ void adj_euler_block(const double *__restrict__ U, const double *__restrict__ w,
                                                const double *__restrict__ Wtr, double *__restrict__ Xtr,
                                                double *__restrict__ vout, const KArgs &a, long bid) {
  using S = Shape<D, N>;
  using L = AdjLds<D, N, false>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  extern __shared__ double lds[];
  const int EB = a.EB;
  double *lops = lds;
  double *lU = lops + S::NOPS_PAD;
  double *lT = lU + EB * L::U;
  double *lw = lT + EB * L::R;
  const long e0 = bid * EB;
  const long neb = min((long)EB, (long)a.E - e0);
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  StageRegs<D, N> sr;
  stage_U_load<D, N>(U, a, e0, neb, sr);
  double wr[V];
#pragma unroll
  for (int v = 0; v < V; v++) wr[v] = valid ? w[(e * V + v) * nS + t] : 0.0;
  const unsigned mask = valid ? owned_faces<D, N>(a.nbr + e * nF, 0) : 0u;
  const unsigned owned = face_list<D>(mask);
  const int cnt = __popc(mask) * S::nFF;
  // quads with Roe: the metric is loaded after the face adjoint, which with it held takes 178
  // registers instead of 168 and so two waves per SIMD instead of three
  constexpr bool kLate = FC == 1 && D == 2;
  double ij[D][D], detJ;
  if (!kLate && valid) load_metric<D>(a, e, t, nS, ij, detJ, false);
  double cp[V];
  if (t < cnt) owned_partner_trace<D, N>(U, a, e, list_fpt<D, N>(owned, t), cp);
  stage_U_store<D, N>(U, a, lops, lU, e0, neb, L::U, sr);
  const double *u = lU + el * L::U;
  double *to = lT + el * L::R, *we = lw + el * L::GB;
  if (valid) {
#pragma unroll
    for (int v = 0; v < V; v++) we[v * nS + t] = wr[v];
    for (int k = t; k < V * nF; k += nS) to[k] = 0.0;
  }
  __syncthreads();
  const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
  double Ub[V];
  if (valid) {
#pragma unroll 1
    for (int k = t; k < cnt; k += nS) {
      const int f = list_fpt<D, N>(owned, k);
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
      const double *fg = a.fgeo + e * (D + 1) * nF + f;
      double n[D], Uo[V], Up[V], Uob[V], Upb[V], Gb[V];
#pragma unroll
      for (int d = 0; d < D; d++) n[d] = fg[d * nF];
      if (k == t) {
#pragma unroll
        for (int v = 0; v < V; v++) Up[v] = cp[v];
      } else {
        owned_partner_trace<D, N>(U, a, e, f, Up);
      }
#pragma unroll
      for (int v = 0; v < V; v++) Uo[v] = line_extrap<N>(lE, u + v * nS, base, str);
      owned_flux_vjp<D, N, false, 0, FC>(a, Wtr, e, f, n, Uo, Up, Uob, Upb, Gb);
#pragma unroll
      for (int v = 0; v < V; v++) {
        Xtr[(e * V + v) * nF + f] = Upb[v];
        to[v * nF + f] = Uob[v];
      }
    }
    // volume adjoint: Dss^T w along the lines, the flux reversed
    if (kLate) {
      asm volatile("" ::: "memory");
      load_metric<D>(a, e, t, nS, ij, detJ, false);
    }
    double Us[V];
#pragma unroll
    for (int v = 0; v < V; v++) {
      Us[v] = u[v * nS + t];
      Ub[v] = 0.0;
    }
    const Prim<D> p = primitives<D>(Us, a.gamma);
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
      const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
      double tFb[V];
#pragma unroll
      for (int v = 0; v < V; v++) tFb[v] = line_T_Dss<N>(lops, id, we + v * nS, t - id * str, str);
      conv_proj_vjp<D>(Us, p, ij[d], tFb, a.gamma, Ub);
    }
  }
  __syncthreads();
  if (!valid) return;
#pragma unroll
  for (int d = 0; d < D; d++) {
    const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
    const double l0 = tab_lE<N>(lops, 0)[id], l1 = tab_lE<N>(lops, 1)[id];
    const int f0 = fpt_end<D, N>(ia, ib, ic, d, 0), f1 = fpt_end<D, N>(ia, ib, ic, d, 1);
#pragma unroll
    for (int v = 0; v < V; v++) Ub[v] += l0 * to[v * nF + f0] + l1 * to[v * nF + f1];
  }
#pragma unroll
  for (int v = 0; v < V; v++) vout[(e * V + v) * nS + t] = Ub[v];
}

template <int D, int N, bool VISC, int BM, int FC>
__device__ __forceinline__ void adj_main_block(const double *__restrict__ U, const double *__restrict__ w,
                                               double *__restrict__ Wtr, double *__restrict__ Xtr,
                                               double *__restrict__ vout, const KArgs &a, long bid) {
  if constexpr (VISC) adj_visc_block<D, N, BM, FC>(U, w, Wtr, Xtr, vout, a, bid);
  else adj_euler_block<D, N, FC>(U, w, Wtr, Xtr, vout, a, bid);
}

// Occupancy target of the main adjoint kernels: three waves per SIMD (168 VGPRs) where they
// fit it with at most a few spills, else two (256 VGPRs): held to three, 26^3 hexes p = 2
// Euler with Roe took 129 us instead of 80 (58 spills), 100^2 quads p = 2 with Rusanov + LDG
// 29 us instead of 25 (42 spills), while 20^2 x 27 hexes p = 3 Euler went from 80 to 76.
// Euler quads with Roe, two / three waves, VJP: 117x102 of p=4 34.7 / 31.2 us, 185x161 of p=2
// 34.9 / 32.7.
template <int D, int N, bool VISC, int FC>
struct AdjWaves {
  static constexpr int value = VISC ? (FC == 0 && D == 2 && (N == 4 || N == 5) ? 3 : 2) : (FC == 0 || D == 2 ? 3 : 2);
};

template <int D, int N, bool VISC, int BM, int FC>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) __attribute__((amdgpu_waves_per_eu(AdjWaves<D, N, VISC, FC>::value)))
void k_adj_main(const double *__restrict__ U, const double *__restrict__ w, double *__restrict__ Wtr,
                double *__restrict__ Xtr, double *__restrict__ vout, KArgs a) {
  adj_main_block<D, N, VISC, BM, FC>(U, w, Wtr, Xtr, vout, a, xcd_block(blockIdx.x, gridDim.x));
}

// The same kernel for workgroups of one wave (the default tile where a wave is well filled, see
// default_tile): its barriers need no cross-wave synchronisation.
template <int D, int N, bool VISC, int BM, int FC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(AdjWaves<D, N, VISC, FC>::value)))
void k_adj_main_w64(const double *__restrict__ U, const double *__restrict__ w, double *__restrict__ Wtr,
                    double *__restrict__ Xtr, double *__restrict__ vout, KArgs a) {
  adj_main_block<D, N, VISC, BM, FC>(U, w, Wtr, Xtr, vout, a, xcd_block(blockIdx.x, gridDim.x));
}

// v += E^T (the owner's cotangent of this element's trace) at the points the partner owns.
template <int D, int N, int BM>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) void k_adj_gather(const double *__restrict__ Xtr, double *__restrict__ vout,
                                                            KArgs a) {
  using S = Shape<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V;
  constexpr int owner = (BM == 2) ? 1 : 0;
  extern __shared__ double lds[];
  const int EB = a.EB;
  double *lops = lds;
  double *lT = lops + S::NOPS_PAD;
  const int tid = threadIdx.x, NT = blockDim.x;
  for (int i = tid; i < S::NOPS; i += NT) lops[i] = a.ops[i];
  const long e0 = xcd_block(blockIdx.x, gridDim.x) * EB;
  const long neb = min((long)EB, (long)a.E - e0);
  const int el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  double *T = lT + el * S::ele(V * nF);
  if (valid) {
#pragma unroll
    for (int k = 0; k < S::FPT; k++) {
      const int f = t + k * nS;
      if (f >= nF) continue;
      long ep; int sl, fp;
      unpack_nbr<D, N>(a.nbr[e * nF + f], ep, sl, fp);
#pragma unroll
      for (int v = 0; v < V; v++)
        T[v * nF + f] = (BM != kAdjAllPoints && sl == owner) ? 0.0 : Xtr[(ep * V + v) * nF + fp];
    }
  }
  __syncthreads();
  if (!valid) return;
  const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
  double acc[V];
#pragma unroll
  for (int v = 0; v < V; v++) acc[v] = vout[(e * V + v) * nS + t];
#pragma unroll
  for (int d = 0; d < D; d++) {
    const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
    const double l0 = tab_lE<N>(lops, 0)[id], l1 = tab_lE<N>(lops, 1)[id];
    const int f0 = fpt_end<D, N>(ia, ib, ic, d, 0), f1 = fpt_end<D, N>(ia, ib, ic, d, 1);
#pragma unroll
    for (int v = 0; v < V; v++) acc[v] += l0 * T[v * nF + f0] + l1 * T[v * nF + f1];
  }
#pragma unroll
  for (int v = 0; v < V; v++) vout[(e * V + v) * nS + t] = acc[v];
}

// ---------------------------------------------------------------- general LDG beta
// With beta not +-1/2 both sides' gradients enter every common flux (src/faces.cpp:
// 1476-1614) and the common solution mixes both traces, Ucomm = (1/2 - beta) UL +
// (1/2 + beta) UR (src/faces.cpp:1366-1474).  The reverse runs after the forward trace
// and gradient-trace launches (Utr, Gtr at every flux point) and k_adj_prep:
//   k_adj_face     : per flux-point pair, by its slot-0 side: the common flux reversed for
//                    both sides' states and gradient traces; the cotangents overwrite the
//                    traces in place (Utr -> d/dUtr, Gtr -> d/dGtr);
//   k_adj_main_gen : per element: volume adjoint, the gradient-trace cotangents collected
//                    along the normal lines, the gradient reversed into U and into the
//                    common solution, whose cotangent splits (1/2 -+ beta) between this
//                    element's trace (with the face part, E^T into v) and the partner's
//                    (Xtr, at every point);
//   k_adj_gather   : v += E^T Xtr(partner) at every point (BM = kAdjAllPoints).

template <int D, int N, int FC>
__global__ __launch_bounds__(kMaxThreads) void k_adj_face(const double *__restrict__ Wtr, KArgs a) {
  using S = Shape<D, N>;
  constexpr int nF = S::nF, V = S::V;
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)a.E * nF) return;
  const long e = i / nF;
  const int f = (int)(i - e * nF);
  long ep; int sl, fp;
  unpack_nbr<D, N>(a.nbr[e * nF + f], ep, sl, fp);
  if (sl != 0) return;  // each pair is reversed once, by its slot-0 (left) side
  const double *fg = a.fgeo + e * (D + 1) * nF + f;
  double n[D];
#pragma unroll
  for (int d = 0; d < D; d++) n[d] = fg[d * nF];
  double UL[V], UR[V], Fb[V], ULb[V], URb[V], G1b[V], G2b[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    UL[v] = a.Utr[(e * V + v) * nF + f];
    UR[v] = a.Utr[(ep * V + v) * nF + fp];
    // both sides' copies of the flux are the same function of (UL, UR, GL, GR)
    Fb[v] = Wtr[(e * V + v) * nF + f] + Wtr[(ep * V + v) * nF + fp];
    ULb[v] = URb[v] = G1b[v] = G2b[v] = 0.0;
  }
  common_flux_vjp<D, true, 0, FC>(UL, UR, n, 1.0, a, Fb, ULb, URb, G1b, G2b);
  // each side's viscous normal flux G = -T(U, grad) . n, reversed (gradient from Gtr)
  double GLb[V][D], GRb[V][D];
  {
    const Prim<D> pL = primitives<D>(UL, a.gamma);
    viscous_vjp<D>(
        UL, pL,
        [&](int j, double *dUj) {
#pragma unroll
          for (int v = 0; v < V; v++) dUj[v] = a.Gtr[((e * D + j) * V + v) * nF + f];
        },
        [&](int v, int j) { return -G1b[v] * n[j]; },
        [&](int j, const double *gbj) {
#pragma unroll
          for (int v = 0; v < V; v++) GLb[v][j] = gbj[v];
        },
        a, ULb);
  }
  {
    const Prim<D> pR = primitives<D>(UR, a.gamma);
    viscous_vjp<D>(
        UR, pR,
        [&](int j, double *dUj) {
#pragma unroll
          for (int v = 0; v < V; v++) dUj[v] = a.Gtr[((ep * D + j) * V + v) * nF + fp];
        },
        [&](int v, int j) { return -G2b[v] * n[j]; },
        [&](int j, const double *gbj) {
#pragma unroll
          for (int v = 0; v < V; v++) GRb[v][j] = gbj[v];
        },
        a, URb);
  }
  // in place: this pair's two entries are read and written by this thread only
#pragma unroll
  for (int v = 0; v < V; v++) {
    a.Utr[(e * V + v) * nF + f] = ULb[v];
    a.Utr[(ep * V + v) * nF + fp] = URb[v];
  }
#pragma unroll
  for (int j = 0; j < D; j++)
#pragma unroll
    for (int v = 0; v < V; v++) {
      a.Gtr[((e * D + j) * V + v) * nF + f] = GLb[v][j];
      a.Gtr[((ep * D + j) * V + v) * nF + fp] = GRb[v][j];
    }
}

// LDS per element: U [V][nS]; R, which holds the common solution [V][nF], then one
// direction's gradient-trace cotangents [D][V][2 nFF] at a time, then the trace cotangent
// [V][nF]; GB, which holds w [V][nS], then the gradient cotangent [D][V][nS].
template <int D, int N>
struct AdjGenLds {
  using S = Shape<D, N>;
  static constexpr int U = S::ele(S::V * S::nS);
  static constexpr int R = S::ele((2 * D * S::V * S::nFF > S::V * S::nF) ? 2 * D * S::V * S::nFF : S::V * S::nF);
  static constexpr int GB = S::ele(D * S::V * S::nS);
  static constexpr int per_ele = U + R + GB;  // doubles
};

template <int D, int N>
__device__ __forceinline__ void adj_main_general_block(const double *__restrict__ U, const double *__restrict__ w,
                                                       double *__restrict__ Xtr, double *__restrict__ vout,
                                                       const KArgs &a, long bid) {
  using S = Shape<D, N>;
  using L = AdjGenLds<D, N>;
  constexpr int nS = S::nS, nF = S::nF, V = S::V, nFF = S::nFF;
  extern __shared__ double lds[];
  const int EB = a.EB;
  double *lops = lds;
  double *lU = lops + S::NOPS_PAD;
  double *lR = lU + EB * L::U;
  double *lGB = lR + EB * L::R;
  const long e0 = bid * EB;
  const long neb = min((long)EB, (long)a.E - e0);
  const int tid = threadIdx.x, el = tid / nS, t = tid - el * nS;
  const long e = e0 + el;
  const bool valid = el < neb;
  const double *u = lU + el * L::U;
  double *c = lR + el * L::R, *T = c, *to = c;
  double *gb = lGB + el * L::GB;
  StageRegs<D, N> sr;
  stage_U_load<D, N>(U, a, e0, neb, sr);
  if (valid) {
#pragma unroll
    for (int v = 0; v < V; v++) gb[v * nS + t] = w[(e * V + v) * nS + t];
  }
  stage_U_store<D, N>(U, a, lops, lU, e0, neb, L::U, sr);
  __syncthreads();
  const int ia = t % N, ib = (t / N) % N, ic = (D == 3) ? t / (N * N) : 0;
  const double beta = a.ldg_b;
  // 1. common solution, the partner's trace extrapolated from its U (Utr now holds cotangents)
  if (valid) {
#pragma unroll
    for (int k = 0; k < S::FPT; k++) {
      const int f = t + k * nS;
      if (f >= nF) continue;
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const double *lE = tab_lE<N>(lops, side);
      long ep; int sl, fp;
      unpack_nbr<D, N>(a.nbr[e * nF + f], ep, sl, fp);
      double pt[V];
      partner_trace<D, N>(U, a.ops, ep, fp, pt);
#pragma unroll
      for (int v = 0; v < V; v++) {
        const double own = line_extrap<N>(lE, u + v * nS, base, str);
        const double l = sl ? pt[v] : own, r = sl ? own : pt[v];
        c[v * nF + f] = 0.5 * (l + r) - beta * (l - r);
      }
    }
  }
  __syncthreads();
  // 2. forward physical gradient at this thread's spt; tFb[d1] = Dss^T w along the d1 lines
  double Ub[V];
  {
    double ij[D][D], detJ, g[V][D], tFb[D][V];
    if (valid) {
      load_metric<D>(a, e, t, nS, ij, detJ, true);
      spt_gradient<D, N>(lops, u, c, t, ij, detJ, g);
#pragma unroll
      for (int d = 0; d < D; d++) {
        const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
        const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
#pragma unroll
        for (int v = 0; v < V; v++) tFb[d][v] = line_T_Dss<N>(lops, id, gb + v * nS, t - id * str, str);
      }
    }
    __syncthreads();  // the common solution and w are consumed
    // 3. volume adjoint: F(U, grad) reversed for the cotangent tFb
    if (valid) {
      double Us[V];
#pragma unroll
      for (int v = 0; v < V; v++) {
        Us[v] = u[v * nS + t];
        Ub[v] = 0.0;
      }
      const Prim<D> p = primitives<D>(Us, a.gamma);
#pragma unroll
      for (int d = 0; d < D; d++) conv_proj_vjp<D>(Us, p, ij[d], tFb[d], a.gamma, Ub);
      viscous_vjp<D>(
          Us, p,
          [&](int j, double *dUj) {
#pragma unroll
            for (int v = 0; v < V; v++) dUj[v] = g[v][j];
          },
          [&](int v, int j) {
            double s = 0.0;
#pragma unroll
            for (int d1 = 0; d1 < D; d1++) s += tFb[d1][v] * ij[d1][j];
            return -s;
          },
          [&](int j, const double *gbj) {
#pragma unroll
            for (int v = 0; v < V; v++) gb[(j * V + v) * nS + t] = gbj[v];
          },
          a, Ub);
    }
  }
  // 4. the gradient-trace cotangents (k_adj_face, in Gtr) belong to the spts of their normal
  //    lines: one direction's faces at a time go through LDS and every spt collects the two
  //    ends of its line (by the face pair's order, so the sums are fixed)
  {
    double gv[V][D];
    if (valid) {
#pragma unroll
      for (int j = 0; j < D; j++)
#pragma unroll
        for (int v = 0; v < V; v++) gv[v][j] = gb[(j * V + v) * nS + t];
    }
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int fa = fpt_end<D, N>(0, 0, 0, d, 0) / nFF, fb = fpt_end<D, N>(0, 0, 0, d, 1) / nFF;  // the faces
      if (d > 0) __syncthreads();  // the previous direction's are consumed
      if (valid) {
        for (int i = t; i < 2 * nFF; i += nS) {
          const int f = (i < nFF) ? fa * nFF + i : fb * nFF + (i - nFF);
#pragma unroll
          for (int r = 0; r < D * V; r++) T[r * 2 * nFF + i] = a.Gtr[(e * D * V + r) * nF + f];
        }
      }
      __syncthreads();
      if (valid) {
        const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
        const double l0 = tab_lE<N>(lops, 0)[id], l1 = tab_lE<N>(lops, 1)[id];
        const int i0 = fpt_end<D, N>(ia, ib, ic, d, 0) - fa * nFF, i1 = fpt_end<D, N>(ia, ib, ic, d, 1) - fb * nFF + nFF;
#pragma unroll
        for (int j = 0; j < D; j++)
#pragma unroll
          for (int v = 0; v < V; v++) {
            const double *Tr = T + (j * V + v) * 2 * nFF;
            gv[v][j] += l0 * Tr[i0];
            gv[v][j] += l1 * Tr[i1];
          }
      }
    }
    // 5. reference-space gradient cotangent: grb[d2][v] = sum_d1 adj[d2][d1] gb[v][d1] / detJ
    if (valid) {
      double ij[D][D], detJ;
      load_metric<D>(a, e, t, nS, ij, detJ, true);
      const double inv_det = 1.0 / detJ;
#pragma unroll
      for (int d2 = 0; d2 < D; d2++)
#pragma unroll
        for (int v = 0; v < V; v++) {
          double s = 0.0;
#pragma unroll
          for (int d1 = 0; d1 < D; d1++) s += ij[d2][d1] * gv[v][d1];
          gb[(d2 * V + v) * nS + t] = s * inv_det;
        }
    }
  }
  __syncthreads();
  // 6. Dss^T into U; Dsf^T into the common solution's cotangent, split between this
  //    element's trace (added to its face cotangent from Utr) and the partner's (Xtr)
  if (valid) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
      const int str = (d == 0) ? 1 : ((d == 1) ? N : N * N);
      const int base = t - id * str;
#pragma unroll
      for (int v = 0; v < V; v++) Ub[v] += line_T_Dss<N>(lops, id, gb + (d * V + v) * nS, base, str);
    }
#pragma unroll
    for (int k = 0; k < S::FPT; k++) {
      const int f = t + k * nS;
      if (f >= nF) continue;
      int dim, side, base, str;
      fpt_info<D, N>(f, dim, side, base, str);
      const int sl = nbr_slot<D, N>(a.nbr[e * nF + f]);
      const double ao = sl ? (0.5 + beta) : (0.5 - beta), ap = sl ? (0.5 - beta) : (0.5 + beta);
#pragma unroll
      for (int v = 0; v < V; v++) {
        const double cb = line_Dsf<N>(lops, side, gb + (dim * V + v) * nS, base, str);
        to[v * nF + f] = a.Utr[(e * V + v) * nF + f] + ao * cb;
        Xtr[(e * V + v) * nF + f] = ap * cb;
      }
    }
  }
  __syncthreads();
  if (!valid) return;
  // 7. own trace cotangent E^T into v
#pragma unroll
  for (int d = 0; d < D; d++) {
    const int id = (d == 0) ? ia : ((d == 1) ? ib : ic);
    const double l0 = tab_lE<N>(lops, 0)[id], l1 = tab_lE<N>(lops, 1)[id];
    const int f0 = fpt_end<D, N>(ia, ib, ic, d, 0), f1 = fpt_end<D, N>(ia, ib, ic, d, 1);
#pragma unroll
    for (int v = 0; v < V; v++) Ub[v] += l0 * to[v * nF + f0] + l1 * to[v * nF + f1];
  }
#pragma unroll
  for (int v = 0; v < V; v++) vout[(e * V + v) * nS + t] = Ub[v];
}

template <int D, int N>
__global__ __launch_bounds__((Shape<D, N>::kThreads)) __attribute__((amdgpu_waves_per_eu(2)))
void k_adj_main_gen(const double *__restrict__ U, const double *__restrict__ w, double *__restrict__ Xtr,
                    double *__restrict__ vout, KArgs a) {
  adj_main_general_block<D, N>(U, w, Xtr, vout, a, xcd_block(blockIdx.x, gridDim.x));
}
