// dg_ader.hpp -- ADER Cauchy-Kowalevski time integral as one fused kernel.
//
// Restates integrate_taylor_cauchykovalewski with spectral_evaluation
// (source/wave_equation_operations.cc:961-1262): per cell
//   contrib = (t2-t1) u + 1/2[(t2-te)^2-(t1-te)^2] u'
//             + sum_{j>=2} fac_j [(t2-te)^{j+1}-(t1-te)^{j+1}] u^(j),
// where u^(j) are obtained by applying the local collocation operator
// repeatedly at the Gauss points; every second derivative the field is
// L2-projected (on the unit cell) to two polynomial degrees less
// (source/wave_equation_operations.cc:287-313, 1238-1255), and the
// lower-degree contributions are interpolated back at the end.
//
// GPU layout, node form: one lane per top-level Gauss node; the working field is
// double buffered in LDS; the level-0 contribution stays in registers, lower
// levels' contributions live in LDS.  On box cells each derivative runs in line
// form (one lane per line of the level, then one per node) where that was
// measured faster.  Line form, large launches of box cells: one lane per line
// throughout, the velocities in registers (ck_lines; CkLinesFrom draws the line).
#pragma once
#include <type_traits>
#include <utility>

#include "dg_common.hpp"
#include "dg_operator_gen.hpp"
#include "gauss_cx.hpp"

namespace exw {

// Offsets of the CK tables (per level l: n_l = K+1-2l points).
struct CkTab {
  int n_levels;
  int off_D[8];  // D_l[q*n_l+i] = l_i'(x_q)
  int off_X[8];  // Gauss points of level l
  int off_P[8];  // P_l (level l-1 -> l), [i*n_{l-1}+q] = l^lo_i(x^hi_q) w^hi_q / w^lo_i
  int off_V[8];  // V_l (level l -> l-1), [q*n_l+i] = l^lo_i(x^hi_q)
  int size;
};

template <int K>
struct CkShape {
  static constexpr int N_STEPS = K >= 2 ? K - 1 : 1;  // steps 0 .. max(0, K-2)
  static constexpr int N_LEVELS = (N_STEPS - 1) / 2 + 1;
  static constexpr int n_of(int l) { return K + 1 - 2 * l; }
  // points per direction of level l (at least 1), nodes in DIM dimensions, and
  // the offset of level l >= 1 among the lower levels' contributions
  static constexpr int nl(int l) { return K + 1 - 2 * l > 1 ? K + 1 - 2 * l : 1; }
  static constexpr int nd(int dim, int l) { return dim == 2 ? nl(l) * nl(l) : nl(l) * nl(l) * nl(l); }
  static constexpr int low_off(int dim, int l) {
    int s = 0;
    for (int j = 1; j < l; ++j) s += nd(dim, j);
    return s;
  }
  static constexpr int TAB_SIZE = [] {
    int s = 0;
    for (int l = 0; l < N_LEVELS; ++l) {
      const int n = K + 1 - 2 * l;
      s += n * n + n;
      if (l > 0) s += 2 * n * (n + 2);
    }
    return s;
  }();
};

// Cells per workgroup of the CK kernel.  Its 18 barrier-separated passes per
// cell wait on every wave of the group, so fewer cells per group pay: in 3D
// one cell per group from 100 nodes on (k=4, 64^3: 1.041 against 1.117 ms
// with two), two below (k=3: 0.315 against 0.323 ms with four); 2D keeps the
// operator's grouping.
template <int DIM, int K>
struct CkGroup {
  static constexpr int ND = Shape<DIM, K>::ND;
  static constexpr int MAXC = DIM == 3 ? (ND >= 100 ? 1 : 2) : 16;
  static constexpr int CPB = Shape<DIM, K>::CPB < MAXC ? Shape<DIM, K>::CPB : MAXC;
  static constexpr int BLOCK = ((CPB * ND + 63) / 64) * 64;
  // 3D k=6 sits one register above 6 waves per SIMD (81 VGPRs): held to 6 it
  // spills 2 and runs 0.633 against 0.735 ms at 32^3 (FP64); elsewhere no hint
  static constexpr int MIN_WAVES = (DIM == 3 && K == 6) ? 6 : 1;
};

template <int DIM, int N>
__device__ __forceinline__ constexpr int ipow_c() {
  return DIM == 2 ? N * N : N * N * N;
}

namespace ck {

using exw::static_for;

// Physical derivative at node qq of a level field of NN points per direction
// (in[f][...] in LDS): outv_d = rho^-1 d_d p, outp = rho c^2 div v (the
// time derivative is minus this).  Cartesian: d_d = (1/h_d) d/dxi_d.
template <int DIM, int NN, int LD, bool CART, typename Number>
__device__ __forceinline__ void derive(const Number (*in)[LD], const Number *Dl, const Number *Xl,
                                       int qq, const Number *ih, Number rho_inv, Number rc2,
                                       const double *V, Number *outv, Number &outp) {
  const int qd[3] = {qq % NN, (qq / NN) % NN, DIM == 3 ? qq / (NN * NN) : 0};
  constexpr int st[3] = {1, NN, NN * NN};
  if constexpr (CART) {
    Number div = Number(0);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const int q0 = qq - qd[d] * st[d];
      const Number *Dr = Dl + qd[d] * NN;
      Number gp = Number(0), gv = Number(0);
#pragma unroll
      for (int m = 0; m < NN; ++m) {
        const Number dm = Dr[m];
        gp += dm * in[DIM][q0 + m * st[d]];
        gv += dm * in[d][q0 + m * st[d]];
      }
      outv[d] = rho_inv * gp * ih[d];
      div += gv * ih[d];
    }
    outp = rc2 * div;
  } else {
    Number gr[DIM + 1][DIM];
#pragma unroll
    for (int e = 0; e < DIM; ++e) {
      const int q0 = qq - qd[e] * st[e];
      Number dr[NN];
#pragma unroll
      for (int m = 0; m < NN; ++m) dr[m] = Dl[qd[e] * NN + m];
#pragma unroll
      for (int f = 0; f <= DIM; ++f) {
        Number g = Number(0);
#pragma unroll
        for (int m = 0; m < NN; ++m) g += dr[m] * in[f][q0 + m * st[e]];
        gr[f][e] = g;
      }
    }
    Number xi[DIM], J[DIM * DIM], Ji[DIM * DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) xi[d] = Xl[qd[d]];
    multilinear_jacobian<DIM>(V, xi, J, Ji);
    Number div = Number(0);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      Number pg = Number(0);
#pragma unroll
      for (int e = 0; e < DIM; ++e) {
        pg += gr[DIM][e] * Ji[e * DIM + d];
        div += gr[d][e] * Ji[e * DIM + d];
      }
      outv[d] = rho_inv * pg;
    }
    outp = rc2 * div;
  }
}

// The same Cartesian derivative in line form, for lane `line` < DIM * NN^(DIM-1)
// of a cell: along its line (direction d) the lane reads p and v_d of `in` into
// registers once and, at the line's nodes, writes rho^-1 (d/dxi_d p) into
// out[d] and d/dxi_d v_d over in[d] (only this lane reads those entries of
// in[d]); derive_nodes then applies 1/h and forms the divergence.  The 1D
// matrix is the compile-time one of NN Gauss points (CartTable, built by the
// same routines as the level's table), and every sum and product runs in
// derive's order: N reads per line instead of N per node and direction.
template <int DIM, int NN, int LD, typename Number>
__device__ __forceinline__ void derive_line(Number (*in)[LD], Number (*out)[LD], int line,
                                            Number rho_inv) {
  constexpr int NT = DIM == 2 ? NN : NN * NN;
  constexpr const CartConst<NN> &T = CartTable<NN>::value;
  const int d = line / NT, t = line - d * NT;
  int base, sd;
  if constexpr (DIM == 2) {
    base = d == 0 ? t * NN : t;
    sd = d == 0 ? 1 : NN;
  } else {
    const int t0 = t % NN, t1 = t / NN;
    base = d == 0 ? t0 * NN + t1 * NN * NN : (d == 1 ? t0 + t1 * NN * NN : t0 + t1 * NN);
    sd = d == 0 ? 1 : (d == 1 ? NN : NN * NN);
  }
  Number pl[NN], vl[NN];
#pragma unroll
  for (int m = 0; m < NN; ++m) {
    pl[m] = in[DIM][base + m * sd];
    vl[m] = in[d][base + m * sd];
  }
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    Number gp = Number(0), gv = Number(0);
#pragma unroll
    for (int m = 0; m < NN; ++m) {
      const Number dm = Number(T.D[i * NN + m]);
      gp += dm * pl[m];
      gv += dm * vl[m];
    }
    out[d][base + i * sd] = rho_inv * gp;
    in[d][base + i * sd] = gv;
  }
}

// The node half of the line form (after a barrier): outv_d = (rho^-1 d/dxi_d p)
// / h_d from out[d], and outp = rho c^2 sum_d (d/dxi_d v_d) / h_d from in[d].
template <int DIM, int LD, typename Number>
__device__ __forceinline__ void derive_nodes(const Number (*in)[LD], const Number (*out)[LD],
                                             int qq, const Number *ih, Number rc2, Number *outv,
                                             Number &outp) {
  Number div = Number(0);
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    outv[d] = out[d][qq] * ih[d];
    div += in[d][qq] * ih[d];
  }
  outp = rc2 * div;
}

// whether the lines of a level of NN points fit the cell's lanes
template <int DIM, int NN, int ND>
constexpr bool lines_fit() {
  return DIM * (DIM == 2 ? NN : NN * NN) <= ND;
}

// where the line form was measured faster (CK kernel alone): FP64 everywhere
// (3D k=4: 1.11 against 1.31 ms at 64^3, k=6: 0.66 against 0.93 ms at 32^3,
// 3D k=3 equal); FP32 only in 3D from k=4 (at 3D k=3 and 2D it lost 8-10 %)
template <int DIM, int K, typename Number>
constexpr bool derive_lines_pay() {
  return std::is_same_v<Number, double> || (DIM == 3 && K >= 4);
}

// One tensor pass along direction DIR of the matrix M (NO x NI, row-major) on
// every field: the input has sizes (A0, A1, A2) with A_DIR = NI, the output
// the same with NO in direction DIR.  Lane o computes output entry o.
template <int DIM, int DIR, int NI, int NO, int A0, int A1, int A2, int LD, typename Number,
          int LDI = LD>
__device__ __forceinline__ void pass(const Number *M, const Number (*in)[LDI], Number (*out)[LD],
                                     int o) {
  constexpr int O0 = DIR == 0 ? NO : A0, O1 = DIR == 1 ? NO : A1, O2 = DIR == 2 ? NO : A2;
  constexpr int TOTAL = O0 * O1 * (DIM == 3 ? O2 : 1);
  constexpr int SI[3] = {1, A0, A0 * A1};
  if (o >= TOTAL) return;
  int idx[3] = {o % O0, (o / O0) % O1, DIM == 3 ? o / (O0 * O1) : 0};
  const int r = idx[DIR];
  idx[DIR] = 0;
  const int b = idx[0] * SI[0] + idx[1] * SI[1] + (DIM == 3 ? idx[2] * SI[2] : 0);
  // the lane's matrix row once in registers (the output may alias nothing
  // the compiler can prove, so it would reload the row for every field)
  Number mr[NI];
#pragma unroll
  for (int c = 0; c < NI; ++c) mr[c] = M[r * NI + c];
#pragma unroll
  for (int f = 0; f <= DIM; ++f) {
    Number acc = Number(0);
#pragma unroll
    for (int c = 0; c < NI; ++c) acc += mr[c] * in[f][b + c * SI[DIR]];
    out[f][o] = acc;
  }
}

// The same pass, its output entry o returned in res (all fields) instead of
// stored: the last interpolation pass, whose entry o is lane o's own node.
template <int DIM, int DIR, int NI, int NO, int A0, int A1, int A2, int LDI, typename Number>
__device__ __forceinline__ bool pass_reg(const Number *M, const Number (*in)[LDI], int o,
                                         Number *res) {
  constexpr int O0 = DIR == 0 ? NO : A0, O1 = DIR == 1 ? NO : A1, O2 = DIR == 2 ? NO : A2;
  constexpr int TOTAL = O0 * O1 * (DIM == 3 ? O2 : 1);
  constexpr int SI[3] = {1, A0, A0 * A1};
  if (o >= TOTAL) return false;
  int idx[3] = {o % O0, (o / O0) % O1, DIM == 3 ? o / (O0 * O1) : 0};
  const int r = idx[DIR];
  idx[DIR] = 0;
  const int b = idx[0] * SI[0] + idx[1] * SI[1] + (DIM == 3 ? idx[2] * SI[2] : 0);
  Number mr[NI];
#pragma unroll
  for (int c = 0; c < NI; ++c) mr[c] = M[r * NI + c];
#pragma unroll
  for (int f = 0; f <= DIM; ++f) {
    Number acc = Number(0);
#pragma unroll
    for (int c = 0; c < NI; ++c) acc += mr[c] * in[f][b + c * SI[DIR]];
    res[f] = acc;
  }
  return true;
}

}  // namespace ck

// The cell's factors of the CK derivatives: 1/rho, rho c^2 and (Cartesian)
// 1/h_d; 1 for lanes without a cell.  Reciprocals by the hardware estimate
// and two Newton steps (recip), not IEEE divisions: every lane computes them.
template <int DIM, bool CART, typename Number>
__device__ __forceinline__ void ck_factors(const DevMesh &mesh, int cell, bool active,
                                           Number &rho_inv, Number &rc2, Number (&ih)[DIM]) {
  Number rho = Number(1), cc = Number(1);
#pragma unroll
  for (int d = 0; d < DIM; ++d) ih[d] = Number(1);
  if (active) {
    rho = Number(mesh.rho[cell]);
    cc = Number(mesh.speed[cell]);
    if constexpr (CART) {
#pragma unroll
      for (int d = 0; d < DIM; ++d) ih[d] = recip(Number(mesh.h[(size_t)cell * DIM + d]));
    }
  }
  rho_inv = recip(rho);
  rc2 = rho * cc * cc;
}

// The Cauchy-Kowalevski work of the group's cells once the lane's node value
// u of its cell is known (in registers): the Taylor levels in LDS, the time
// integral over [t1, t2] about te written to tempsrc.  Shared by
// ader_ck_kernel and the fused ADER sweep, so both give the same bits.
template <int DIM, int K, typename Number, bool CART>
__device__ __forceinline__ void ck_cell(
    const DevMesh &mesh, const double *__restrict__ recon, const Number *s_ck, const CkTab &ckt,
    double t2, double t1, double te, Number (*s_a)[Shape<DIM, K>::NF][Shape<DIM, K>::ND],
    Number (*s_b)[Shape<DIM, K>::NF][Shape<DIM, K>::ND],
    Number (*s_c)[Shape<DIM, K>::NF]
                 [CkShape<K>::low_off(DIM, CkShape<K>::N_LEVELS) > 0
                      ? CkShape<K>::low_off(DIM, CkShape<K>::N_LEVELS)
                      : 1],
    const double *Vc, int lc, int lcc, int q, bool lane_ok, bool active, size_t cbase,
    Number rho_inv, Number rc2, const Number (&ih)[DIM], const Number (&u)[Shape<DIM, K>::NF],
    double *__restrict__ tempsrc) {
  using S = Shape<DIM, K>;
  using CS = CkShape<K>;
  constexpr int N = S::N, ND = S::ND, NF = S::NF;
  constexpr int NL = CS::N_LEVELS, NSTEPS = CS::N_STEPS;
  constexpr int LOW = CS::low_off(DIM, NL) > 0 ? CS::low_off(DIM, NL) : 1;
  if (lane_ok) {
#pragma unroll
    for (int f = 0; f < NF; ++f) s_a[lc][f][q] = u[f];
  }
  __syncthreads();

  // contrib (level 0) and the first derivative
  const double a2 = t2 - te, a1 = t1 - te;
  const Number c1 = Number(0.5 * (a2 * a2 - a1 * a1));
  Number contrib[NF], up[NF];
  if (recon) {
#pragma unroll
    for (int f = 0; f < NF; ++f) up[f] = active ? Number(recon[cbase + f * ND + q]) : Number(0);
  } else {
    Number ov[DIM], op;
    if constexpr (CART && ck::lines_fit<DIM, N, ND>() && ck::derive_lines_pay<DIM, K, Number>()) {
      if (lane_ok && q < DIM * (DIM == 2 ? N : N * N))
        ck::derive_line<DIM, N, ND>(s_a[lc], s_b[lc], q, rho_inv);
      __syncthreads();
      ck::derive_nodes<DIM, ND>(s_a[lcc], s_b[lcc], q, ih, rc2, ov, op);
    } else {
      ck::derive<DIM, N, ND, CART>(s_a[lcc], s_ck + ckt.off_D[0], s_ck + ckt.off_X[0], q, ih,
                                   rho_inv, rc2, Vc, ov, op);
    }
#pragma unroll
    for (int d = 0; d < DIM; ++d) up[d] = -ov[d];
    up[DIM] = -op;
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) contrib[f] = Number(a2 - a1) * u[f] + c1 * up[f];
  // the node form of the derivative reads other nodes' entries of s_a: wait
  // for every lane before overwriting; the line form's node half (and the
  // reconstruction input) read only the lane's own entries
  if constexpr (!(CART && ck::lines_fit<DIM, N, ND>() && ck::derive_lines_pay<DIM, K, Number>()))
    __syncthreads();
  if (lane_ok) {
#pragma unroll
    for (int f = 0; f < NF; ++f) s_a[lc][f][q] = -up[f];
  }
  __syncthreads();

  // the derivative steps; cur/nxt alternate between s_a and s_b at every step
  // and every projection pass
  double fac = -0.5, p2 = a2 * a2, p1 = a1 * a1;
  int parity = 0;  // 0: current field in s_a
  ck::static_for<NSTEPS>([&](auto S_) {
    constexpr int STEP = decltype(S_)::value;
    constexpr int LEVEL = STEP / 2;
    constexpr int n = CS::nl(LEVEL), nd = CS::nd(DIM, LEVEL);
    fac /= -double(STEP + 3);
    p2 *= a2;
    p1 *= a1;
    const Number fac_t = Number(fac * (p2 - p1));
    Number(*cur)[ND] = parity ? s_b[lcc] : s_a[lcc];
    Number(*nxt)[ND] = parity ? s_a[lcc] : s_b[lcc];
    constexpr bool LINES = CART && ck::lines_fit<DIM, n, ND>() && ck::derive_lines_pay<DIM, K, Number>();
    if constexpr (LINES) {
      if (lane_ok && q < DIM * (DIM == 2 ? n : n * n))
        ck::derive_line<DIM, n, ND>(cur, nxt, q, rho_inv);
      __syncthreads();
    }
    if (q < nd) {
      Number ov[DIM], op;
      if constexpr (LINES)
        ck::derive_nodes<DIM, ND>(cur, nxt, q, ih, rc2, ov, op);
      else
        ck::derive<DIM, n, ND, CART>(cur, s_ck + ckt.off_D[LEVEL], s_ck + ckt.off_X[LEVEL], q,
                                     ih, rho_inv, rc2, Vc, ov, op);
      if (lane_ok) {
        // (the line phase left rho^-1 d/dxi_d p there: this lane's own entries)
#pragma unroll
        for (int d = 0; d < DIM; ++d) nxt[d][q] = ov[d];
        nxt[DIM][q] = op;
      }
      if constexpr (LEVEL == 0) {
#pragma unroll
        for (int d = 0; d < DIM; ++d) contrib[d] += fac_t * ov[d];
        contrib[DIM] += fac_t * op;
      } else if (lane_ok) {
        constexpr bool FIRST = (STEP & 1) == 0;  // the first step of a level sets
        constexpr int OFF = CS::low_off(DIM, LEVEL);
#pragma unroll
        for (int d = 0; d < DIM; ++d)
          s_c[lc][d][OFF + q] = (FIRST ? Number(0) : s_c[lc][d][OFF + q]) + fac_t * ov[d];
        s_c[lc][DIM][OFF + q] = (FIRST ? Number(0) : s_c[lc][DIM][OFF + q]) + fac_t * op;
      }
    }
    __syncthreads();
    parity ^= 1;
    // project to the next level after an odd step that is not the last one
    if constexpr ((STEP & 1) == 1 && STEP < K - 2) {
      constexpr int NLO = n - 2;
      const Number *P = s_ck + ckt.off_P[LEVEL + 1];
      ck::static_for<DIM>([&](auto D_) {
        constexpr int DIR = decltype(D_)::value;
        // sizes before this pass: directions < DIR already reduced
        constexpr int A0 = DIR > 0 ? NLO : n, A1 = DIR > 1 ? NLO : n, A2 = n;
        Number(*in)[ND] = parity ? s_b[lcc] : s_a[lcc];
        Number(*out)[ND] = parity ? s_a[lcc] : s_b[lcc];
        if (lane_ok) ck::pass<DIM, DIR, n, NLO, A0, A1, A2, ND>(P, in, out, q);
        __syncthreads();
        parity ^= 1;
      });
    }
  });

  // interpolate the lower levels' contributions back up and add: the first
  // pass of a level reads its contribution where it lies in s_c, the last one
  // hands lane o its own output entry (level 0: the lane's node)
  if constexpr (NL > 1) {
    ck::static_for<NL - 1>([&](auto L_) {
      constexpr int LV = NL - 1 - decltype(L_)::value;  // NL-1 .. 1
      constexpr int NLO = CS::nl(LV), NHI = NLO + 2;
      constexpr int OFF = CS::low_off(DIM, LV);
      const Number *Vt = s_ck + ckt.off_V[LV];
      const Number(*lvl)[LOW] = reinterpret_cast<const Number(*)[LOW]>(&s_c[lcc][0][OFF]);
      bool in_b = true;  // the latest pass output is in s_b (else s_a)
      ck::static_for<DIM>([&](auto D_) {
        constexpr int DIR = decltype(D_)::value;
        constexpr int A0 = DIR > 0 ? NHI : NLO, A1 = DIR > 1 ? NHI : NLO, A2 = NLO;
        if constexpr (DIR < DIM - 1) {
          if constexpr (DIR == 0) {
            if (lane_ok) ck::pass<DIM, DIR, NLO, NHI, A0, A1, A2, ND, Number, LOW>(Vt, lvl, s_b[lcc], q);
            in_b = true;
          } else {
            if (lane_ok)
              ck::pass<DIM, DIR, NLO, NHI, A0, A1, A2, ND>(Vt, in_b ? s_b[lcc] : s_a[lcc],
                                                         in_b ? s_a[lcc] : s_b[lcc], q);
            in_b = !in_b;
          }
          __syncthreads();
        } else {
          Number res[NF];
          bool have = false;
          if (lane_ok)
            have = ck::pass_reg<DIM, DIR, NLO, NHI, A0, A1, A2, ND>(
                Vt, in_b ? s_b[lcc] : s_a[lcc], q, res);
          if (have) {
            if constexpr (LV - 1 == 0) {
#pragma unroll
              for (int f = 0; f < NF; ++f) contrib[f] += res[f];
            } else {
#pragma unroll
              for (int f = 0; f < NF; ++f) s_c[lc][f][CS::low_off(DIM, LV - 1) + q] += res[f];
            }
          }
          // the next level's first pass reads s_c; the last level needs no wait
          if constexpr (LV - 1 > 0) __syncthreads();
        }
      });
    });
  }

  if (active) {
#pragma unroll
    for (int f = 0; f < NF; ++f) tempsrc[cbase + f * ND + q] = double(contrib[f]);
  }
}

template <int DIM, int K, typename Number, bool CART>
__global__ void __launch_bounds__((CkGroup<DIM, K>::BLOCK))
    __attribute__((amdgpu_waves_per_eu(CkGroup<DIM, K>::MIN_WAVES)))
    ader_ck_kernel(const DevMesh mesh, const double *__restrict__ src,
                   const double *__restrict__ recon, const double *__restrict__ cktab,
                   const CkTab ckt, double t2, double t1, double te_all, const CellSel sel,
                   double *__restrict__ tempsrc) {
  using S = Shape<DIM, K>;
  using CS = CkShape<K>;
  constexpr int N = S::N, ND = S::ND, NF = S::NF, CPB = CkGroup<DIM, K>::CPB;
  constexpr int NL = CS::N_LEVELS, NSTEPS = CS::N_STEPS;
  // the lower levels' contributions, one after the other in s_c
  constexpr int LOW = CS::low_off(DIM, NL) > 0 ? CS::low_off(DIM, NL) : 1;

  __shared__ Number s_a[CPB][NF][ND];
  __shared__ Number s_b[CPB][NF][ND];
  __shared__ Number s_c[CPB][NF][LOW];
  __shared__ double s_V[CART ? 1 : CPB][CART ? 1 : (1 << DIM) * DIM];
  __shared__ Number s_ck[CS::TAB_SIZE];

  const int tid = threadIdx.x;
  for (int i = tid; i < CS::TAB_SIZE && i < ckt.size; i += blockDim.x) s_ck[i] = Number(cktab[i]);
  const int lc = tid / ND;
  const int q = tid - lc * ND;
  const bool lane_ok = lc < CPB;
  const int lcc = lane_ok ? lc : 0;  // LDS slot used by spare lanes (they store nothing)
  // entry -> cell (identity, or through the selection list)
  auto cell_of = [&](int e) { return sel.list ? (e < sel.n ? sel.list[e] : -1) : e; };
  const int cell = cell_of(blockIdx.x * CPB + lc);
  const bool active = lane_ok && cell >= 0 && cell < mesh.n_cells;
  const double te = active && sel.cluster ? sel.te[sel.cluster[cell]] : te_all;

  if constexpr (!CART) {
    constexpr int NVD = (1 << DIM) * DIM;
    for (int i = tid; i < CPB * NVD; i += blockDim.x) {
      const int c2 = cell_of(blockIdx.x * CPB + i / NVD);
      s_V[i / NVD][i % NVD] =
          c2 >= 0 && c2 < mesh.n_cells ? mesh.vertices[(size_t)c2 * NVD + i % NVD] : 0.0;
    }
  }
  Number rho_inv, rc2, ih[DIM];
  ck_factors<DIM, CART>(mesh, cell, active, rho_inv, rc2, ih);
  const double *Vc = CART ? nullptr : s_V[CART ? 0 : lcc];

  const size_t cbase = (size_t)cell * NF * ND;
  Number u[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) u[f] = Number(0);
  if (active) {
#pragma unroll
    for (int f = 0; f < NF; ++f) u[f] = Number(src[cbase + f * ND + q]);
  }
  ck_cell<DIM, K, Number, CART>(mesh, recon, s_ck, ckt, t2, t1, te, s_a, s_b, s_c, Vc, lc, lcc,
                                q, lane_ok, active, cbase, rho_inv, rc2, ih, u, tempsrc);
}

// ---------------------------------------------------------------------------
// From how many groups of the node form (CkGroup) on a launch over box cells runs
// the line form; 1 << 30: never.  The line form's matrices are constants of its
// unrolled code, 10 to 100 KB of it that every launch fetches once: a launch that
// leaves most of the chip idle waits for the instructions (2D k=7, 100 cells, FP32:
// 13.0 us against 6.6, k=12 38.7 against 14.2), and at 2D k=12 the code does not
// stay in the instruction cache at all (FP32 47524 cells: 802 us against 515).  The
// node form reads its matrices from LDS in short loops.  us, node form / line form:
//   FP64 2D k=4   256 cells 5.9 / 6.1,  3969 6.9 / 6.6;  k=6 841 9.5 / 9.9,
//        2025 11.6 / 10.1, 54289 135 / 58
//        2D k=8  1225 16.4 / 17.4,  2304 20.6 / 19.7;  k=10 1521 28.4 / 31.1,
//        2704 47 / 32;  k=11 676 22.5 / 34.3, 1296 39.7 / 35
//        3D k=4   216 6.4 / 6.8, 1000 8.2 / 7.9;  k=6 216 11.4 / 11.8, 343
//        14.2 / 13.2;  k=7 216 14.4 / 15.5, 512 19.8 / 17.9
//   FP32 2D k=4  3969 6.0 / 6.7,  13225 9.6 / 7.9;  k=6 3721 9.7 / 11.5, 6724
//        15 / 11.9;  k=7 2916 9.8 / 13.7, 5184 16.3 / 14.3;  k=9 6724 38.7 / 39.8,
//        26569 132 / 106;  k=10 5476 45.6 / 50.3, 66049 446 / 337;  k=11 2304
//        26.6 / 32.4, 4624 48.9 / 33.7
//        3D k=4  1000 7.2 / 7.8, 2197 10.5 / 10.0;  k=6 729 14.0 / 15.2, 1331
//        22.9 / 20.6;  k=7 512 15.5 / 17.1, 1000 26.8 / 20.1
// Never: 3D k=5 (lines fill 36 of a wave's 64 lanes: 4913 cells 38.9 / 41.8), k=8, 9
// (two waves per direction, registers: 592 / 632 at k=9, 5832 cells), 2D k=12, and
// FP32 2D k=3 (83521 cells 13.0 / 14.1).  FP32 3D k=3 loses to 30000 cells (15625 13.0 /
// 15.1) and gains with the fused kernel from 10^5 on (262144: 501 / 492 per step).
template <int DIM, int K, typename Number>
struct CkLinesFrom {
  static constexpr int NEVER = 1 << 30;
  static constexpr bool D = std::is_same_v<Number, double>;
  static constexpr int groups() {
    if constexpr (DIM == 2) {
      if (D) return K <= 3 || K == 5 ? 0 : K <= 7 ? 320 : K <= 10 ? 1024 : K == 11 ? 1280 : NEVER;
      return K <= 2 ? 0 : K == 3 ? NEVER : K <= 5 ? 1024 : K <= 8 ? 1280 : K <= 10 ? 8192
             : K == 11 ? 3584 : NEVER;
    } else {
      if (D) return K <= 2 ? 0 : K == 3 ? 128 : K == 4 ? 512 : K == 6 || K == 7 ? 384 : NEVER;
      return K <= 2 ? 0 : K == 3 ? 50000 : K == 4 ? 1792 : K == 6 ? 1280 : K == 7 ? 768 : NEVER;
    }
  }
  static constexpr bool ALWAYS = groups() == 0, EXISTS = groups() < NEVER;
  static bool pays(int n_cells) {
    return ALWAYS || (EXISTS && n_cells / CkGroup<DIM, K>::CPB >= groups());
  }
};

// The Cauchy-Kowalevski work of box cells in line form.  Lane (d, t) of a cell
// owns line t of direction d.  On a box v_d is only ever differentiated along d
// and only ever receives d/dxi_d p, so v_d and its Taylor contribution live in
// the registers of the direction-d lines from the first derivative to the last;
// LDS carries the lines' shares of div v, which every line through a node adds
// up for its own copy of p, and the passes between levels.  One barrier per
// derivative.
// (The form with one lane per node moved every field through LDS four times per
// derivative and kept the LDS pipe 88 % busy.)
// CK alone, ms before -> now (FP64; FP32): 3D k=3 64^3 0.311 -> 0.247 (0.182 -> 0.185),
// k=4 64^3 0.979 -> 0.778 (0.617 -> 0.541), k=6 32^3 0.636 -> 0.401 (0.384 -> 0.304),
// 2D k=5 512^2 0.324 -> 0.149 (0.176 -> 0.111): 1.8 to 5.8 TB/s of 16 B/DoF.  LDS
// accesses are halved (4.8e8 -> 2.2e8 cycles at 3D k=4); what bounds it now is the
// FP64 VALU (about two thirds busy) and its occupancy of 5-6 waves per SIMD.

// projection to two degrees less (P, with the mass weights) and interpolation
// back (V) between NLO + 2 and NLO Gauss points, at compile time
template <int NLO>
struct CkLevelConst {
  static constexpr int NHI = NLO + 2;
  double P[NLO * NHI], V[NHI * NLO];
  constexpr CkLevelConst() : P(), V() {
    double xl[NLO] = {}, wl[NLO] = {}, xh[NHI] = {}, wh[NHI] = {};
    cx::gauss01(NLO, xl, wl);
    cx::gauss01(NHI, xh, wh);
    for (int q = 0; q < NHI; ++q) {
      cx::lagrange(NLO, xl, xh[q], V + q * NLO, nullptr);
      for (int i = 0; i < NLO; ++i) P[i * NHI + q] = V[q * NLO + i] * wh[q] / wl[i];
    }
  }
};
template <int NLO>
struct CkLevelTable {
  static constexpr CkLevelConst<NLO> value{};
};

// a level's node grid in LDS: rows of odd length (no bank conflicts along x)
template <int DIM, int NN>
struct CkGrid {
  static constexpr int NX = NN | 1;
  static constexpr int SIZE = DIM == 2 ? NX * NN : NX * NN * NN;
  static constexpr int st(int d) { return d == 0 ? 1 : (d == 1 ? NX : NX * NN); }
  // first entry of line t of direction d
  static __device__ __forceinline__ int base(int d, int t) {
    if constexpr (DIM == 2) return d == 0 ? t * NX : t;
    const int t1 = small_div<NN>(t), t0 = t - t1 * NN;
    return d == 0 ? t0 * NX + t1 * NX * NN : (d == 1 ? t0 + t1 * NX * NN : t0 + t1 * NX);
  }
  static __device__ __forceinline__ int stride(int d) {
    return d == 0 ? 1 : (d == 1 ? NX : NX * NN);
  }
  static __device__ __forceinline__ int node(int q) { return NX == NN ? q : q + small_div<NN>(q); }
};

namespace ck {

// One tensor pass along direction (f's own + OFF) of field f of NF in a (grid
// strides of NG points per direction): the lines whose coordinate along f's own
// direction is < M0 and along the third one < M1 go from NI to NO entries in
// place, one task each over the cell's NL line lanes.  f's own direction is f,
// the pressure's (f = DIM) is 0.
template <int DIM, int NG, int OFF, int NI, int NO, int M0, int M1, int NL, typename Number>
__device__ __forceinline__ void line_tasks(const double *M, Number *a, int ld, int id) {
  using G = CkGrid<DIM, NG>;
  constexpr int MM = DIM == 2 ? M0 : M0 * M1, TASKS = (DIM + 1) * MM;
#pragma unroll
  for (int task0 = 0; task0 < TASKS; task0 += NL) {
    const int task = task0 + id;
    if (task >= TASKS) break;
    const int f = small_div<MM>(task), r = task - f * MM, j = small_div<M0>(r), i = r - j * M0;
    const int own = f == DIM ? 0 : f;
    int e = own + OFF, o = own + (OFF == 1 ? 2 : 1);
    if (e >= DIM) e -= DIM;
    if (o >= DIM) o -= DIM;
    Number *x = a + f * ld + i * G::stride(own) + (DIM == 2 ? 0 : j * G::stride(o));
    const int st = G::stride(e);
    Number in[NI];
#pragma unroll
    for (int m = 0; m < NI; ++m) in[m] = x[m * st];
#pragma unroll
    for (int q = 0; q < NO; ++q) {
      Number s = Number(M[q * NI]) * in[0];
#pragma unroll
      for (int m = 1; m < NI; ++m) s = fma_of(Number(M[q * NI + m]), in[m], s);
      x[q * st] = s;
    }
  }
}

}  // namespace ck

// a: [DIM+1][SIZE], the fields at the cell's nodes (CkGrid of K+1 points; a
// barrier behind it) on entry, the time integral over [t1, t2] about te there on
// return (a barrier behind it); b: [DIM][SIZE].  Every lane of the group
// calls it; the lanes with ok own line t < (K+1)^(DIM-1) of direction d of
// their cell.  put_recon (or none): stores the given first time derivative at
// the cell's nodes into a.  rih = 1/(rho h_d) and kih = rho c^2 / h_d, so that
// v_d' = -rih d/dxi_d p and p' is minus the sum of kih d/dxi_d v_d.  (Lines that
// carry rho h_d v_d would save the product by rih, 1 % of the step, but round the
// leading term twice more, on the way in and out.)
template <int DIM, int K, typename Number, typename PutRecon>
__device__ __forceinline__ void ck_lines(Number *a, Number *b, bool ok, int d, int t, Number rih,
                                         Number kih, double t2, double t1, double te,
                                         bool recon, PutRecon put_recon) {
  // (shared by kernels that must agree bit for bit: every FMA spelled out)
#pragma clang fp contract(off)
  using CS = CkShape<K>;
  constexpr int N = K + 1, NL = CS::N_LEVELS, NSTEPS = CS::N_STEPS;
  constexpr int LD = CkGrid<DIM, N>::SIZE;
  constexpr int LINES = DIM * (DIM == 2 ? N : N * N);
  const int id = d * (DIM == 2 ? N : N * N) + t;
  Number v[N], p[N], cv[NL][N], cp[NL][N];  // level l uses the first nl(l) entries
  auto get = [&](auto NN_, Number *vv, Number *pp) __attribute__((always_inline)) {
    constexpr int n = decltype(NN_)::value;
    const int o = CkGrid<DIM, n>::base(d, t), st = CkGrid<DIM, n>::stride(d);
#pragma unroll
    for (int i = 0; i < n; ++i) {
      vv[i] = a[d * LD + o + i * st];
      pp[i] = a[DIM * LD + o + i * st];
    }
  };
  // one derivative of (v, p): the lines' shares of div v through buf, one barrier
  auto derive = [&](auto NN_, Number *buf) __attribute__((always_inline)) {
#pragma clang fp contract(off)
    constexpr int n = decltype(NN_)::value;
    constexpr const CartConst<n> &T = CartTable<n>::value;
    using G = CkGrid<DIM, n>;
    const bool on = ok && t < (DIM == 2 ? n : n * n);
    const int o = G::base(d, t), st = G::stride(d);
    Number q[n];
    if (on) {
      Number w[n];
#pragma unroll
      for (int i = 0; i < n; ++i) {
        Number gv = Number(T.D[i * n]) * v[0], gp = Number(T.D[i * n]) * p[0];
#pragma unroll
        for (int m = 1; m < n; ++m) {
          gv = fma_of(Number(T.D[i * n + m]), v[m], gv);
          gp = fma_of(Number(T.D[i * n + m]), p[m], gp);
        }
        q[i] = gv * kih;
        w[i] = gp * rih;
        buf[d * LD + o + i * st] = q[i];
      }
#pragma unroll
      for (int i = 0; i < n; ++i) v[i] = w[i];
    }
    __syncthreads();
    if (on) {
      const Number *b1 = buf + (d == 0 ? 1 : 0) * LD + o, *b2 = buf + (d == 2 ? 1 : 2) * LD + o;
#pragma unroll
      for (int i = 0; i < n; ++i) {
        Number s = b1[i * st];
        if constexpr (DIM == 3) s += b2[i * st];
        p[i] = s + q[i];
      }
    }
  };
  using N0 = std::integral_constant<int, N>;
  const double a2 = t2 - te, a1 = t1 - te;
  const Number c0 = Number(a2 - a1), c1 = Number(0.5 * (a2 * a2 - a1 * a1));
  if (ok) {
    get(N0{}, v, p);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      cv[0][i] = v[i];
      cp[0][i] = p[i];
    }
  }
  // the first derivative: u' = -derive(u), or the given one; carried negated
  if (recon) {
    __syncthreads();
    put_recon();
    __syncthreads();
    if (ok) {
      get(N0{}, v, p);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        v[i] = -v[i];
        p[i] = -p[i];
      }
    }
  } else {
    derive(N0{}, b);
  }
  // (the leading term's product in the FMA: one rounding of its size)
  if (ok)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      cv[0][i] = fma_of(c0, cv[0][i], -c1 * v[i]);
      cp[0][i] = fma_of(c0, cp[0][i], -c1 * p[i]);
    }

  double fac = -0.5, p2 = a2 * a2, p1 = a1 * a1;
  // the buffer of the latest derivative: b or a (its readers may not have passed
  // the next barrier yet)
  static_for<NSTEPS>([&](auto S_) __attribute__((always_inline)) {
#pragma clang fp contract(off)
    constexpr int STEP = decltype(S_)::value, LEVEL = STEP / 2, n = CS::nl(LEVEL);
    using NN = std::integral_constant<int, n>;
    fac /= -double(STEP + 3);
    p2 *= a2;
    p1 *= a1;
    const Number ft = Number(fac * (p2 - p1));
    // level 0: b, then a, b; lower levels: b, a
    constexpr bool IN_A = LEVEL == 0 ? STEP % 2 == 0 : STEP % 2 == 1;
    derive(NN{}, IN_A ? a : b);
    constexpr bool FIRST = LEVEL > 0 && STEP % 2 == 0;  // a lower level's first step sets
    if (ok) {
#pragma unroll
      for (int i = 0; i < n; ++i) cv[LEVEL][i] = FIRST ? ft * v[i] : fma_of(ft, v[i], cv[LEVEL][i]);
    }
    // (uniform over the line waves; a lane without a line adds into sums that nobody
    // reads: testing ok here costs 25 registers)
    if (d == 0) {
#pragma unroll
      for (int i = 0; i < n; ++i) cp[LEVEL][i] = FIRST ? ft * p[i] : fma_of(ft, p[i], cp[LEVEL][i]);
    }
    if constexpr ((STEP & 1) == 1 && STEP < K - 2) {
      // project to the next level: along the line in registers, then the other
      // directions field by field in a
      constexpr int NLO = n - 2;
      constexpr const CkLevelConst<NLO> &L = CkLevelTable<NLO>::value;
      using G = CkGrid<DIM, n>;
      if constexpr (IN_A) __syncthreads();
      if (ok && t < (DIM == 2 ? n : n * n)) {
        const int o = G::base(d, t), st = G::stride(d);
#pragma unroll
        for (int i = 0; i < NLO; ++i) {
          Number x = Number(L.P[i * n]) * v[0];
#pragma unroll
          for (int m = 1; m < n; ++m) x = fma_of(Number(L.P[i * n + m]), v[m], x);
          a[d * LD + o + i * st] = x;
        }
        if (d == 0)
#pragma unroll
          for (int i = 0; i < NLO; ++i) {
            Number y = Number(L.P[i * n]) * p[0];
#pragma unroll
            for (int m = 1; m < n; ++m) y = fma_of(Number(L.P[i * n + m]), p[m], y);
            a[DIM * LD + o + i * st] = y;
          }
      }
      __syncthreads();
      if (ok) ck::line_tasks<DIM, n, 1, n, NLO, NLO, n, LINES>(L.P, a, LD, id);
      __syncthreads();
      if constexpr (DIM == 3) {
        if (ok) ck::line_tasks<DIM, n, 2, n, NLO, NLO, NLO, LINES>(L.P, a, LD, id);
        __syncthreads();
      }
      if (ok && t < (DIM == 2 ? NLO : NLO * NLO)) {
        const int u1 = small_div<NLO>(t), u0 = t - u1 * NLO, ea = d == 0 ? 1 : 0, eb = d == 2 ? 1 : 2;
        const int o = u0 * G::stride(ea) + (DIM == 2 ? 0 : u1 * G::stride(eb)), st = G::stride(d);
#pragma unroll
        for (int i = 0; i < NLO; ++i) {
          v[i] = a[d * LD + o + i * st];
          p[i] = a[DIM * LD + o + i * st];
        }
      }
    }
  });
  constexpr int LAST = NSTEPS - 1, LASTL = LAST / 2;
  constexpr bool LAST_IN_A = LASTL == 0 ? LAST % 2 == 0 : LAST % 2 == 1;

  // interpolate the lower levels' contributions back up: the other directions
  // field by field in a, along the line in registers
  static_for<NL - 1>([&](auto L_) __attribute__((always_inline)) {
    constexpr int LV = NL - 1 - decltype(L_)::value, NLO = CS::nl(LV), NHI = NLO + 2;
    constexpr const CkLevelConst<NLO> &L = CkLevelTable<NLO>::value;
    using G = CkGrid<DIM, NHI>;
    if constexpr (LV < NL - 1 || LAST_IN_A) __syncthreads();
    if (ok && t < (DIM == 2 ? NLO : NLO * NLO)) {
      const int u1 = small_div<NLO>(t), u0 = t - u1 * NLO, ea = d == 0 ? 1 : 0, eb = d == 2 ? 1 : 2;
      const int o = u0 * G::stride(ea) + (DIM == 2 ? 0 : u1 * G::stride(eb)), st = G::stride(d);
#pragma unroll
      for (int i = 0; i < NLO; ++i) {
        a[d * LD + o + i * st] = cv[LV][i];
        if (d == 0) a[DIM * LD + o + i * st] = cp[LV][i];
      }
    }
    __syncthreads();
    if (ok) ck::line_tasks<DIM, NHI, 1, NLO, NHI, NLO, NLO, LINES>(L.V, a, LD, id);
    __syncthreads();
    if constexpr (DIM == 3) {
      if (ok) ck::line_tasks<DIM, NHI, 2, NLO, NHI, NLO, NHI, LINES>(L.V, a, LD, id);
      __syncthreads();
    }
    if (ok && t < (DIM == 2 ? NHI : NHI * NHI)) {
      const int o = G::base(d, t), st = G::stride(d);
      auto add = [&](int f, Number *c) __attribute__((always_inline)) {
        Number x[NLO];
#pragma unroll
        for (int i = 0; i < NLO; ++i) x[i] = a[f * LD + o + i * st];
        // (summed by itself: one rounding of the larger terms' size)
#pragma unroll
        for (int i = 0; i < NHI; ++i) {
          Number y = Number(L.V[i * NLO]) * x[0];
#pragma unroll
          for (int m = 1; m < NLO; ++m) y = fma_of(Number(L.V[i * NLO + m]), x[m], y);
          c[i] += y;
        }
      };
      add(d, cv[LV - 1]);
      if (d == 0) add(DIM, cp[LV - 1]);
    }
  });
  // (without lower levels others may still read the last shares in a; else every
  // lane has only read the lines that it writes now)
  if constexpr (NL == 1 && LAST_IN_A) __syncthreads();
  if (ok) {
    const int o = CkGrid<DIM, N>::base(d, t), st = CkGrid<DIM, N>::stride(d);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      a[d * LD + o + i * st] = cv[0][i];
      if (d == 0) a[DIM * LD + o + i * st] = cp[0][i];
    }
  }
  __syncthreads();
}

// The layout of ader_ck_lines_kernel: GenShape's line waves (direction uniform
// per wave, as many cells as fill them), the fields copied flat 16 bytes at a time.
template <int DIM, int K>
struct CkLinesShape {
  using G = GenShape<DIM, K>;
  static constexpr int BLOCK = G::LINE_LANES, CPB = G::CPB;
  static constexpr int PPC = G::PPC, NPP = (CPB * PPC + BLOCK - 1) / BLOCK;
  static constexpr int LD = CkGrid<DIM, K + 1>::SIZE;
  // 3D k=4: 98 -> 94 registers, the sixth group of a CU (0.825 -> 0.778 ms).  Elsewhere
  // the next step of waves spills (3D k=5 4, k=6 61, 2D k=5 19 registers).
  static constexpr int MIN_WAVES = DIM == 3 && K == 4 ? 5 : 1;
};

// ader_ck_kernel for box cells (same arguments but the tables)
template <int DIM, int K, typename Number>
__global__ void __launch_bounds__((CkLinesShape<DIM, K>::BLOCK), (CkLinesShape<DIM, K>::MIN_WAVES))
    ader_ck_lines_kernel(const DevMesh mesh, const double *__restrict__ src,
                         const double *__restrict__ recon, double t2, double t1, double te_all,
                         const CellSel sel, double *__restrict__ tempsrc) {
  using S = GenShape<DIM, K>;
  using C = CkLinesShape<DIM, K>;
  constexpr int N = S::N, ND = S::ND, NT = S::NT, NF = S::NF, WPD = S::WPD, CPB = C::CPB;
  constexpr int BLOCK = C::BLOCK, PPC = C::PPC, NPP = C::NPP, LD = C::LD;
  typedef double dbl2 __attribute__((ext_vector_type(2)));
  typedef dbl2 dbl2u __attribute__((aligned(8)));
  __shared__ Number s_a[CPB][NF][LD];
  __shared__ Number s_b[CPB][DIM][LD];

  const int tid = threadIdx.x;
  const int n_entries = sel.list ? sel.n : mesh.n_cells, c0 = blockIdx.x * CPB;
  // (a slot past the last entry repeats it and stores nothing)
  auto cell_of = [&](int lc) __attribute__((always_inline)) {
    const int e = CPB == 1 ? c0 : min(c0 + lc, n_entries - 1);
    return sel.list ? sel.list[e] : e;
  };
  const int d = __builtin_amdgcn_readfirstlane((tid >> 6) / WPD);
  const int li = tid - d * (WPD * 64);
  static_assert(NF * ND <= 4096 && NPP * BLOCK <= 4096, "small_div's range");
  const int lc = CPB == 1 ? 0 : min(small_div<NT>(li), CPB - 1), t = li - lc * NT;
  const bool ok = t < NT;

  size_t idx[NPP];
  int dst[NPP];
  auto copy_in = [&](const double *u) __attribute__((always_inline)) {
    dbl2 x[NPP];
#pragma unroll
    for (int j = 0; j < NPP; ++j) __builtin_memcpy(&x[j], u + idx[j], 16);
#pragma unroll
    for (int j = 0; j < NPP; ++j)
      if (dst[j] >= 0) {
        Number *o = &s_a[0][0][0] + dst[j];
        o[0] = Number(x[j].x);
        o[1] = Number(x[j].y);
      }
  };
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    const int q = tid + j * BLOCK, l = CPB == 1 ? 0 : min(small_div<PPC>(q), CPB - 1);
    int e = 2 * (q - l * PPC);
    const bool on = e < NF * ND;
    if (!on || ((NF * ND) % 2 && e == NF * ND - 1)) e = NF * ND - 2;  // (the odd last pair overlaps)
    dst[j] = on ? l * (NF * LD) + CkGrid<DIM, N>::node(e) : -1;
    idx[j] = (size_t)cell_of(l) * (NF * ND) + e;
  }
  copy_in(src);
  const int cell = cell_of(lc);
  const double te = sel.cluster ? sel.te[sel.cluster[cell]] : te_all;
  const Number rho = Number(mesh.rho[cell]), cc = Number(mesh.speed[cell]);
  const Number ih = recip(Number(mesh.h[(size_t)cell * DIM + d]));
  __syncthreads();
  ck_lines<DIM, K, Number>(s_a[lc][0], s_b[lc][0], ok, d, t, recip(rho) * ih, (rho * cc * cc) * ih, t2, t1,
                           te, recon != nullptr, [&]() { copy_in(recon); });
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    const int q = tid + j * BLOCK, l = CPB == 1 ? 0 : min(small_div<PPC>(q), CPB - 1);
    if (dst[j] < 0 || (CPB > 1 && c0 + l >= n_entries)) continue;
    const Number *k = &s_a[0][0][0] + dst[j];
    if ((NF * ND) % 2 && q - l * PPC == PPC - 1) {  // the odd last entry alone
      tempsrc[idx[j] + 1] = double(k[1]);
      continue;
    }
    const dbl2 o = {double(k[0]), double(k[1])};
    *(dbl2u *)(tempsrc + idx[j]) = o;
  }
}

}  // namespace exw
