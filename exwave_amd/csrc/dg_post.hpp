// dg_post.hpp -- post-processed pressure and its error.
//
// compute_post_pressure (source/wave_equation_operations.cc:786-848): per cell
// the local Neumann problem (grad phi, grad p*) = (grad phi, -rho v_t) on
// Q_{k+1} with the nodal basis of the k+2 Gauss-Lobatto points
// (fe_post_disp, source/explicit_wave.cc:165) and QGauss(k+2), v_t the
// velocity part of apply(solution); then the constant is set so that the cell
// average of p* equals that of p_h.
//
// Layout: with P = k+2 the Gauss-Lobatto nodes and the QGauss(P) points form
// grids of the same size P^dim, so thread t of a cell owns node t AND point t.
// Every CG vector (u, r, p, Ap) lives in registers, one value per thread; the
// symmetric geometry factor G = J^-1 J^-T det w of point t too.  The
// sum-factorised passes of the Laplacian exchange values through LDS:
//   nodes -> points: P^dim values, one pass per direction with the GL
//   interpolation matrix; gradient: collocation derivative of the QGauss(P)
//   points; flux G grad; the transposes back.
//
// Solver: the reference fixes the first unknown and runs CG to |r|/|r0| <
// 1e-11 (include/elementwise_cg.templates.h:66-145).  The result after the
// average adjustment is the same for every Neumann solution, so this kernel
// runs CG on the zero-sum subspace instead (the matrix's null space is the
// constant vector): condition numbers 20-500x smaller than with the fixed
// unknown, so the same iteration count reaches 1e-13.  The stopping rule is
// per cell (abs, rel, cap), the division guard that of the reference
// (adjust_division_by_zero, :44-61).
#pragma once
#include "dg_common.hpp"
#include "dg_misc.hpp"

namespace exw {

template <int DIM, int K>
struct PostShape {
  static constexpr int N = K + 1, P = K + 2, E = K + 3;
  static constexpr int ND = DIM == 2 ? N * N : N * N * N;
  static constexpr int NP = DIM == 2 ? P * P : P * P * P;
  static constexpr int NE = DIM == 2 ? E * E : E * E * E;
  static constexpr int LANES = (NP + 63) / 64 * 64;  // whole waves per cell
  static constexpr int WAVES = LANES / 64;
  static constexpr int CPB = LANES >= 256 ? 1 : 256 / LANES;
  static constexpr int BLOCK = LANES * CPB;
  static_assert(BLOCK <= 1024, "cell does not fit a workgroup");
};

// Table (built on the host, per degree): offsets into one array
template <int K>
struct PostTab {
  static constexpr int N = K + 1, P = K + 2, E = K + 3;
  static constexpr int XQ = 0;             // QGauss(P) points on [0,1]
  static constexpr int WQ = XQ + P;        // and weights
  static constexpr int PV = WQ + P;        // PV[q*P+i] = l^GL_i(xq_q)
  static constexpr int DQ = PV + P * P;    // DQ[q*P+j] = l^Q_j'(xq_q) (collocation)
  static constexpr int IQ = DQ + P * P;    // IQ[q*N+i] = l^G(N)_i(xq_q)
  static constexpr int XE = IQ + P * N;    // QGauss(E) points (error rule)
  static constexpr int WE = XE + E;
  static constexpr int IE = WE + E;        // IE[q*P+i] = l^GL_i(xe_q)
  static constexpr int SV = IE + E * P;    // SV[q*P+m]: eigenvector m of the 1D Laplacian at xq_q
  static constexpr int LAM = SV + P * P;   // its eigenvalues, LAM[0] = 0 (the constant)
  static constexpr int EG = LAM + P;       // EG[i*P+q] = l^Q_q(x^GL_i)
  static constexpr int SIZE = EG + P * P;
  static constexpr int LDS = XE;           // what the plain CG kernel stages
};

struct PostSolver {
  double abs_tol, rel_tol;
  int max_iter;  // stop after max_iter + 1 iterations at most
};

namespace post {

// One pass along direction D of a square (P x P) matrix on a P^dim tensor at
// the thread's point ti: out = sum_j M(ti_D, j) in(ti with ti_D = j); TR uses
// M^T.
template <int DIM, int P, int D, bool TR>
__device__ __forceinline__ double sq(const double *M, const double *in, const int *ti) {
  constexpr int st = D == 0 ? 1 : (D == 1 ? P : P * P);
  const int base = ti[0] + P * ti[1] + (DIM == 3 ? P * P * ti[2] : 0) - ti[D] * st;
  double s = 0.0;
#pragma unroll
  for (int j = 0; j < P; ++j) s += (TR ? M[j * P + ti[D]] : M[ti[D] * P + j]) * in[base + j * st];
  return s;
}

// Rectangular pass D of an NO x NI matrix on the tensor whose directions < D
// already have NO points and directions >= D still NI: output entry o (of
// NO^(D+1) NI^(DIM-D-1)) or 0 when o is out of range.
template <int DIM, int NI, int NO, int D>
__device__ __forceinline__ double rect(const double *M, const double *in, int o) {
  constexpr int LO = D == 0 ? 1 : (D == 1 ? NO : NO * NO);
  constexpr int COUNT = LO * NO * (D == DIM - 1 ? 1 : (DIM - D - 1 == 1 ? NI : NI * NI));
  if (o >= COUNT) return 0.0;
  const int lower = o % LO, id = (o / LO) % NO, upper = o / (LO * NO);
  const double *src = in + lower + LO * NI * upper;
  double s = 0.0;
#pragma unroll
  for (int j = 0; j < NI; ++j) s += M[id * NI + j] * src[LO * j];
  return s;
}

// Sum over the lanes of one cell (WAVES waves), every lane gets the total;
// fixed order (butterfly, then the waves in order): deterministic.
template <int WAVES, int CPB, int NV>
__device__ __forceinline__ void reduce(double *v, double (*red)[WAVES][3], int lc, int t) {
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
  if constexpr (WAVES > 1) {
    if ((t & 63) == 0)
#pragma unroll
      for (int k = 0; k < NV; ++k) red[lc][t >> 6][k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) s += red[lc][w][k];
      v[k] = s;
    }
  }
}

}  // namespace post

// grid: ceil(n_cells / CPB) groups of BLOCK threads; dudt = apply(sol)
template <int DIM, int K>
__global__ void __launch_bounds__((PostShape<DIM, K>::BLOCK))
    post_pressure_kernel(const DevMesh mesh, const double *__restrict__ tab,
                         const double *__restrict__ sol, const double *__restrict__ dudt,
                         double *__restrict__ post, int *__restrict__ iterations,
                         const PostSolver cfg) {
  using S = PostShape<DIM, K>;
  using T = PostTab<K>;
  constexpr int N = S::N, P = S::P, NP = S::NP, ND = S::ND, NF = DIM + 1, LANES = S::LANES;
  constexpr int WAVES = S::WAVES, CPB = S::CPB, NG = DIM * (DIM + 1) / 2;
  __shared__ double s_tab[T::LDS];
  __shared__ double s_buf[CPB][DIM + 1][NP];
  __shared__ double s_red[2][CPB][WAVES][3];
  const int tid = threadIdx.x, lc = tid / LANES, t = tid % LANES;
  const int cell_raw = blockIdx.x * CPB + lc;
  const bool cell_ok = cell_raw < mesh.n_cells;
  const int cell = cell_ok ? cell_raw : mesh.n_cells - 1;  // spare groups redo the last cell
  const bool act = t < NP;
  const int tc = act ? t : NP - 1;
  const int ti[3] = {tc % P, (tc / P) % P, DIM == 3 ? tc / (P * P) : 0};
  for (int i = tid; i < T::LDS; i += S::BLOCK) s_tab[i] = tab[i];
  const double *xq = s_tab + T::XQ, *wq = s_tab + T::WQ, *PV = s_tab + T::PV,
               *DQ = s_tab + T::DQ, *IQ = s_tab + T::IQ;
  double *B[DIM + 1];
#pragma unroll
  for (int b = 0; b <= DIM; ++b) B[b] = s_buf[lc][b];
  int rb = 0;  // alternating reduction buffer
  auto reduce1 = [&](double x) {
    double v[1] = {x};
    post::reduce<WAVES, CPB, 1>(v, s_red[rb], lc, t);
    rb ^= 1;
    return v[0];
  };

  __syncthreads();

  // geometry at QGauss(P) point ti
  double G[NG], Ji[DIM * DIM], jxw;
  {
    double xi[3], J[9], w = 1.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      xi[d] = xq[ti[d]];
      w *= wq[ti[d]];
    }
    const double det =
        multilinear_jacobian<DIM>(mesh.vertices + (size_t)cell * (1 << DIM) * DIM, xi, J, Ji);
    jxw = det * w;
    int g = 0;
#pragma unroll
    for (int e = 0; e < DIM; ++e)
#pragma unroll
      for (int e2 = e; e2 < DIM; ++e2) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < DIM; ++i) s += Ji[e * DIM + i] * Ji[e2 * DIM + i];
        G[g++] = s * jxw;
      }
  }

  // v_t (velocity of dudt) and p_h at the QGauss(P) points: N^dim -> P^dim
  double vt[DIM], ph = 0.0;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const double *src = (f < DIM ? dudt : sol) + ((size_t)cell * NF + f) * ND;
    __syncthreads();  // previous readers of B[0], B[1] are done
    if (t < ND) B[0][t] = src[t];
    __syncthreads();
    double val;
    if constexpr (DIM == 2) {
      const double a = post::rect<2, N, P, 0>(IQ, B[0], t);
      if (t < P * N) B[1][t] = a;
      __syncthreads();
      val = post::rect<2, N, P, 1>(IQ, B[1], tc);
    } else {
      const double a = post::rect<3, N, P, 0>(IQ, B[0], t);
      if (t < P * N * N) B[1][t] = a;
      __syncthreads();
      const double b = post::rect<3, N, P, 1>(IQ, B[1], t);
      if (t < P * P * N) B[2][t] = b;
      __syncthreads();
      val = post::rect<3, N, P, 2>(IQ, B[2], tc);
    }
    if (f < DIM)
      vt[f] = val;
    else
      ph = val;
  }
  __syncthreads();

  // The flux part of the operator: given F_e (the reference-space flux at the
  // thread's point, already in B[0..DIM-1]), sum_e grad_e^T F_e back to the
  // nodes, via B[DIM] and the transposed interpolation passes.
  auto grad_transpose = [&]() -> double {
    __syncthreads();
    double y = 0.0;
    y += post::sq<DIM, P, 0, true>(DQ, B[0], ti);
    y += post::sq<DIM, P, 1, true>(DQ, B[1], ti);
    if constexpr (DIM == 3) y += post::sq<DIM, P, 2, true>(DQ, B[2], ti);
    if (act) B[DIM][t] = y;
    __syncthreads();
    if constexpr (DIM == 2) {
      const double a = post::sq<2, P, 1, true>(PV, B[2], ti);
      if (act) B[0][t] = a;
      __syncthreads();
      return post::sq<2, P, 0, true>(PV, B[0], ti);
    } else {
      const double a = post::sq<3, P, 2, true>(PV, B[3], ti);
      if (act) B[0][t] = a;
      __syncthreads();
      const double b = post::sq<3, P, 1, true>(PV, B[0], ti);
      if (act) B[1][t] = b;
      __syncthreads();
      return post::sq<3, P, 0, true>(PV, B[1], ti);
    }
  };
  // nodal values -> values at the QGauss(P) points (the thread's own point).
  // 2D stages in B[1] (B[0] may still be read by the last transposed pass),
  // 3D in B[0].
  auto to_points = [&](double x) -> double {
    constexpr int st = DIM == 2 ? 1 : 0;
    if (act) B[st][t] = x;
    __syncthreads();
    if constexpr (DIM == 2) {
      const double a = post::sq<2, P, 0, false>(PV, B[1], ti);
      if (act) B[0][t] = a;
      __syncthreads();
      const double b = post::sq<2, P, 1, false>(PV, B[0], ti);
      if (act) B[2][t] = b;
      __syncthreads();
      return b;
    } else {
      const double a = post::sq<3, P, 0, false>(PV, B[0], ti);
      if (act) B[1][t] = a;
      __syncthreads();
      const double b = post::sq<3, P, 1, false>(PV, B[1], ti);
      if (act) B[2][t] = b;
      __syncthreads();
      const double c = post::sq<3, P, 2, false>(PV, B[2], ti);
      if (act) B[3][t] = c;
      __syncthreads();
      return c;
    }
  };
  // Neumann Laplacian of the nodal vector x at node t
  auto laplace = [&](double x) -> double {
    to_points(x);  // values at the points now in B[DIM]
    double g[DIM];
    g[0] = post::sq<DIM, P, 0, false>(DQ, B[DIM], ti);
    g[1] = post::sq<DIM, P, 1, false>(DQ, B[DIM], ti);
    if constexpr (DIM == 3) g[2] = post::sq<DIM, P, 2, false>(DQ, B[DIM], ti);
    double f[DIM];
    if constexpr (DIM == 2) {
      f[0] = G[0] * g[0] + G[1] * g[1];
      f[1] = G[1] * g[0] + G[2] * g[1];
    } else {
      f[0] = G[0] * g[0] + G[1] * g[1] + G[2] * g[2];
      f[1] = G[1] * g[0] + G[3] * g[1] + G[4] * g[2];
      f[2] = G[2] * g[0] + G[4] * g[1] + G[5] * g[2];
    }
    __syncthreads();  // everyone has read B[DIM]; B[0..DIM-1] are free
#pragma unroll
    for (int e = 0; e < DIM; ++e)
      if (act) B[e][t] = f[e];
    return grad_transpose();
  };

  // right-hand side (grad phi, -rho v_t): reference-space flux Ji (-rho v_t) jxw
  const double rho = mesh.rho[cell];
  {
    double f[DIM];
#pragma unroll
    for (int e = 0; e < DIM; ++e) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < DIM; ++i) s += Ji[e * DIM + i] * (-rho * vt[i]);
      f[e] = s * jxw;
    }
#pragma unroll
    for (int e = 0; e < DIM; ++e)
      if (act) B[e][t] = f[e];
  }
  double rhs = grad_transpose();
  if (!act) rhs = 0.0;
  const double mean = reduce1(rhs) / NP;  // project onto the zero-sum subspace
  if (act) rhs -= mean;

  // CG on the zero-sum subspace
  double u = 0.0, r = rhs, p = rhs;
  double rr = reduce1(r * r);
  const double nr0 = sqrt(rr);
  const double guard = fmax(1e-5 * cfg.abs_tol * cfg.abs_tol, 1e4 * 2.2250738585072014e-308);
  bool done = false;
  int it = 0;
  for (;;) {
    double Ap = laplace(p);
    if (!act) Ap = 0.0;
    double pAp = reduce1(p * Ap);
    if (!done) {
      if (pAp < guard) pAp = 1.0;
      const double alpha = rr / pAp;
      u += alpha * p;
      r -= alpha * Ap;
    }
    double v2[2] = {r, r * r};
    post::reduce<WAVES, CPB, 2>(v2, s_red[rb], lc, t);
    rb ^= 1;
    if (!done) {
      const double m = v2[0] / NP;
      if (act) r -= m;
      const double rn = fmax(v2[1] - v2[0] * m, 0.0);
      ++it;
      if (sqrt(rn) < cfg.abs_tol || sqrt(rn) < cfg.rel_tol * nr0 || it > cfg.max_iter) {
        done = true;
      } else {
        const double beta = rn / rr;
        rr = rn;
        p = act ? r + beta * p : 0.0;
      }
    }
    if (__syncthreads_and((int)done)) break;  // every cell of the group converged
  }

  // constant offset from the cell averages (:821-841)
  const double uq = to_points(u);
  double v3[3] = {act ? jxw : 0.0, act ? jxw * ph : 0.0, act ? jxw * uq : 0.0};
  post::reduce<WAVES, CPB, 3>(v3, s_red[rb], lc, t);
  const double adjust = (v3[1] - v3[2]) / v3[0];
  if (cell_ok && act) post[(size_t)cell * NP + t] = u + adjust;
  if (cell_ok && t == 0 && iterations) iterations[cell] = it;
}

// Lanes of the preconditioned solver: one per column of the cell (P^(dim-1)
// columns of P points along the last direction), several cells to a wave where
// they fit; LDS rows of odd length PP keep the row-wise reads free of bank
// conflicts.
template <int DIM, int K>
struct PostColumns {
  static constexpr int P = K + 2, PP = P | 1;
  static constexpr int LPC = DIM == 2 ? P : P * P;
  static constexpr int NPL = DIM == 2 ? P * PP : P * P * PP;  // LDS entries of a tensor
  static constexpr int CPB = LPC <= 64 ? 64 / LPC : 1;
  static constexpr int BLOCK = LPC <= 64 ? 64 : (LPC + 63) / 64 * 64;
  // columns of up to 6 points (3D) or 9 (2D) are held to 256 registers, two waves per
  // SIMD (the two largest spill 11 and 4 vector registers; the matrices' scalar
  // registers spill to vector lanes from 2D k=3 and 3D k=2 on)
  static constexpr int MIN_WAVES = P <= (DIM == 2 ? 9 : 6) ? 2 : 1;
};

namespace post {

// y = M x or M^T x for one line in registers, M row-major NO x NI, wave-uniform:
// scalar loads at every use.  The empty asm hides where M points, or the
// compiler hoists the matrices out of the iteration and spills their scalar
// registers to vector lanes, two lane reads per product.
template <int NO, int NI, bool TR>
__device__ __forceinline__ void line(const double *Mg, const double *x, double *y) {
  asm volatile("" : "+s"(Mg));
  const auto *M = (const __attribute__((address_space(4))) double *)Mg;
#pragma unroll
  for (int q = 0; q < NO; ++q) {
    double a = 0.0;
#pragma unroll
    for (int i = 0; i < NI; ++i) a += (TR ? M[i * NO + q] : M[q * NI + i]) * x[i];
    y[q] = a;
  }
}

// Sums of NV values over the LPC consecutive lanes of a cell, to all of them,
// (and, like theirs, to the wave's spare lanes, which share their slot) in a
// fixed order: within a wave a halving tree of the lanes from `first`, then (one
// cell over several waves) the waves in order.
template <int LPC, int BLOCK, int NV>
__device__ __forceinline__ void column_sum(double *v, int idx, int first, double (*red)[4]) {
  if constexpr (LPC <= 64) {
#pragma unroll
    for (int n = LPC; n > 1;) {
      const int h = (n + 1) / 2;
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        const double o = __shfl_down(v[k], h, 64);
        if (idx + h < n) v[k] += o;
      }
      n = h;
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = __shfl(v[k], first, 64);
  } else {
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
    __syncthreads();  // the sums before have been read
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int k = 0; k < NV; ++k) red[threadIdx.x >> 6][k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < BLOCK / 64; ++w) s += red[w][k];
      v[k] = s;
    }
  }
}

}  // namespace post

// The post-processed pressure by preconditioned CG (the default; a call that
// asks for the CG iteration counts runs post_pressure_kernel, whose plain CG
// they count).
//
// The same Neumann problem, posed for the values at the P^dim Gauss points
// (one basis of the same space: no interpolation passes in the operator, which
// is sum_e,e' D_e^T G_ee' D_e') and preconditioned with the inverse of its
// separable part: with the cell's mean metric g_e = sum_q G_ee(q) the operator
// sum_e g_e W..(D^T W D)..W is diagonal in the tensor product of the 1D
// eigenvectors SV (SV^T W SV = 1), so z = SV3 (1 / sum_e g_e lambda) SV3^T r,
// the constant left out.  On box cells that is the exact inverse (one
// iteration); on the deformed membranes 8-14 iterations reach the 1e-13 that
// plain CG needs 60-150 for.  Both stops are on r.z, the energy norm of the error in
// that metric, relative to the first one.  A cell
// whose p.Ap is at the bottom of the exponent range (a state that has decayed
// to 1e-150) ends with what it has: the ratio of two such numbers is noise.
//
// Lanes hold columns: every tensor is P registers per lane along the last
// direction, a pass along it is register FMAs, and the other directions
// exchange through LDS (one read and one write per entry and pass instead of
// 2 P reads).  A cell of up to 64 columns is one wave: no barriers.
// Bound by the FP64 issue of two waves per SIMD (the column's metric and CG
// vectors fill their registers).  3D k=4, 16^3 deformed cells: 0.19 ms against
// 4.34 ms of plain CG on one lane per point (LDS reads of matrix and data for
// every product, 20 barriers per iteration); against dense solves in 64 bits its
// p* is off by 4.6e-15, plain CG's by 1.3e-14.
template <int DIM, int K>
__global__ void __launch_bounds__((PostColumns<DIM, K>::BLOCK))
    __attribute__((amdgpu_waves_per_eu(PostColumns<DIM, K>::MIN_WAVES)))
    post_pcg_kernel(const DevMesh mesh, const double *__restrict__ tab,
                    const double *__restrict__ sol, const double *__restrict__ dudt,
                    double *__restrict__ post, const PostSolver cfg) {
  using S = PostColumns<DIM, K>;
  using T = PostTab<K>;
  constexpr int N = K + 1, P = S::P, PP = S::PP, LPC = S::LPC, CPB = S::CPB, BLOCK = S::BLOCK;
  constexpr int NF = DIM + 1, NG = DIM * (DIM + 1) / 2, NVD = (1 << DIM) * DIM;
  constexpr int ND = DIM == 2 ? N * N : N * N * N, NP = DIM == 2 ? P * P : P * P * P;
  __shared__ double s_t[CPB][DIM][S::NPL];  // exchange buffers
  __shared__ double s_w[CPB][S::NPL];       // det J times the weights at the points
  __shared__ double s_V[CPB][NVD];
  __shared__ double s_red[BLOCK / 64][4];
  const double *IQ = tab + T::IQ, *SV = tab + T::SV, *LAM = tab + T::LAM, *EG = tab + T::EG,
               *D = tab + T::DQ;

  const int tid = threadIdx.x;
  const int lc_raw = tid / LPC;
  const bool act = lc_raw < CPB && tid < CPB * LPC;
  const int lc = act ? lc_raw : CPB - 1, idx = act ? tid - lc * LPC : LPC - 1;
  const int cell_raw = blockIdx.x * CPB + lc;
  const bool cell_ok = cell_raw < mesh.n_cells;
  const int cell = cell_ok ? cell_raw : mesh.n_cells - 1;  // spare slots redo the last cell
  double(*t)[S::NPL] = s_t[lc];
  // a line of direction e for lane idx: first entry and stride
  const int i0 = idx % P, i1 = idx / P;
  auto base = [&](int e) {
    if constexpr (DIM == 2) return e == 1 ? i0 : PP * i0;
    else return e == 2 ? i0 + PP * i1 : (e == 1 ? i0 + PP * P * i1 : PP * (i0 + P * i1));
  };
  constexpr int st[3] = {1, PP, PP * P};
  constexpr int LAST = DIM - 1;
  auto get = [&](const double *b, int e, double *x) {
#pragma unroll
    for (int j = 0; j < P; ++j) x[j] = b[base(e) + j * st[e]];
  };
  auto put = [&](double *b, int e, const double *x) {
    if (act)
#pragma unroll
      for (int j = 0; j < P; ++j) b[base(e) + j * st[e]] = x[j];
  };

  if (act)
    for (int i = idx; i < NVD; i += LPC) s_V[lc][i] = mesh.vertices[(size_t)cell * NVD + i];

  // v_t (velocity of dudt) and p_h from their N^dim nodes to the P^dim points
  double val[NF][P];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const double *src = (f < DIM ? dudt : sol) + ((size_t)cell * NF + f) * ND;
    __syncthreads();  // the field before has been read
    if (act)
      for (int n = idx; n < ND; n += LPC) {
        const int x = n % N, y = (n / N) % N, z = n / (N * N);
        t[0][x + PP * (y + P * z)] = src[n];
      }
    __syncthreads();
    double a[N], b[P];
    // x lines: N^(dim-1) of them, (y, z) = (idx % N, idx / N)
    constexpr int LX = DIM == 2 ? N : N * N;
    if (act && idx < LX) {
      double *r = t[0] + PP * (DIM == 2 ? idx : idx % N + P * (idx / N));
#pragma unroll
      for (int j = 0; j < N; ++j) a[j] = r[j];
      post::line<P, N, false>(IQ, a, b);
#pragma unroll
      for (int j = 0; j < P; ++j) r[j] = b[j];
    }
    __syncthreads();
    if constexpr (DIM == 3) {
      // y lines: (x, z) with z < N
      if (act && idx < P * N) {
        double *r = t[0] + base(1);
#pragma unroll
        for (int j = 0; j < N; ++j) a[j] = r[j * PP];
        post::line<P, N, false>(IQ, a, b);
#pragma unroll
        for (int j = 0; j < P; ++j) r[j * PP] = b[j];
      }
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < N; ++j) a[j] = t[0][base(LAST) + j * st[LAST]];
    post::line<P, N, false>(IQ, a, val[f]);
  }

  // metric G at the column's points, the right-hand side's flux (over val)
  const double rho = mesh.rho[cell];
  double G[NG][P], ph_sum = 0.0, vol = 0.0;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    double xi[3], J[9], Ji[9], w = tab[T::WQ + j];
    const double *xq = tab + T::XQ;
    xi[0] = xq[i0];
    w *= tab[T::WQ + i0];
    if constexpr (DIM == 3) {
      xi[1] = xq[i1];
      w *= tab[T::WQ + i1];
    }
    xi[LAST] = xq[j];
    const double jxw = multilinear_jacobian<DIM>(s_V[lc], xi, J, Ji) * w;
    int g = 0;
    double f[DIM];
#pragma unroll
    for (int e = 0; e < DIM; ++e) {
#pragma unroll
      for (int e2 = e; e2 < DIM; ++e2) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < DIM; ++i) s += Ji[e * DIM + i] * Ji[e2 * DIM + i];
        G[g++][j] = s * jxw;
      }
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < DIM; ++i) s += Ji[e * DIM + i] * (-rho * val[i][j]);
      f[e] = s * jxw;
    }
#pragma unroll
    for (int e = 0; e < DIM; ++e) val[e][j] = f[e];
    if (act) s_w[lc][base(LAST) + j * st[LAST]] = jxw;
    vol += jxw;
    ph_sum += jxw * val[DIM][j];
  }
  // the preconditioner's mean metric, then the inverse eigenvalue sums at the
  // x line's entries
  double invd[P];
  {
    double g[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < P; ++j) {
      g[0] += G[0][j];
      g[1] += G[DIM][j];
      if constexpr (DIM == 3) g[2] += G[5][j];
    }
    if (!act) g[0] = g[1] = g[2] = 0.0;
    post::column_sum<LPC, BLOCK, DIM>(g, idx, lc * LPC, s_red);
    const double rest = DIM == 2 ? g[1] * LAM[i0] : g[1] * LAM[i0] + g[2] * LAM[i1];
#pragma unroll
    for (int m = 0; m < P; ++m) invd[m] = (m == 0 && idx == 0) ? 0.0 : 1.0 / (g[0] * LAM[m] + rest);
  }

  // sum_e D_e^T f_e: f_0.. through the buffers, f_LAST in registers
  auto div = [&](double (*f)[P], double *out) {
#pragma unroll
    for (int e = 0; e < LAST; ++e) put(t[e], LAST, f[e]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < LAST; ++e) {
      double x[P], y[P];
      get(t[e], e, x);
      post::line<P, P, true>(D, x, y);
      put(t[e], e, y);
    }
    post::line<P, P, true>(D, f[LAST], out);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < LAST; ++e) {
      double x[P];
      get(t[e], LAST, x);
#pragma unroll
      for (int j = 0; j < P; ++j) out[j] += x[j];
    }
    __syncthreads();
  };
  auto laplace = [&](const double *x, double *out) {
    double g[DIM][P];
    put(t[LAST], LAST, x);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < LAST; ++e) {
      double a[P], b[P];
      get(t[LAST], e, a);
      post::line<P, P, false>(D, a, b);
      put(t[e], e, b);
    }
    post::line<P, P, false>(D, x, g[LAST]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < LAST; ++e) get(t[e], LAST, g[e]);
#pragma unroll
    for (int j = 0; j < P; ++j) {
      if constexpr (DIM == 2) {
        const double a = g[0][j], b = g[1][j];
        g[0][j] = G[0][j] * a + G[1][j] * b;
        g[1][j] = G[1][j] * a + G[2][j] * b;
      } else {
        const double a = g[0][j], b = g[1][j], c = g[2][j];
        g[0][j] = G[0][j] * a + G[1][j] * b + G[2][j] * c;
        g[1][j] = G[1][j] * a + G[3][j] * b + G[4][j] * c;
        g[2][j] = G[2][j] * a + G[4][j] * b + G[5][j] * c;
      }
    }
    div(g, out);  // (each lane overwrites the entries it has read itself)
  };
  // z = SV3 invd SV3^T r
  auto precond = [&](const double *r, double *z) {
    double a[P], b[P];
    post::line<P, P, true>(SV, r, a);
    put(t[0], LAST, a);
    __syncthreads();
    if constexpr (DIM == 3) {
      get(t[0], 1, a);
      post::line<P, P, true>(SV, a, b);
      put(t[0], 1, b);
      __syncthreads();
    }
    get(t[0], 0, a);
    post::line<P, P, true>(SV, a, b);
#pragma unroll
    for (int m = 0; m < P; ++m) b[m] *= invd[m];
    post::line<P, P, false>(SV, b, a);
    put(t[0], 0, a);
    __syncthreads();
    if constexpr (DIM == 3) {
      get(t[0], 1, a);
      post::line<P, P, false>(SV, a, b);
      put(t[0], 1, b);
      __syncthreads();
    }
    get(t[0], LAST, a);
    post::line<P, P, false>(SV, a, z);
    __syncthreads();
  };
  auto dot = [&](const double *x, const double *y) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < P; ++j) s += x[j] * y[j];
    double v[1] = {act ? s : 0.0};
    post::column_sum<LPC, BLOCK, 1>(v, idx, lc * LPC, s_red);
    return v[0];
  };
  double u[P], r[P], p[P];
  div(val, r);  // (val[0..DIM-1] holds the right-hand side's flux)
#pragma unroll
  for (int j = 0; j < P; ++j) u[j] = 0.0;
  precond(r, p);
  double rz = dot(r, p);
  // |r| < abs_tol is tested on r.z too, in the first residual's proportion (a sum of
  // its own costs the iterations 4 %)
  const double abs2 = cfg.abs_tol * cfg.abs_tol;
  const double stop = rz * fmax(cfg.rel_tol * cfg.rel_tol, abs2 / dot(r, r));
  const double guard = fmax(1e-5 * abs2, 1e4 * 2.2250738585072014e-308);  // as plain CG's
  // a zero right-hand side (or NaN) leaves u = 0 (or NaN, through r)
  bool done = !(rz > 0.0);
  if (done && !(rz == 0.0)) u[0] = rz - rz;
  for (int it = 0; it <= cfg.max_iter; ++it) {
    if (__syncthreads_and((int)done)) break;  // every cell of the group converged
    double q[P];
    laplace(p, q);
    const double pAp = dot(p, q);
    if (!done) {
      const double alpha = pAp < guard ? 0.0 : rz / pAp;
#pragma unroll
      for (int j = 0; j < P; ++j) {
        u[j] += alpha * p[j];
        r[j] -= alpha * q[j];
      }
    }
    precond(r, q);
    const double rn = dot(r, q);
    if (!done) {
      const double beta = rn / rz;
      rz = rn;
      done = pAp < guard || !(rn > stop);
#pragma unroll
      for (int j = 0; j < P; ++j) p[j] = q[j] + beta * p[j];
    }
  }

  // constant offset from the cell averages (:821-841), then the values at the
  // Gauss-Lobatto nodes
  double uq = 0.0;
#pragma unroll
  for (int j = 0; j < P; ++j) uq += s_w[lc][base(LAST) + j * st[LAST]] * u[j];
  double v3[3] = {act ? vol : 0.0, act ? ph_sum : 0.0, act ? uq : 0.0};
  post::column_sum<LPC, BLOCK, 3>(v3, idx, lc * LPC, s_red);
  const double adjust = (v3[1] - v3[2]) / v3[0];
  put(t[0], LAST, u);
  __syncthreads();
  {
    double a[P], b[P];
    get(t[0], 0, a);
    post::line<P, P, false>(EG, a, b);
    put(t[0], 0, b);
    __syncthreads();
    if constexpr (DIM == 3) {
      get(t[0], 1, a);
      post::line<P, P, false>(EG, a, b);
      put(t[0], 1, b);
      __syncthreads();
    }
    get(t[0], LAST, a);
    post::line<P, P, false>(EG, a, b);
    if (act && cell_ok)
#pragma unroll
      for (int j = 0; j < P; ++j) post[(size_t)cell * NP + j * LPC + idx] = b[j] + adjust;
  }
}

// Whether p* is summed directly at each point of the error rule instead of by tensor
// passes: in 2D from k=5 on, where a cell's 7 to 14 lines leave most of a group idle
// through the passes' barriers, and the direct sums have few terms.  us per call with
// the readback (about 28), direct / passes: 2D k=4 19881 cells 53.3 / 46.1, k=5 196
// 29.8 / 32.2, k=7 7744 56.5 / 74.3, k=12 2916 67.7 / 79.2; 3D k=4 2744 141 / 64.
template <int DIM, int K>
constexpr bool post_error_direct() {
  return DIM == 2 && K >= 5;
}

// ||p* - p_exact||^2 partial sums with QGauss(k+3) (source/explicit_wave.cc:477-484)
template <int DIM, int K>
__global__ void __launch_bounds__(256)
    post_error_kernel(const DevMesh mesh, const double *__restrict__ tab, const DevModes modes,
                      double t, const double *__restrict__ post, double *__restrict__ partial) {
  using S = PostShape<DIM, K>;
  using T = PostTab<K>;
  constexpr int P = S::P, E = S::E, NVD = (1 << DIM) * DIM;
  using R = Refine<DIM, P, E, 1>;
  constexpr int CPB = R::CPB, NP = R::NDI, NE = R::NDO;
  __shared__ double red[1][256];
  __shared__ double s_a[R::A], s_b[R::B], s_V[CPB][NVD], s_amp[8][DIM + 1];
  modes_factors<DIM>(modes, t, s_amp);
  const double *xe = tab + T::XE, *we = tab + T::WE;
  double err = 0.0;
  if constexpr (post_error_direct<DIM, K>()) {
    for (int i = threadIdx.x; i < E * P; i += 256) s_a[i] = tab[T::IE + i];
    __syncthreads();
    const size_t total = (size_t)mesh.n_cells * NE;
    for (size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x; gid < total;
         gid += (size_t)gridDim.x * 256) {
      const int cell = int(gid / NE), q = int(gid % NE);
      const int qi[2] = {q % E, q / E};
      double xi[2], x[2], J[4], Ji[4], ex[DIM + 1];
      xi[0] = xe[qi[0]];
      xi[1] = xe[qi[1]];
      const double *V = mesh.vertices + (size_t)cell * NVD, *pc = post + (size_t)cell * NP;
      multilinear_point<DIM>(V, xi, x);
      const double jxw = fabs(multilinear_jacobian<DIM>(V, xi, J, Ji)) * we[qi[0]] * we[qi[1]];
      double val = 0.0;
      for (int n = 0; n < NP; ++n)
        val += s_a[qi[0] * P + n % P] * s_a[qi[1] * P + n / P] * pc[n];
      modes_all<DIM>(modes, s_amp, x, ex);
      const double d = val - ex[DIM];
      err += d * d * jxw;
    }
    block_partials<1>(&err, red, partial);
    return;
  }
  for (int c0 = blockIdx.x * CPB; c0 < mesh.n_cells; c0 += gridDim.x * CPB) {
    const int nc = min(CPB, mesh.n_cells - c0);
    __syncthreads();  // the points of the cells before have been read
    for (int i = threadIdx.x; i < nc * NVD; i += 256)
      s_V[i / NVD][i % NVD] = mesh.vertices[(size_t)c0 * NVD + i];
    for (int i = threadIdx.x; i < CPB * NP; i += 256)
      s_a[i] = i < nc * NP ? post[(size_t)c0 * NP + i] : 0.0;
    __syncthreads();
    const double *out = R::run(tab + T::IE, s_a, s_b);
#pragma unroll 1
    for (int i = threadIdx.x; i < nc * NE; i += 256) {
      const int c = i / NE, q = i - c * NE;
      const int qi[3] = {q % E, (q / E) % E, q / (E * E)};
      double xi[3], x[3], J[9], Ji[9], w = 1.0, ex[DIM + 1];
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        xi[d] = xe[qi[d]];
        w *= we[qi[d]];
      }
      multilinear_point<DIM>(s_V[c], xi, x);
      const double jxw = fabs(multilinear_jacobian<DIM>(s_V[c], xi, J, Ji)) * w;
      modes_all<DIM>(modes, s_amp, x, ex);
      const double d = out[i] - ex[DIM];
      err += d * d * jxw;
    }
  }
  block_partials<1>(&err, red, partial);
}

}  // namespace exw
