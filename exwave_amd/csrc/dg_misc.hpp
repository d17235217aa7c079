// dg_misc.hpp -- setup and norm kernels: initial projection, L2 errors, energy.
//
// project_initial_field (source/wave_equation_operations.cc:902-935): with the
// Gauss-collocated basis the QGauss(k+1) L2 projection is the value of the
// function at the mapped Gauss points.
// L2 errors (VectorTools::integrate_difference with QGauss(k+2),
// source/explicit_wave.cc:452-496): per cell, interpolate to the k+2 Gauss
// points by tensor passes in LDS, compare with the exact modes, reduce per
// workgroup; a second single-group pass sums the partials in a fixed order
// (deterministic).
#pragma once
#include "dg_common.hpp"

namespace exw {

struct DevModes {
  int n_modes;
  double amp[8];
  int m[8][3];
  double rho, c;
};

// The modes' factors that do not depend on the point, per mode and component
// (s_amp in LDS, filled by the group's first lanes; a barrier must follow).
template <int DIM>
__device__ __forceinline__ void modes_factors(const DevModes &e, double t,
                                              double (*s_amp)[DIM + 1]) {
  constexpr double PI = 3.14159265358979323846;
  const int k = threadIdx.x / (DIM + 1), comp = threadIdx.x % (DIM + 1);
  if (k >= e.n_modes) return;
  double mm = 0.0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) mm += double(e.m[k][d]) * e.m[k][d];
  mm = sqrt(mm);
  const double omega = e.c * PI * mm;
  s_amp[k][comp] = comp == DIM ? e.amp[k] * cos(omega * t)
                               : -e.amp[k] * e.m[k][comp] / (e.rho * e.c * mm) * sin(omega * t);
}

// All components of the modes at x: one sine and cosine per mode and direction
// serve every component.
template <int DIM>
__device__ __forceinline__ void modes_all(const DevModes &e, const double (*s_amp)[DIM + 1],
                                          const double *x, double *val) {
  constexpr double PI = 3.14159265358979323846;
#pragma unroll
  for (int f = 0; f <= DIM; ++f) val[f] = 0.0;
  for (int k = 0; k < e.n_modes; ++k) {
    double sn[DIM], cs[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) sincos(e.m[k][d] * PI * x[d], &sn[d], &cs[d]);
#pragma unroll
    for (int f = 0; f <= DIM; ++f) {
      double v = s_amp[k][f];
#pragma unroll
      for (int d = 0; d < DIM; ++d) v *= d != f ? sn[d] : cs[d];
      val[f] += v;
    }
  }
}

template <int DIM, int K>
__global__ void __launch_bounds__(256)
    project_kernel(const DevMesh mesh, const double *__restrict__ tab, const DevModes modes,
                   double t, double *__restrict__ dst) {
  using S = Shape<DIM, K>;
  constexpr int N = S::N, ND = S::ND, NF = S::NF;
  __shared__ double s_amp[8][DIM + 1];
  modes_factors<DIM>(modes, t, s_amp);
  __syncthreads();
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (size_t)mesh.n_cells * ND) return;
  const int cell = int(gid / ND), q = int(gid % ND);
  const int qi[3] = {q % N, (q / N) % N, q / (N * N)};
  double xi[3], x[3], val[NF];
#pragma unroll
  for (int d = 0; d < DIM; ++d) xi[d] = tab[TabOff<N>::X + qi[d]];
  multilinear_point<DIM>(mesh.vertices + (size_t)cell * (1 << DIM) * DIM, xi, x);
  modes_all<DIM>(modes, s_amp, x, val);
#pragma unroll
  for (int f = 0; f < NF; ++f) dst[((size_t)cell * NF + f) * ND + q] = val[f];
}

// One tensor pass of the matrix M (NO x NI, row-major, wave-uniform) on COUNT
// tensors in LDS: one task per line, its NI entries read into registers once.
// LO = entries below the direction (already NO-sized), HI = above (still NI).
template <int LO, int HI, int NI, int NO, int COUNT>
__device__ __forceinline__ void line_pass(const double *M, const double *in, double *out) {
  for (int task = threadIdx.x; task < COUNT * LO * HI; task += blockDim.x) {
    const int s = task / (LO * HI), t = task - s * (LO * HI), hi = t / LO, lo = t - hi * LO;
    const double *src = in + s * (LO * HI * NI) + hi * (LO * NI) + lo;
    double *dst = out + s * (LO * HI * NO) + hi * (LO * NO) + lo;
    double x[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) x[i] = src[i * LO];
#pragma unroll
    for (int q = 0; q < NO; ++q) {
      double a = 0.0;
#pragma unroll
      for (int i = 0; i < NI; ++i) a += M[q * NI + i] * x[i];
      dst[q * LO] = a;
    }
  }
}

// Evaluation of cell polynomials (NI points per direction) on a finer tensor
// grid of NO points by tensor passes between two LDS buffers, NFLD fields of a
// cell in rounds of FC fields (as many as keep both buffers within 48 KB),
// CPB small cells at a time.
// Per cell NFLD * sum_d NO^(d+1) NI^(DIM-d) products instead of NO^DIM NI^DIM:
// the L2 errors of 3D k=4, 16^3 cells take 47 us instead of 407 (of which the
// modes' sines, evaluated once per point for all components, are the rest), the
// error of p* 70 instead of 193.
template <int DIM, int NI, int NO, int NFLD>
struct Refine {
  static constexpr int pw(int b, int e) { return e == 0 ? 1 : b * pw(b, e - 1); }
  static constexpr int NDI = pw(NI, DIM), NDO = pw(NO, DIM);
  static constexpr int SA = DIM == 2 ? (NDI > NDO ? NDI : NDO)
                                     : (NDI > NO * NO * NI ? NDI : NO * NO * NI);
  static constexpr int SB = DIM == 2 ? NO * NI : (NDO > NO * NI * NI ? NDO : NO * NI * NI);
  static constexpr int fits(int fc) { return (SA + SB) * fc * 8 <= 48 * 1024; }
  static constexpr int FC = fits(NFLD) ? NFLD : (NFLD % 2 == 0 && fits(2) ? 2 : 1);
  static constexpr int CPB = FC < NFLD || NDO >= 256 ? 1 : 256 / NDO;
  static constexpr int A = SA * FC * CPB, B = SB * FC * CPB;
  // the FC*CPB tensors in a -> the result's buffer (b in 3D, a in 2D);
  // barriers after every pass
  static __device__ __forceinline__ const double *run(const double *M, double *a, double *b) {
    constexpr int C = FC * CPB;
    if constexpr (DIM == 2) {
      line_pass<1, NI, NI, NO, C>(M, a, b);
      __syncthreads();
      line_pass<NO, 1, NI, NO, C>(M, b, a);
      __syncthreads();
      return a;
    } else {
      line_pass<1, NI * NI, NI, NO, C>(M, a, b);
      __syncthreads();
      line_pass<NO, NI, NI, NO, C>(M, b, a);
      __syncthreads();
      line_pass<NO * NO, 1, NI, NO, C>(M, a, b);
      __syncthreads();
      return b;
    }
  }
};

// The sums of NV per-lane values over the 256 lanes, in a fixed order, to
// partial[blockIdx][NV].
template <int NV>
__device__ __forceinline__ void block_partials(const double *v, double (*red)[256],
                                               double *__restrict__ partial) {
#pragma unroll
  for (int k = 0; k < NV; ++k) red[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
#pragma unroll
      for (int k = 0; k < NV; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) partial[blockIdx.x * NV + k] = red[k][0];
}

// errtab: xe[N+1], we[N+1], I[(N+1)*N] (I[q*N+i] = l_i(xe_q))
template <int DIM, int K>
__global__ void __launch_bounds__(256)
    l2_error_kernel(const DevMesh mesh, const double *__restrict__ errtab, const DevModes modes,
                    double t, const double *__restrict__ u, double *__restrict__ partial) {
  using S = Shape<DIM, K>;
  constexpr int N = S::N, ND = S::ND, NF = S::NF;
  constexpr int NE = N + 1;
  using R = Refine<DIM, N, NE, NF>;
  constexpr int NDE = R::NDO, CPB = R::CPB, NVD = (1 << DIM) * DIM;
  __shared__ double red[3][256];
  __shared__ double s_a[R::A], s_b[R::B], s_V[CPB][NVD], s_amp[8][DIM + 1];
  modes_factors<DIM>(modes, t, s_amp);
  double sum[3] = {0.0, 0.0, 0.0};  // |p_h - p|^2, |v_h - v|^2, |p|^2
  const double *xe = errtab, *we = errtab + NE, *I = errtab + 2 * NE;
  for (int c0 = blockIdx.x * CPB; c0 < mesh.n_cells; c0 += gridDim.x * CPB) {
    const int nc = min(CPB, mesh.n_cells - c0);
    __syncthreads();  // the points of the cells before have been read
    for (int i = threadIdx.x; i < nc * NVD; i += 256)
      s_V[i / NVD][i % NVD] = mesh.vertices[(size_t)c0 * NVD + i];
    static_for<NF / R::FC>([&](auto R_) __attribute__((always_inline)) {
      constexpr int f0 = decltype(R_)::value * R::FC;
      if constexpr (f0 > 0) __syncthreads();  // the round before has been read
      for (int i = threadIdx.x; i < CPB * R::FC * ND; i += 256) {
        const int c = i / (R::FC * ND);
        s_a[i] = c < nc ? u[((size_t)(c0 + c) * NF + f0) * ND + (i - c * (R::FC * ND))] : 0.0;
      }
      __syncthreads();
      const double *out = R::run(I, s_a, s_b);
#pragma unroll 1
      for (int i = threadIdx.x; i < nc * NDE; i += 256) {
        const int c = i / NDE, q = i - c * NDE;
        const int qi[3] = {q % NE, (q / NE) % NE, q / (NE * NE)};
        double xi[3], x[3], J[9], Ji[9], w = 1.0, ex[NF];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          xi[d] = xe[qi[d]];
          w *= we[qi[d]];
        }
        multilinear_point<DIM>(s_V[c], xi, x);
        const double jxw = fabs(multilinear_jacobian<DIM>(s_V[c], xi, J, Ji)) * w;
        modes_all<DIM>(modes, s_amp, x, ex);
#pragma unroll
        for (int f = 0; f < R::FC; ++f) {
          const double dl = out[(c * R::FC + f) * NDE + q] - ex[f0 + f];
          sum[f0 + f == DIM ? 0 : 1] += dl * dl * jxw;
          if (f0 + f == DIM) sum[2] += ex[DIM] * ex[DIM] * jxw;
        }
      }
    });
  }
  block_partials<3>(sum, red, partial);
}

template <int DIM, int K>
__global__ void __launch_bounds__(256)
    energy_kernel(const DevMesh mesh, const double *__restrict__ tab,
                  const double *__restrict__ u, double *__restrict__ partial) {
  using S = Shape<DIM, K>;
  constexpr int N = S::N, ND = S::ND, NF = S::NF;
  __shared__ double red[1][256];
  double E = 0.0;
  const size_t total = (size_t)mesh.n_cells * ND;
  for (size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x; gid < total;
       gid += (size_t)gridDim.x * blockDim.x) {
    const int cell = int(gid / ND), q = int(gid % ND);
    const int qi[3] = {q % N, (q / N) % N, q / (N * N)};
    double xi[3], J[9], Ji[9], w = 1.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      xi[d] = tab[TabOff<N>::X + qi[d]];
      w *= tab[TabOff<N>::W + qi[d]];
    }
    const double *V = mesh.vertices + (size_t)cell * (1 << DIM) * DIM;
    const double jxw = fabs(multilinear_jacobian<DIM>(V, xi, J, Ji)) * w;
    const double *uc = u + (size_t)cell * NF * ND;
    double v2 = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) v2 += uc[d * ND + q] * uc[d * ND + q];
    const double p = uc[DIM * ND + q];
    const double rho = mesh.rho[cell], c = mesh.speed[cell];
    E += 0.5 * jxw * (rho * v2 + p * p / (rho * c * c));
  }
  block_partials<1>(&E, red, partial);
}

// estimate_error (source/wave_equation_operations.cc:871-898): per cell
// err = sqrt(int_K |grad p_h - v_t|^2) at the QGauss(k+1) points (the nodes),
// dudt = apply(sol).  One lane per node; the cell's sum is taken by its first
// lane in node order (deterministic).
template <int DIM, int K>
__global__ void __launch_bounds__((Shape<DIM, K>::BLOCK))
    estimate_error_kernel(const DevMesh mesh, const double *__restrict__ tab,
                          const double *__restrict__ sol, const double *__restrict__ dudt,
                          double *__restrict__ err) {
  using S = Shape<DIM, K>;
  using TO = TabOff<S::N>;
  constexpr int N = S::N, ND = S::ND, NF = S::NF, CPB = S::CPB;
  __shared__ double s_p[CPB][ND];
  __shared__ double s_e[CPB][ND];
  __shared__ double s_tab[TO::SIZE];
  const int tid = threadIdx.x, lc = tid / ND, q = tid - lc * ND;
  const int cell = blockIdx.x * CPB + lc;
  const bool active = lc < CPB && cell < mesh.n_cells;
  for (int i = tid; i < TO::SIZE; i += blockDim.x) s_tab[i] = tab[i];
  if (active) s_p[lc][q] = sol[((size_t)cell * NF + DIM) * ND + q];
  __syncthreads();
  if (active) {
    const int qi[3] = {q % N, (q / N) % N, DIM == 3 ? q / (N * N) : 0};
    double xi[DIM], J[DIM * DIM], Ji[DIM * DIM], w = 1.0, gref[DIM];
#pragma unroll
    for (int e = 0; e < DIM; ++e) {
      xi[e] = s_tab[TO::X + qi[e]];
      w *= s_tab[TO::W + qi[e]];
      const int se = pow_n<N>(e), q0 = q - qi[e] * se;
      double g = 0.0;
#pragma unroll
      for (int m = 0; m < N; ++m) g += s_tab[TO::D + qi[e] * N + m] * s_p[lc][q0 + m * se];
      gref[e] = g;
    }
    const double det =
        multilinear_jacobian<DIM>(mesh.vertices + (size_t)cell * (1 << DIM) * DIM, xi, J, Ji);
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      double gp = 0.0;
#pragma unroll
      for (int e = 0; e < DIM; ++e) gp += Ji[e * DIM + i] * gref[e];
      const double dl = gp - dudt[((size_t)cell * NF + i) * ND + q];
      s += dl * dl;
    }
    s_e[lc][q] = s * fabs(det) * w;
  }
  __syncthreads();
  if (active && q == 0) {
    double s = 0.0;
    for (int i = 0; i < ND; ++i) s += s_e[lc][i];
    err[cell] = sqrt(s);
  }
}

// u += I b on the pressure of the source cells selected by `sel` (bit s:
// source cell s): the time-integrated point source, one lane per node
static __global__ void __launch_bounds__(256)
    source_add_kernel(double *__restrict__ u, const int *__restrict__ cells,
                      const double *__restrict__ b, int n_src, int nd, int dim, unsigned sel,
                      double I) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = i / nd, q = i - s * nd;
  if (s >= n_src || !((sel >> s) & 1u)) return;
  u[((size_t)cells[s] * (dim + 1) + dim) * nd + q] += I * b[(size_t)s * nd + q];
}

// fixed-order final sum of `n` partial vectors of width `w`
static __global__ void __launch_bounds__(256)
    sum_partials_kernel(const double *__restrict__ partial, int n, int w, double *__restrict__ out) {
  __shared__ double red[256];
  for (int k = 0; k < w; ++k) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += partial[i * w + k];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
      if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[k] = red[0];
    __syncthreads();
  }
}

}  // namespace exw
