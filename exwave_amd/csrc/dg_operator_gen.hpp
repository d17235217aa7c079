// dg_operator_gen.hpp -- fused operator + RK epilogue for general multilinear
// cells (every degree whose cell fits a workgroup of one lane per node), and the rule
// by which a launch runs it or a kernel with one lane per node (GenForms).
//
// The arithmetic is that of evaluate_cell / evaluate_inner_face /
// evaluate_boundary_face (source/wave_equation_operations.cc:424-629) on a
// cell whose Jacobian varies from point to point:
//   dv/dt = -rho^-1 J^-T grad_xi p            + lifting of the face terms
//   dp/dt = weak div of rho c^2 w det(J) J^-1 v + lifting of the face terms
// followed by the inverse mass 1/(w det J) (collocated Gauss basis) and the
// RK epilogue.  Lanes alternate between flat copies, the cells' lines (a line of
// direction d owns the two face points at its ends) and the cells' nodes:
//   A (flat): the cells and all their neighbours in 16-byte loads; the cells go
//     to LDS, the neighbours follow through one LDS buffer direction by
//     direction, where (lane = line) the traces at the line's two ends are
//     summed; a few lanes form the Jacobian column coefficients and the faces'
//     linear flux maps meanwhile;
//   B (lane = line): the line's nodes once from LDS: the reference gradient of
//     p along it and the own traces at both ends; the Jacobian column along
//     the line (constant on it) and the cofactor rows at its ends (Nanson:
//     det J J^-T e_d = j_{d+1} x j_{d+2}), the fluxes of both face points;
//   C (lane = node): the Jacobian from the three line columns through the
//     node, the pressure gradient, the test-gradient values rho c^2 w det J
//     (J^-1 v);
//   D (lane = line): the weak derivative along the line with the lifted
//     pressure fluxes of its two ends (still in registers);
//   E (lane = node): velocity lifting, inverse mass, dv/dt and dp/dt over the
//     cell's fields in LDS; (flat): the epilogue, 16 bytes at a time.
// No atomics.
//
// What bounds it: the address unit takes a quad of lanes per clock, so 8-byte
// loads and stores move 32 B per clock and CU and the neighbours' six cells at
// that width were a third of the time (3D k=4, 33x31x29 cells: 183 us with one
// lane per node and 8-byte gathers along the lines; 118 with the gathers left
// out, 97 for the streaming alone).  Copied flat, 16 bytes per lane, every
// byte costs half; the line form cuts the LDS traffic of the node form (every
// derivative and trace re-read N values per point) to a third.  Same workload:
// 143 us; 3D k=6 32^3 with the FP32 operator 626 -> 369 us; 3D k=2 45^3 200 ->
// 104; 2D k=5 340^2 201 -> 118.
#pragma once
#include <type_traits>

#include "dg_common.hpp"
#include "gauss_cx.hpp"

namespace exw {

// The lanes of a group: WPD waves per direction hold its lines, so that the
// direction is uniform over a wave and compile-time inside it (strides and
// cofactors are constants); cells of fewer than 64 face points per direction
// share the waves.  In the node phases lane l takes nodes l + j BLOCK, j < NPL,
// of the group's CPB cells, in the flat copies entry pairs likewise.  Group
// sizes as measured: half the cells per group lost 20-30 % at 3D k = 2..4 (part-
// filled line waves), twice as many 12-60 % (fewer groups per CU); 3D k=6 lost
// 40 % with 384 instead of its three line waves, 3D k=8 the same with six waves
// instead of eight (two groups per CU: unevenly spread over the SIMDs).
// SMALL: a wave's worth of nodes per group instead of a wave of lines per direction,
// for launches of few groups (GenSmall).
template <int DIM, int K, bool SMALL = false>
struct GenShape {
  static constexpr int N = K + 1;
  static constexpr int ND = DIM == 2 ? N * N : N * N * N;
  static constexpr int NT = DIM == 2 ? N : N * N;
  static constexpr int NF = DIM + 1;
  static constexpr int NFACE = 2 * DIM;
  static constexpr int WPD = (NT + 63) / 64;
  static constexpr int CPB = SMALL ? (ND >= 64 ? 1 : 64 / ND) : (NT >= 64 ? 1 : 64 / NT);
  static constexpr int LINE_LANES = DIM * WPD * 64;
  static constexpr int NODES = CPB * ND;
  // nodes beyond the line waves get waves of their own up to 256 lanes (512 for
  // the cells of 512 nodes and more); degree 1 takes 256 for its copies and its
  // few-lane tasks, which outnumber its nodes (3D 113 -> 93 us, 60^3 cells)
  static constexpr int NODE_CAP = ND >= 512 ? 512 : 256;
  static constexpr int NODE_LANES =
      NODES >= NODE_CAP || (K == 1 && !SMALL) ? NODE_CAP : (NODES + 63) / 64 * 64;
  static constexpr int BLOCK = K == 6 && DIM == 3 ? LINE_LANES
                               : LINE_LANES > NODE_LANES ? LINE_LANES : NODE_LANES;
  static constexpr int NPL = (NODES + BLOCK - 1) / BLOCK;
  // node fields in LDS with rows of odd length (x lines free of bank conflicts)
  static constexpr int NX = N % 2 ? N : N + 1;
  static constexpr int NDP = ND / N * NX;
  // the flat copies: PPC pairs of entries per cell, NPP per lane, all three
  // directions' neighbours in flight where their registers allow
  static constexpr int PPC = (NF * ND + 1) / 2, NPP = (CPB * PPC + BLOCK - 1) / BLOCK;
  static constexpr bool PREFETCH_ALL = NPP <= 2;
  // waves per SIMD to hold the registers to, one or two below the compiler's
  // own choice (no vector register spills; the matrices' constants spill scalar
  // registers to vector lanes, 8 to 30 at k=5, 100 to 800 from 2D k=8 and 3D k=8 on)
  static constexpr int MIN_WAVES = DIM == 3 ? (K <= 5 ? 5 : 4) : (K <= 3 ? 6 : 4);
};

// Whether a launch over n cells runs the small groups: while the full ones are few
// its time is that of one group from start to end, which a smaller one finishes
// earlier; with more cells the small groups' emptier lanes cost more.  Degrees whose
// small launches run this kernel (GenForms).  2D, ten launches in us, small against
// full groups: k=4 506 cells (43 full groups) 54.0 against 64.8, k=5 361 cells (37)
// 56 against 71; near 230 full groups the small ones take 77 and 82, the full ones
// 68 and 76: the lines cross between 100 and 160 full groups.  3D, us per RK stage,
// full / small, FP64 and FP32: k=2 125 cells (18 groups) 6.3 / 5.8, 6.1 / 5.7, 729 (104)
// 6.4 / 6.3, 6.2 / 6.0, 1331 (190) 6.6 / 7.3, 6.4 / 6.6; k=3 125 (31) 7.0 / 6.2, 6.7 /
// 5.9, 512 (128) 7.3 / 6.7, 6.9 / 6.1, 1000 (250) 7.7 / 8.5, 7.4 / 7.5; k=4 216 (108)
// 7.4 / 7.0, 7.1 / 6.8, 343 (172) 7.8 / 8.1, 7.4 / 7.4.  2D FP32 k=4 400 cells (33) 6.4 /
// 5.6, k=5 361 (37) 7.0 / 5.8.  2D k=3: within 4 % of each other below the line.
template <int DIM, int K>
struct GenSmall {
  static constexpr bool EXISTS = (DIM == 2 ? K >= 3 && K <= 5 : K >= 2) &&
                                 GenShape<DIM, K>::CPB > GenShape<DIM, K, true>::CPB;
  static bool pays(int n) { return EXISTS && n < 128 * GenShape<DIM, K>::CPB; }
};

// Which launches over general cells run the kernels with one lane per node
// (dg_operator_gen_node_kernel, below 48 nodes dg_operator_kernel) instead of this
// file's line form: those over from <= n < to cells; `single`: the launch only writes
// the operator's result.  One output that accumulates (the last stage of a time step,
// the sweep of an ADER step) goes by the two-output line: it costs the line form no more
// than its neighbours in the step, and the node form 3 to 15 % (ADER step, us, node /
// line form: FP64 2D k=1 332929 cells 67.6 / 62.7, k=3 18769 22.8 / 20.4, k=5 8281 35.9 /
// 31.2).  The line form's matrices are constants of its unrolled code, which every
// launch fetches once, and its chain of barriers is longer: small launches wait for
// both, and at 2D k >= 9 the code leaves the instruction cache.  The node forms read
// their tables from LDS in short loops.  us per RK stage (two outputs) and, behind
// the bar, per plain sweep, node form / line form:
//   FP64 2D k=1 58212 cells 10.5 / 11.3 (just before the node form's 64-cell groups need a
//        second round of the CUs), 332929 60 / 50 | 41 / 43;  k=3 11449 8.1 / 8.0 | 5 %
//        lost;  k=4 676 6.1 / 5.5, 1600 6.0 / 6.4, 3969 6.9 / 7.8, 7396 10.9 / 9.4;  k=5 2809 8.8
//        / 8.7 | 21 % lost, 9216 15.8 / 12.1;  k=6 2025 7.4 / 8.8, 6724 13.5 / 12.4;
//        k=7 2916 9.2 / 9.6, 5184 12.9 / 11.0;  k=8 2304 10.9 / 11.7, 4096 15.7 /
//        13.5;  k=9 1849 9.7 / 12.0, 3364 14.6 / 13.6;  k=10 841 7.9 / 12.4, 5476 24.7
//        / 29.3, 21904 93 / 91 | 71 / 83;  k=11 1296 11.7 / 13.3, 4624 28.0 / 29.5,
//        18496 107 / 95 | 86 / 84;  k=12 100 6.5 / 14.0, 7921 52.0 / 52.6, 15876 104 /
//        94 | 82 / 88
//     3D k=5 343 9.0 / 10.1, 2197 26.0 / 26.2, 4913 55.7 / 51.4 | 27000 220 / 225; k=6
//       343 10.8 / 11.4, 729 17.1 / 14.4;  k=7 216 10.3 / 12.7, 512 18.9 / 17.1; k=8
//       729 32.1 / 34.6, 2744 113 / 104 | 101 / 100;  k=9 5832 408 / 412
//   FP32 2D k=3 11449 6.9 / 7.1 | 6.2 / 6.7;  k=4 1600 5.9 / 6.4, 7396 7.8 / 8.5,
//        13225 11.7 / 10.2;  k=5 1089 6.1 / 6.5, 5041 8.0 / 8.3, 9216 13.0 / 10.0;
//        k=6 2025 7.1 / 8.2, 6724 12.9 / 10.4;  k=7 1600 7.0 / 8.0, 5184 12.4 / 10.0;
//        k=8 2304 8.4 / 14.3, 8281 26.1 / 25.6 | 17 % lost, 32761 96 / 73 | 69 / 66;
//        k=9 13225 44.1 / 45.2, 26569 86 / 79 | 61 / 71;  k=10 21904 86 / 89, 66049
//        266 / 257 | 176 / 224;  k=11 9216 49 / 51, 18496 95 / 88 | 73 / 80;  k=12 36
//        6.1 / 19.8, 47524 281 / 286
//     3D k=5 729 9.8 / 9.9, 1000 12.1 / 11.2 | 13 % lost, 2197 23.6 / 21.6;  k=6 343
//       9.6 / 10.3, 729 16.4 / 12.7;  k=7 1728 39 / 41, 4096 86 / 82;  k=8 729 28.7 /
//       29.7, 1331 50.8 / 49.6;  k=9 216 16.2 / 18.5, 512 29.3 / 27.4
// From a sweep in steps of 12 % of the cells, line form's time over the node form's just
// below and above the line: FP64 2D k=4 5112 cells 1.15, 5700 0.78 (one round
// of the node form's groups ends between), k=7 3248 1.02, 4095 0.96, k=8 2304 1.07, 2915
// 0.97, k=9 2304 1.05, 2915 0.95, 3D k=7 252 1.22, 288 0.96, k=8 1573 1.02, 1728 0.97;
// FP32 2D k=8 9024 1.01, 10100 0.93,
// k=9 14160 1.02, 15875 0.92, k=11 9024 1.05, 10100 0.96, 3D k=8 810 1.04, 1000 0.96, k=9 252
// 1.16, 441 0.95.  FP32 2D k=8 and 9 just below one full round of the line form's groups: 5700
// 1.02, 6399 0.93, 7140 0.86, 8010 1.00; 5112 1.05, 5700 0.95, 6399 1.21.  Plain sweeps: FP64 2D
// k=1 22201 0.96, 27889 1.04, k=3 15875 1.09, 17689 0.93, k=5 5112 1.07, 5700 0.85, k=7 3660
// 1.00, 5112 0.92, k=11 11236 1.00, 14160 0.99; FP32 k=3 15875 1.08, 17689 0.89, k=5 5112 1.07,
// 5700 0.86, k=8 12656 1.04, 14160 0.97.
template <int DIM, int K, typename Number>
struct GenForms {
  static constexpr int NEVER = 1 << 30;
  static constexpr bool D = std::is_same_v<Number, double>;
  static constexpr int from(bool single) {
    if constexpr (DIM == 2) {
      if (K == 1) return D ? (single ? 24000 : 50000) : NEVER;
      if (K == 3) return single ? 6000 : NEVER;
      if (K == 4) return 1200;
      if (K == 5) return D && !single ? NEVER : 600;
      return K >= 6 ? 0 : NEVER;
    }
    return K >= 5 ? 0 : NEVER;
  }
  static constexpr int to(bool single) {
    constexpr int N = NEVER;
    // [FP64 two outputs, FP64 single, FP32 two outputs, FP32 single][degree]
    constexpr int to_2d[4][13] = {
        {0, 65536, 0, 0, 5121, 0, 5500, 3500, 2600, 2500, 12000, 9000, 9000},
        {0, N, 0, 16385, 5121, 5121, 5500, 3700, 2500, 2500, N, 12000, N},
        {0, 0, 0, 0, 11000, 5121, 4096, 3584, 9100, 14500, 32768, 9800, N},
        {0, 0, 0, 16385, 11000, 5121, 4096, 3584, 13000, N, N, N, N}};
    constexpr int to_3d[4][10] = {{0, 0, 0, 0, 0, 2500, 576, 257, 1600, N},
                                  {0, 0, 0, 0, 0, N, 576, 257, 2800, N},
                                  {0, 0, 0, 0, 0, 800, 576, 3500, 950, 380},
                                  {0, 0, 0, 0, 0, 2000, 576, 4800, 1152, 280}};
    const int row = (D ? 0 : 2) + (single ? 1 : 0);
    if constexpr (DIM == 2) return to_2d[row][K];
    else return to_3d[row][K];
  }
  // launches whose line groups just fill the CUs once (four a CU) stay in the line form
  static constexpr int ROUND =
      DIM == 2 && (K == 8 || K == 9) && !D ? 1024 * GenShape<DIM, K>::CPB : 0;
  // (the node form's offsets into the vectors have 32 bits)
  static bool node(int n, bool single) {
    return n >= from(single) && n < to(single) &&
           (single || n <= ROUND / 8 * 7 || n > ROUND) &&
           uint64_t(n) * (GenShape<DIM, K>::NF * GenShape<DIM, K>::ND) < (uint64_t(1) << 32);
  }
  static constexpr bool NODE_EXISTS = from(false) < to(false) || from(true) < to(true);
};

// Jinv[e*DIM+i] = dxi_e/dx_i of J; returns det J (as multilinear_jacobian)
template <int DIM, typename T>
__device__ __forceinline__ T jacobian_invert(const T *J, T *Jinv) {
  T det;
  if constexpr (DIM == 2) {
    det = J[0] * J[3] - J[1] * J[2];
    const T id = recip(det);
    Jinv[0] = J[3] * id;
    Jinv[1] = -J[1] * id;
    Jinv[2] = -J[2] * id;
    Jinv[3] = J[0] * id;
  } else {
    const T a = J[0], b = J[1], c = J[2], d = J[3], e = J[4], f = J[5], g = J[6], h = J[7],
            k = J[8];
    const T A = e * k - f * h, B = f * g - d * k, C = d * h - e * g;
    det = a * A + b * B + c * C;
    const T id = recip(det);
    Jinv[0] = A * id;
    Jinv[3] = B * id;
    Jinv[6] = C * id;
    Jinv[1] = (c * h - b * k) * id;
    Jinv[4] = (a * k - c * g) * id;
    Jinv[7] = (b * g - a * h) * id;
    Jinv[2] = (b * f - c * e) * id;
    Jinv[5] = (c * d - a * f) * id;
    Jinv[8] = (a * e - b * d) * id;
  }
  return det;
}

// 1/sqrt(x): the hardware estimate refined by Newton steps, as recip
__device__ __forceinline__ double recip_sqrt(double x) {
  double y = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int it = 0; it < 2; ++it) y = __builtin_fma(0.5 * y, __builtin_fma(-x * y, y, 1.0), y);
  return y;
}
__device__ __forceinline__ float recip_sqrt(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  return __builtin_fmaf(0.5f * y, __builtin_fmaf(-x * y, y, 1.0f), y);
}

// 1/|c| and |c|.  Low-degree 3D cells in FP32 take their length out of the square by a
// power of two (exact), so that cells of 3e-11 or 3e10 have an area as those of 1 do.
template <int DIM, int K, typename T>
__device__ __forceinline__ void norm_of(const T *c, T &inv, T &len) {
  T n2 = T(0);
  if constexpr (DIM == 3 && K <= 2 && std::is_same_v<T, float>) {
    const int e = __builtin_amdgcn_frexp_expf(fmaxf(fmaxf(fabsf(c[0]), fabsf(c[1])), fabsf(c[2])));
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      const float x = __builtin_amdgcn_ldexpf(c[i], -e);
      n2 += x * x;
    }
    const float y = recip_sqrt(n2);
    inv = __builtin_amdgcn_ldexpf(y, -e);
    len = __builtin_amdgcn_ldexpf(n2 * y, e);
  } else {
#pragma unroll
    for (int i = 0; i < DIM; ++i) n2 += c[i] * c[i];
    inv = recip_sqrt(n2);
    len = n2 * inv;
  }
}

template <int DIM, int K, typename Number, bool SMALL = false>
__global__ void __launch_bounds__((GenShape<DIM, K, SMALL>::BLOCK))
    __attribute__((amdgpu_waves_per_eu(GenShape<DIM, K, SMALL>::MIN_WAVES)))
    dg_operator_gen_kernel(const DevMesh mesh, const double *__restrict__ src,
                           const Epilogue epi) {
  using S = GenShape<DIM, K, SMALL>;
  constexpr int N = S::N, ND = S::ND, NT = S::NT, NF = S::NF, NFACE = S::NFACE;
  constexpr int BLOCK = S::BLOCK, CPB = S::CPB, NX = S::NX, NDP = S::NDP, NV = 1 << DIM;
  constexpr int WPD = S::WPD, NPL = S::NPL, NODES = S::NODES;
  constexpr int PPC = S::PPC, NPP = S::NPP;
  typedef double dbl2 __attribute__((ext_vector_type(2)));
  typedef dbl2 dbl2u __attribute__((aligned(8)));
  constexpr const CartConst<N> &T = CartTable<N>::value;

  __shared__ Number s_u[CPB][NF][NDP];
  // first the staged neighbour fields of one direction's two faces, then
  // (phases B to E) the arrays below
  struct Work {
    // by direction: the gradient of p along it (B), the test-gradient values
    // (C), the lines' dp/dt shares (D), each over its own entries
    Number g[CPB][DIM][NDP];
    Number F[CPB][NFACE][DIM][NT];  // the velocity fluxes of the face points
    Number jd[CPB][DIM][DIM][NT];   // per line the Jacobian column along it
  };
  __shared__ union {
    Number nb[2][CPB][NF][NDP];
    Work w;
  } s_v;
  auto &s_g = s_v.w.g;
  auto &s_F = s_v.w.F;
  auto &s_jd = s_v.w.jd;
  __shared__ Number s_jc[CPB][DIM][1 << (DIM - 1)][DIM];
  __shared__ Number s_fc[CPB][NFACE][8];       // the faces' flux maps
  __shared__ Number s_x[N], s_w[N], s_l[2][N];

  const int tid = threadIdx.x;
  const int c0 = xcd_remap(blockIdx.x, gridDim.x) * CPB;
  // (a slot past the last cell repeats it and stores nothing)
  auto cell_of = [&](int lc) {
    if constexpr (CPB == 1) return c0;
    return min(c0 + lc, mesh.n_cells - 1);
  };
  if constexpr (CPB == 1)
    if (epi.cell_scale && epi.cell_scale[c0] == 0.0) return;  // uniform over the group

  // the lane's line: direction dir (uniform over the wave), cell slot, line t
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dir = wave / WPD;
  const int li = tid - dir * (WPD * 64);
  static_assert(NF * ND <= 4096 && NPP * BLOCK <= 4096, "small_div's range");
  const int lcB = CPB == 1 ? 0 : small_div<NT>(li), t = li - lcB * NT, t0 = small_mod<N>(t),
            t1 = small_div<N>(t);
  const bool line_ok = dir < DIM && (CPB == 1 ? t < NT : lcB < CPB);
  // f(direction) at compile time, for the waves that hold lines
  auto lines = [&](auto f) __attribute__((always_inline)) {
    if (!line_ok) return;
    if (dir == 0) f(std::integral_constant<int, 0>{});
    else if (dir == 1) f(std::integral_constant<int, 1>{});
    else if constexpr (DIM == 3) f(std::integral_constant<int, 2>{});
  };
  // a line's first node and stride with rows of R entries (N in memory, NX in LDS)
  auto line_base = [&](auto D_, int R) __attribute__((always_inline)) {
    constexpr int d = decltype(D_)::value;
    if constexpr (DIM == 2) return d == 0 ? t * R : t;
    else return d == 0 ? t0 * R + t1 * R * N : (d == 1 ? t0 + t1 * R * N : t0 + t1 * R);
  };

  // ---------------- A ----------------
  // the few-lane tasks (a face's flux map, a Jacobian coefficient), from the
  // group's last lanes down (where a wave without lines is, if any): their
  // loads first, ahead of the cells' own, finished after those are issued
  constexpr int NT1 = CPB * NFACE, NT2 = CPB * DIM * DIM, NTASK = (NT1 + NT2 + BLOCK - 1) / BLOCK;
  double tv[NTASK][NV / 2][2];
  int tnb[NTASK];
#pragma unroll
  for (int j = 0; j < NTASK; ++j) {
    const int r = BLOCK - 1 - tid + j * BLOCK;
    tnb[j] = -1;
    if (r < NT1) {
      const int lc = r / NFACE, cell = cell_of(lc);
      tnb[j] = mesh.neighbor[(size_t)cell * NFACE + (r - lc * NFACE)];
      tv[j][0][0] = mesh.rho[cell];
      tv[j][0][1] = mesh.speed[cell];
    } else if (r < NT1 + NT2) {
      const int r2 = r - NT1, lc = r2 / (DIM * DIM), ei = r2 - lc * (DIM * DIM), e = ei / DIM;
      const double *V = mesh.vertices + (size_t)cell_of(lc) * NV * DIM + ei % DIM;
      const int a = e == 0 ? 1 : 0, b = e == 2 ? 1 : 2;  // the other coordinates, ascending
#pragma unroll
      for (int v = 0; v < NV / 2; ++v) {
        const int v0 = ((v & 1) << a) | (DIM == 3 ? ((v >> 1) << b) : 0);
        tv[j][v][0] = V[v0 * DIM];
        tv[j][v][1] = V[(v0 | (1 << e)) * DIM];
      }
    }
  }
  // the group's cells and all their neighbours, copied as flat pairs of entries
  // (boundary and hanging faces read the cell itself: their flux maps ignore
  // the values)
  dbl2 own[NPP], nbv[NPP][NFACE];
  const double *un[NPP][NFACE], *un0[NPP];
  int dst[NPP];  // the pair's place in a [CPB][NF][NDP] LDS array; -1: none
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    const int p = tid + j * BLOCK, lc = CPB == 1 ? 0 : min(small_div<PPC>(p), CPB - 1);
    int e = 2 * (p - lc * PPC);
    const bool ok = e < NF * ND;
    if (!ok) e = NF * ND - 2;
    if ((NF * ND) % 2 && e == NF * ND - 1) e = NF * ND - 2;  // (the last pair overlaps)
    dst[j] = ok ? lc * (NF * NDP) + (NX == N ? e : e + small_div<N>(e)) : -1;
    const int cell = cell_of(lc);
    const double *uc = src + (size_t)cell * (NF * ND) + e;
#pragma unroll
    for (int f = 0; f < NFACE; ++f) {
      const int nb = mesh.neighbor[(size_t)cell * NFACE + f];
      un[j][f] = src + (size_t)(nb >= 0 ? nb : cell) * (NF * ND) + e;
    }
    un0[j] = uc;
    __builtin_memcpy(&own[j], uc, 16);
  }
  auto load_faces = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NPP; ++j)
#pragma unroll
      for (int s = 0; s < 2; ++s) __builtin_memcpy(&nbv[j][2 * d + s], un[j][2 * d + s], 16);
  };
  auto put2 = [&](Number *b, int j, dbl2 v) __attribute__((always_inline)) {
    if (dst[j] < 0) return;
    // (rows of odd N end between the two entries; the LDS rows are then contiguous)
    b[dst[j]] = Number(v.x);
    b[dst[j] + 1] = Number(v.y);
  };
#pragma unroll
  for (int d = 0; d < (S::PREFETCH_ALL ? DIM : 1); ++d) load_faces(d);
  double tm[NTASK][2];
#pragma unroll
  for (int j = 0; j < NTASK; ++j) {
    const int r = BLOCK - 1 - tid + j * BLOCK;
    if (r < NT1) {
      const int nb = tnb[j] >= 0 ? tnb[j] : cell_of(r / NFACE);
      tm[j][0] = mesh.rho[nb];
      tm[j][1] = mesh.speed[nb];
    }
  }
#pragma unroll
  for (int j = 0; j < NTASK; ++j) {
    const int r = BLOCK - 1 - tid + j * BLOCK;
    if (r >= NT1 && r < NT1 + NT2) {
      const int r2 = r - NT1, lc = r2 / (DIM * DIM), ei = r2 - lc * (DIM * DIM);
      double D[NV / 2];
#pragma unroll
      for (int v = 0; v < NV / 2; ++v) D[v] = tv[j][v][1] - tv[j][v][0];
      Number(*c)[DIM] = s_jc[lc][ei / DIM];
      const int i = ei % DIM;
      c[0][i] = Number(D[0]);
      c[1][i] = Number(D[1] - D[0]);
      if constexpr (DIM == 3) {
        c[2][i] = Number(D[2] - D[0]);
        c[3][i] = Number((D[3] - D[2]) - (D[1] - D[0]));
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NPP; ++j) put2(&s_u[0][0][0], j, own[j]);
  if (tid < N) {
    s_x[tid] = Number(T.x[tid]);
    s_w[tid] = Number(T.w[tid]);
    s_l[0][tid] = Number(T.L[tid]);
    s_l[1][tid] = Number(T.L[N + tid]);
  }
#pragma unroll
  for (int j = 0; j < NTASK; ++j) {
    const int r = BLOCK - 1 - tid + j * BLOCK;
    if (r < NT1) {
      const int lc = r / NFACE, f = r - lc * NFACE;
      double a[4], b[4];
      flux_matrix<double>(tv[j][0][0], tv[j][0][1], tm[j][0], tm[j][1], tnb[j] >= 0 ? 0 : -tnb[j],
                          a, b);
      // a hanging face contributes nothing here (nc_face_kernel adds it)
      const double on = tnb[j] == -NC_BID ? 0.0 : 1.0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s_fc[lc][f][i] = Number(on * a[i]);
        s_fc[lc][f][4 + i] = Number(on * b[i]);
      }
    }
  }
  // direction by direction through LDS: the neighbours' traces at the ends of
  // its lines, all fields
  Number um[2][NF];
  static_for<DIM>([&](auto R_) __attribute__((always_inline)) {
    constexpr int r = decltype(R_)::value, lsd = r == 0 ? 1 : (r == 1 ? NX : NX * N);
    constexpr const CartConst<N> &T = CartTable<N>::value;
#pragma unroll
    for (int j = 0; j < NPP; ++j)
#pragma unroll
      for (int s = 0; s < 2; ++s) put2(&s_v.nb[s][0][0][0], j, nbv[j][2 * r + s]);
    if constexpr (!S::PREFETCH_ALL && r + 1 < DIM) load_faces(r + 1);
    __syncthreads();
    if (line_ok && dir == r) {
      const int lbase = line_base(R_, NX);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          Number a = Number(0);
#pragma unroll
          for (int i = 0; i < N; ++i)
            a += Number(T.L[(1 - s) * N + i]) * s_v.nb[s][lcB][f][lbase + i * lsd];
          um[s][f] = a;
        }
    }
    __syncthreads();
  });

  // ---------------- B: lines ----------------
  Number fp[2] = {Number(0), Number(0)};  // the pressure fluxes of the line's ends
  lines([&](auto D_) __attribute__((always_inline)) {
    constexpr int d = decltype(D_)::value, lsd = d == 0 ? 1 : (d == 1 ? NX : NX * N);
    constexpr const CartConst<N> &T = CartTable<N>::value;
    const int lbase = line_base(D_, NX);
    Number up[2][NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      Number x[N];
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = s_u[lcB][f][lbase + i * lsd];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        Number a = Number(0);
#pragma unroll
        for (int i = 0; i < N; ++i) a += Number(T.L[s * N + i]) * x[i];
        up[s][f] = a;
      }
      if (f == DIM) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
          Number a = Number(0);
#pragma unroll
          for (int m = 0; m < N; ++m) a += Number(T.D[i * N + m]) * x[m];
          s_g[lcB][d][lbase + i * lsd] = a;
        }
      }
    }
    // geometry: the column along the line, and per end the area vector
    // sg det J J^-T e_d (|.| the area element, direction the outward normal)
    Number jd[DIM], av[2][DIM], wt;
    const Number(*c)[DIM] = s_jc[lcB][d];
    if constexpr (DIM == 3) {
      constexpr int e1 = (d + 1) % 3, e2 = (d + 2) % 3;
      const Number xa = s_x[t0], xb = s_x[t1], xab = xa * xb;  // tangential, ascending
      wt = s_w[t0] * s_w[t1];
#pragma unroll
      for (int i = 0; i < DIM; ++i) jd[i] = c[0][i] + xa * c[1][i] + xb * c[2][i] + xab * c[3][i];
      // column e at xi_d = s and at the tangential coordinate o other than e:
      // (c_0 + x_o c_o) + s (c_d + x_o c_3); of the two coordinates other than
      // e the lower has coefficient 1, the upper 2
      Number j1[2][DIM], j2[2][DIM];
      auto ends = [&](auto E_, auto O_, Number(*j)[DIM]) __attribute__((always_inline)) {
        constexpr int e = decltype(E_)::value, o = decltype(O_)::value;
        constexpr int mo = o < d ? 1 : 2, md = 3 - mo;
        const Number xo = o < e ? xa : xb;
        const Number(*ce)[DIM] = s_jc[lcB][e];
#pragma unroll
        for (int i = 0; i < DIM; ++i) {
          j[0][i] = ce[0][i] + xo * ce[mo][i];
          j[1][i] = j[0][i] + (ce[md][i] + xo * ce[3][i]);
        }
      };
      using E1 = std::integral_constant<int, e1>;
      using E2 = std::integral_constant<int, e2>;
      ends(E1{}, E2{}, j1);
      ends(E2{}, E1{}, j2);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        av[s][0] = j1[s][1] * j2[s][2] - j1[s][2] * j2[s][1];
        av[s][1] = j1[s][2] * j2[s][0] - j1[s][0] * j2[s][2];
        av[s][2] = j1[s][0] * j2[s][1] - j1[s][1] * j2[s][0];
      }
    } else {
      const Number xa = s_x[t];
      wt = s_w[t];
      const Number(*ce)[DIM] = s_jc[lcB][1 - d];
      constexpr Number turn = d == 0 ? Number(1) : Number(-1);
#pragma unroll
      for (int i = 0; i < DIM; ++i) jd[i] = c[0][i] + xa * c[1][i];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        // cofactor row d: (j_1y, -j_1x) of column 1 for d = 0, (-j_0y, j_0x) for d = 1
        av[s][0] = turn * (s ? ce[0][1] + ce[1][1] : ce[0][1]);
        av[s][1] = -turn * (s ? ce[0][0] + ce[1][0] : ce[0][0]);
      }
    }
#pragma unroll
    for (int i = 0; i < DIM; ++i) s_jd[lcB][d][i][t] = jd[i];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      Number det = Number(0), inv, na;
#pragma unroll
      for (int i = 0; i < DIM; ++i) det += av[s][i] * jd[i];
      norm_of<DIM, K>(av[s], inv, na);
      const Number sg = (s != 0) == (det > Number(0)) ? Number(1) : Number(-1);
      Number vp = Number(0), vm = Number(0);
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        vp += up[s][i] * av[s][i];
        vm += um[s][i] * av[s][i];
      }
      vp *= sg * inv;
      vm *= sg * inv;
      const Number *fc = s_fc[lcB][2 * d + s];
      const Number pn = fc[0] * vp + fc[1] * up[s][DIM] + fc[2] * vm + fc[3] * um[s][DIM];
      const Number pp = fc[4] * vp + fc[5] * up[s][DIM] + fc[6] * vm + fc[7] * um[s][DIM];
      const Number k = pn * sg * wt;
#pragma unroll
      for (int i = 0; i < DIM; ++i) s_F[lcB][2 * d + s][i][t] = k * av[s][i];
      fp[s] = pp * na * wt;
    }
  });
  __syncthreads();

  // ---------------- C: nodes ----------------
  Number kv[NPL][DIM], jxw[NPL];
#pragma unroll
  for (int j = 0; j < NPL; ++j) {
    const int n = tid + j * BLOCK, lc = CPB == 1 ? 0 : small_div<ND>(n), q = n - lc * ND;
    const int r = small_div<N>(q), qi[3] = {q - r * N, DIM == 3 ? small_mod<N>(r) : r,
                                             DIM == 3 ? small_div<N>(r) : 0};
    const int ql = NX == N ? q : q + r;
    if (n >= NODES) continue;
    const int cell = cell_of(lc);
    const Number rho = Number(mesh.rho[cell]), cc = Number(mesh.speed[cell]);
    Number J[DIM * DIM], Ji[DIM * DIM], wq = Number(1);
#pragma unroll
    for (int e = 0; e < DIM; ++e) {
      const int tq = DIM == 2 ? qi[1 - e]
                              : (e == 0 ? qi[1] + N * qi[2] : (e == 1 ? qi[0] + N * qi[2]
                                                                      : qi[0] + N * qi[1]));
      wq *= s_w[qi[e]];
#pragma unroll
      for (int i = 0; i < DIM; ++i) J[i * DIM + e] = s_jd[lc][e][i][tq];
    }
    jxw[j] = wq * jacobian_invert<DIM>(J, Ji);
    const Number rho_inv = recip(rho), gw = rho * cc * cc * jxw[j];
    Number v[DIM];
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      kv[j][i] = Number(0);
      v[i] = s_u[lc][i][ql];
    }
#pragma unroll
    for (int e = 0; e < DIM; ++e) {
      const Number g = s_g[lc][e][ql];
      Number a = Number(0);
#pragma unroll
      for (int i = 0; i < DIM; ++i) {
        kv[j][i] += Ji[e * DIM + i] * g;
        a += Ji[e * DIM + i] * v[i];
      }
      s_g[lc][e][ql] = gw * a;
    }
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
      kv[j][i] *= -rho_inv;
      // (not to be sunk past the barriers, which would hold J^-1 over them)
      asm volatile("" : "+v"(kv[j][i]));
    }
  }
  __syncthreads();

  // ---------------- D: lines ----------------
  // the epilogue operands, in flight during the last phases
  dbl2 bv[NPP];
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    bv[j] = dbl2{0.0, 0.0};
    if (epi.b) __builtin_memcpy(&bv[j], epi.b + (un0[j] - src), 16);
  }
  lines([&](auto D_) __attribute__((always_inline)) {
    constexpr int d = decltype(D_)::value, lsd = d == 0 ? 1 : (d == 1 ? NX : NX * N);
    constexpr const CartConst<N> &T = CartTable<N>::value;
    const int lbase = line_base(D_, NX);
    Number x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = s_g[lcB][d][lbase + i * lsd];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      Number a = Number(T.L[i]) * fp[0] + Number(T.L[N + i]) * fp[1];
#pragma unroll
      for (int m = 0; m < N; ++m) a += Number(T.D[m * N + i]) * x[m];
      s_g[lcB][d][lbase + i * lsd] = a;
    }
  });
  __syncthreads();

  // ---------------- E: nodes ----------------
#pragma unroll
  for (int j = 0; j < NPL; ++j) {
    const int n = tid + j * BLOCK, lc = CPB == 1 ? 0 : small_div<ND>(n), q = n - lc * ND;
    const int r = small_div<N>(q), qi[3] = {q - r * N, DIM == 3 ? small_mod<N>(r) : r,
                                             DIM == 3 ? small_div<N>(r) : 0};
    const int ql = NX == N ? q : q + r;
    if (n >= NODES) continue;
    Number fv[DIM], kp = Number(0);
#pragma unroll
    for (int i = 0; i < DIM; ++i) fv[i] = Number(0);
#pragma unroll
    for (int e = 0; e < DIM; ++e) {
      const int tq = DIM == 2 ? qi[1 - e]
                              : (e == 0 ? qi[1] + N * qi[2] : (e == 1 ? qi[0] + N * qi[2]
                                                                      : qi[0] + N * qi[1]));
      kp += s_g[lc][e][ql];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const Number l = s_l[s][qi[e]];
#pragma unroll
        for (int i = 0; i < DIM; ++i) fv[i] += l * s_F[lc][2 * e + s][i][tq];
      }
    }
    const Number ij = recip(jxw[j]);
#pragma unroll
    for (int i = 0; i < DIM; ++i) s_u[lc][i][ql] = kv[j][i] + fv[i] * ij;
    s_u[lc][DIM][ql] = kp * ij;
  }
  __syncthreads();

  // ---------------- epilogue, pairs of entries ----------------
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    const int p = tid + j * BLOCK, lc = CPB == 1 ? 0 : min(small_div<PPC>(p), CPB - 1);
    if (dst[j] < 0 || (CPB > 1 && c0 + lc >= mesh.n_cells)) continue;
    const double cscale = epi.cell_scale ? epi.cell_scale[c0 + lc] : 1.0;
    if (cscale == 0.0) continue;
    const double ea1 = epi.a1 * cscale, ea2 = epi.a2 * cscale, ea3 = epi.a3 * cscale;
    const Number *kk = &s_u[0][0][0] + dst[j];
    const size_t idx = un0[j] - src;
    if ((NF * ND) % 2 && p - lc * PPC == PPC - 1) {
      // the odd last entry alone: its pair's other one belongs to the pair before
      const size_t i = idx + 1;
      const double k = double(kk[1]), o1 = bv[j].y + ea1 * k;
      const double cv = epi.o2 && !epi.o2_from_o1 ? epi.c[i] : o1;
      __builtin_nontemporal_store(o1, epi.o1 + i);
      if (epi.o2) __builtin_nontemporal_store(cv + ea2 * k, epi.o2 + i);
      if (epi.o2 && epi.o3) __builtin_nontemporal_store(cv + ea3 * k, epi.o3 + i);
      continue;
    }
    const dbl2 k = {double(kk[0]), double(kk[1])};
    const dbl2 o1 = bv[j] + ea1 * k;
    dbl2 cv = o1;
    if (epi.o2 && !epi.o2_from_o1) __builtin_memcpy(&cv, epi.c + idx, 16);
    __builtin_nontemporal_store(o1, (dbl2u *)(epi.o1 + idx));
    if (epi.o2) {
      __builtin_nontemporal_store(dbl2(cv + ea2 * k), (dbl2u *)(epi.o2 + idx));
      if (epi.o3) __builtin_nontemporal_store(dbl2(cv + ea3 * k), (dbl2u *)(epi.o3 + idx));
    }
  }
}

}  // namespace exw
