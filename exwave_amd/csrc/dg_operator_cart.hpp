// dg_operator_cart.hpp -- fused operator + RK epilogue for Cartesian (box)
// cells: the hot path of the 3D k=4 benchmark.
//
// On a box cell J = diag(h) and the normal of face 2d+s is +-e_d, so the
// operator splits by direction (evaluate_cell and the face fluxes,
// source/wave_equation_operations.cc:424-551, 569-629):
//   dv_d/dt = -rho^-1 d_d p / h_d                     + lifting of faces +-d
//   dp/dt   = sum_d rho c^2 (weak d_d v_d) / h_d      + lifting of faces +-d
// and every term of direction d only needs v_d and p on lines parallel to e_d.
//
// One workgroup per cell batch, three phases:
//   A (lane = node): coalesced loads of the cell's nodes, of the epilogue
//     operand and of the six neighbours' (v_n, p) nodes, staged in LDS;
//   B (lane = line): each of the dim*N^(dim-1) lines of the cell is read
//     from LDS into registers once; the collocation derivative, the weak
//     derivative, both face traces, both fluxes and the face lifting are
//     register FMAs with wave-uniform 1D matrices taken from the kernel
//     arguments; the line's dv_d/dt and its share of dp/dt go back to LDS over
//     the neighbour staging it has just consumed (only this lane reads it);
//   C (lane = node): sum the pressure shares, fused RK epilogue (FP64,
//     RKVectorUpdater semantics, source/time_integrators.cc:128-155) with
//     streaming stores.
// Global traffic is coalesced exactly like a streaming kernel; LDS traffic is
// one read + one write per value and line instead of N reads per derivative.
#pragma once
#include "dg_operator_gen.hpp"

namespace exw {

// The least number of groups of dg_operator_cartp_kernel (below) on a launch with two
// outputs that runs it (NEVER: none).  Below, its larger groups are spread unevenly over
// the CUs.  (With one output the staged kernel moves less, and the pair kernel gains nowhere by
// more than it loses elsewhere.)  RK stage, its time over the staged kernel's at so
// many groups:
//   FP64 2D k=2 439 1.04, 793 0.96, 7059 0.89;  k=3 484 1.03, 589 0.98, 1296 0.87;
//        k=4 281 1.21, 785 1.05, 1452 1.07, 1901 0.97, 44409 0.97;  k=5 281 1.19,
//        505 0.98, 1210 0.72;  3D k=2 247 to 586 1.00, 980 0.91, 53322 0.97
//   FP32 2D k=2 652 1.02, 974 0.93;  k=3 265 1.06, 589 0.95;  k=4 1103 0.97, 1452
//        1.12, 1901 0.93;  k=5 349 1.02, 505 0.96;  k=9 384 1.22, 726 0.86, 2205 1.07,
//        3314 0.97, 22205 0.95;  k=11 260 0.90, 1378 0.91;  3D k=2 586 1.03, 980 0.93;
//        k=4 1099 1.11, 6084 1.02, 39754 0.98;  k=5 343 0.98, 1331 0.88
// Degree 1 gains at every size.  Never (FP32; some sizes gain up to 15 %, others lose
// up to 37 %): 2D k=7 562 1.12, 25992 1.11;  k=8 265 1.37, 586 0.87, 16418 1.06;
// k=10 305 1.32, 541 0.83, 15457 1.19;  k=12 273 1.30, 651 0.80, 13807 1.02;  2D k=6;
// 3D k=3.  FP64 2D k >= 6 and 3D k >= 3 run the pipelined kernel.
template <int DIM, int K, typename Number>
constexpr int cart_pairs_from() {
  constexpr int NEVER = 1 << 30;
  if constexpr (std::is_same_v<Number, double>) {
    if (DIM == 3) return K == 1 ? 0 : K == 2 ? 450 : NEVER;
    return K == 1 ? 0 : K == 2 ? 700 : K == 3 ? 560 : K == 4 ? 1800 : K == 5 ? 500 : NEVER;
  } else {
    if (DIM == 3) return K == 1 ? 0 : K == 2 ? 700 : K == 4 ? 10000 : K == 5 ? 500 : NEVER;
    return K == 1 ? 0 : K == 2 ? 850 : K == 3 ? 560 : K == 4 ? 1800 : K == 5 ? 500
           : K == 9 ? 2600 : K == 11 ? 256 : NEVER;
  }
}

// Whether a launch of so many groups runs it: not just beyond one full round of them
// over the CUs (5, 6 or 7 a CU), where the last, nearly empty round costs more than the
// pairs gain (3D k=2 FP64 1449 groups 1.08, FP32 1591 1.10; 2D k=3 FP32 1893 1.05).
template <int DIM, int K, typename Number>
constexpr bool cart_pairs_pay(int groups) {
  constexpr bool D = std::is_same_v<Number, double>;
  constexpr int round =
      DIM == 3 && K == 2 ? (D ? 1280 : 1536) : DIM == 2 && K == 3 && !D ? 1792 : 0;
  return groups >= cart_pairs_from<DIM, K, Number>() &&
         !(round && groups > round && groups <= round + round / 6);
}

// whether the degree's kernels spell out their FMAs (flux_row)
template <int DIM, int K>
constexpr bool CART_FMAS = !(DIM == 2 ? K == 7 : K >= 8);

#ifndef EXW_CART_GROUP
#define EXW_CART_GROUP 128
#endif

template <int DIM, int K>
struct CartShape {
  static constexpr int N = K + 1;
  static constexpr int ND = DIM == 2 ? N * N : N * N * N;
  static constexpr int NT = DIM == 2 ? N : N * N;  // lines per direction
  static constexpr int NF = DIM + 1;
  static constexpr int NLINE = DIM * NT;           // lines per cell
  // node lanes per cell: cells of >= 48 nodes occupy whole waves (their
  // neighbour rows stay wave-uniform scalar loads); smaller cells are packed
  static constexpr bool WAVE_ALIGNED = ND >= 48;
  static constexpr int LANES = WAVE_ALIGNED ? ((ND + 63) / 64) * 64 : (ND > NLINE ? ND : NLINE);
  // cells per workgroup: about EXW_CART_GROUP lanes per group
  static constexpr int CPB = LANES >= EXW_CART_GROUP ? 1 : EXW_CART_GROUP / LANES;
  static constexpr int BLOCK = ((CPB * LANES + 63) / 64) * 64;
  // cells per group one after the other (their loads issued together; one
  // was measured fastest: fewer cells in flight per CU with more)
  static constexpr int ITER = 1;
  static_assert(CPB * NLINE <= BLOCK, "the packed line phase must fit the group");
};


// The LDS of one group of the Cartesian kernel.
template <int DIM, int K, typename Number>
struct CartLds {
  using S = CartShape<DIM, K>;
  Number u[S::CPB][S::NF][S::ND];
  // neighbour (v_n, p) nodes of face f; phase B overwrites [2d][0] with the
  // lines' dv_d/dt and [2d][1] with their dp/dt share
  Number nb[S::CPB][2 * DIM][2][S::ND];
  // per face: the numerical flux as a linear map of the traces (own v_n, own
  // p, neighbour v_n, neighbour p) -> (v lifting, p lifting), with 1/h and the
  // normal's sign folded in
  Number fc[S::CPB][2 * DIM][8];
  // whether each cell slot is active (several cells per group only: with one,
  // every lane knows)
  int act[S::CPB > 1 ? S::CPB : 0];
};

// The operator part of dg_operator_cart_kernel for the group's cells: phases
// A and B, then k = M^-1 A(src) at the lane's node (phase C's first half).
// Returns the lane's cell slot lc, cell, whether it is active (a node lane of
// an active cell), the cell scale, the epilogue operand b at the node (0
// without b) and k.  Three barriers' worth of LDS use; the caller may reuse
// the LDS after a barrier.
template <int DIM, int K, typename Number>
__device__ __forceinline__ void cart_cell(const DevMesh &mesh, const double *__restrict__ src,
                                          const Epilogue &epi, int group,
                                          CartLds<DIM, K, Number> &L, int &lc_out, int &cell_out,
                                          bool &active_out, double &cscale_out,
                                          double (&bv)[CartShape<DIM, K>::NF],
                                          Number (&k)[CartShape<DIM, K>::NF]) {
  using S = CartShape<DIM, K>;
  constexpr int N = S::N, ND = S::ND, NT = S::NT, NF = S::NF, LANES = S::LANES, CPB = S::CPB;
  constexpr int NFACE = 2 * DIM;
  // the 1D matrices are compile-time constants (folded into the unrolled loops)
  constexpr const CartConst<N> &T = CartTable<N>::value;
  auto &s_u = L.u;
  auto &s_nb = L.nb;
  auto &s_fc = L.fc;
  auto &s_act = L.act;

  const int tid = threadIdx.x;
  int lc = tid / LANES;
  // a wave-aligned cell slot is uniform over the wave: say so, so that the
  // cell's index, neighbour row and material are scalar loads
  if constexpr (S::WAVE_ALIGNED) lc = __builtin_amdgcn_readfirstlane(lc);
  const int lane = tid - lc * LANES;
  const bool lane_ok = lc < CPB;
  const int lane_c = lane < ND ? lane : ND - 1;

  // ---------------- A: the loads of the group's cells ----------------
  // Every load is unconditional and in bounds (no branch between the loads,
  // so all of them are in flight together): lanes past the last node read the
  // last node, inactive slots read cell 0, and boundary faces read the cell
  // itself -- their neighbour inputs have zero flux coefficients.
  int nbr[NFACE];
  double uo[NF], nv[NFACE][2];
  const int e = group * CPB + lc;
  const int cell = epi.cell_list ? (e < epi.n_list ? epi.cell_list[e] : -1) : e;
  bool active = lane_ok && cell >= 0 && cell < mesh.n_cells;
  double cscale = 1.0;
  if (active && epi.cell_scale) {
    cscale = epi.cell_scale[cell];
    active = cscale != 0.0;
  }
#pragma unroll
  for (int f = 0; f < NFACE; ++f) nbr[f] = active ? mesh.neighbor[(size_t)cell * NFACE + f] : -1;
  const int cell_c = active ? cell : 0;
  const size_t cbase_c = (size_t)cell_c * NF * ND;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    uo[f] = src[cbase_c + f * ND + lane_c];
    bv[f] = 0.0;
  }
  if (epi.b) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      bv[f] = __builtin_nontemporal_load(epi.b + cbase_c + f * ND + lane_c);
  }
#pragma unroll
  for (int f = 0; f < NFACE; ++f) {
    const double *un = src + (size_t)(nbr[f] >= 0 ? nbr[f] : cell_c) * NF * ND;
    nv[f][0] = un[(f >> 1) * ND + lane_c];
    nv[f][1] = un[DIM * ND + lane_c];
  }

  if (CPB > 1 && lane_ok && lane == 0) s_act[lc] = active ? 1 : 0;
  if (active && lane < NFACE) {
    // face lane: columns of the linear flux map (evaluate_inner_face /
    // evaluate_boundary_face, source/wave_equation_operations.cc:480-629)
    const int f = lane, d = f >> 1;
    int nb = nbr[0];
#pragma unroll
    for (int g = 1; g < NFACE; ++g)
      if (lane == g) nb = nbr[g];
    const double rho = mesh.rho[cell], cc = mesh.speed[cell];
    const double rho_m = nb >= 0 ? mesh.rho[nb] : rho, c_m = nb >= 0 ? mesh.speed[nb] : cc;
    const double ih = recip(mesh.h[(size_t)cell * DIM + d]);
    const double sg = (f & 1) ? 1.0 : -1.0;
    // a hanging face contributes nothing here (nc_face_kernel adds it)
    const double ihf = nb == -NC_BID ? 0.0 : ih;
    double a[4], b[4];
    flux_matrix<double>(rho, cc, rho_m, c_m, nb >= 0 ? 0 : -nb, a, b);
    // inputs (v_d, p, neighbour v_d, neighbour p): v.n = sg v_d on both sides
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double in = (j == 0 || j == 2) ? sg : 1.0;
      s_fc[lc][f][j] = Number(a[j] * in * sg * ihf);
      s_fc[lc][f][4 + j] = Number(b[j] * in * ihf);
    }
  }
  if (lane_ok) {  // lanes past the last node store the last node's (same) values
#pragma unroll
    for (int f = 0; f < NF; ++f) s_u[lc][f][lane_c] = Number(uo[f]);
#pragma unroll
    for (int f = 0; f < NFACE; ++f) {
      s_nb[lc][f][0][lane_c] = Number(nv[f][0]);
      s_nb[lc][f][1][lane_c] = Number(nv[f][1]);
    }
  }
  __syncthreads();

  // ---------------- B: one lane per line, the group's lines packed ----------------
  const int lcB = tid / S::NLINE, line = tid - lcB * S::NLINE;
  if (lcB < CPB && (CPB > 1 ? s_act[lcB] != 0 : active)) {
    const int d = line / NT, t = line - d * NT;
    int base, sd;
    if constexpr (DIM == 2) {
      base = d == 0 ? t * N : t;
      sd = d == 0 ? 1 : N;
    } else {
      const int t0 = t % N, t1 = t / N;
      base = d == 0 ? t0 * N + t1 * N * N : (d == 1 ? t0 + t1 * N * N : t0 + t1 * N);
      sd = d == 0 ? 1 : (d == 1 ? N : N * N);
    }
    // the cell term's factors of direction d, -1/(rho h_d) and rho c^2/h_d
    // (the line's own; as few bytes of LDS as possible keep 10 groups per CU)
    Number cvv, cvp;
    {
      const int eB = group * CPB + lcB;
      const int cB = CPB > 1 ? (epi.cell_list ? epi.cell_list[eB] : eB) : cell;
      const double rho = mesh.rho[cB], cc = mesh.speed[cB];
      const double ih = recip(mesh.h[(size_t)cB * DIM + d]);
      cvv = Number(-ih * recip(rho));
      cvp = Number(rho * cc * cc * ih);
    }
    Number vl[N], pl[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int n = base + i * sd;
      vl[i] = s_u[lcB][d][n];
      pl[i] = s_u[lcB][DIM][n];
    }
    Number kv[N], kp[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      Number gp = Number(0), dv = Number(0);
#pragma unroll
      for (int m = 0; m < N; ++m) {
        gp += Number(T.D[i * N + m]) * pl[m];
        dv += Number(T.DT[i * N + m]) * vl[m];
      }
      kv[i] = cvv * gp;
      kp[i] = cvp * dv;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int f = 2 * d + s;
      Number vo = Number(0), po = Number(0), vn = Number(0), pn = Number(0);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int n = base + i * sd;
        const Number ls = Number(T.L[s * N + i]), lo = Number(T.L[(1 - s) * N + i]);
        vo += ls * vl[i];
        po += ls * pl[i];
        vn += lo * s_nb[lcB][f][0][n];
        pn += lo * s_nb[lcB][f][1][n];
      }
      const Number *c = s_fc[lcB][f];
      const Number fv = flux_row<CART_FMAS<DIM, K>>(c, vo, po, vn, pn);
      const Number fp = flux_row<CART_FMAS<DIM, K>>(c + 4, vo, po, vn, pn);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const Number lw = Number(T.LW[s * N + i]);
        kv[i] = lift_end<CART_FMAS<DIM, K>>(kv[i], lw, fv);
        kp[i] = lift_end<CART_FMAS<DIM, K>>(kp[i], lw, fp);
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int n = base + i * sd;
      s_nb[lcB][2 * d][0][n] = kv[i];
      s_nb[lcB][2 * d][1][n] = kp[i];
    }
  }
  __syncthreads();

  // ---------------- C (first half): k at the lane's node ----------------
  active = active && lane < ND;
  if (active) {
    Number kp = s_nb[lc][0][1][lane];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      k[d] = s_nb[lc][2 * d][0][lane];
      if (d > 0) kp += s_nb[lc][2 * d][1][lane];
    }
    k[DIM] = kp;
  }
  lc_out = lc;
  cell_out = cell;
  active_out = active;
  cscale_out = cscale;
}

template <int DIM, int K, typename Number>
__global__ void __launch_bounds__((CartShape<DIM, K>::BLOCK))
    dg_operator_cart_kernel(const DevMesh mesh, const double *__restrict__ src,
                            const Epilogue epi) {
  using S = CartShape<DIM, K>;
  constexpr int ND = S::ND, NF = S::NF, LANES = S::LANES;
  static_assert(S::ITER == 1, "one cell per lane slot and group");
  __shared__ CartLds<DIM, K, Number> lds;
  int lc, cell;
  bool active;
  double cscale, bv[NF];
  Number k[NF];
  cart_cell<DIM, K, Number>(mesh, src, epi, xcd_remap(blockIdx.x, gridDim.x), lds, lc, cell,
                            active, cscale, bv, k);

  // ---------------- C: fused epilogue ----------------
  if (active) {
    const int lane = threadIdx.x - lc * LANES;
    const double ea1 = epi.a1 * cscale, ea2 = epi.a2 * cscale, ea3 = epi.a3 * cscale;
    const size_t cbase = (size_t)cell * NF * ND;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const size_t idx = cbase + f * ND + lane;
      const double kk = double(k[f]);
      const double o1 = bv[f] + ea1 * kk;
      __builtin_nontemporal_store(o1, epi.o1 + idx);
      if (epi.o2) {
        const double cv = epi.o2_from_o1 ? o1 : epi.c[idx];
        __builtin_nontemporal_store(cv + ea2 * kk, epi.o2 + idx);
        if (epi.o3) __builtin_nontemporal_store(cv + ea3 * kk, epi.o3 + idx);
      }
    }
  }
}

// dg_operator_cartp_kernel: the same sweep for large launches of small cells,
// everything that touches memory in 16-byte pairs of entries.  The address unit
// takes a quad of lanes per clock, so the 8-byte accesses of one lane per node
// cost twice the time of pairs, and cells of a few nodes fill the node-aligned
// lanes badly (2D k=5: 36 lines on a group's 128 lanes).  Here the cells, their
// neighbours' fields, the accumulator and the outputs are flat copies, and the
// lines have GenShape's line waves (direction uniform per wave).  It costs more
// barriers than dg_operator_cart_kernel (all neighbour fields of the group
// staged at once where they take up to 24 KB, FULL; else one direction's at a
// time) and larger groups, so it pays where memory accesses dominate.
// cart_pairs_from says which launches run it.  RK stage, us, dg_operator_cart_kernel ->
// this one: 2D 301x287 k=5 102 -> 80,
// 512^2 k=3 109 -> 93, 700^2 k=2 192 -> 168, 1000^2 k=1 186 -> 111; 3D 45^3 k=2
// 109 -> 99, 60^3 k=1 97 -> 62, FP32 32^3 k=5 204 -> 182.
template <int DIM, int K, typename Number>
struct CartLines {
  using G = GenShape<DIM, K>;
  static constexpr int N = G::N, ND = G::ND, NF = G::NF, NFACE = G::NFACE, CPB = G::CPB;
  static constexpr int BLOCK = G::BLOCK, NDP = G::NDP;
  // the staged fields: PPF pairs of entries per field, one direction's two faces
  // with two fields each per round
  static constexpr int PPF = (ND + 1) / 2;
  static constexpr int NPF = (CPB * 4 * PPF + BLOCK - 1) / BLOCK;
  static constexpr int FULL_BYTES = CPB * (NF + 2 * NFACE) * NDP * int(sizeof(Number));
  static constexpr bool FULL = FULL_BYTES <= 24 * 1024;
  static constexpr int ROUND_FIELDS = FULL ? 2 * NFACE : 4;
};

template <int DIM, int K, typename Number>
__global__ void __launch_bounds__((CartLines<DIM, K, Number>::BLOCK))
    dg_operator_cartp_kernel(const DevMesh mesh, const double *__restrict__ src,
                            const Epilogue epi) {
  using S = GenShape<DIM, K>;
  using C = CartLines<DIM, K, Number>;
  constexpr int N = S::N, ND = S::ND, NT = S::NT, NF = S::NF, NFACE = S::NFACE;
  constexpr int BLOCK = S::BLOCK, CPB = S::CPB, NX = S::NX, NDP = S::NDP, WPD = S::WPD;
  constexpr int PPC = S::PPC, NPP = S::NPP, PPF = C::PPF, NPF = C::NPF;
  constexpr bool FULL = C::FULL;
  typedef double dbl2 __attribute__((ext_vector_type(2)));
  typedef dbl2 dbl2u __attribute__((aligned(8)));

  __shared__ Number s_u[CPB][NF][NDP];
  // the neighbours' v_n (0) and p (1) of faces 2d + s, as [d][s][0/1] (FULL) or of
  // the round's direction as [s][0/1]; then the lines' dp/dt shares: direction d's
  // over [d][0][1] (FULL: its own lines' entries) or [d]
  __shared__ Number s_nb[C::ROUND_FIELDS][CPB][NDP];
  __shared__ Number s_fc[CPB][NFACE][8];
  __shared__ Number s_vc[CPB][DIM][2];
  auto kp_slot = [](int d) { return FULL ? 4 * d + 1 : d; };

  const int tid = threadIdx.x;
  const int c0 = xcd_remap(blockIdx.x, gridDim.x) * CPB;
  const int n_entries = epi.cell_list ? epi.n_list : mesh.n_cells;
  // (a slot past the last entry repeats it and stores nothing)
  auto cell_of = [&](int lc) __attribute__((always_inline)) {
    const int e = CPB == 1 ? c0 : min(c0 + lc, n_entries - 1);
    return epi.cell_list ? epi.cell_list[e] : e;
  };
  if constexpr (CPB == 1)
    if (epi.cell_scale && epi.cell_scale[cell_of(0)] == 0.0) return;  // uniform over the group

  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dir = wave / WPD;
  const int li = tid - dir * (WPD * 64);
  static_assert(NF * ND <= 4096 && NPP * BLOCK <= 4096, "small_div's range");
  const int lcB = CPB == 1 ? 0 : small_div<NT>(li), t = li - lcB * NT, t0 = small_mod<N>(t),
            t1 = small_div<N>(t);
  const bool line_ok = dir < DIM && (CPB == 1 ? t < NT : lcB < CPB);
  auto line_base = [&](auto D_) __attribute__((always_inline)) {
    constexpr int d = decltype(D_)::value;
    if constexpr (DIM == 2) return d == 0 ? t * NX : t;
    else return d == 0 ? t0 * NX + t1 * NX * N : (d == 1 ? t0 + t1 * NX * N : t0 + t1 * NX);
  };

  // ---------------- A ----------------
  // the faces' flux maps, one lane each from the group's last lanes down: their
  // loads first, ahead of the cells' own
  constexpr int NT1 = CPB * NFACE, NTASK = (NT1 + BLOCK - 1) / BLOCK;
  double tv[NTASK][5];
  int tnb[NTASK];
#pragma unroll
  for (int j = 0; j < NTASK; ++j) {
    const int r = BLOCK - 1 - tid + j * BLOCK;
    tnb[j] = -1;
    if (r < NT1) {
      const int lc = r / NFACE, f = r - lc * NFACE, cell = cell_of(lc);
      tnb[j] = mesh.neighbor[(size_t)cell * NFACE + f];
      tv[j][0] = mesh.rho[cell];
      tv[j][1] = mesh.speed[cell];
      tv[j][4] = mesh.h[(size_t)cell * DIM + (f >> 1)];
    }
  }
  // the cells, flat, 16 bytes per lane
  dbl2 own[NPP];
  size_t idx[NPP];  // the pair's place in the vectors
  int dst[NPP];     // and in s_u; -1: none
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    const int p = tid + j * BLOCK, lc = CPB == 1 ? 0 : min(small_div<PPC>(p), CPB - 1);
    int e = 2 * (p - lc * PPC);
    const bool ok = e < NF * ND;
    if (!ok || ((NF * ND) % 2 && e == NF * ND - 1)) e = NF * ND - 2;  // (the odd last pair overlaps)
    dst[j] = ok ? lc * (NF * NDP) + (NX == N ? e : e + small_div<N>(e)) : -1;
    idx[j] = (size_t)cell_of(lc) * (NF * ND) + e;
    __builtin_memcpy(&own[j], src + idx[j], 16);
  }
  // the neighbours' fields of direction d's faces, flat per field (boundary and
  // hanging faces read the cell itself: their flux maps ignore the values)
  dbl2 nbv[DIM][NPF];
  auto load_faces = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NPF; ++j) {
      const int q = tid + j * BLOCK, g = min(small_div<PPF>(q), 4 * CPB - 1);  // field g of the round
      const int lc = g / 4, s = (g >> 1) & 1, c = g & 1;
      int e = 2 * min(q - g * PPF, PPF - 1);
      if (ND % 2 && e == ND - 1) e = ND - 2;
      const int cell = cell_of(lc), nb = mesh.neighbor[(size_t)cell * NFACE + 2 * d + s];
      const double *un = src + (size_t)(nb >= 0 ? nb : cell) * (NF * ND) + (c ? DIM : d) * ND + e;
      __builtin_memcpy(&nbv[d][j], un, 16);
    }
  };
  auto put_faces = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NPF; ++j) {
      const int q = tid + j * BLOCK, g = small_div<PPF>(q);
      int e = 2 * (q - g * PPF);
      if (ND % 2 && e == ND - 1) e = ND - 2;
      if (g < 4 * CPB) {
        Number *o = &s_nb[(FULL ? 4 * d : 0) + (g & 3)][g >> 2][NX == N ? e : e + small_div<N>(e)];
        o[0] = Number(nbv[d][j].x);
        o[1] = Number(nbv[d][j].y);
      }
    }
  };
#pragma unroll
  for (int d = 0; d < DIM; ++d) load_faces(d);
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
  for (int j = 0; j < NPP; ++j)
    if (dst[j] >= 0) {
      Number *o = &s_u[0][0][0] + dst[j];
      o[0] = Number(own[j].x);
      o[1] = Number(own[j].y);
    }
#pragma unroll
  for (int j = 0; j < NTASK; ++j) {
    const int r = BLOCK - 1 - tid + j * BLOCK;
    if (r < NT1) {
      // columns of the linear flux map (evaluate_inner_face /
      // evaluate_boundary_face, source/wave_equation_operations.cc:480-629)
      const int lc = r / NFACE, f = r - lc * NFACE, d = f >> 1, nb = tnb[j];
      const double rho = tv[j][0], cc = tv[j][1];
      const double ih = recip(tv[j][4]);
      const double sg = (f & 1) ? 1.0 : -1.0;
      // a hanging face contributes nothing here (nc_face_kernel adds it)
      const double ihf = nb == -NC_BID ? 0.0 : ih;
      double a[4], b[4];
      flux_matrix<double>(rho, cc, tm[j][0], tm[j][1], nb >= 0 ? 0 : -nb, a, b);
      // inputs (v_d, p, neighbour v_d, neighbour p): v.n = sg v_d on both sides
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double in = (i == 0 || i == 2) ? sg : 1.0;
        s_fc[lc][f][i] = Number(a[i] * in * sg * ihf);
        s_fc[lc][f][4 + i] = Number(b[i] * in * ihf);
      }
      if ((f & 1) == 0) {  // the cell term's factors of direction d
        s_vc[lc][d][0] = Number(-ih * recip(rho));
        s_vc[lc][d][1] = Number(rho * cc * cc * ih);
      }
    }
  }
  Number tr[2][2];  // the neighbours' traces (v_n, p) at the line's ends
  auto traces = [&](auto D_) __attribute__((always_inline)) {
    constexpr int d = decltype(D_)::value, sd = d == 0 ? 1 : (d == 1 ? NX : NX * N);
    constexpr const CartConst<N> &T = CartTable<N>::value;
    const int base = line_base(D_);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const Number *x = s_nb[(FULL ? 4 * d : 0) + 2 * s + c][lcB] + base;
        Number a = Number(0);
#pragma unroll
        for (int i = 0; i < N; ++i) a += Number(T.L[(1 - s) * N + i]) * x[i * sd];
        tr[s][c] = a;
      }
  };
  if constexpr (FULL) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) put_faces(d);
    __syncthreads();
  } else {
    static_for<DIM>([&](auto R_) __attribute__((always_inline)) {
      put_faces(decltype(R_)::value);
      __syncthreads();
      if (line_ok && dir == decltype(R_)::value) traces(R_);
      __syncthreads();
    });
  }
  // the accumulator, in flight during the line phase
  dbl2 bv[NPP];
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    bv[j] = dbl2{0.0, 0.0};
    if (epi.b) bv[j] = __builtin_nontemporal_load((const dbl2u *)(epi.b + idx[j]));
  }

  // ---------------- B: one lane per line ----------------
  static_for<DIM>([&](auto D_) __attribute__((always_inline)) {
    constexpr int d = decltype(D_)::value, sd = d == 0 ? 1 : (d == 1 ? NX : NX * N);
    constexpr const CartConst<N> &T = CartTable<N>::value;
    if (!line_ok || dir != d) return;
    if constexpr (FULL) traces(D_);
    const int base = line_base(D_);
    const Number cvv = s_vc[lcB][d][0], cvp = s_vc[lcB][d][1];
    Number vl[N], pl[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      vl[i] = s_u[lcB][d][base + i * sd];
      pl[i] = s_u[lcB][DIM][base + i * sd];
    }
    Number fv[2], fp[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      Number vo = Number(0), po = Number(0);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        vo += Number(T.L[s * N + i]) * vl[i];
        po += Number(T.L[s * N + i]) * pl[i];
      }
      const Number *c = s_fc[lcB][2 * d + s];
      fv[s] = flux_row<true>(c, vo, po, tr[s][0], tr[s][1]);
      fp[s] = flux_row<true>(c + 4, vo, po, tr[s][0], tr[s][1]);
    }
    Number(*ks)[NDP] = s_nb[kp_slot(d)];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      Number dv = Number(0);
#pragma unroll
      for (int m = 0; m < N; ++m) dv += Number(T.DT[i * N + m]) * vl[m];
      const Number k = lift_ends<true>(cvp * dv, Number(T.LW[i]), fp[0], Number(T.LW[N + i]), fp[1]);
      ks[lcB][base + i * sd] = k;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      Number gp = Number(0);
#pragma unroll
      for (int m = 0; m < N; ++m) gp += Number(T.D[i * N + m]) * pl[m];
      const Number k = lift_ends<true>(cvv * gp, Number(T.LW[i]), fv[0], Number(T.LW[N + i]), fv[1]);
      s_u[lcB][d][base + i * sd] = k;  // (over v_d, which only this lane reads)
    }
  });
  __syncthreads();

  // ---------------- C: fused epilogue, pairs of entries ----------------
  // M^-1 A(src) at entry e (LDS place l) of a cell
  auto value = [&](int lc, int e, int l) __attribute__((always_inline)) {
    if (e < DIM * ND) return double((&s_u[0][0][0])[l]);
    const int n = l - lc * (NF * NDP) - DIM * NDP;
    Number kp = s_nb[kp_slot(0)][lc][n];
#pragma unroll
    for (int d = 1; d < DIM; ++d) kp += s_nb[kp_slot(d)][lc][n];
    return double(kp);
  };
#pragma unroll
  for (int j = 0; j < NPP; ++j) {
    const int p = tid + j * BLOCK, lc = CPB == 1 ? 0 : min(small_div<PPC>(p), CPB - 1);
    if (dst[j] < 0 || (CPB > 1 && c0 + lc >= n_entries)) continue;
    const double cscale = epi.cell_scale ? epi.cell_scale[cell_of(lc)] : 1.0;
    if (cscale == 0.0) continue;
    const double ea1 = epi.a1 * cscale, ea2 = epi.a2 * cscale, ea3 = epi.a3 * cscale;
    const bool odd = (NF * ND) % 2 && p - lc * PPC == PPC - 1;
    const int e = odd ? NF * ND - 2 : 2 * (p - lc * PPC);
    const double k1 = value(lc, e + 1, dst[j] + 1);
    if (odd) {
      // the odd last entry alone: its pair's other one belongs to the pair before
      const size_t i = idx[j] + 1;
      const double o1 = bv[j].y + ea1 * k1;
      const double cv = epi.o2 && !epi.o2_from_o1 ? epi.c[i] : o1;
      __builtin_nontemporal_store(o1, epi.o1 + i);
      if (epi.o2) __builtin_nontemporal_store(cv + ea2 * k1, epi.o2 + i);
      if (epi.o2 && epi.o3) __builtin_nontemporal_store(cv + ea3 * k1, epi.o3 + i);
      continue;
    }
    const double k0 = value(lc, e, dst[j]);
    const dbl2 o1 = {bv[j].x + ea1 * k0, bv[j].y + ea1 * k1};
    dbl2 cv = o1;
    if (epi.o2 && !epi.o2_from_o1) __builtin_memcpy(&cv, epi.c + idx[j], 16);
    __builtin_nontemporal_store(o1, (dbl2u *)(epi.o1 + idx[j]));
    if (epi.o2) {
      const dbl2 o2 = {cv.x + ea2 * k0, cv.y + ea2 * k1};
      __builtin_nontemporal_store(o2, (dbl2u *)(epi.o2 + idx[j]));
      if (epi.o3) {
        const dbl2 o3 = {cv.x + ea3 * k0, cv.y + ea3 * k1};
        __builtin_nontemporal_store(o3, (dbl2u *)(epi.o3 + idx[j]));
      }
    }
  }
}

}  // namespace exw
