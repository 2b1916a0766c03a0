// gather.hip -- row-owner ("gather") assembly of the tangent and residual into CSR.
//
// Same element arithmetic as the reference's per-element loop (Elem_Solid_3D_Disp.cpp:196-374,
// ElementBase2.cpp:278-552) and the same assembled K and R as SolverPetsc::assembleMatrixAndVector
// (SolverPetsc.cpp:357-378, 434-502) with the first-iteration Dirichlet lift (ElementBase.cpp:567-594,
// 717-782), organised for the GPU in two kernels:
//
//   element kernel: per element, the 3x3 tangent blocks of its node pairs (each unordered pair once:
//       K_e is symmetric), its u-p couplings and its residual with the lift, as one dense record.
//   row kernel (one wavefront per 64 laid-out items of one or more nodes): every item is one element
//       around a node and one node of it; its block is read from the element's record, the blocks of
//       each column are summed in element order in LDS, and the node's CSR rows and right-hand side go
//       out with consecutive lanes on consecutive values.
//
// Nothing is read-modify-written, so there is no zero fill, no colouring and no atomics on the FP64
// path, and the result is bitwise reproducible.  Each column block's contributions are summed in
// element order, the reference's own order for a given row (femSolidmechanics2.cpp:1061); (n, m) and
// (m, n) sum the same records in the same order, so the matrix is exactly symmetric.

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>

#include "fem_device.hpp"

namespace mpf {

namespace {

using namespace dev;

constexpr int kMaxAdj = 64;   // elements around one node
constexpr int kMaxNB = 128;   // nodes coupled to one node (column blocks of its rows)

// Element record (doubles).  Node pairs by the distance d = (b - a) mod NPE of their local indices:
//   U  [NPE][H][9]   block (a, (a + d) mod NPE), d < H = NPE / 2, row-major 3x3: the H blocks of a node are
//                    contiguous, so that a row of the matrix reads few lines of each element
//      [NPE / 2][9]  block (a, a + H), a < H; block (b, a) of a stored (a, b) is its transpose
//   Q  [NPE][4][3]   Tet10/P1: Kup(3a + i, q); Kpu is its transpose
//   P  [4][4]        Tet10/P1: Kpp
//   R  [NPE][3]      residual, and RP [4] the pressure rows' (Tet10/P1); lift included on a first
//                    iteration.  Q1/P0: condensed, Fu - Kup Fp / Kpp, as its blocks are
// MIXED with NPE = 8 is the Hex8 Q1/P0 element (one pressure per element, condensed; the system has
// displacement rows only), with NPE = 10 the Tet10/P1 element (pressure rows on the corner nodes).
// Records and their two parts are multiples of 128 bytes (a line completed at different times reaches memory
// twice): 352 doubles Hex8, 544 Tet10, 688 Tet10/P1.
template <int NPE, bool MIXED>
struct Rec {
  static constexpr bool P0 = MIXED && NPE == 8;
  static constexpr bool P1 = MIXED && NPE != 8;
  static constexpr int H = NPE / 2;
  static constexpr int ROW = H * 9;                         // a node's stored blocks
  static constexpr int UN = NPE * ROW;
  static constexpr int T0 = (UN + 15) / 16 * 16;            // then pairs (a, a + H), Q, P, R, RP
  static constexpr int Q0 = T0 + (H * 9 + 1) / 2 * 2;
  static constexpr int P0f = Q0 + (P1 ? NPE * 12 : 0);
  static constexpr int R0 = P0f + (P1 ? 16 : 0);
  static constexpr int RP0 = R0 + NPE * 3;
  static constexpr int TN = (RP0 + (P1 ? 4 : 0) - T0 + 1) / 2 * 2;  // its length
  static constexpr int TS = (T0 + TN + 15) / 16 * 16;
  static_assert(UN % 2 == 0 && TN % 2 == 0, "16-byte groups");
};

// Where block (a, b) of a record starts, and whether the stored block is its transpose.
template <int NPE, bool MIXED>
__device__ __forceinline__ int pair_slot(int a, int b, bool& tr) {
  constexpr int H = NPE / 2;
  int d = b - a;
  if (d < 0) d += NPE;
  tr = d > H || (d == H && a >= H);
  const int dd = tr ? NPE - d : d, aa = tr ? b : a;
  return dd < H ? (aa * H + dd) * 9 : Rec<NPE, MIXED>::T0 + aa * 9;
}

// Gauss-point data of one element in LDS, per point: g of every node by component ([3][NPE], so that the
// lanes (element, node) of a wavefront read consecutive addresses), the six components of b, the
// tangent scalars (s1..s5; mixed s1..s4, dv, dv0, thetahat, resip), and the residual's tensor T (dv sigma, six
// components; with the lift nine, not symmetric, and the mixed element's div of the lift).
template <int NPE, bool MIXED, bool LIFT, int NGP>
struct GaussLds {
  static constexpr int SS = MIXED ? 8 : 5;
  static constexpr int B0 = 3 * NPE, S0 = B0 + 6, T0 = S0 + SS;
  static constexpr int PER = T0 + (LIFT ? (MIXED ? 10 : 9) : 6);
  // element stride: the elements of half a wavefront start on different LDS banks
  static constexpr int pad(int n) {
    while (n % 32 != NPE && n % 32 != 32 - NPE) ++n;
    return n;
  }
  static constexpr int SLP = pad(NGP * PER);
};

// Element kernel.  A workgroup takes EPB elements; lane (element, Gauss point) runs the geometry and the
// material (gauss_state) and puts its point's data in LDS.  Then two groups of lanes (element, node a)
// accumulate over the Gauss points in order: the first the pair blocks of the shorter distances and the
// residual, the second the other distances and the couplings (one lane with all of a node's blocks keeps so
// many registers that a compute unit holds two thirds of the wavefronts).  The records then go through LDS
// to memory as 16-byte stores of whole contiguous lines.
//   BLOCKS = false: only R (and RP) of the records (a residual assembly), one group of lanes.
//   LIFT: the residual also loses K_e times the prescribed increments (dispApplied on prescribed dofs): with
//     H_ki = sum_b ubar_b,k g_b,i per Gauss point it is T += s1 H^T + (s2 tr H + s3 b:H) I + s3 tr(H) b + s4 H b + s5 H.
// Bound by FP64 arithmetic (about 30 kFLOP a Hex8 element: 1.6 of its 3.1 ms on 128^3) and, Tet10, by the record writes
// (7.1 GB in 2.5 ms on 60^3 x 6).
template <int NPE, bool MIXED>
struct ElemSplit {
  static constexpr int ND = NPE / 2 + 1;
  static constexpr int DH = NPE == 8 ? 2 : 3;  // distances of the first group
  static constexpr int NA = DH > ND - DH ? DH : ND - DH;
};

template <int NPE, bool MIXED>
struct NodeSums {
  double acc[ElemSplit<NPE, MIXED>::NA][9];
  double r[3], rp;                  // residual, pressure row (first group)
  double up[12], pp[4];             // Tet10/P1 couplings (second group)
  double kup[3], kpp, fp, fpl;      // Q1/P0 (both groups)
};

// Node a's sums over the NG Gauss points whose data starts at o (element stride applied): distances D0 <= d < D1.
template <int NPE, bool MIXED, bool LIFT, int NG, int D0, int D1, bool RES, bool COUP>
__device__ __forceinline__ void node_sums(const double* o, int a, NodeSums<NPE, MIXED>& N) {
  using Rc = Rec<NPE, MIXED>;
  using Gl = GaussLds<NPE, MIXED, LIFT, NG>;
  constexpr int H = Rc::H;
#pragma unroll
  for (int d = 0; d < D1 - D0; ++d)
#pragma unroll
    for (int t = 0; t < 9; ++t) N.acc[d][t] = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) N.r[i] = N.kup[i] = 0.0;
#pragma unroll
  for (int i = 0; i < 12; ++i) N.up[i] = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) N.pp[i] = 0.0;
  N.rp = N.kpp = N.fp = N.fpl = 0.0;
#pragma unroll 1
  for (int gp = 0; gp < NG; ++gp, o += Gl::PER) {
    const double ga[3] = {o[a], o[NPE + a], o[2 * NPE + a]};
    const double* S = o + Gl::S0;
    const double* t = o + Gl::T0;
    if constexpr (RES) {
      if constexpr (LIFT) {
#pragma unroll
        for (int i = 0; i < 3; ++i) N.r[i] -= t[3 * i] * ga[0] + t[3 * i + 1] * ga[1] + t[3 * i + 2] * ga[2];
      } else {
        N.r[0] -= t[0] * ga[0] + t[3] * ga[1] + t[4] * ga[2];
        N.r[1] -= t[3] * ga[0] + t[1] * ga[1] + t[5] * ga[2];
        N.r[2] -= t[4] * ga[0] + t[5] * ga[1] + t[2] * ga[2];
      }
    }
    if constexpr (D1 > D0) {
      double B6[6], ba[3];
#pragma unroll
      for (int q = 0; q < 6; ++q) B6[q] = o[Gl::B0 + q];
      bsym_times(B6, ga, ba);
      const double s1 = S[0], s2 = S[1], s3 = S[2], s4 = S[3], s5 = MIXED ? 0.0 : S[4];
#pragma unroll
      for (int d = D0; d < D1; ++d) {
        if (d == H && a >= H) continue;
        int b = a + d;
        if (b >= NPE) b -= NPE;
        const double gb[3] = {o[b], o[NPE + b], o[2 * NPE + b]};
        double bb[3];
        bsym_times(B6, gb, bb);
        tangent_gp<!MIXED>(ga, ba, gb, bb, s1, s2, s3, s4, s5, N.acc[d - D0]);
      }
    }
    if constexpr (Rc::P1 && (RES || COUP)) {  // ElementBase2.cpp:500-539
      double Np[4];
      tet_Np(gp, Np);
      const double Na = a == 0 ? Np[0] : a == 1 ? Np[1] : a == 2 ? Np[2] : Np[3];
      const double dv = S[4], dv0 = S[5], th = S[6], resip = S[7];
      if constexpr (RES) {
        if (a < 4) {
          N.rp -= (dv0 * Na) * resip;
          if constexpr (LIFT) N.rp -= (dv * Na) * t[9];
        }
      }
      if constexpr (COUP) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const double b1 = dv * ga[i];
#pragma unroll
          for (int q = 0; q < 4; ++q) N.up[3 * q + i] += b1 * Np[q];
        }
        if (a < 4) {
#pragma unroll
          for (int q = 0; q < 4; ++q) N.pp[q] -= ((dv0 * Na) * th) * Np[q];
        }
      }
    }
    if constexpr (Rc::P0) {  // Kup_a = sum dv g_a, Kpp = -sum dv0 thetahat, Fp = -sum dv0 resip (Np = 1)
      const double dv = S[4], dv0 = S[5];
#pragma unroll
      for (int i = 0; i < 3; ++i) N.kup[i] += dv * ga[i];
      N.kpp -= dv0 * S[6];
      if constexpr (RES) {
        N.fp -= dv0 * S[7];
        if constexpr (LIFT) N.fpl += dv * t[9];
      }
    }
  }
}

// Q1/P0: the condensation's share of the group's blocks (Elem_Solid_3D_Mixed0.cpp:93-104), from every
// node's Kup of the element at kup.
template <int NPE, bool MIXED, int D0, int D1>
__device__ __forceinline__ void condense_blocks(const double* kup, int a, NodeSums<NPE, MIXED>& N) {
#pragma unroll
  for (int d = D0; d < D1; ++d) {
    if (d == NPE / 2 && a >= NPE / 2) continue;
    int b = a + d;
    if (b >= NPE) b -= NPE;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double w = kup[3 * b + j] / N.kpp;
#pragma unroll
      for (int i = 0; i < 3; ++i) N.acc[d - D0][3 * i + j] -= N.kup[i] * w;
    }
  }
}

template <int NPE, int NGP, bool MIXED, int EPB, bool BLOCKS, bool LIFT>
__global__ void __launch_bounds__((EPB * NPE + 63) / 64 * 64 * (BLOCKS ? 2 : 1))
    __attribute__((amdgpu_waves_per_eu(BLOCKS ? 3 : 2)))
    k_elem_records(ElemArgs A, int32_t nElem, const double* __restrict__ dispApplied,
                   const int32_t* __restrict__ nodeinfo, double* __restrict__ KE, double* __restrict__ qKup,
                   double* __restrict__ qKpp, double* __restrict__ qFp) {
  using Rc = Rec<NPE, MIXED>;
  using Gl = GaussLds<NPE, MIXED, LIFT, NGP>;
  using Sp = ElemSplit<NPE, MIXED>;
  constexpr int NL = EPB * NGP, NC = EPB * NPE, GRP = (NC + 63) / 64 * 64, WG = GRP * (BLOCKS ? 2 : 1);
  static_assert(NL <= WG, "Gauss-point lanes");
  constexpr int H = Rc::H, ND = Sp::ND, DH = Sp::DH;
  constexpr int FLD = (MIXED ? 3 : 2) + (LIFT ? 1 : 0);  // nodal fields: X, u, (u_prev), (ubar)
  constexpr int ER = NPE == 8 ? EPB : EPB / 2;  // elements whose blocks go out together
  static_assert(EPB % ER == 0, "rounds");
  constexpr int nU = ER * Rc::UN, nT = EPB * Rc::TN, nOut = nU > nT ? nU : nT;
  constexpr int n1 = EPB * Gl::SLP, n2 = BLOCKS ? nOut : 0, n3 = EPB * (FLD * NPE * 3 + 4);
  constexpr int n12 = n1 > n2 ? n1 : n2, NS = n12 > n3 ? n12 : n3;
  __shared__ double2 sm2[(NS + 1) / 2];
  __shared__ double sdN[NGP][3][NPE];
  double* const sm = reinterpret_cast<double*>(sm2);
  const int tid = threadIdx.x;
  const int base = blockIdx.x * EPB;
  if (tid < NGP) {
    double d[3][NPE];
    if (NPE == 8) {
      hex8_dN(tid, (double(*)[8])d);
    } else {
      double x1, x2, x3;
      tet_gp(tid, x1, x2, x3);
      tet10_dN(x1, x2, x3, (double*)d[0], (double*)d[1], (double*)d[2]);
    }
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int a = 0; a < NPE; ++a) sdN[tid][r][a] = d[r][a];
  }
  // nodal data, one (element, node) pair per lane: sm as [field][element][node][3], then the pressures
  constexpr int FS = EPB * NPE * 3;
  double* const sP = sm + FLD * FS;
  if (tid < NC) {
    const int k = tid / NPE, a = tid - k * NPE;
    const int e = base + k < nElem ? base + k : base;  // idle slots repeat the first element
    const size_t nd = (size_t)A.conn[(size_t)e * NPE + a];
    const int info = LIFT ? nodeinfo[nd] : 0;
    double v[FLD][3], pv = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      v[0][c] = A.X[3 * nd + c];
      v[1][c] = A.u[3 * nd + c];
      if constexpr (MIXED) v[2][c] = A.uprev[3 * nd + c];
      if constexpr (LIFT) v[FLD - 1][c] = ((info >> c) & 1) ? 0.0 : dispApplied[3 * nd + c];
    }
    if (Rc::P1 && a < 4) pv = A.pres[nd];
    if (Rc::P0 && a == 0) pv = A.pres[e];
#pragma unroll
    for (int f = 0; f < FLD; ++f)
#pragma unroll
      for (int c = 0; c < 3; ++c) sm[f * FS + tid * 3 + c] = v[f][c];
    if (Rc::P1 && a < 4) sP[4 * k + a] = pv;
    if (Rc::P0 && a == 0) sP[4 * k] = pv;
  }
  __syncthreads();
  const int sk = tid / NGP, sgp = tid % NGP;
  const bool stage = tid < NL;
  GaussState Q;
  double T[9], trH = 0.0;  // T: residual tensor (row i, column m)
  if (stage) {
    const int e = base + sk < nElem ? base + sk : base;
    const double wgp = (NPE == 8) ? 1.0 : 0.2500000000000000 * (1.0 / 6.0);  // QuadratureUtil.cpp:466-492, 706-709
    double mu, K;
    elem_material(A, e, mu, K);
    const auto field = [&](int f) { return reinterpret_cast<const double(*)[3]>(sm + f * FS + sk * NPE * 3); };
    gauss_state<NPE, NGP, MIXED, 2>(field(0), field(1), MIXED ? field(2) : nullptr, MIXED ? sP + 4 * sk : nullptr,
                                 sdN[sgp], sgp, wgp, mu, K, A.Utype, Rc::P0 ? false : A.consistent != 0, Q);
    if (Q.negJ && base + sk < nElem) flag_bad(A.bad, e);
    const NHPoint& P = Q.nh;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int m = 0; m < 3; ++m) T[3 * i + m] = Q.dv * P.sig[i][m];
    if constexpr (LIFT) {
      const double(*ub)[3] = field(FLD - 1);
      double Hh[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};  // Hh[k][i]
      bool any = false;
#pragma unroll
      for (int a = 0; a < NPE; ++a) any = any || ub[a][0] != 0.0 || ub[a][1] != 0.0 || ub[a][2] != 0.0;
      if (any) {
#pragma unroll 2
        for (int a = 0; a < NPE; ++a) {
          double g[3];
          const double da[3] = {sdN[sgp][0][a], sdN[sgp][1][a], sdN[sgp][2][a]};
          grad_jinv(&Q.Bi[0][0], da, g);
#pragma unroll
          for (int kk = 0; kk < 3; ++kk)
#pragma unroll
            for (int i = 0; i < 3; ++i) Hh[kk][i] += ub[a][kk] * g[i];
        }
        trH = Hh[0][0] + Hh[1][1] + Hh[2][2];
        double bH = 0.0;
#pragma unroll
        for (int kk = 0; kk < 3; ++kk)
#pragma unroll
          for (int l = 0; l < 3; ++l) bH += P.b[kk][l] * Hh[kk][l];
        const double iso = P.s2 * trH + P.s3 * bH;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int m = 0; m < 3; ++m) {
            const double hb = Hh[i][0] * P.b[0][m] + Hh[i][1] * P.b[1][m] + Hh[i][2] * P.b[2][m];
            T[3 * i + m] += P.s1 * Hh[m][i] + P.s3 * trH * P.b[i][m] + P.s4 * hb + P.s5 * Hh[i][m] + (i == m ? iso : 0.0);
          }
      }
    }
  }
  __syncthreads();
  if (stage) {
    double* o = sm + sk * Gl::SLP + sgp * Gl::PER;
#pragma unroll
    for (int c = 0; c < NPE; ++c) {
      double g[3];
      const double dc[3] = {sdN[sgp][0][c], sdN[sgp][1][c], sdN[sgp][2][c]};
      grad_jinv(&Q.Bi[0][0], dc, g);
      o[c] = g[0]; o[NPE + c] = g[1]; o[2 * NPE + c] = g[2];
    }
    const NHPoint& P = Q.nh;
    double* B = o + Gl::B0;
    B[0] = P.b[0][0]; B[1] = P.b[1][1]; B[2] = P.b[2][2];
    B[3] = P.b[0][1]; B[4] = P.b[0][2]; B[5] = P.b[1][2];
    double* S = o + Gl::S0;
    S[0] = P.s1; S[1] = P.s2; S[2] = P.s3; S[3] = P.s4;
    if constexpr (MIXED) {
      S[4] = Q.dv; S[5] = Q.dv0; S[6] = Q.thetahat; S[7] = Q.resip;
    } else {
      S[4] = P.s5;
    }
    double* t = o + Gl::T0;
    if constexpr (LIFT) {
#pragma unroll
      for (int i = 0; i < 9; ++i) t[i] = T[i];
      if constexpr (MIXED) t[9] = trH;
    } else {
      t[0] = T[0]; t[1] = T[4]; t[2] = T[8]; t[3] = T[1]; t[4] = T[2]; t[5] = T[5];
    }
  }
  __syncthreads();
  const bool second = BLOCKS && tid >= GRP;  // uniform per wavefront
  const int ct = second ? tid - GRP : tid;
  const int k = ct / NPE, a = ct - k * NPE;
  const bool comp = ct < NC, live = comp && base + k < nElem;
  NodeSums<NPE, MIXED> N;
  if (comp) {
    const double* o = sm + k * Gl::SLP;
    if constexpr (!BLOCKS) node_sums<NPE, MIXED, LIFT, NGP, 0, 0, true, false>(o, a, N);
    else if (!second) node_sums<NPE, MIXED, LIFT, NGP, 0, DH, true, false>(o, a, N);
    else node_sums<NPE, MIXED, LIFT, NGP, DH, ND, false, true>(o, a, N);
  }
  __syncthreads();
  if constexpr (Rc::P0) {
    if (comp && !second) {
#pragma unroll
      for (int i = 0; i < 3; ++i) sm[ct * 3 + i] = N.kup[i];
    }
    __syncthreads();
    if (comp) {
      const double* kup = sm + k * NPE * 3;
      if (!second) {  // the lift takes Kpu ubar from the pressure equation
        const double fps = (LIFT ? N.fp - N.fpl : N.fp) / N.kpp;
#pragma unroll
        for (int i = 0; i < 3; ++i) N.r[i] = N.r[i] - N.kup[i] * fps;
        if (live) {
          const size_t e = (size_t)(base + k);
#pragma unroll
          for (int i = 0; i < 3; ++i) qKup[e * 24 + 3 * a + i] = N.kup[i];
          if (a == 0) { qKpp[e] = N.kpp; qFp[e] = N.fp; }
        }
        if constexpr (BLOCKS) condense_blocks<NPE, MIXED, 0, DH>(kup, a, N);
      } else {
        condense_blocks<NPE, MIXED, DH, ND>(kup, a, N);
      }
    }
    __syncthreads();
  }
  if constexpr (!BLOCKS) {
    if (live) {
      double* o = KE + (size_t)(base + k) * Rc::TS;
#pragma unroll
      for (int i = 0; i < 3; ++i) o[Rc::R0 + 3 * a + i] = N.r[i];
      if (Rc::P1 && a < 4) o[Rc::RP0 + a] = N.rp;
    }
  } else {
    // self blocks: their (i, k) and (k, i) entries agree to rounding; the mean makes them exactly symmetric
    if (!second) {
      double* c = N.acc[0];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = i + 1; j < 3; ++j) c[3 * i + j] = c[3 * j + i] = 0.5 * (c[3 * i + j] + c[3 * j + i]);
    }
    const int nv = nElem - base < EPB ? nElem - base : EPB;
    // out: n2w 16-byte groups of each of elements k0 .. k1 - 1, contiguous in LDS, to the records' offset off
    const auto copy_out = [&](int k0, int k1, int n2w, int off) {
      const int kn = min(k1, nv) - k0;
      for (int t = tid; t < kn * n2w; t += WG) {
        const int kk = t / n2w, c = t - kk * n2w;
        reinterpret_cast<double2*>(KE + (size_t)(base + k0 + kk) * Rc::TS + off)[c] = sm2[t];
      }
    };
#pragma unroll
    for (int k0 = 0; k0 < EPB; k0 += ER) {
      if (comp && k >= k0 && k < k0 + ER) {
        double* o = sm + (k - k0) * Rc::UN + a * Rc::ROW;
        if (second) {
#pragma unroll
          for (int d = DH; d < H; ++d)
#pragma unroll
            for (int t = 0; t < 9; ++t) o[d * 9 + t] = N.acc[d - DH][t];
        } else {
#pragma unroll
          for (int d = 0; d < DH; ++d)
#pragma unroll
            for (int t = 0; t < 9; ++t) o[d * 9 + t] = N.acc[d][t];
        }
      }
      __syncthreads();
      copy_out(k0, k0 + ER, Rc::UN / 2, 0);
      __syncthreads();
    }
    if (comp) {
      double* o = sm + k * Rc::TN - Rc::T0;
      if (second) {
        if (a < H) {
#pragma unroll
          for (int t = 0; t < 9; ++t) o[Rc::T0 + a * 9 + t] = N.acc[H - DH][t];
        }
        if constexpr (Rc::P1) {
#pragma unroll
          for (int t = 0; t < 12; ++t) o[Rc::Q0 + a * 12 + t] = N.up[t];
          if (a < 4) {
#pragma unroll
            for (int q = 0; q < 4; ++q) o[Rc::P0f + 4 * a + q] = N.pp[q];
          }
        }
      } else {
        if (Rc::P1 && a < 4) o[Rc::RP0 + a] = N.rp;
#pragma unroll
        for (int i = 0; i < 3; ++i) o[Rc::R0 + 3 * a + i] = N.r[i];
      }
    }
    __syncthreads();
    copy_out(0, EPB, Rc::TN / 2, Rc::T0);
  }
}

// Morton (Z-curve) code of a node: 21 bits per axis of its position in the bounding box, interleaved.
__device__ __forceinline__ uint64_t spread3(uint64_t v) {
  v &= 0x1fffffull;
  v = (v | (v << 32)) & 0x1f00000000ffffull;
  v = (v | (v << 16)) & 0x1f0000ff0000ffull;
  v = (v | (v << 8)) & 0x100f00f00f00f00full;
  v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
  v = (v | (v << 2)) & 0x1249249249249249ull;
  return v;
}

__global__ void k_morton(int32_t nNode, const double* __restrict__ X, double x0, double y0, double z0, double sx,
                         double sy, double sz, uint64_t* __restrict__ code, int32_t* __restrict__ id) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nNode) return;
  const double q[3] = {(X[3 * (size_t)i] - x0) * sx, (X[3 * (size_t)i + 1] - y0) * sy, (X[3 * (size_t)i + 2] - z0) * sz};
  uint64_t c[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) c[d] = (uint64_t)fmin(fmax(q[d] + 0.5, 0.0), 2097151.0);
  code[i] = spread3(c[0]) | (spread3(c[1]) << 1) | (spread3(c[2]) << 2);
  id[i] = i;
}

// Batched meshes (node ranges [moff[m], moff[m + 1])): mesh index above a Morton code of the node on
// its own mesh's lattice (origin mq[4m..4m+2], inverse spacing mq[4m+3], 15 bits per axis), so the
// order runs mesh by mesh even where the meshes overlap in space.
__global__ void k_morton_mesh(int32_t nNode, int32_t nmesh, const int32_t* __restrict__ moff,
                              const double* __restrict__ mq, const double* __restrict__ X,
                              uint64_t* __restrict__ code, int32_t* __restrict__ id) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nNode) return;
  int lo = 0, hi = nmesh - 1;  // last mesh whose first node is <= i
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (moff[mid] <= i) lo = mid; else hi = mid - 1;
  }
  const double* q = mq + 4 * lo;
  uint64_t c[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) c[d] = (uint64_t)fmin(fmax((X[3 * (size_t)i + d] - q[d]) * q[3] + 0.5, 0.0), 32767.0);
  code[i] = ((uint64_t)lo << 45) | spread3(c[0]) | (spread3(c[1]) << 1) | (spread3(c[2]) << 2);
  id[i] = i;
}

// XCD-aware order of the workgroups: consecutive ones land on different XCDs (round robin), so each XCD is
// given a contiguous 1/8 of the work.  Work is laid out in Morton order of the nodes, so that share is a
// compact region of the mesh, whose elements' records that XCD's L2 holds while its nodes' rows read them.
__device__ __forceinline__ int64_t xcd_share(int64_t b, int64_t nb) {
  const int64_t per = (nb + 7) / 8;
  return (b % 8) * per + b / 8;
}

// Ascending bitonic sort of n (a power of two, >= 64) keys in LDS by one wavefront.
__device__ __forceinline__ void wave_sort(int32_t* key, int n, int lane) {
  for (int k = 2; k <= n; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = lane; t < n; t += 64) {
        const int u = t ^ j;
        if (u > t) {
          const int32_t x = key[t], y = key[u];
          if ((x > y) == ((t & k) == 0)) { key[t] = y; key[u] = x; }
        }
      }
      __syncthreads();
    }
}

constexpr int kItemCap = 1024;   // kMaxAdj * NPE rounded up to a power of two (Tet10: 640 -> 1024)
constexpr int kGroupNodes = 8;   // nodes per layout group (consecutive in Morton order)

template <bool MIXED>
__device__ __forceinline__ bool has_rows(int info) {
  return (info & 7) || (MIXED && ((info >> 3) & 1));
}

// Build step 1 (one wavefront per node n):
//   nelA[nptr[n] + s]       = e * 16 + a: the elements around n in ascending id, a = local index of n in e
//   keys[nptr[n] * NPE + t] = (j << 16) | (s << 4) | b for every element s around n and node b of it that
//                             has rows (and so columns), sorted: j = position of node conn[e][b] in the sorted
//                             coupled-node list of n (the column block of n's rows the item adds to)
//   cnt[n]                  = number of those items (0 for a node without rows)
// overflow: 1 too many elements or coupled nodes, 2 inconsistent tables, 4 a node with rows in no element.
template <int NPE, bool MIXED>
__global__ void __launch_bounds__(64) k_node_items(int32_t nNode, const int32_t* __restrict__ nptr,
                                                   const int32_t* __restrict__ nel, const int32_t* __restrict__ nbptr,
                                                   const int32_t* __restrict__ nb, const int32_t* __restrict__ conn,
                                                   const int32_t* __restrict__ nodeinfo, int32_t* __restrict__ nelA,
                                                   int32_t* __restrict__ keys, int64_t* __restrict__ cnt,
                                                   int32_t* __restrict__ overflow) {
  static_assert(kMaxAdj * NPE <= kItemCap, "item capacity");
  __shared__ int32_t sE[kMaxAdj], sNB[kMaxNB], sK[kItemCap];
  const int lane = threadIdx.x;
  const int n = blockIdx.x;
  if (n >= nNode) return;
  const int e0 = nptr[n], m = nptr[n + 1] - e0;
  const int b0 = nbptr[n], nnb = nbptr[n + 1] - b0;
  if (m > kMaxAdj || nnb > kMaxNB) {
    if (lane == 0) { atomicOr(overflow, 1); cnt[n] = 0; }
    return;
  }
  sE[lane] = lane < m ? nel[e0 + lane] : 0x7fffffff;
  for (int j = lane; j < nnb; j += 64) sNB[j] = nb[b0 + j];
  __syncthreads();
  wave_sort(sE, 64, lane);
  if (lane < m) {
    const int32_t* c = conn + (size_t)sE[lane] * NPE;
    int a = 0;
    for (int t = 0; t < NPE; ++t)
      if (c[t] == n) a = t;
    nelA[e0 + lane] = sE[lane] * 16 + a;
  }
  const bool rows = has_rows<MIXED>(nodeinfo[n]);
  if (rows && m == 0 && lane == 0) atomicOr(overflow, 4);
  const int nall = rows ? m * NPE : 0;
  int P2 = 64;
  while (P2 < nall) P2 <<= 1;
  int own = 0;
  for (int t = lane; t < P2; t += 64) {
    int32_t key = 0x7fffffff;
    if (t < nall) {
      const int s = t / NPE, b = t % NPE;
      const int vb = conn[(size_t)sE[s] * NPE + b];
      if (has_rows<MIXED>(nodeinfo[vb])) {
        int lo = 0, hi = nnb;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (sNB[mid] < vb) lo = mid + 1; else hi = mid;
        }
        if (lo >= nnb || sNB[lo] != vb) atomicOr(overflow, 2);  // not a coupled node: inconsistent tables
        key = (min(lo, nnb - 1) << 16) | (s << 4) | b;
        ++own;
      }
    }
    sK[t] = key;
  }
  for (int off = 32; off > 0; off >>= 1) own += __shfl_xor(own, off, 64);
  __syncthreads();
  wave_sort(sK, P2, lane);
  for (int t = lane; t < own; t += 64) keys[(size_t)e0 * NPE + t] = sK[t];
  if (lane == 0) cnt[n] = own;
}

// Build step 2 (one wavefront per layout group, the nodes order[8g .. 8g+7]): each node's sorted items are placed one
// after the other, except that a run (one column block of one node) never crosses a 64-item wavefront.
//   FILL = false: glen[g] = the group's length padded to a multiple of 64
//   FILL = true:  the laid-out items,
//     fitem[goff[g] + q] = {e * 16 + a, (blk << 4) | b}  (element e around node n, a = n's local index
//     in e, blk = nbptr[n] + j the column block of n's rows node b of e lands in), for step 4;
//     padding slots, always at the end of a wavefront, keep {-1, -1}.
// A round looks at the next 64 items of a node and places the whole runs among them that fit; one lane walking a group's items
// one after the other took 0.8 and 0.9 ms, a chain of loads (Tet10/P1, whole pattern preparation: 4^3 x 6 elements 7.25 -> 5.65 ms,
// 30^3 x 6 25.4 -> 22.4).
template <int NPE, bool FILL>
__global__ void __launch_bounds__(256) k_group_layout(int64_t ngroups, int32_t nNode, const int32_t* __restrict__ order,
                                                      const int32_t* __restrict__ nptr,
                                                      const int32_t* __restrict__ nbptr,
                                                      const int32_t* __restrict__ keys,
                                                      const int64_t* __restrict__ cnt,
                                                      const int32_t* __restrict__ nelA,
                                                      const int64_t* __restrict__ goff, int64_t* __restrict__ glen,
                                                      int2* __restrict__ fitem) {
  const int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (g >= ngroups) return;  // uniform per wavefront, no barrier below
  const int64_t base = FILL ? goff[g] : 0;
  int64_t pos = 0;
  const int64_t q1 = (g + 1) * kGroupNodes < nNode ? (g + 1) * kGroupNodes : nNode;
  for (int64_t q = g * kGroupNodes; q < q1; ++q) {
    const int n = order[q];
    const int c = (int)cnt[n];
    const int32_t* K = keys + (size_t)nptr[n] * NPE;
    for (int t = 0; t < c;) {
      const int m = c - t < 64 ? c - t : 64;
      const int32_t key = lane < m ? K[t + lane] : -1;
      const int j = key >> 16, jp = __shfl_up(j, 1, 64);
      const unsigned long long heads = __ballot(lane > 0 && lane < m && j != jp);  // the first item starts a run too
      const int first = heads ? __ffsll(heads) - 1 : m;                            // its run's items
      const int room = 64 - (int)(pos & 63);
      if (first > room) {
        pos += room;
        continue;
      }
      // whole runs: to the last start of one, unless the node ends here; of them what fits
      const int whole = t + m == c || !heads ? m : 63 - __clzll(heads);
      const int take = whole <= room ? whole : 63 - __clzll(heads & (~0ull >> (63 - room)));
      if (FILL && lane < take)
        fitem[base + pos + lane] =
            make_int2(nelA[nptr[n] + ((key >> 4) & 63)], ((nbptr[n] + ((key >> 16) & 127)) << 4) | (key & 15));
      pos += take;
      t += take;
    }
  }
  if (!FILL && lane == 0) glen[g] = (pos + 63) & ~(int64_t)63;
}

// Build step 3 (one wavefront per node n): where each column block (n, j) of n's rows lives in the CSR,
//   displacement elements:  {A, (La << 9) | flags}
//   Tet10/P1:               {A, Bp, (D << 16) | La, flags}
//   flags = (self << 8) | (isPn << 7) | (isPb << 6) | (mn << 3) | mb
// A = start of n's first free u row + column offset of j's u dofs (-1 if n has no free u dof),
// Bp = the same in n's pressure row (-1 if n carries no pressure), D = offset of j's pressure column
// relative to A (same in every row of n), La = length of n's rows, mn / mb = free masks of n / j,
// self: j is n itself (its column run also sums n's right-hand side).
template <bool MIXED>
__global__ void __launch_bounds__(64) k_block_table(int32_t nNode, const int32_t* __restrict__ nbptr,
                                                    const int32_t* __restrict__ nb,
                                                    const int32_t* __restrict__ nodeinfo,
                                                    const int32_t* __restrict__ nda, const int32_t* __restrict__ idp,
                                                    int32_t dispDOF, const int32_t* __restrict__ rowptr,
                                                    int32_t* __restrict__ btab) {
  const int lane = threadIdx.x;
  const int n = blockIdx.x;
  if (n >= nNode) return;
  const int info_n = nodeinfo[n];
  const int mn = info_n & 7, La = info_n >> 4;
  const bool isPn = MIXED && ((info_n >> 3) & 1);
  const int b0 = nbptr[n], nnb = nbptr[n + 1] - b0;
  const int fr = (mn & 1) ? 0 : (mn & 2) ? 1 : (mn & 4) ? 2 : -1;
  const int RU = fr >= 0 ? rowptr[nda[3 * (size_t)n + fr]] : -1;
  const int RP = isPn ? rowptr[dispDOF + idp[n]] : -1;
  int Ucols = 0;
  for (int c = 0; c < nnb; c += 64) {
    const int j = c + lane;
    int nu = j < nnb ? __popc(nodeinfo[nb[b0 + j]] & 7) : 0;
    for (int off = 32; off > 0; off >>= 1) nu += __shfl_xor(nu, off, 64);
    Ucols += nu;
  }
  int cu0 = 0, cp0 = 0;
  for (int c = 0; c < nnb; c += 64) {
    const int j = c + lane;
    int inf = 0, nu = 0, np = 0;
    if (j < nnb) {
      inf = nodeinfo[nb[b0 + j]];
      nu = __popc(inf & 7);
      np = MIXED ? ((inf >> 3) & 1) : 0;
    }
    int iu = nu, ip = np;
    for (int off = 1; off < 64; off <<= 1) {
      const int tu = __shfl_up(iu, off, 64), tp = __shfl_up(ip, off, 64);
      if (lane >= off) { iu += tu; ip += tp; }
    }
    if (j < nnb) {
      const int upos = cu0 + iu - nu, ppos = cp0 + ip - np;
      const int mb = inf & 7;
      const size_t blk = (size_t)b0 + j;
      const int self = nb[b0 + j] == n;
      if (MIXED) {
        const int isPb = (inf >> 3) & 1;
        btab[4 * blk] = RU >= 0 ? RU + upos : -1;
        btab[4 * blk + 1] = RP >= 0 ? RP + upos : -1;
        btab[4 * blk + 2] = ((Ucols + ppos - upos) << 16) | La;
        btab[4 * blk + 3] = (self << 8) | ((int)isPn << 7) | (isPb << 6) | (mn << 3) | mb;
      } else {
        btab[2 * blk] = RU >= 0 ? RU + upos : -1;
        btab[2 * blk + 1] = (La << 9) | (self << 8) | (mn << 3) | mb;
      }
    }
    cu0 += __shfl(iu, 63, 64);
    cp0 += __shfl(ip, 63, 64);
  }
}

// Build step 4 (one wavefront per laid-out wavefront w): its runs (columns) and self runs (the column of the
// node itself) are counted (COUNT), then tabled in their order in the wavefront:
//   rtab[whead[w].x + r]  = the block table entry of run r
//   stab[whead[w].y + q]  = {n's first free row, n's pressure row or -1, first item | items << 8 | free mask << 16, n}
//   whead[w].zw           = the positions that start a run, as a 64-bit mask
//   mtab[mhead[w] + q]    = Tet10/P1, the q-th run whose column node m carries a pressure: where n's u columns
//                           start in m's pressure row (Kpu(m, n) is the transpose of the run's Kup(n, m))
//   fitem                 = {offset of the item's block in the records (unsigned), slot | a << 10 | b << 14 |
//                            transposed << 18 | self << 19 | first of its run << 20 | position << 21}, padding {0, -1},
//                            in the order of the offsets
// so that the row kernel reads its tables with consecutive lanes and does no index arithmetic.  A vector load's
// address processing takes one pass per distinct 128-byte line among each four consecutive lanes (measured on
// MI355X), and the kernel is bound by it: in record order a node's neighbouring blocks of an element are
// neighbouring lanes.
template <int NPE, bool MIXED, bool COUNT>
__global__ void __launch_bounds__(64) k_wave_table(int64_t nwaves, int2* __restrict__ fitem,
                                                   const int32_t* __restrict__ btab, const int32_t* __restrict__ conn,
                                                   const int32_t* __restrict__ nodeinfo,
                                                   const int32_t* __restrict__ nda, const int32_t* __restrict__ idp,
                                                   const int32_t* __restrict__ nbptr, const int32_t* __restrict__ nb,
                                                   int32_t dispDOF, int64_t* __restrict__ nrun,
                                                   int64_t* __restrict__ nself, const int64_t* __restrict__ roff,
                                                   const int64_t* __restrict__ soff, int4* __restrict__ whead,
                                                   int32_t* __restrict__ rtab, int4* __restrict__ stab,
                                                   int64_t* __restrict__ npres, const int64_t* __restrict__ poff,
                                                   int32_t* __restrict__ mhead, int32_t* __restrict__ mtab) {
  using Rc = Rec<NPE, MIXED>;
  constexpr int BT = Rc::P1 ? 4 : 2;
  const int64_t w = blockIdx.x;
  if (w >= nwaves) return;
  const int lane = threadIdx.x;
  const int2 it = fitem[w * 64 + lane];
  const bool on = it.x >= 0;
  const int blk = on ? (it.y >> 4) : -1;
  const int pblk = __shfl_up(blk, 1, 64);
  const bool head = on && (lane == 0 || pblk != blk);
  const int e = it.x >> 4, a = it.x & 15, b = it.y & 15;
  const bool self = on && a == b;
  const unsigned long long hm = __ballot(head), sm = __ballot(head && self), am = __ballot(self);
  const bool pcol = Rc::P1 && head && ((btab[BT * (size_t)blk + (BT - 1)] >> 6) & 1);
  const unsigned long long pm = __ballot(pcol);
  if (COUNT) {
    if (lane == 0) {
      nrun[w] = __popcll(hm);
      nself[w] = __popcll(sm);
      if (Rc::P1) npres[w] = __popcll(pm);
    }
    return;
  }
  const unsigned long long below = (1ull << lane) - 1;
  if (lane == 0) whead[w] = make_int4((int)roff[w], (int)soff[w], (int)(uint32_t)hm, (int)(uint32_t)(hm >> 32));
  if (head) {
    int32_t* d = rtab + BT * (size_t)(roff[w] + __popcll(hm & below));
#pragma unroll
    for (int q = 0; q < BT; ++q) d[q] = btab[BT * (size_t)blk + q];
  }
  if constexpr (Rc::P1) {
    if (lane == 0) mhead[w] = (int)poff[w];
    if (pcol) {
      const int n = conn[(size_t)e * NPE + a], m = nb[blk];
      int lo = nbptr[m], hi = nbptr[m + 1];
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (nb[mid] < n) lo = mid + 1; else hi = mid;
      }
      mtab[poff[w] + __popcll(pm & below)] = lo < nbptr[m + 1] && nb[lo] == n ? btab[BT * (size_t)lo + 1] : -1;
    }
  }
  if (head && self) {
    const size_t n = (size_t)conn[(size_t)e * NPE + a];
    const int mn = nodeinfo[n] & 7;
    const int fr = (mn & 1) ? 0 : (mn & 2) ? 1 : 2;
    const unsigned long long mine = am >> lane;  // the run's items are consecutive self items
    int cnt = 1;
    while (lane + cnt < 64 && ((mine >> cnt) & 1) && !((hm >> (lane + cnt)) & 1)) ++cnt;
    stab[soff[w] + __popcll(sm & below)] =
        make_int4(mn ? nda[3 * n + fr] : -1, Rc::P1 && idp[n] >= 0 ? dispDOF + idp[n] : -1,
                  lane | (cnt << 8) | (mn << 16), (int)n);
  }
  bool tr = false;
  const int slot = on ? pair_slot<NPE, MIXED>(a, b, tr) : 0;
  const uint32_t off = on ? (uint32_t)e * (uint32_t)Rc::TS + (uint32_t)slot : 0xffffffffu;
  int rank = 0;
  for (int j = 0; j < 64; ++j) {
    const uint32_t oj = (uint32_t)__shfl((int)off, j, 64);
    rank += (oj < off || (oj == off && j < lane)) ? 1 : 0;
  }
  fitem[w * 64 + rank] = on ? make_int2((int)off, slot | (a << 10) | (b << 14) | ((int)tr << 18) | ((int)self << 19) |
                                                      ((int)head << 20) | (lane << 21))
                            : make_int2(0, -1);
}

struct RowArgs {
  int64_t nwaves;
  const int2* fitem;
  const int4* whead;
  const int32_t* rtab;
  const int4* stab;
  const int32_t* mhead;   // Tet10/P1
  const int32_t* mtab;
  const double* KE;
  double* vals;
  double* rhs;
  const double* fext;     // unit-load external force per node dof, or null; rhs += lam fext
  double lam;
  const double* lam_dev;  // when given, the load factor in device memory (captured graphs)
};

typedef double double2_u __attribute__((ext_vector_type(2), aligned(8)));  // 16-byte load at an 8-byte address

// The LDS writes of a wavefront are read by the same wavefront below: they execute in order, the fences
// keep the compiler from moving them.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Row kernel: kRowWaves independent wavefronts a workgroup, each on 64 laid-out items.  A lane reads its
// item's block (72 contiguous bytes of the element's record) and stores it at its item's position in LDS, where runs
// of equal column are consecutive items in element order.  Lane (run, column dof) then sums the run for the
// (up to) three rows of the node and writes the values: consecutive lanes write consecutive values of a
// row, and a wavefront that holds a whole node writes its rows entirely.
// Bound by the vector loads' address processing (2.0 of the 3.0 ms on Hex8 128^3 with every record in cache; a
// block is 72 scattered bytes) and by memory: 9 GB read and 4.1 GB written, exactly the values.  Tet10/P1, 60^3 x 6:
// 4.7 ms, 5.2 GB written for 4.3 GB of values (Kpu goes into rows that other wavefronts fill).
// The two kernels replace Gauss-point records from which every item formed its block (Hex8: eight-wavefront chunks
// with their elements in LDS, symmetric pairs written to both rows from one sum; Tet10: every item from global
// memory).  A whole assembly call, before -> now: Hex8 10^3 53 -> 39.5 us, 128^3 8.00 -> 6.00 ms; Q1/P0 45 x 31 x 52
// 359 -> 250 us, 80^3 2.28 -> 1.54 ms; Tet10 30^3 x 6 877 -> 682 us; Tet10/P1 60^3 x 6 7.33 -> 7.08 ms (7.0 to 7.15 over
// several runs).  A residual alone (kernels, Hex8 128^3): 1.57 -> 1.21 ms.  Measured and not taken (Hex8 128^3 / Tet10/P1 60^3 x 6, row kernel): non-temporal value stores 3.82 / 5.73 against 3.57 / 5.39 ms;
// 1, 2, 8 wavefronts a workgroup 4.11, 3.93, 4.04 against 3.57 with 4; block offsets by distance before node 3.28 /
// 4.94 against 2.97 / 4.66 by node.
constexpr int kRowWaves = 4;
template <int NPE, bool MIXED>
__global__ void __launch_bounds__(64 * kRowWaves) k_rows(RowArgs F) {
  using Rc = Rec<NPE, MIXED>;
  constexpr bool P1 = Rc::P1;
  constexpr int BT = P1 ? 4 : 2;  // ints of a run's table entry
  constexpr int NR = P1 ? 4 : 3;  // right-hand-side rows of a node
  __shared__ double sPartA[kRowWaves][64 * 9];
  __shared__ int32_t sStartA[kRowWaves][65];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t nwg = (F.nwaves + kRowWaves - 1) / kRowWaves;
  const int64_t w = xcd_share(blockIdx.x, nwg) * kRowWaves + wid;
  if (w >= F.nwaves) return;  // no workgroup barrier below
  double* const part = sPartA[wid];
  int32_t* const start = sStartA[wid];
  const int2 it = F.fitem[w * 64 + lane];
  const int4 hd = F.whead[w];
  const bool on = it.y >= 0;
  const bool head = on && ((it.y >> 20) & 1);
  const int a = (it.y >> 10) & 15, b = (it.y >> 14) & 15;
  const double* blkp = F.KE + (uint32_t)it.x;
  double v[9];
  if (on) {
    const double2_u* p2 = reinterpret_cast<const double2_u*>(blkp);
    const double2_u x0 = p2[0], x1 = p2[1], x2 = p2[2], x3 = p2[3];
    v[0] = x0.x; v[1] = x0.y; v[2] = x1.x; v[3] = x1.y; v[4] = x2.x; v[5] = x2.y; v[6] = x3.x; v[7] = x3.y;
    v[8] = blkp[8];
  }
  const double* rec = blkp - (it.y & 1023);
  double q4[P1 ? 4 : 1];  // Kup(n's u rows, b's pressure column), Kpp
  if constexpr (P1) {
#pragma unroll
    for (int t = 0; t < 4; ++t) q4[t] = 0.0;
    if (on && b < 4) {
      const double* q = rec + Rc::Q0 + (a * 4 + b) * 3;
      const double2_u x0 = *reinterpret_cast<const double2_u*>(q);
      q4[0] = x0.x; q4[1] = x0.y; q4[2] = q[2];
      if (a < 4) q4[3] = rec[Rc::P0f + 4 * (a < b ? a : b) + (a < b ? b : a)];
    }
  }
  const bool self = on && ((it.y >> 19) & 1);
  double rr[NR];
  if (self) {
#pragma unroll
    for (int i = 0; i < 3; ++i) rr[i] = rec[Rc::R0 + 3 * a + i];
    if constexpr (P1) rr[3] = a < 4 ? rec[Rc::RP0 + a] : 0.0;
  }
  const unsigned long long hm = (uint32_t)hd.z | ((unsigned long long)(uint32_t)hd.w << 32);
  const int pos = (it.y >> 21) & 63;
  const int nruns = __popcll(hm), nself = __popcll(__ballot(head && self)), nitems = __popcll(__ballot(on));
  if ((hm >> lane) & 1) start[__popcll(hm & ((1ull << lane) - 1))] = lane;
  if (lane == 0) start[nruns] = nitems;
  if (on) {
    double* o = part + pos * 9;
    const bool tr = (it.y >> 18) & 1;
    o[0] = v[0];
    o[4] = v[4];
    o[8] = v[8];
    const int t1 = tr ? 3 : 1, t2 = tr ? 6 : 2, t5 = tr ? 7 : 5;  // the stored block or its transpose
    o[t1] = v[1];
    o[4 - t1] = v[3];
    o[t2] = v[2];
    o[8 - t2] = v[6];
    o[t5] = v[5];
    o[12 - t5] = v[7];
  }
  wave_lds_fence();
  double* __restrict__ V = F.vals;
  const int c = lane % 3;
  for (int r = lane / 3, r0 = 0; r0 < nruns; r += 21, r0 += 21) {  // 21 runs at a time, lane 63 idle
    if (lane == 63 || r >= nruns) continue;
    int A0, La, masks;
    if constexpr (P1) {
      const int4 x = reinterpret_cast<const int4*>(F.rtab)[hd.x + r];
      A0 = x.x; La = x.z & 0xffff; masks = x.w;
    } else {
      const int2 x = reinterpret_cast<const int2*>(F.rtab)[hd.x + r];
      A0 = x.x; La = x.y >> 9; masks = x.y & 0x1ff;
    }
    int s = start[r];
    const int s1 = start[r + 1];
    const double* q = part + s * 9 + c;
    double y0 = q[0], y1 = q[3], y2 = q[6];
    for (++s; s < s1; ++s) {
      q += 9;
      y0 += q[0];
      y1 += q[3];
      y2 += q[6];
    }
    if ((masks & 0x3f) == 0x3f) {  // free node, free column
      double* row = V + A0 + c;
      row[0] = y0;
      row[La] = y1;
      row[2 * La] = y2;
    } else {
      const int mn = (masks >> 3) & 7, mb = masks & 7;
      if ((mb >> c) & 1) {
        double* row = V + A0 + rank3(mb, c);
        if (mn & 1) row[0] = y0;
        if (mn & 2) row[rank3(mn, 1) * La] = y1;
        if (mn & 4) row[rank3(mn, 2) * La] = y2;
      }
    }
  }
  if constexpr (P1) {  // couplings: Kup and Kpp of every item in the same LDS, the pressure column of run lane
    wave_lds_fence();
    if (on) {
#pragma unroll
      for (int i = 0; i < 4; ++i) part[pos * 4 + i] = q4[i];
    }
    wave_lds_fence();
    const int4 x = lane < nruns ? reinterpret_cast<const int4*>(F.rtab)[hd.x + lane] : make_int4(0, 0, 0, 0);
    const bool pcol = (x.w >> 6) & 1;
    const unsigned long long pm = __ballot(pcol);
    if (pcol) {
      const int M = F.mtab[F.mhead[w] + __popcll(pm & ((1ull << lane) - 1))];
      double y[4] = {0.0, 0.0, 0.0, 0.0};
      for (int s = start[lane]; s < start[lane + 1]; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] += part[s * 4 + i];
      const int mn = (x.w >> 3) & 7, D = x.z >> 16, La = x.z & 0xffff;
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if ((mn >> i) & 1) {
          V[x.x + rank3(mn, i) * La + D] = y[i];
          V[M + rank3(mn, i)] = y[i];
        }
      if ((x.w >> 7) & 1) V[x.y + D] = y[3];
    }
  }
  // right-hand side: lane (self run, row) sums the run's residual rows
  if (nself == 0) return;
  wave_lds_fence();
  if (self) {
#pragma unroll
    for (int i = 0; i < NR; ++i) part[pos * NR + i] = rr[i];
  }
  wave_lds_fence();
  for (int t = lane; t < nself * NR; t += 64) {
    const int q = t / NR, i = t - q * NR;
    const int4 x = F.stab[hd.y + q];
    const int s0 = x.z & 255, cnt = (x.z >> 8) & 255, mn = x.z >> 16;
    double y = part[s0 * NR + i];
    for (int s = s0 + 1; s < s0 + cnt; ++s) y += part[s * NR + i];
    if (i == 3) {
      if (x.y >= 0) F.rhs[x.y] = y;
    } else if ((mn >> i) & 1) {
      if (F.fext) y += (F.lam_dev ? *F.lam_dev : F.lam) * F.fext[3 * (size_t)x.w + i];
      F.rhs[x.x + rank3(mn, i)] = y;
    }
  }
}

struct RhsArgs {
  int32_t nNode;
  const int32_t* nptr;
  const int32_t* nelA;
  const int32_t* nodeinfo;
  const int32_t* nda;
  const int32_t* idp;
  int32_t dispDOF;
  const double* KE;
  double* rhs;
  const double* fext;
  double lam;
  const double* lam_dev;
  int32_t isolated_only;      // the row kernel has written every node with an element
};

// Right-hand-side kernel (one lane per node): n's rows of the element residuals, summed in element
// order.  With isolated_only, the nodes in no element (zeros, and their external force).
template <int NPE, bool MIXED>
__global__ void __launch_bounds__(256) k_rhs(RhsArgs R) {
  using Rc = Rec<NPE, MIXED>;
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= R.nNode) return;
  const int info = R.nodeinfo[n];
  const int mn = info & 7;
  const bool isPn = Rc::P1 && ((info >> 3) & 1);
  if (!mn && !isPn) return;
  const int e0 = R.nptr[n], m = R.nptr[n + 1] - e0;
  if (R.isolated_only && m > 0) return;
  double r[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int s = 0; s < m; ++s) {
    const int ea = R.nelA[e0 + s], a = ea & 15;
    const double* rec = R.KE + (size_t)(ea >> 4) * Rc::TS;
#pragma unroll
    for (int i = 0; i < 3; ++i) r[i] += rec[Rc::R0 + 3 * a + i];
    if (isPn && a < 4) r[3] += rec[Rc::RP0 + a];
  }
  const double l = R.lam_dev ? *R.lam_dev : R.lam;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if ((mn >> i) & 1) R.rhs[R.nda[3 * (size_t)n + i]] = R.fext ? r[i] + l * R.fext[3 * (size_t)n + i] : r[i];
  if (isPn) R.rhs[R.dispDOF + R.idp[n]] = r[3];
}

}  // namespace

size_t elem_record_doubles(int etype) {
  if (etype == MPF_HEX8) return (size_t)Rec<8, false>::TS;
  return etype == MPF_TET10 ? (size_t)Rec<10, false>::TS : (size_t)Rec<10, true>::TS;
}

static mpf_status gather_unsupported(mpf_problem* p, const char* why) {
  std::fprintf(stderr, "libmpf: %s; using the coloured scatter\n", why);
  PatternBufs& P = p->pat;
  P.g_order.release();
  P.g_nelA.release();
  P.g_fitem.release();
  P.g_whead.release();
  P.g_rtab.release();
  P.g_stab.release();
  P.g_mhead.release();
  P.g_mtab.release();
  p->KE.release();
  p->asm_mode = MPF_ASSEMBLY_COLORED_SCATTER;
  return MPF_OK;
}

mpf_status ensure_gather_tables(mpf_problem* p) {
  PatternBufs& P = p->pat;
  if (P.gather_ready) return MPF_OK;
  hipStream_t s = p->stream;
  const int npe = p->npe, nNode = p->nNode;
  const bool mixed = p->etype == MPF_TET10P1;
  const int64_t nadj = (int64_t)p->nElem * npe;
  int64_t nbtot = 0;
  {
    int32_t last = 0;
    if (nNode > 0) MPF_HIP(hipMemcpyAsync(&last, P.nbptr.ptr + nNode, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    MPF_HIP(hipStreamSynchronize(s));
    nbtot = last;
  }
  if (p->nElem >= (1 << 27)) return gather_unsupported(p, "more than 2^27 elements");
  if (nbtot >= (1 << 27)) return gather_unsupported(p, "more than 2^27 node-pair blocks");
  if (nNode == 0 || p->nElem == 0) return gather_unsupported(p, "empty mesh");
  if ((uint64_t)p->nElem * elem_record_doubles(p->etype) >= (1ull << 32))
    return gather_unsupported(p, "element records past 2^32 doubles");

  // processing order: Morton order of the node coordinates
  MPF_TRY(P.g_order.alloc(nNode));
  {
    DevBuf<uint64_t> code, code2;
    DevBuf<int32_t> ids;
    MPF_TRY(code.alloc(nNode));
    MPF_TRY(code2.alloc(nNode));
    MPF_TRY(ids.alloc(nNode));
    // positions quantised to a lattice of spacing h = (bounding-box volume / elements)^(1/3), about
    // the element size: on a structured grid each node gets its own lattice point, so 8 consecutive
    // nodes of the order form an aligned 2x2x2 block, whose items share most of their elements' records
    double ext[3], h = 0.0;
    for (int c = 0; c < 3; ++c) ext[c] = p->xmax[c] - p->xmin[c];
    const double emax = std::max(ext[0], std::max(ext[1], ext[2]));
    if (ext[0] > 0.0 && ext[1] > 0.0 && ext[2] > 0.0) h = std::cbrt(ext[0] * ext[1] * ext[2] / (double)p->nElem);
    if (!(h > 0.0)) h = emax / std::cbrt((double)p->nElem);
    if (!(h > 0.0)) h = 1.0;
    h = std::max(h, emax / 2097151.0);
    const double sc[3] = {1.0 / h, 1.0 / h, 1.0 / h};
    std::vector<int32_t> moff, eoff;
    const bool multi = p->batch && batch_node_offsets(p, moff) == MPF_OK && batch_elem_offsets(p, eoff) == MPF_OK &&
                       moff.size() > 2 && moff.size() < (1u << 18);
    DevBuf<int32_t> moff_d;
    DevBuf<double> mq_d;
    if (multi) {  // each mesh on its own lattice, h_m = (box volume / elements)^(1/3) of that mesh
      const int nm = (int)moff.size() - 1;
      std::vector<double> Xh((size_t)nNode * 3), mq(4 * (size_t)nm);
      MPF_TRY(p->X.download(Xh.data(), Xh.size(), s));
      MPF_HIP(hipStreamSynchronize(s));
      for (int m = 0; m < nm; ++m) {
        double lo3[3] = {1e300, 1e300, 1e300}, hi3[3] = {-1e300, -1e300, -1e300};
        for (int32_t v = moff[m]; v < moff[m + 1]; ++v)
          for (int d = 0; d < 3; ++d) {
            lo3[d] = std::min(lo3[d], Xh[3 * (size_t)v + d]);
            hi3[d] = std::max(hi3[d], Xh[3 * (size_t)v + d]);
          }
        const int32_t ne = eoff[m + 1] - eoff[m];
        double e[3], hm = 0.0;
        for (int d = 0; d < 3; ++d) e[d] = moff[m + 1] > moff[m] ? hi3[d] - lo3[d] : 0.0;
        const double em = std::max(e[0], std::max(e[1], e[2]));
        if (e[0] > 0.0 && e[1] > 0.0 && e[2] > 0.0 && ne > 0) hm = std::cbrt(e[0] * e[1] * e[2] / (double)ne);
        if (!(hm > 0.0)) hm = ne > 0 ? em / std::cbrt((double)ne) : 1.0;
        if (!(hm > 0.0)) hm = 1.0;
        hm = std::max(hm, em / 32767.0);
        for (int d = 0; d < 3; ++d) mq[4 * (size_t)m + d] = moff[m + 1] > moff[m] ? lo3[d] : 0.0;
        mq[4 * (size_t)m + 3] = 1.0 / hm;
      }
      MPF_TRY(moff_d.upload(moff.data(), moff.size(), s));
      MPF_TRY(mq_d.upload(mq.data(), mq.size(), s));
      hipLaunchKernelGGL(k_morton_mesh, dim3(grid_for(nNode, 256)), dim3(256), 0, s, nNode, nm, moff_d.ptr, mq_d.ptr,
                         p->X.ptr, code.ptr, ids.ptr);
    } else {
      hipLaunchKernelGGL(k_morton, dim3(grid_for(nNode, 256)), dim3(256), 0, s, nNode, p->X.ptr, p->xmin[0],
                         p->xmin[1], p->xmin[2], sc[0], sc[1], sc[2], code.ptr, ids.ptr);
    }
    size_t tmp = 0;
    MPF_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, code.ptr, code2.ptr, ids.ptr, P.g_order.ptr, nNode, 0, 63,
                                               s));
    DevBuf<char> t;
    MPF_TRY(t.alloc(tmp > 0 ? tmp : 1));
    MPF_HIP(hipcub::DeviceRadixSort::SortPairs(t.ptr, tmp, code.ptr, code2.ptr, ids.ptr, P.g_order.ptr, nNode, 0, 63,
                                               s));
    MPF_HIP(hipStreamSynchronize(s));
  }

  // step 1: sorted items per node
  DevBuf<int32_t> keys, ovf;
  DevBuf<int64_t> cnt;
  MPF_TRY(P.g_nelA.alloc(nadj));
  MPF_TRY(keys.alloc((size_t)nadj * npe));
  MPF_TRY(cnt.alloc(nNode));
  MPF_TRY(ovf.alloc(1));
  MPF_HIP(hipMemsetAsync(ovf.ptr, 0, sizeof(int32_t), s));
  if (mixed)
    hipLaunchKernelGGL((k_node_items<10, true>), dim3(nNode), dim3(64), 0, s, nNode, P.nptr.ptr, P.nel.ptr,
                       P.nbptr.ptr, P.nb.ptr, p->conn.ptr, P.nodeinfo.ptr, P.g_nelA.ptr, keys.ptr, cnt.ptr, ovf.ptr);
  else if (npe == 10)
    hipLaunchKernelGGL((k_node_items<10, false>), dim3(nNode), dim3(64), 0, s, nNode, P.nptr.ptr, P.nel.ptr,
                       P.nbptr.ptr, P.nb.ptr, p->conn.ptr, P.nodeinfo.ptr, P.g_nelA.ptr, keys.ptr, cnt.ptr, ovf.ptr);
  else
    hipLaunchKernelGGL((k_node_items<8, false>), dim3(nNode), dim3(64), 0, s, nNode, P.nptr.ptr, P.nel.ptr,
                       P.nbptr.ptr, P.nb.ptr, p->conn.ptr, P.nodeinfo.ptr, P.g_nelA.ptr, keys.ptr, cnt.ptr, ovf.ptr);
  MPF_HIP(hipGetLastError());
  int32_t o = 0;
  MPF_HIP(hipMemcpyAsync(&o, ovf.ptr, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  MPF_HIP(hipStreamSynchronize(s));
  if (o & 1) return gather_unsupported(p, "a node has more than 64 elements or 128 coupled nodes");
  if (o & 2) return MPF_ERR_STATE;
  P.g_isolated = (o & 4) != 0;

  // step 2: layout groups of 8 nodes in Morton order, their padded lengths and offsets
  const int64_t ngroups = ((int64_t)nNode + kGroupNodes - 1) / kGroupNodes;
  DevBuf<int64_t> glen, goff;
  MPF_TRY(glen.alloc(ngroups + 1));
  MPF_TRY(goff.alloc(ngroups + 1));
  const auto layout = [&](bool fill) {
#define MPF_GL(NPE, F)                                                                                          \
  hipLaunchKernelGGL((k_group_layout<NPE, F>), dim3((unsigned)((ngroups + 3) / 4)), dim3(256), 0, s, ngroups, nNode, \
                     P.g_order.ptr, P.nptr.ptr, P.nbptr.ptr, keys.ptr, cnt.ptr, P.g_nelA.ptr, goff.ptr, glen.ptr,    \
                     P.g_fitem.ptr)
    if (npe == 10) { if (fill) MPF_GL(10, true); else MPF_GL(10, false); }
    else { if (fill) MPF_GL(8, true); else MPF_GL(8, false); }
#undef MPF_GL
  };
  layout(false);
  MPF_HIP(hipMemsetAsync(glen.ptr + ngroups, 0, sizeof(int64_t), s));
  auto exclusive_sum = [&](const int64_t* in, int64_t* out, int64_t n) -> mpf_status {
    size_t tmp = 0;
    MPF_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, in, out, n, s));
    DevBuf<char> t;
    MPF_TRY(t.alloc(tmp > 0 ? tmp : 1));
    MPF_HIP(hipcub::DeviceScan::ExclusiveSum(t.ptr, tmp, in, out, n, s));
    MPF_HIP(hipStreamSynchronize(s));
    return MPF_OK;
  };
  MPF_TRY(exclusive_sum(glen.ptr, goff.ptr, ngroups + 1));
  int64_t total = 0;
  MPF_HIP(hipMemcpyAsync(&total, goff.ptr + ngroups, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  MPF_HIP(hipStreamSynchronize(s));
  if (total >= ((int64_t)1 << 31) - 64) return gather_unsupported(p, "more than 2^31 laid-out items");

  // laid-out items
  MPF_TRY(P.g_fitem.alloc(total > 0 ? (size_t)total : 64));
  MPF_HIP(hipMemsetAsync(P.g_fitem.ptr, 0xff, (total > 0 ? (size_t)total : 64) * sizeof(int2), s));
  layout(true);
  MPF_HIP(hipGetLastError());
  P.g_nwaves = total / 64;

  // step 3: column-block table; step 4: the row kernel's tables
  DevBuf<int32_t> btab;
  MPF_TRY(btab.alloc((size_t)(nbtot > 0 ? nbtot : 1) * (mixed ? 4 : 2)));
  if (mixed)
    hipLaunchKernelGGL(k_block_table<true>, dim3(nNode), dim3(64), 0, s, nNode, P.nbptr.ptr, P.nb.ptr, P.nodeinfo.ptr,
                       P.nda.ptr, P.idp.ptr, P.dispDOF, P.rowptr.ptr, btab.ptr);
  else
    hipLaunchKernelGGL(k_block_table<false>, dim3(nNode), dim3(64), 0, s, nNode, P.nbptr.ptr, P.nb.ptr, P.nodeinfo.ptr,
                       P.nda.ptr, nullptr, P.dispDOF, P.rowptr.ptr, btab.ptr);
  MPF_HIP(hipGetLastError());
  if (P.g_nwaves > 0) {
    DevBuf<int64_t> nrun, nself, roff, soff, npres, poff;
    const int64_t nw = P.g_nwaves;
    MPF_TRY(nrun.alloc(nw + 1));
    MPF_TRY(nself.alloc(nw + 1));
    MPF_TRY(roff.alloc(nw + 1));
    MPF_TRY(soff.alloc(nw + 1));
    MPF_HIP(hipMemsetAsync(nrun.ptr + nw, 0, sizeof(int64_t), s));
    MPF_HIP(hipMemsetAsync(nself.ptr + nw, 0, sizeof(int64_t), s));
    MPF_TRY(P.g_whead.alloc(nw));
    if (mixed) {
      MPF_TRY(npres.alloc(nw + 1));
      MPF_TRY(poff.alloc(nw + 1));
      MPF_TRY(P.g_mhead.alloc(nw));
      MPF_HIP(hipMemsetAsync(npres.ptr + nw, 0, sizeof(int64_t), s));
    }
    const auto table = [&](bool count) {
#define MPF_WT(NPE, MX, C)                                                                                           \
  hipLaunchKernelGGL((k_wave_table<NPE, MX, C>), dim3((unsigned)nw), dim3(64), 0, s, nw, P.g_fitem.ptr, btab.ptr, \
                     p->conn.ptr, P.nodeinfo.ptr, P.nda.ptr, P.idp.ptr, P.nbptr.ptr, P.nb.ptr, P.dispDOF, nrun.ptr,  \
                     nself.ptr, roff.ptr, soff.ptr, P.g_whead.ptr, P.g_rtab.ptr, P.g_stab.ptr, npres.ptr, poff.ptr,   \
                     P.g_mhead.ptr, P.g_mtab.ptr)
      if (mixed) { if (count) MPF_WT(10, true, true); else MPF_WT(10, true, false); }
      else if (npe == 10) { if (count) MPF_WT(10, false, true); else MPF_WT(10, false, false); }
      else { if (count) MPF_WT(8, false, true); else MPF_WT(8, false, false); }
#undef MPF_WT
    };
    table(true);
    MPF_TRY(exclusive_sum(nrun.ptr, roff.ptr, nw + 1));
    MPF_TRY(exclusive_sum(nself.ptr, soff.ptr, nw + 1));
    if (mixed) MPF_TRY(exclusive_sum(npres.ptr, poff.ptr, nw + 1));
    int64_t tot[3] = {0, 0, 0};
    if (mixed) MPF_HIP(hipMemcpyAsync(&tot[2], poff.ptr + nw, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    MPF_HIP(hipMemcpyAsync(&tot[0], roff.ptr + nw, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    MPF_HIP(hipMemcpyAsync(&tot[1], soff.ptr + nw, sizeof(int64_t), hipMemcpyDeviceToHost, s));
    MPF_HIP(hipStreamSynchronize(s));
    MPF_TRY(P.g_rtab.alloc((size_t)tot[0] * (mixed ? 4 : 2)));
    MPF_TRY(P.g_stab.alloc((size_t)tot[1]));
    if (mixed) MPF_TRY(P.g_mtab.alloc((size_t)std::max<int64_t>(tot[2], 1)));
    table(false);
    MPF_HIP(hipGetLastError());
    MPF_HIP(hipStreamSynchronize(s));
  }
  MPF_TRY(p->KE.alloc((size_t)p->nElem * elem_record_doubles(p->etype)));
  MPF_HIP(hipStreamSynchronize(s));
  P.gather_ready = true;
  return MPF_OK;
}

// The two kernels of one element type.  Elements a workgroup: Hex8, 8 (64 Gauss-point lanes and 64 node lanes);
// Tet10, 12 (48 and 120 lanes of 128).
template <int NPE, int NGP, bool MIXED, int EPB>
static void launch_type(const ElemArgs& A, mpf_problem* p, const double* dispApplied, const RowArgs& F,
                        const RhsArgs& R, bool flat, hipStream_t s) {
  const int32_t nElem = p->nElem;
  const dim3 grid(grid_for(nElem, EPB));
  const int block = (EPB * NPE + 63) / 64 * 64;
  const int32_t* info = p->pat.nodeinfo.ptr;
  double *KE = p->KE.ptr, *qu = p->q_Kup.ptr, *qp = p->q_Kpp.ptr, *qf = p->q_Fp.ptr;
#define MPF_ELEM(BLOCKS, LIFT)                                                                                   \
  hipLaunchKernelGGL((k_elem_records<NPE, NGP, MIXED, EPB, BLOCKS, LIFT>), grid, dim3(block *(BLOCKS ? 2 : 1)), 0, \
                     s, A, nElem, dispApplied, info, KE, qu, qp, qf)
  if (flat && dispApplied) MPF_ELEM(true, true);
  else if (flat) MPF_ELEM(true, false);
  else if (dispApplied) MPF_ELEM(false, true);
  else MPF_ELEM(false, false);
#undef MPF_ELEM
  if (flat) {
    const int64_t nwg = (F.nwaves + kRowWaves - 1) / kRowWaves;
    hipLaunchKernelGGL((k_rows<NPE, MIXED>), dim3((unsigned)((nwg + 7) / 8 * 8)), dim3(64 * kRowWaves), 0, s, F);
  }
  if (!flat || R.isolated_only)
    hipLaunchKernelGGL((k_rhs<NPE, MIXED>), dim3(grid_for(p->nNode, 256)), dim3(256), 0, s, R);
}

mpf_status launch_gather_assembly(mpf_problem* p, const ElemArgs& A, const double* dispApplied, int writeK, double lam,
                                  const double* lam_dev, hipStream_t s) {
  const PatternBufs& P = p->pat;
  if (!P.gather_ready) return MPF_ERR_STATE;
  if (p->nElem <= 0 || p->nNode <= 0) return MPF_OK;
  if (p->bc_dof_h.empty()) dispApplied = nullptr;  // nothing prescribed: no lift
  const double* fext = p->has_fext && P.dispDOF > 0 ? p->fext_unit.ptr : nullptr;
  RowArgs F{};
  F.nwaves = P.g_nwaves;
  F.fitem = P.g_fitem.ptr; F.whead = P.g_whead.ptr; F.rtab = P.g_rtab.ptr; F.stab = P.g_stab.ptr;
  F.mhead = P.g_mhead.ptr; F.mtab = P.g_mtab.ptr;
  F.KE = p->KE.ptr; F.vals = p->vals.ptr; F.rhs = p->rhs.ptr;
  F.fext = fext; F.lam = lam; F.lam_dev = lam_dev;
  const bool flat = writeK && F.nwaves > 0;
  RhsArgs R{};
  R.nNode = p->nNode;
  R.nptr = P.nptr.ptr; R.nelA = P.g_nelA.ptr; R.nodeinfo = P.nodeinfo.ptr; R.nda = P.nda.ptr;
  R.idp = P.idp.ptr; R.dispDOF = P.dispDOF; R.KE = p->KE.ptr; R.rhs = p->rhs.ptr;
  R.fext = fext; R.lam = lam; R.lam_dev = lam_dev;
  R.isolated_only = flat && P.g_isolated ? 1 : 0;
  if (p->etype == MPF_TET10) launch_type<10, 4, false, 12>(A, p, dispApplied, F, R, flat, s);
  else if (p->etype == MPF_TET10P1) launch_type<10, 4, true, 12>(A, p, dispApplied, F, R, flat, s);
  else if (p->p0) launch_type<8, 8, true, 8>(A, p, dispApplied, F, R, flat, s);
  else launch_type<8, 8, false, 8>(A, p, dispApplied, F, R, flat, s);
  MPF_HIP(hipGetLastError());
  return MPF_OK;
}

}  // namespace mpf
