// Fused per-element HDG assembly + static condensation (FP64).
//
// One workgroup owns one element at a time (grid-stride over elements).  The
// element's operator blocks are built at the cubature points and condensed
// onto the face traces without leaving LDS; only the condensed blocks
// S, S0, U, Q, U0, Q0 are written to HBM (element-major, coalesced).
//
// Math (reference: HDGBase.cpp:67-158, HDGDiffusion.cpp:31-145,
// HDGConvection.cpp:31-104, Source.cpp:5-48, HDGSolver.cpp:331-348), with
// Sqq = I_d (x) M, so Sqq^-1 [Squ | Sql] is d independent mass solves:
//   A_k = M^-1 Cg_k,  B_k = M^-1 Sql_k,  K = Suu - sum_k Suq_k A_k
//   U = -K^-1 (Sul - sum_k (Suq_k M^-1) Sql_k),  U0 = K^-1 F_u
//   Q_k = -A_k U - B_k,  Q0_k = -A_k U0
//   S = Slu U + sum_k Slq_k Q_k + Sll,  S0 = -Slu U0 - sum_k Slq_k Q0_k
// Face blocks are kept as per-face weighted face masses
//   FM[f][s][a][b] = sum_q w_s(f,q) psi_a psi_b,
//   s = 0: tau, 1: b.n, 2..2+d-1: n_k, 2+d..2+2d-1: (D n)_k   (all times dS).
#include "dense_gj.h"
#include "hdg_element.h"
#include "hfx_internal.h"

namespace hfx {

namespace {

template <int D, int P, int NT>
struct Layout {
  using Z = ESz<D, P>;
  static constexpr int NN = Z::NN, NNF = Z::NNF, NIP = Z::NIP, NIPF = Z::NIPF, NF = Z::NF, NL = Z::NL;
  static constexpr int NS = 2 + 2 * D;
  static constexpr int NC1 = NN + D * NN + NN;  // [M | Cg_0..Cg_{d-1} | I]
  static constexpr int NC2 = NN + NL + 1;       // [K | -R | Fu]
  // persistent regions
  static constexpr int O_TAB = 0;
  static constexpr int O_FM = O_TAB + Z::TAB;
  static constexpr int O_AUG1 = O_FM + NF * NS * NNF * NNF;
  static constexpr int O_AUG2 = O_AUG1 + NN * NC1;
  static constexpr int O_R5 = O_AUG2 + NN * NC2;  // SUQ[D][NN][NN] SUU[NN][NN] FU[NN]
  static constexpr int O_SUQ = O_R5;
  static constexpr int O_SUU = O_SUQ + D * NN * NN;
  static constexpr int O_FU = O_SUU + NN * NN;
  static constexpr int O_R4 = O_FU + NN;
  // R4 phase 1: gathered inputs and IP data
  static constexpr int O_X = O_R4;
  static constexpr int O_DN = O_X + NN * D;
  static constexpr int O_BN = O_DN + NN * D * D;
  static constexpr int O_TAU = O_BN + NN * D;
  static constexpr int O_FQ = O_TAU + NF * NNF;
  static constexpr int O_RQ = O_FQ + NIP;
  static constexpr int O_DV = O_RQ + NIP;
  static constexpr int O_JI = O_DV + NIP;
  static constexpr int O_DQ = O_JI + NIP * D * D;
  static constexpr int O_BQ = O_DQ + NIP * D * D;
  static constexpr int O_GR = O_BQ + NIP * D;
  static constexpr int O_FWT = O_GR + NIP * NN * D;
  static constexpr int END1 = O_FWT + NF * NIPF * NS;
  // R4 phase 2: Z_k = Suq_k M^-1
  static constexpr int O_Z = O_R4;
  static constexpr int END2 = O_Z + D * NN * NN;
  // R4 phase 3: Q_k (LDS copy) and Q0_k
  static constexpr int O_QL = O_R4;
  static constexpr int O_Q0L = O_QL + D * NN * NL;
  static constexpr int END3 = O_Q0L + D * NN;
  static constexpr int TOTAL = END1 > END2 ? (END1 > END3 ? END1 : END3) : (END2 > END3 ? END2 : END3);
};

template <int D>
__device__ inline double det_small(const double* J) {
  if (D == 2) return J[0] * J[3] - J[1] * J[2];
  return J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) + J[2] * (J[3] * J[7] - J[4] * J[6]);
}

template <int D>
__device__ inline void inv_small(const double* J, double dt, double* Ji) {
  const double r = 1.0 / dt;
  if (D == 2) {
    Ji[0] = J[3] * r; Ji[1] = -J[1] * r; Ji[2] = -J[2] * r; Ji[3] = J[0] * r;
  } else {
    Ji[0] = (J[4] * J[8] - J[5] * J[7]) * r; Ji[1] = (J[2] * J[7] - J[1] * J[8]) * r; Ji[2] = (J[1] * J[5] - J[2] * J[4]) * r;
    Ji[3] = (J[5] * J[6] - J[3] * J[8]) * r; Ji[4] = (J[0] * J[8] - J[2] * J[6]) * r; Ji[5] = (J[2] * J[3] - J[0] * J[5]) * r;
    Ji[6] = (J[3] * J[7] - J[4] * J[6]) * r; Ji[7] = (J[1] * J[6] - J[0] * J[7]) * r; Ji[8] = (J[0] * J[4] - J[1] * J[3]) * r;
  }
}

// Orders whose working set does not fit the 160 KB of LDS keep it in a
// device workspace, one slab per workgroup (the same layout, read and written
// through the caches); the workgroup barriers order those accesses as they
// order the LDS ones.
template <int D, int P>
constexpr bool element_in_workspace() {
  return (size_t)Layout<D, P, 64>::TOTAL * sizeof(double) > 160 * 1024;
}

// The two eliminations touch every entry of their matrices once a step, so
// the workspace orders hold those in LDS: both, where both fit (2-D p 7 to 9,
// 3-D p = 4), else the one at work, copied in and out (2-D p = 10, 3-D p = 5).
// The tables are read where they are (one copy for every workgroup) and the
// IP data lies in LDS too: a slab of 286 KB per workgroup, 18 MB for the 64
// workgroups of an XCD, went through its 4 MB of L2 for every phase.
// Measured, 1,296 3-D p=4 cells: 4.48 ms with everything in the workspace,
// 2.81 ms with the matrices in LDS and two workgroups per CU, 1.93 ms with the
// rest.
template <int D, int P>
struct ElemLds {
  using L = Layout<D, P, 64>;
  static constexpr int A1 = L::NN * L::NC1, A2 = L::NN * L::NC2;
  static constexpr bool WS = element_in_workspace<D, P>();
  static constexpr bool BOTH = (size_t)(A1 + A2) * sizeof(double) <= 156 * 1024;
  // Phase 1 (gathered inputs and IP data, without the gradients, which are
  // formed from the tables where they are used) is over before AUG2 is filled
  // (BOTH) or AUG1 copied in, and lies in their place.
  static constexpr int O_P1 = BOTH ? A1 : 0;
  static constexpr int N_P1 = (L::O_GR - L::O_X) + L::NF * L::NIPF * L::NS;
  static_assert(!WS || N_P1 <= (BOTH ? A2 : A1), "phase 1 does not fit its overlay");
  static constexpr size_t BYTES = (size_t)(!WS ? L::TOTAL : BOTH ? A1 + A2 : A1 > A2 ? A1 : A2) * sizeof(double);
};

// Waves per SIMD that the registers are held to.  Left alone the kernel takes
// up to 350, one wave per SIMD, and a workgroup of four leaves no second one
// beside it (7,442 2-D p=3 cells with a tensor: 0.376 ms so, 0.264 ms with two).
constexpr int ELEMENT_WAVES = 2;

// Columns of the volume blocks per thread: as few as let one pass of the
// workgroup cover them, at most 5 (their sums stay in registers).
constexpr int volume_columns(int nn, int nt) {
  int jb = 1;
  while (jb < 5 && nn * ((nn + jb - 1) / jb) > nt) ++jb;
  return jb;
}

// gauss_jordan on a workspace matrix through the LDS buffer
template <int NR, int NC, int NT>
__device__ void gauss_jordan_via(double* A, double* lds, int* perm) {
  for (int t = threadIdx.x; t < NR * NC; t += NT) lds[t] = A[t];
  __syncthreads();
  gauss_jordan<NR, NC, NT>(lds, perm);
  for (int t = threadIdx.x; t < NR * (NC - NR); t += NT) {
    const int o = (t / (NC - NR)) * NC + NR + t % (NC - NR);
    A[o] = lds[o];
  }
  __syncthreads();
}

template <int D, int P, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(ELEMENT_WAVES)))
void hdg_element_kernel(ElemArgs a) {
  using L = Layout<D, P, NT>;
  using Z = ESz<D, P>;
  constexpr int NN = L::NN, NNF = L::NNF, NIP = L::NIP, NIPF = L::NIPF, NF = L::NF, NL = L::NL, NS = L::NS;
  constexpr int NC1 = L::NC1, NC2 = L::NC2;
  extern __shared__ double lds_ws[];
  double* sm = lds_ws;
  using E = ElemLds<D, P>;
  if constexpr (E::WS) sm = a.gws + (size_t)blockIdx.x * L::TOTAL;
  __shared__ int fn[NF * NNF];
  __shared__ int pos[NF * NN];
  __shared__ int vopp[NF];
  __shared__ int perm1[NN], perm2[NN];
  const int tid = threadIdx.x;

  if constexpr (!E::WS)
    for (int t = tid; t < Z::TAB; t += NT) sm[L::O_TAB + t] = a.tabs[t];
  for (int t = tid; t < NF * NN; t += NT) pos[t] = -1;
  __syncthreads();
  for (int t = tid; t < NF * NNF; t += NT) {
    fn[t] = a.faceNodes[t];
    pos[(t / NNF) * NN + a.faceNodes[t]] = t % NNF;
  }
  __syncthreads();
  if (tid < NF) {
    int v = -1;
    for (int i = 0; i < NN && v < 0; ++i)
      if (pos[tid * NN + i] < 0) v = i;
    vopp[tid] = v;
  }
  __syncthreads();

  const double* TB = E::WS ? a.tabs : sm + L::O_TAB;
  const double* PHI = TB + Z::T_PHI;
  const double* DPHI = TB + Z::T_DPHI;
  const double* FPHI = TB + Z::T_FPHI;
  const double* FDPHI = TB + Z::T_FDPHI;
  const double* W = TB + Z::T_W;
  const double* FW = TB + Z::T_FW;
  double* FM = sm + L::O_FM;
  double* AUG1 = E::WS && E::BOTH ? lds_ws : sm + L::O_AUG1;
  double* AUG2 = E::WS && E::BOTH ? lds_ws + E::A1 : sm + L::O_AUG2;
  double* SUQ = sm + L::O_SUQ;
  double* SUU = sm + L::O_SUU;
  double* FU = sm + L::O_FU;
  double* P1 = E::WS ? lds_ws + E::O_P1 : sm + L::O_X;
  double* X = P1;
  double* DN = P1 + (L::O_DN - L::O_X);
  double* BN = P1 + (L::O_BN - L::O_X);
  double* TAU = P1 + (L::O_TAU - L::O_X);
  double* FQ = P1 + (L::O_FQ - L::O_X);
  double* RQ = P1 + (L::O_RQ - L::O_X);
  double* DV = P1 + (L::O_DV - L::O_X);
  double* JI = P1 + (L::O_JI - L::O_X);
  double* DQ = P1 + (L::O_DQ - L::O_X);
  double* BQ = P1 + (L::O_BQ - L::O_X);
  double* GR = sm + L::O_GR;  // not in the workspace orders
  double* FWT = P1 + ((E::WS ? L::O_GR : L::O_FWT) - L::O_X);
  double* ZB = sm + L::O_Z;
  double* QL = sm + L::O_QL;
  double* Q0L = sm + L::O_Q0L;

  const int e_end = a.el_offset + a.nEl;
  for (int e = a.el_offset + blockIdx.x; e < e_end; e += gridDim.x) {
    // ---------------------------------------------------------- gather
    for (int t = tid; t < NN * D; t += NT) {
      int i = t / D, k = t % D;
      X[t] = a.coords[(size_t)a.cells[(size_t)e * NN + i] * D + k];
    }
    for (int t = tid; t < NN * D * D; t += NT) {
      int i = t / (D * D), r = (t / D) % D, c = t % D;
      double v = (r == c) ? 1.0 : 0.0;
      if (!a.useDiff) v = 0.0;
      else if (a.ndD == 1) v = (r == c) ? a.Dn[a.cells[(size_t)e * NN + i]] : 0.0;
      else if (a.ndD == D * D) v = a.Dn[(size_t)a.cells[(size_t)e * NN + i] * D * D + c * D + r];
      DN[t] = v;  // DN[i][r][c] = D_rc at node i
    }
    for (int t = tid; t < NN * D; t += NT)
      BN[t] = a.hasB ? a.bn[(size_t)a.cells[(size_t)e * NN + t / D] * D + t % D] : 0.0;
    for (int t = tid; t < NF * NNF; t += NT) {
      int f = t / NNF, j = t % NNF;
      int fc = a.cell2face[(size_t)e * NF + f];
      int side = (a.tau_sides == 2 && a.face2cell[2 * (size_t)fc] != e) ? 1 : 0;
      int p = a.face_perm[((size_t)e * NF + f) * NNF + j];
      TAU[t] = a.tau[((size_t)fc * NNF + p) * a.tau_sides + side];
    }
    for (int t = tid; t < NIP; t += NT) {
      double fq = (a.hasF && a.kind != 0) ? a.f_ip[(size_t)e * NIP + t] : 0.0;
      if (a.u_old && a.ts_idt != 0.0) {  // implicit Euler: + u_old(x_q) / dt
        double uo = 0.0;
        for (int j = 0; j < NN; ++j) uo += PHI[t * NN + j] * a.u_old[(size_t)e * NN + j];
        fq += a.ts_idt * uo;
      }
      FQ[t] = fq;
      RQ[t] = (a.hasR ? a.r_ip[(size_t)e * NIP + t] : 0.0) + a.ts_idt;
    }
    __syncthreads();
    // ------------------------- IP fields: J (into JI), D, b, one entry each
    constexpr int NG = 2 * D * D + D;
    for (int t = tid; t < NIP * NG; t += NT) {
      const int q = t / NG, c = t % NG;
      const double *row, *src;
      double* dst;
      int rs, ss;
      if (c < D * D) {
        row = DPHI + q * NN * D + c / D; rs = D; src = X + c % D; ss = D; dst = JI + q * D * D + c;
      } else if (c < 2 * D * D) {
        row = PHI + q * NN; rs = 1; src = DN + (c - D * D); ss = D * D; dst = DQ + q * D * D + (c - D * D);
      } else {
        row = PHI + q * NN; rs = 1; src = BN + (c - 2 * D * D); ss = D; dst = BQ + q * D + (c - 2 * D * D);
      }
      double s = 0.0;
#pragma unroll 4
      for (int i = 0; i < NN; ++i) s += row[i * rs] * src[i * ss];
      *dst = s;
    }
    // ------------------------------------------------- IP geometry (faces)
    for (int t = tid; t < NF * NIPF; t += NT) {
      int f = t / NIPF, q = t % NIPF;
      double Jf[(D - 1) * D];
      for (int u = 0; u < (D - 1) * D; ++u) Jf[u] = 0.0;
      for (int j = 0; j < NNF; ++j) {
        const double* xj = X + fn[f * NNF + j] * D;
        for (int r = 0; r < D - 1; ++r)
          for (int c = 0; c < D; ++c) Jf[r * D + c] += FDPHI[(q * NNF + j) * (D - 1) + r] * xj[c];
      }
      double nv[D];
      double meas;
      if (D == 2) {
        meas = sqrt(Jf[0] * Jf[0] + Jf[1] * Jf[1]);
        nv[0] = Jf[1];
        nv[1] = -Jf[0];
      } else {
        double g00 = 0, g01 = 0, g11 = 0;
        for (int c = 0; c < D; ++c) {
          g00 += Jf[c] * Jf[c];
          g01 += Jf[c] * Jf[D + c];
          g11 += Jf[D + c] * Jf[D + c];
        }
        meas = sqrt(g00 * g11 - g01 * g01);
        nv[0] = Jf[1] * Jf[D + 2] - Jf[2] * Jf[D + 1];
        nv[1] = Jf[2] * Jf[D + 0] - Jf[0] * Jf[D + 2];
        nv[2] = Jf[0] * Jf[D + 1] - Jf[1] * Jf[D + 0];
      }
      double nn = 0.0;
      for (int c = 0; c < D; ++c) nn += nv[c] * nv[c];
      nn = 1.0 / sqrt(nn);
      double prod = 0.0;
      const int v0 = fn[f * NNF], vn = vopp[f];
      for (int c = 0; c < D; ++c) {
        nv[c] *= nn;
        prod += (X[vn * D + c] - X[v0 * D + c]) * nv[c];
      }
      if (prod > 0)
        for (int c = 0; c < D; ++c) nv[c] = -nv[c];
      double tq = 0.0, bq[D], dq[D * D];
      for (int c = 0; c < D; ++c) bq[c] = 0.0;
      for (int u = 0; u < D * D; ++u) dq[u] = 0.0;
      for (int j = 0; j < NNF; ++j) {
        double ps = FPHI[q * NNF + j];
        int node = fn[f * NNF + j];
        tq += ps * TAU[f * NNF + j];
        for (int c = 0; c < D; ++c) bq[c] += ps * BN[node * D + c];
        for (int u = 0; u < D * D; ++u) dq[u] += ps * DN[node * D * D + u];
      }
      const double dvf = FW[q] * meas;
      double bn = 0.0;
      for (int c = 0; c < D; ++c) bn += bq[c] * nv[c];
      double* w = FWT + (f * NIPF + q) * NS;
      w[0] = dvf * tq;
      w[1] = dvf * bn;
      for (int k = 0; k < D; ++k) {
        w[2 + k] = dvf * nv[k];
        double s = 0.0;
        for (int c = 0; c < D; ++c) s += dq[k * D + c] * nv[c];
        w[2 + D + k] = dvf * s;
      }
    }
    __syncthreads();
    for (int q = tid; q < NIP; q += NT) {
      double J[D * D];
      for (int t = 0; t < D * D; ++t) J[t] = JI[q * D * D + t];
      const double dt = det_small<D>(J);
      DV[q] = W[q] * dt;
      inv_small<D>(J, dt, JI + q * D * D);
    }
    __syncthreads();
    // physical gradients GR[q][i][k] = (J^-1 grad_xi phi_i)_k
    for (int t = tid; t < (E::WS ? 0 : NIP * NN); t += NT) {
      int q = t / NN, i = t % NN;
      for (int k = 0; k < D; ++k) {
        double s = 0.0;
        for (int r = 0; r < D; ++r) s += JI[q * D * D + k * D + r] * DPHI[(q * NN + i) * D + r];
        GR[t * D + k] = s;
      }
    }
    // weighted face masses, every weight of one (f, a, b) by one thread
    for (int t = tid; t < NF * NNF * NNF; t += NT) {
      const int b = t % NNF, aa = (t / NNF) % NNF, f = t / (NNF * NNF);
      double acc[NS];
      for (int s = 0; s < NS; ++s) acc[s] = 0.0;
#pragma unroll 2
      for (int q = 0; q < NIPF; ++q) {
        const double pa = FPHI[q * NNF + aa], pb = FPHI[q * NNF + b];
        const double* w = FWT + (f * NIPF + q) * NS;
        for (int s = 0; s < NS; ++s) acc[s] += w[s] * pa * pb;
      }
      for (int s = 0; s < NS; ++s) FM[((f * NS + s) * NNF + aa) * NNF + b] = acc[s];
    }
    __syncthreads();
    // -------------------------------------------------- volume blocks
    constexpr int JB = volume_columns(NN, NT), JG = (NN + JB - 1) / JB;  // JB columns per thread share row i's part
    for (int t = tid; t < NN * JG; t += NT) {
      const int i = t / JG, j0 = t % JG;
      double m[JB], suu[JB], cg[JB][D], sq[JB][D];
      int ju[JB];
#pragma unroll
      for (int u = 0; u < JB; ++u) {
        ju[u] = j0 + u * JG < NN ? j0 + u * JG : NN - 1;
        m[u] = suu[u] = 0.0;
        for (int k = 0; k < D; ++k) cg[u][k] = sq[u][k] = 0.0;
      }
#pragma unroll 1
      for (int q = 0; q < NIP; ++q) {
        const double w = DV[q], pi = PHI[q * NN + i];
        double g[D], dg[D], bg = 0.0;
        for (int k = 0; k < D; ++k) {
          if constexpr (E::WS) {
            g[k] = 0.0;
            for (int r = 0; r < D; ++r) g[k] += JI[q * D * D + k * D + r] * DPHI[(q * NN + i) * D + r];
          } else {
            g[k] = GR[(q * NN + i) * D + k];
          }
        }
        for (int k = 0; k < D; ++k) {
          dg[k] = 0.0;
          for (int c = 0; c < D; ++c) dg[k] += DQ[q * D * D + k * D + c] * g[c];
          bg += BQ[q * D + k] * g[k];
        }
        const double rb = RQ[q] * pi - bg;
#pragma unroll
        for (int u = 0; u < JB; ++u) {
          const double pj = w * PHI[q * NN + ju[u]];
          m[u] += pi * pj;
          for (int k = 0; k < D; ++k) {
            cg[u][k] += g[k] * pj;
            sq[u][k] += dg[k] * pj;
          }
          suu[u] += rb * pj;
        }
      }
#pragma unroll
      for (int u = 0; u < JB; ++u) {
        if (j0 + u * JG >= NN) continue;
        const int j = ju[u];
        for (int f = 0; f < NF; ++f) {
          const int ai = pos[f * NN + i], bj = pos[f * NN + j];
          if (ai >= 0 && bj >= 0) {
            const double* F0 = FM + (f * NS) * NNF * NNF + ai * NNF + bj;
            suu[u] += F0[0];
            for (int k = 0; k < D; ++k) sq[u][k] -= F0[(2 + D + k) * NNF * NNF];
          }
        }
        AUG1[i * NC1 + j] = m[u];
        for (int k = 0; k < D; ++k) {
          AUG1[i * NC1 + NN + k * NN + j] = cg[u][k];
          SUQ[(k * NN + i) * NN + j] = sq[u][k];
        }
        AUG1[i * NC1 + NN + D * NN + j] = (i == j) ? 1.0 : 0.0;
        SUU[i * NN + j] = suu[u];
      }
    }
    for (int i = tid; i < NN; i += NT) {
      double s = 0.0;
#pragma unroll 4
      for (int q = 0; q < NIP; ++q) s += DV[q] * FQ[q] * PHI[q * NN + i];
      FU[i] = s;
    }
    __syncthreads();
    if (a.ts_gen) {
      // general time transform of the u rows: F_u first (it applies the
      // model's rows to w), then the rows; M is the mass block of AUG1
      const double* w = a.ts_w + (size_t)e * Z::NLOC;
      const double* uo = a.u_old + (size_t)e * NN;
      for (int i = tid; i < NN; i += NT) {
        double c = 0.0, mu = 0.0;
#pragma unroll 4
        for (int j = 0; j < NN; ++j) {
          c += SUU[i * NN + j] * w[j];
          mu += AUG1[i * NC1 + j] * uo[j];
          for (int k = 0; k < D; ++k) c += SUQ[(k * NN + i) * NN + j] * w[NN + j * D + k];
        }
        for (int f = 0; f < NF; ++f) {
          const int ai = pos[f * NN + i];
          if (ai < 0) continue;
#pragma unroll 4
          for (int b = 0; b < NNF; ++b)
            c += (-FM[((f * NS + 0) * NNF + ai) * NNF + b] + FM[((f * NS + 1) * NNF + ai) * NNF + b]) *
                 w[NN * (D + 1) + f * NNF + b];
        }
        FU[i] = a.ts_phi * FU[i] + a.ts_mu * mu - c;
      }
      __syncthreads();
      for (int t = tid; t < NN * NN; t += NT) SUU[t] = a.ts_auu * SUU[t] + a.ts_mu * AUG1[(t / NN) * NC1 + t % NN];
      for (int t = tid; t < D * NN * NN; t += NT) SUQ[t] *= a.ts_arest;
      __syncthreads();
    }

    if (a.Kloc) {
      // assembly-only path: write the local matrix in the reference layout
      constexpr int NLOC = Z::NLOC;
      constexpr int OQ = NN, OL = NN * (D + 1);
      double* K = a.Kloc + (size_t)(e - a.el_offset) * NLOC * NLOC;
      for (int t = tid; t < NLOC * NLOC; t += NT) {
        const int r = t / NLOC, c = t % NLOC;
        double v = 0.0;
        if (r < OQ) {
          const int i = r;
          if (c < OQ) v = SUU[i * NN + c];
          else if (c < OL) v = SUQ[(((c - OQ) % D) * NN + i) * NN + (c - OQ) / D];
          else {
            const int f = (c - OL) / NNF, b = (c - OL) % NNF, ai = pos[f * NN + i];
            if (ai >= 0)
              v = a.ts_arest * (-FM[((f * NS + 0) * NNF + ai) * NNF + b] + FM[((f * NS + 1) * NNF + ai) * NNF + b]);
          }
        } else if (r < OL) {
          const int i = (r - OQ) / D, k = (r - OQ) % D;
          if (c < OQ) v = AUG1[i * NC1 + NN + k * NN + c];
          else if (c < OL) { if ((c - OQ) % D == k) v = AUG1[i * NC1 + (c - OQ) / D]; }
          else {
            const int f = (c - OL) / NNF, b = (c - OL) % NNF, ai = pos[f * NN + i];
            if (ai >= 0) v = -FM[((f * NS + 2 + k) * NNF + ai) * NNF + b];
          }
        } else {
          const int f = (r - OL) / NNF, aa = (r - OL) % NNF;
          if (c < OQ) {
            const int bj = pos[f * NN + c];
            if (bj >= 0) v = FM[((f * NS + 0) * NNF + aa) * NNF + bj];
          } else if (c < OL) {
            const int j = (c - OQ) / D, k = (c - OQ) % D, bj = pos[f * NN + j];
            if (bj >= 0) v = -FM[((f * NS + 2 + D + k) * NNF + aa) * NNF + bj];
          } else {
            const int g = (c - OL) / NNF, b = (c - OL) % NNF;
            if (g == f) v = -FM[((f * NS + 0) * NNF + aa) * NNF + b] + FM[((f * NS + 1) * NNF + aa) * NNF + b];
          }
        }
        // time schemes: the reference's u rows are ts_dt x (these rows)
        K[t] = (a.ts_dt > 0.0 && r < OQ) ? a.ts_dt * v : v;
      }
      double* F = a.Floc + (size_t)(e - a.el_offset) * NLOC;
      for (int t = tid; t < NLOC; t += NT) F[t] = t < NN ? (a.ts_dt > 0.0 ? a.ts_dt * FU[t] : FU[t]) : 0.0;
      __syncthreads();
      continue;
    }

    // ---------------------------------- [M | Cg | I] -> [I | A | M^-1]
    if constexpr (E::WS && !E::BOTH) gauss_jordan_via<NN, NC1, NT>(AUG1, lds_ws, perm1);
    else gauss_jordan<NN, NC1, NT>(AUG1, perm1);
    // K = Suu - sum_k Suq_k A_k ;  Z_k = Suq_k M^-1
    for (int t = tid; t < NN * NN; t += NT) {
      const int i = t / NN, j = t % NN;
      double s = SUU[t];
      for (int k = 0; k < D; ++k) {
        double z = 0.0;
#pragma unroll 4
        for (int l = 0; l < NN; ++l) {
          const double sq = SUQ[(k * NN + i) * NN + l];
          const double* row = AUG1 + perm1[l] * NC1 + NN;
          s -= sq * row[k * NN + j];
          z += sq * row[D * NN + j];
        }
        ZB[k * NN * NN + t] = z;
      }
      AUG2[i * NC2 + j] = s;
    }
    __syncthreads();
    // -R = -(Sul - sum_k Z_k Sql_k) ; Fu.  IB rows per thread share the face masses.
    constexpr int IB = 4, IG = (NN + IB - 1) / IB;
    for (int t = tid; t < IG * NL; t += NT) {
      const int i0 = t / NL, c = t % NL, f = c / NNF, b = c % NNF;
      int iu[IB];
      double r[IB];
#pragma unroll
      for (int u = 0; u < IB; ++u) {
        const int i = i0 + u * IG;
        iu[u] = i < NN ? i : NN - 1;
        r[u] = 0.0;
        const int ai = pos[f * NN + iu[u]];
        if (ai >= 0) r[u] = a.ts_arest * (-FM[((f * NS + 0) * NNF + ai) * NNF + b] + FM[((f * NS + 1) * NNF + ai) * NNF + b]);
      }
      for (int k = 0; k < D; ++k)
#pragma unroll 4
        for (int aa = 0; aa < NNF; ++aa) {
          const double fm = FM[((f * NS + 2 + k) * NNF + aa) * NNF + b];
          const double* z = ZB + k * NN * NN + fn[f * NNF + aa];
#pragma unroll
          for (int u = 0; u < IB; ++u) r[u] += z[iu[u] * NN] * fm;
        }
#pragma unroll
      for (int u = 0; u < IB; ++u)
        if (i0 + u * IG < NN) AUG2[iu[u] * NC2 + NN + c] = -r[u];
    }
    for (int i = tid; i < NN; i += NT) AUG2[i * NC2 + NN + NL] = FU[i];
    __syncthreads();
    // ---------------------------------------- [K | -R | Fu] -> [I | U | U0]
    if constexpr (E::WS && !E::BOTH) gauss_jordan_via<NN, NC2, NT>(AUG2, lds_ws, perm2);
    else gauss_jordan<NN, NC2, NT>(AUG2, perm2);
    // Q_k = -A_k U - M^-1 Sql_k ;  Q0_k = -A_k U0 ; write U, U0, Q, Q0
    double* Ue = a.U + (size_t)e * NN * NL;
    double* Qe = a.Q + (size_t)e * NN * D * NL;
    for (int t = tid; t < NN * NL; t += NT) Ue[t] = AUG2[perm2[t / NL] * NC2 + NN + t % NL];
    for (int t = tid; t < NN; t += NT) a.U0[(size_t)e * NN + t] = AUG2[perm2[t] * NC2 + NN + NL];
    for (int t = tid; t < NN * NL; t += NT) {
      const int i = t / NL, c = t % NL, f = c / NNF, b = c % NNF;
      double s[D];
      for (int k = 0; k < D; ++k) s[k] = 0.0;
      const double* row = AUG1 + perm1[i] * NC1 + NN;
#pragma unroll 4
      for (int j = 0; j < NN; ++j) {
        const double uj = AUG2[perm2[j] * NC2 + NN + c];
        for (int k = 0; k < D; ++k) s[k] -= row[k * NN + j] * uj;
      }
#pragma unroll 4
      for (int aa = 0; aa < NNF; ++aa) {
        const double mi = row[D * NN + fn[f * NNF + aa]];
        for (int k = 0; k < D; ++k) s[k] += mi * FM[((f * NS + 2 + k) * NNF + aa) * NNF + b];
      }
      for (int k = 0; k < D; ++k) {
        if constexpr (!E::WS) QL[k * NN * NL + t] = s[k];
        Qe[(size_t)(i * D + k) * NL + c] = s[k];
      }
    }
    for (int t = tid; t < D * NN; t += NT) {
      const int k = t / NN, i = t % NN;
      double s = 0.0;
#pragma unroll 4
      for (int j = 0; j < NN; ++j) s -= AUG1[perm1[i] * NC1 + NN + k * NN + j] * AUG2[perm2[j] * NC2 + NN + NL];
      Q0L[t] = s;
      a.Q0[(size_t)e * NN * D + i * D + k] = s;
    }
    __syncthreads();
    // S = Slu U + sum_k Slq_k Q_k + Sll ; S0 = -Slu U0 - sum_k Slq_k Q0_k
    // (explicit HDG modes: S = Sll, S0 = -Slu sol_old - Slq flux_old)
    double* Se = a.S + (size_t)e * NL * NL;
    constexpr int RB = 3, RG = (NNF + RB - 1) / RB;  // RB rows of a face per thread share U and Q
    for (int t = tid; t < NF * RG * NL; t += NT) {
      const int c = t % NL, f = t / (RG * NL), a0 = (t / NL) % RG;
      int au[RB];
      double s[RB];
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        au[u] = a0 + u * RG < NNF ? a0 + u * RG : NNF - 1;
        s[u] = 0.0;
      }
#pragma unroll 4
      for (int b = 0; b < NNF && !a.hdg_explicit; ++b) {
        const int j = fn[f * NNF + b];
        const double uj = AUG2[perm2[j] * NC2 + NN + c];
        double qj[D];
        for (int k = 0; k < D; ++k) qj[k] = E::WS ? Qe[(size_t)(j * D + k) * NL + c] : QL[(k * NN + j) * NL + c];
#pragma unroll
        for (int u = 0; u < RB; ++u) {
          s[u] += FM[((f * NS + 0) * NNF + au[u]) * NNF + b] * uj;
          for (int k = 0; k < D; ++k) s[u] -= FM[((f * NS + 2 + D + k) * NNF + au[u]) * NNF + b] * qj[k];
        }
      }
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        if (a0 + u * RG >= NNF) continue;
        if (c / NNF == f) {
          const int b = c % NNF;
          s[u] += -FM[((f * NS + 0) * NNF + au[u]) * NNF + b] + FM[((f * NS + 1) * NNF + au[u]) * NNF + b];
        }
        Se[(f * NNF + au[u]) * NL + c] = s[u];
      }
    }
    for (int r = tid; r < NL; r += NT) {
      const int f = r / NNF, aa = r % NNF;
      double s = 0.0;
#pragma unroll 4
      for (int b = 0; b < NNF; ++b) {
        const int j = fn[f * NNF + b];
        const double uj = a.hdg_explicit ? a.sol_old[(size_t)e * NN + j] : AUG2[perm2[j] * NC2 + NN + NL];
        s -= FM[((f * NS + 0) * NNF + aa) * NNF + b] * uj;
        for (int k = 0; k < D; ++k) {
          const double qkj = a.hdg_explicit ? a.flux_old[((size_t)e * NN + j) * D + k] : Q0L[k * NN + j];
          s += FM[((f * NS + 2 + D + k) * NNF + aa) * NNF + b] * qkj;
        }
      }
      a.S0[(size_t)e * NL + r] = s;
    }
    __syncthreads();
  }
}

template <int D, int P>
__global__ void ip_coords_kernel(int nEl, const double* __restrict__ tabs, const double* __restrict__ coords,
                                 const int* __restrict__ cells, double* __restrict__ out) {
  using Z = ESz<D, P>;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nEl * Z::NIP) return;
  const int e = (int)(t / Z::NIP), q = (int)(t % Z::NIP);
  double x[D];
  for (int k = 0; k < D; ++k) x[k] = 0.0;
  for (int i = 0; i < Z::NN; ++i) {
    const double ph = tabs[Z::T_PHI + q * Z::NN + i];
    const int node = cells[(size_t)e * Z::NN + i];
    for (int k = 0; k < D; ++k) x[k] += ph * coords[(size_t)node * D + k];
  }
  for (int k = 0; k < D; ++k) out[(size_t)t * D + k] = x[k];
}

template <int D, int P, int NT>
void launch_t(const ElemArgs& a, int grid_cap, hipStream_t s) {
  constexpr bool gws = element_in_workspace<D, P>();
  const size_t lds = ElemLds<D, P>::BYTES;
  auto kern = hdg_element_kernel<D, P, NT>;
  static PerDeviceLaunch once;
  once.lds_attr((const void*)kern, lds);
  int grid = a.nEl;
  if (grid_cap > 0 && grid > grid_cap) grid = grid_cap;
  if (gws) {
    if (!a.gws || a.gws_slots <= 0) throw std::runtime_error("element kernel: this order needs its device workspace");
    if (grid > a.gws_slots) grid = a.gws_slots;
  }
  if (grid <= 0) return;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), lds, s, a);
  HFX_HIP(hipGetLastError());
}

template <int D, int P>
void launch_dp(const ElemArgs& a, int nt, int grid_cap, hipStream_t s) {
  switch (nt) {
    case 64: launch_t<D, P, 64>(a, grid_cap, s); break;
    case 128: launch_t<D, P, 128>(a, grid_cap, s); break;
    case 256: launch_t<D, P, 256>(a, grid_cap, s); break;
    default: throw std::runtime_error("element kernel: threads per element must be 64, 128 or 256");
  }
}

}  // namespace

size_t element_lds_bytes(int dim, int order) {
#define HFX_CASE(D, P) \
  if (dim == D && order == P) return ElemLds<D, P>::BYTES;
  HFX_CASE(2, 1) HFX_CASE(2, 2) HFX_CASE(2, 3) HFX_CASE(2, 4) HFX_CASE(2, 5)
  HFX_CASE(2, 6) HFX_CASE(2, 7) HFX_CASE(2, 8) HFX_CASE(2, 9) HFX_CASE(2, 10)
  HFX_CASE(3, 1) HFX_CASE(3, 2) HFX_CASE(3, 3) HFX_CASE(3, 4) HFX_CASE(3, 5)
#undef HFX_CASE
  throw std::runtime_error("element kernel: (dim, order) not supported on the GPU path");
}

size_t element_workspace_doubles(int dim, int order) {
#define HFX_CASE(D, P) \
  if (dim == D && order == P) return element_in_workspace<D, P>() ? (size_t)Layout<D, P, 64>::TOTAL : 0;
  HFX_CASE(2, 1) HFX_CASE(2, 2) HFX_CASE(2, 3) HFX_CASE(2, 4) HFX_CASE(2, 5)
  HFX_CASE(2, 6) HFX_CASE(2, 7) HFX_CASE(2, 8) HFX_CASE(2, 9) HFX_CASE(2, 10)
  HFX_CASE(3, 1) HFX_CASE(3, 2) HFX_CASE(3, 3) HFX_CASE(3, 4) HFX_CASE(3, 5)
#undef HFX_CASE
  throw std::runtime_error("element kernel: (dim, order) not supported on the GPU path");
}

void launch_element(int dim, int order, const ElemArgs& a, int nt, int grid_cap, hipStream_t s) {
#define HFX_CASE(D, P) \
  if (dim == D && order == P) { launch_dp<D, P>(a, nt, grid_cap, s); return; }
  HFX_CASE(2, 1) HFX_CASE(2, 2) HFX_CASE(2, 3) HFX_CASE(2, 4) HFX_CASE(2, 5)
  HFX_CASE(2, 6) HFX_CASE(2, 7) HFX_CASE(2, 8) HFX_CASE(2, 9) HFX_CASE(2, 10)
  HFX_CASE(3, 1) HFX_CASE(3, 2) HFX_CASE(3, 3) HFX_CASE(3, 4) HFX_CASE(3, 5)
#undef HFX_CASE
  throw std::runtime_error("element kernel: (dim, order) not supported on the GPU path");
}

void launch_ip_coords(int dim, int order, int nEl, const double* tabs, const double* coords, const int* cells,
                      double* out, hipStream_t s) {
#define HFX_CASE(D, P)                                                                                   \
  if (dim == D && order == P) {                                                                          \
    long long n = (long long)nEl * ESz<D, P>::NIP;                                                       \
    if (n > 0) hipLaunchKernelGGL((ip_coords_kernel<D, P>), dim3(ceil_div(n, 256)), dim3(256), 0, s, nEl, \
                                  tabs, coords, cells, out);                                             \
    HFX_HIP(hipGetLastError());                                                                          \
    return;                                                                                              \
  }
  HFX_CASE(2, 1) HFX_CASE(2, 2) HFX_CASE(2, 3) HFX_CASE(2, 4) HFX_CASE(2, 5)
  HFX_CASE(2, 6) HFX_CASE(2, 7) HFX_CASE(2, 8) HFX_CASE(2, 9) HFX_CASE(2, 10)
  HFX_CASE(3, 1) HFX_CASE(3, 2) HFX_CASE(3, 3) HFX_CASE(3, 4) HFX_CASE(3, 5)
#undef HFX_CASE
  throw std::runtime_error("ip coords: (dim, order) not supported on the GPU path");
}

}  // namespace hfx
