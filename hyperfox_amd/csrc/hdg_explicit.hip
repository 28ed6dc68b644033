// Element kernel of an explicit Runge-Kutta stage in the explicit HDG modes, on
// affine (straight-sided) simplices, FP64, one wavefront per cell.
//
// A stage with a_ss = 0 (RungeKutta.cpp:113-159) drops the model's rows from
// the u equation: Suu = mu M, Suq = Sul = 0, so that U = 0 for every trace
// column and nothing has to be factored; U0 = M^-1 F / mu with
//   F = F_u phi + mu M u_old - [Suu | Suq | Sul] w,
// whose last term is evaluated at the cubature points without forming the
// blocks:
//   F_i = sum_q s(q) phi_i + v(q) . grad phi_i + sum over the faces of i of
//         sum_p h(p) psi_i(p),
//   s = w det (phi f + mu u_old - r w_u), v = w det (b w_u - D w_q),
//   h = dS (tau (w_l - w_u) + D n . w_q - b.n w_l).
// The explicit modes then take S = Sll and S0 from the old solution and flux
// (HDGSolver.cpp:346-353):
//   S0 = -sum_p dS psi (tau u - D n . q).
// Q = -B = n rho G and Q0 = -A U0 as in the implicit kernel (hdg_affine.hip),
// which computes the same blocks by the full condensation.
//
// Bound by its stores: U, Q, the trace matrix and the diagonal sides, 38 KB per
// 3-D p=3 cell (3.2 GB for 82,944 cells, 0.65 ms at the copy rate).  Measured
// there: 4.41 ms with the full condensation, 1.19 ms (2.7 TB/s).
#include "hdg_element.h"
#include "hfx_internal.h"
#include "wave.h"

namespace hfx {

template <int D, int P>
struct RefConst;
#include "data/refel_const.inc"

namespace {

// Wavefronts (cells) per workgroup: they share the tables (36 KB at 3-D p=3),
// so 16 of them fit where two workgroups of 4 would.  Measured at the size
// above: 4 waves 1.28 ms, 8 waves 1.32 ms, 12 waves 1.28 ms, 16 waves 1.19 ms.
constexpr int XW = 16;

// The reference tables in the order of the affine kernel's (capi.cpp), with
// Mhat^-1 behind them, and the scratch of one wavefront.
template <int D, int P>
struct XLay {
  using Z = ESz<D, P>;
  static constexpr int NN = Z::NN, NNF = Z::NNF, NIP = Z::NIP, NIPF = Z::NIPF, NF = Z::NF, NL = Z::NL;
  static constexpr int NFP = NF * NIPF;
  static constexpr int T_PHI = 0;
  static constexpr int T_DPHI = T_PHI + NIP * NN;
  static constexpr int T_FPHI = T_DPHI + NIP * NN * D;
  static constexpr int T_W = T_FPHI + NIPF * NNF;
  static constexpr int T_FW = T_W + NIP;
  static constexpr int T_AH = T_FW + NIPF;
  static constexpr int T_G = T_AH + D * NN * NN;
  static constexpr int T_MI = T_G + NF * NN * NNF;
  static constexpr int TAB = T_MI + NN * NN;
  // per wavefront
  static constexpr int O_VX = 0;                       // vertices
  static constexpr int O_DN = O_VX + (D + 1) * D;      // D, b at the nodes
  static constexpr int O_BN = O_DN + NN;
  static constexpr int O_TAU = O_BN + NN * D;          // tau at the face nodes
  static constexpr int O_W = O_TAU + NL;               // w: u, q, lambda
  static constexpr int O_UO = O_W + Z::NLOC;           // u_old
  static constexpr int O_SO = O_UO + NN;               // sol_old, flux_old
  static constexpr int O_FO = O_SO + NN;
  static constexpr int O_FG = O_FO + NN * D;           // per face: n, measure
  static constexpr int O_SV = O_FG + NF * (D + 1);     // [q] s, v in the reference frame
  static constexpr int O_FT = O_SV + NIP * (D + 1);    // face points: dS (b.n - tau), h, S0 integrand
  static constexpr int O_FU = O_FT + 3 * NFP;
  static constexpr int O_U0 = O_FU + NN;
  static constexpr int O_Y = O_U0 + NN;                // Ahat_a U0
  static constexpr int PER = (O_Y + D * NN + 1) & ~1;
};

// FUSED: the trace matrix is written in place (bvals, dside), else S is
// stored.  A template parameter and not a test of a.bvals: as a run-time value
// inside the lane-strided loops the compiler carried the test from one loop to
// the next as a lane mask of the first loop's last, partly filled trip, and
// lanes outside that mask took the other branch (through null pointers).
template <int D, int P, bool FUSED>
__global__ __launch_bounds__(64 * XW) void hdg_explicit_stage_kernel(ElemArgs a) {
  using L = XLay<D, P>;
  using RC = RefConst<D, P>;
  constexpr int NN = L::NN, NNF = L::NNF, NIP = L::NIP, NIPF = L::NIPF, NF = L::NF, NL = L::NL, NFP = L::NFP;
  constexpr int NLOC = L::Z::NLOC;
  extern __shared__ __align__(16) double sm[];
  __shared__ int s_fn[NF * NNF], s_pos[NF * NN];
  for (int t = threadIdx.x; t < L::TAB; t += 64 * XW) sm[t] = a.tabs[t];
  for (int t = threadIdx.x; t < NF * NNF; t += 64 * XW) s_fn[t] = RC::FN[t / NNF][t % NNF];
  for (int t = threadIdx.x; t < NF * NN; t += 64 * XW) s_pos[t] = RC::POS[t / NN][t % NN];
  __syncthreads();
  int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const double *PHI = sm + L::T_PHI, *DPHI = sm + L::T_DPHI, *FPHI = sm + L::T_FPHI, *WQ = sm + L::T_W;
  const double *FWQ = sm + L::T_FW, *AH = sm + L::T_AH, *GT = sm + L::T_G, *MI = sm + L::T_MI;
  double* ws = sm + ((L::TAB + 1) & ~1) + wv * L::PER;
  double *VX = ws + L::O_VX, *DN = ws + L::O_DN, *BN = ws + L::O_BN, *TAU = ws + L::O_TAU, *W = ws + L::O_W;
  double *UO = ws + L::O_UO, *SO = ws + L::O_SO, *FO = ws + L::O_FO, *FG = ws + L::O_FG, *SV = ws + L::O_SV;
  double *FT = ws + L::O_FT, *FU = ws + L::O_FU, *U0 = ws + L::O_U0, *Y = ws + L::O_Y;
  const int e_end = a.el_offset + a.nEl;
  for (int e = a.el_offset + blockIdx.x * XW + wv; e < e_end; e += gridDim.x * XW) {
    // Neither the tables nor the index arithmetic of the loops below are kept in
    // registers from cell to cell (the compiler would hold 490 of them).
    asm volatile("" : "+v"(lane) : : "memory");
    // ------------------------------------------------------------ gather
    const int* cell = a.cells + (size_t)e * NN;
    for (int t = lane; t < (D + 1) * D; t += 64) VX[t] = a.coords[(size_t)cell[t / D] * D + t % D];
    for (int t = lane; t < NN; t += 64) {
      DN[t] = a.ndD == 1 ? a.Dn[cell[t]] : (a.useDiff ? 1.0 : 0.0);
      UO[t] = a.u_old[(size_t)e * NN + t];
      SO[t] = a.sol_old[(size_t)e * NN + t];
    }
    for (int t = lane; t < NN * D; t += 64) {
      BN[t] = a.hasB ? a.bn[(size_t)cell[t / D] * D + t % D] : 0.0;
      FO[t] = a.flux_old[(size_t)e * NN * D + t];
    }
    for (int t = lane; t < NL; t += 64) {
      const int fc = a.cell2face[(size_t)e * NF + t / NNF];
      const int side = (a.tau_sides == 2 && a.face2cell[2 * (size_t)fc] != e) ? 1 : 0;
      TAU[t] = a.tau[((size_t)fc * NNF + a.face_perm[(size_t)e * NL + t]) * a.tau_sides + side];
    }
    for (int t = lane; t < NLOC; t += 64) W[t] = a.ts_w[(size_t)e * NLOC + t];
    wave_sync();
    // --------------------------------------------------- the blocks of zeros
    // first, so that they drain beside the sums below
    for (int t = lane; t < NN * NL; t += 64) __builtin_nontemporal_store(0.0, a.U + (size_t)e * NN * NL + t);
    for (int t = lane; t < NF * NF * NNF * NNF; t += 64) {
      const int fg = t / (NNF * NNF), f = fg / NF, g = fg % NF, ij = t % (NNF * NNF);
      if (f == g) continue;
      if constexpr (FUSED)
        __builtin_nontemporal_store(0.0, a.bvals + (size_t)a.bpos[(size_t)e * NF * NF + fg] * NNF * NNF + ij);
      else
        a.S[((size_t)e * NL + f * NNF + ij / NNF) * NL + g * NNF + ij % NNF] = 0.0;
    }
    // ---------------------------------------------------------- geometry
    double J[D * D], JI[D * D], det;  // J[r][c] = dx_c / dxi_r
    for (int r = 0; r < D; ++r)
      for (int c = 0; c < D; ++c) J[r * D + c] = 0.5 * (VX[(r + 1) * D + c] - VX[c]);
    if constexpr (D == 2) {
      det = J[0] * J[3] - J[1] * J[2];
      const double r = 1.0 / det;
      JI[0] = J[3] * r; JI[1] = -J[1] * r; JI[2] = -J[2] * r; JI[3] = J[0] * r;
    } else {
      det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) + J[2] * (J[3] * J[7] - J[4] * J[6]);
      const double r = 1.0 / det;
      for (int c = 0; c < 3; ++c)
        for (int k = 0; k < 3; ++k) {
          const int c1 = (c + 1) % 3, c2 = (c + 2) % 3, k1 = (k + 1) % 3, k2 = (k + 2) % 3;
          JI[k * 3 + c] = (J[c1 * 3 + k1] * J[c2 * 3 + k2] - J[c1 * 3 + k2] * J[c2 * 3 + k1]) * r;
        }
    }
    if (lane < NF) {
      // face measure and outward unit normal (HDGBase.cpp:34-65)
      const double* x0 = VX + s_fn[lane * NNF] * D;
      double t0[D], nv[D], meas;
      for (int c = 0; c < D; ++c) t0[c] = 0.5 * (VX[s_fn[lane * NNF + 1] * D + c] - x0[c]);
      if constexpr (D == 2) {
        nv[0] = t0[1];
        nv[1] = -t0[0];
        meas = sqrt(nv[0] * nv[0] + nv[1] * nv[1]);
      } else {
        double t1[D];
        for (int c = 0; c < D; ++c) t1[c] = 0.5 * (VX[s_fn[lane * NNF + 2] * D + c] - x0[c]);
        for (int c = 0; c < 3; ++c) nv[c] = t0[(c + 1) % 3] * t1[(c + 2) % 3] - t0[(c + 2) % 3] * t1[(c + 1) % 3];
        meas = sqrt(nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2]);
      }
      int vo = 0;
      for (int i = D; i >= 0; --i)
        if (s_pos[lane * NN + i] < 0) vo = i;
      double prod = 0.0;
      for (int c = 0; c < D; ++c) prod += (VX[vo * D + c] - x0[c]) * nv[c];
      const double sg = (prod > 0 ? -1.0 : 1.0) / meas;
      for (int c = 0; c < D; ++c) FG[lane * (D + 1) + c] = sg * nv[c];
      FG[lane * (D + 1) + D] = meas;
    }
    wave_sync();
    // ------------------------------------------------- cubature points
    for (int q = lane; q < NIP; q += 64) {
      double d = 0.0, b[D], wu = 0.0, wq[D], uo = 0.0;
      for (int k = 0; k < D; ++k) b[k] = wq[k] = 0.0;
      #pragma unroll 4
      for (int i = 0; i < NN; ++i) {
        const double ph = PHI[q * NN + i];
        d += ph * DN[i];
        wu += ph * W[i];
        uo += ph * UO[i];
        for (int k = 0; k < D; ++k) {
          b[k] += ph * BN[i * D + k];
          wq[k] += ph * W[NN + i * D + k];
        }
      }
      const double wd = WQ[q] * det;
      const double f = (a.hasF && a.kind != 0) ? a.f_ip[(size_t)e * NIP + q] : 0.0;
      const double r = a.hasR ? a.r_ip[(size_t)e * NIP + q] : 0.0;
      SV[q * (D + 1)] = wd * (a.ts_phi * f + a.ts_mu * uo - r * wu);
      double v[D];
      for (int k = 0; k < D; ++k) v[k] = wd * (b[k] * wu - d * wq[k]);
      for (int c = 0; c < D; ++c) {  // grad phi = J^-1 (reference gradient)
        double s = 0.0;
        for (int k = 0; k < D; ++k) s += JI[k * D + c] * v[k];
        SV[q * (D + 1) + 1 + c] = s;
      }
    }
    for (int t = lane; t < NFP; t += 64) {
      const int f = t / NIPF, p = t % NIPF;
      const double* n = FG + f * (D + 1);
      double tq = 0.0, bn = 0.0, d = 0.0, wu = 0.0, wl = 0.0, wn = 0.0, us = 0.0, qn = 0.0;
      #pragma unroll 4
      for (int j = 0; j < NNF; ++j) {
        const double ps = FPHI[p * NNF + j];
        const int i = s_fn[f * NNF + j];
        tq += ps * TAU[f * NNF + j];
        d += ps * DN[i];
        wu += ps * W[i];
        wl += ps * W[NN * (D + 1) + f * NNF + j];
        us += ps * SO[i];
        for (int k = 0; k < D; ++k) {
          bn += ps * BN[i * D + k] * n[k];
          wn += ps * W[NN + i * D + k] * n[k];
          qn += ps * FO[i * D + k] * n[k];
        }
      }
      const double ds = FWQ[p] * n[D];
      FT[t] = ds * (bn - tq);
      FT[NFP + t] = ds * (tq * (wl - wu) + d * wn - bn * wl);
      FT[2 * NFP + t] = ds * (d * qn - tq * us);
    }
    wave_sync();
    // ------------------------------------------------------- F and U0, Q0
    for (int i = lane; i < NN; i += 64) {
      double s = 0.0;
      #pragma unroll 4
      for (int q = 0; q < NIP; ++q) {
        s += SV[q * (D + 1)] * PHI[q * NN + i];
        for (int c = 0; c < D; ++c) s += SV[q * (D + 1) + 1 + c] * DPHI[(q * NN + i) * D + c];
      }
      for (int f = 0; f < NF; ++f) {
        const int j = s_pos[f * NN + i];
        if (j < 0) continue;
        #pragma unroll 4
        for (int p = 0; p < NIPF; ++p) s += FT[NFP + f * NIPF + p] * FPHI[p * NNF + j];
      }
      FU[i] = s;
    }
    wave_sync();
    for (int i = lane; i < NN; i += 64) {
      double s = 0.0;
      #pragma unroll 4
      for (int j = 0; j < NN; ++j) s += MI[i * NN + j] * FU[j];
      s /= a.ts_mu * det;
      U0[i] = s;
      a.U0[(size_t)e * NN + i] = s;
    }
    wave_sync();
    for (int t = lane; t < D * NN; t += 64) {
      double s = 0.0;
      #pragma unroll 4
      for (int j = 0; j < NN; ++j) s += AH[t * NN + j] * U0[j];
      Y[t] = s;
    }
    wave_sync();
    for (int t = lane; t < D * NN; t += 64) {
      const int i = t / D, k = t % D;
      double s = 0.0;
      for (int c = 0; c < D; ++c) s -= JI[k * D + c] * Y[c * NN + i];
      a.Q0[(size_t)e * NN * D + t] = s;
    }
    // ------------------------------------------------------------ S, S0
    for (int t = lane; t < NL; t += 64) {
      const int f = t / NNF, j = t % NNF;
      double s = 0.0;
      #pragma unroll 4
      for (int p = 0; p < NIPF; ++p) s += FT[2 * NFP + f * NIPF + p] * FPHI[p * NNF + j];
      a.S0[(size_t)e * NL + t] = s;
    }
    for (int t = lane; t < NF * NNF * NNF; t += 64) {
      const int f = t / (NNF * NNF), i = (t / NNF) % NNF, j = t % NNF;
      double s = 0.0;
      #pragma unroll 4
      for (int p = 0; p < NIPF; ++p) s += FT[f * NIPF + p] * (FPHI[p * NNF + i] * FPHI[p * NNF + j]);
      if constexpr (FUSED) {
        const int F = a.cell2face[(size_t)e * NF + f], side = a.face2cell[2 * (size_t)F] == e ? 0 : 1;
        const int8_t* pm = a.face_perm + (size_t)e * NL + f * NNF;
        __builtin_nontemporal_store(s, a.dside + (size_t)(2 * F + side) * NNF * NNF + pm[i] * NNF + pm[j]);
      } else {
        a.S[((size_t)e * NL + f * NNF + i) * NL + f * NNF + j] = s;
      }
    }
    // --------------------------------------------------------------- Q
    double* Qe = a.Q + (size_t)e * NN * D * NL;
    for (int t = lane; t < NN * NL; t += 64) {
      const int i = t / NL, c = t % NL, g = c / NNF, b = c % NNF;
      const double gb = (FG[g * (D + 1) + D] / det) * GT[(g * NN + i) * NNF + b];
      for (int k = 0; k < D; ++k) __builtin_nontemporal_store(FG[g * (D + 1) + k] * gb, Qe + (size_t)(i * D + k) * NL + c);
    }
    wave_sync();  // the scratch is reused by the next cell
  }
}

template <int D, int P, bool FUSED>
void launch_x(const ElemArgs& a, int grid_cap, hipStream_t s) {
  using L = XLay<D, P>;
  const size_t lds = (size_t)(((L::TAB + 1) & ~1) + XW * L::PER) * sizeof(double);
  auto kern = hdg_explicit_stage_kernel<D, P, FUSED>;
  static PerDeviceLaunch once;
  once.lds_attr((const void*)kern, lds);
  long long grid = ((long long)a.nEl + XW - 1) / XW;
  const long long cap = grid_cap > 0 ? grid_cap : once.resident_wgs((const void*)kern, 64 * XW, lds);
  if (grid > cap) grid = cap;
  if (grid <= 0) return;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * XW), lds, s, a);
  HFX_HIP(hipGetLastError());
}

}  // namespace

bool explicit_stage(const ElemArgs& a) {
  return a.ts_gen && a.ts_auu == 0.0 && a.ts_arest == 0.0 && a.hdg_explicit != 0 && a.ndD <= 1 && a.ts_idt == 0.0;
}

void launch_explicit_stage(int dim, int order, const ElemArgs& a, int grid_cap, hipStream_t s) {
#define HFX_CASE(D, P)                 \
  if (dim == D && order == P) {        \
    if (a.bvals) launch_x<D, P, true>(a, grid_cap, s);  \
    else launch_x<D, P, false>(a, grid_cap, s);         \
    return;                            \
  }
  HFX_CASE(2, 1) HFX_CASE(2, 2) HFX_CASE(2, 3) HFX_CASE(2, 4) HFX_CASE(2, 5)
  HFX_CASE(3, 1) HFX_CASE(3, 2) HFX_CASE(3, 3)
#undef HFX_CASE
  throw std::runtime_error("explicit stage kernel: (dim, order) not supported");
}

}  // namespace hfx
