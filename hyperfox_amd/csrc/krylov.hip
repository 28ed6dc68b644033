// FP64 Krylov solvers for the trace system.  See krylov.h.
#include <cmath>
#include <vector>

#include "bsr_row.h"
#include "krylov.h"
#include "wave.h"

namespace hfx {

namespace {

constexpr int RT = 256;  // reduction block size

// sum over the wavefront, valid in lane 0: the tree of lane distances 32, 16,
// 8, .., 1, the steps inside a row of 16 lanes as
// DPP moves (row_shl)
__device__ __forceinline__ double wave_sum(double v) {
  v += __shfl_down(v, 32, 64);
  v += __shfl_down(v, 16, 64);
  v += dpp_move<0x108, true>(v);
  v += dpp_move<0x104, true>(v);
  v += dpp_move<0x102, true>(v);
  v += dpp_move<0x101, true>(v);
  return v;
}

// Partials of one dot product are added up by SV = 1024 (real or virtual)
// threads, strided, then wave by wave: the same order, and so the same bits,
// in the one-block kernel (reduce_partials_kernel) and in partial_sums below.
constexpr int SV = 1024;

// block-wide sum, result valid in thread 0
__device__ inline double block_sum(double v, double* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
  __syncthreads();
  return s;
}

template <int BS>
__global__ void spmv_kernel(int nb, const int* __restrict__ rowptr, const int* __restrict__ col,
                            const double* __restrict__ vals, const double* __restrict__ x,
                            const double* __restrict__ b, double* __restrict__ y) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nb * BS) return;
  const int F = (int)(t / BS), r = (int)(t % BS);
  const double acc = bsr_row_sum<BS>(rowptr[F], rowptr[F + 1], r, col, vals, x);
  y[t] = b ? b[t] - acc : acc;
}

// Inverses of the diagonal blocks by Gauss-Jordan with partial pivoting: one
// matrix row per lane in registers, 64 / BS blocks per wavefront.  The
// elimination is in place (column k of the block makes room for the column of
// the inverse that belongs to the pivot row) and swaps no rows: every lane
// scans its block's column k in LDS for the first unused row of largest
// magnitude (a NaN never wins), and the pivot row is broadcast through LDS.
// 169,344 blocks of 10 x 10 (271 MB read and written, 0.06 ms at the copy
// rate): 1.73 ms with one block per thread, whose two arrays lived in
// scratch memory, 0.11 ms now.
constexpr int IW = 4;  // wavefronts per workgroup

template <int BS>
__global__ __launch_bounds__(64 * IW) void invert_diag_kernel(int nb, const int* __restrict__ diag,
                                                              const double* __restrict__ vals,
                                                              double* __restrict__ dinv) {
  constexpr int G = 64 / BS;
  __shared__ double s_col[IW][G * BS], s_row[IW][G * BS];
  __shared__ int s_perm[IW][G * BS];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int g = lane < G * BS ? lane / BS : G - 1, r = lane < G * BS ? lane % BS : BS - 1;
  const int F = (blockIdx.x * IW + wv) * G + g;
  const bool on = lane < G * BS && F < nb;  // the other lanes follow along without stores
  double* col = s_col[wv] + g * BS;
  double* row = s_row[wv] + g * BS;
  int* perm = s_perm[wv] + g * BS;
  const double* src = vals + (size_t)diag[F < nb ? F : nb - 1] * BS * BS + r * BS;
  double a[BS];
#pragma unroll
  for (int c = 0; c < BS; ++c) a[c] = src[c];
  bool used = false;
  int myk = 0;
#pragma unroll
  for (int k = 0; k < BS; ++k) {
    if (lane < G * BS) {
      const double v = fabs(a[k]);
      col[r] = used ? -2.0 : (v >= 0.0 ? v : -1.0);
    }
    wave_sync();
    int p = 0;
    double best = col[0];
#pragma unroll
    for (int i = 1; i < BS; ++i) {
      const double v = col[i];
      p = v > best ? i : p;
      best = v > best ? v : best;
    }
    const bool piv = r == p;
    if (piv) {
      const double inv = 1.0 / a[k];
#pragma unroll
      for (int c = 0; c < BS; ++c) a[c] = c == k ? inv : a[c] * inv;
      used = true;
      myk = k;
      if (lane < G * BS) {
#pragma unroll
        for (int c = 0; c < BS; ++c) row[c] = a[c];
        perm[k] = r;
      }
    }
    wave_sync();
    if (!piv) {
      const double f = a[k];
#pragma unroll
      for (int c = 0; c < BS; ++c) a[c] = c == k ? -f * row[c] : fma(-f, row[c], a[c]);
    }
  }
  wave_sync();
  if (on) {
    double* dst = dinv + ((size_t)F * BS + myk) * BS;
#pragma unroll
    for (int c = 0; c < BS; ++c) dst[perm[c]] = a[c];
  }
}

__global__ void point_diag_kernel(int nb, int bs, const int* __restrict__ diag, const double* __restrict__ vals,
                                  double* __restrict__ dinv) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nb * bs) return;
  const int F = (int)(t / bs), r = (int)(t % bs);
  const double d = vals[((size_t)diag[F] * bs + r) * bs + r];
  dinv[t] = d != 0.0 ? 1.0 / d : 1.0;
}

template <int BS>
__global__ void block_diag_apply_kernel(int nb, const double* __restrict__ dinv, const double* __restrict__ x,
                                        double* __restrict__ y) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nb * BS) return;
  const int F = (int)(t / BS), r = (int)(t % BS);
  y[t] = bsr_row_dot<BS>(dinv + ((size_t)F * BS + r) * BS, x + (size_t)F * BS);
}

__global__ void point_diag_apply_kernel(long long n, const double* __restrict__ d, const double* __restrict__ x,
                                        double* __restrict__ y) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] = d[t] * x[t];
}

// partial[blk] = sum over this block's slice of x . x
__global__ void norm2_kernel(long long n, const double* __restrict__ x, double* __restrict__ partial) {
  __shared__ double red[RT / 64];
  const int G = gridDim.x;
  double acc = 0.0;
  for (long long i = (long long)blockIdx.x * RT + threadIdx.x; i < n; i += (long long)G * RT) acc += x[i] * x[i];
  double s = block_sum(acc, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// out[j] = sum_b partial[j*G + b], fixed order
__global__ void reduce_rows_kernel(int G, const double* __restrict__ partial, double* __restrict__ out) {
  __shared__ double red[RT / 64];
  const int j = blockIdx.x;
  double acc = 0.0;
  for (int b = threadIdx.x; b < G; b += RT) acc += partial[(size_t)j * G + b];
  double s = block_sum(acc, red);
  if (threadIdx.x == 0) out[j] = s;
}

// ---------------------------------------------------------------- BiCGStab
//
// Scalars live on the device (no host round trip per iteration), in two slots
// used by even and odd iterations, so that a block that still reads the last
// iteration's values never races with the block that writes the new ones:
//   sc[8 par + 0] rho = (rhat, r)   sc[8 par + 1] alpha   sc[8 par + 2] omega
//   sc[SC_BRK] breakdown flag (1 when a denominator vanished)
//   sc[SC_STOP] (an int) set by the check kernel: every later kernel returns
//   at once, so the host may run ahead of the check without changing x
//   sc[SC_SUMS..+1], sc[SC_XSUMS..+1] reduced partials of a long vector (the
//   products with A, the x/r update)
// The dot products arrive as one partial per block of the kernel before; each
// block of the kernel that needs the scalar adds them up again in the same
// order (a few KB out of L2, behind its own vector loads) instead of waiting
// for a one-block kernel in between.
enum { SC_RHO = 0, SC_ALPHA, SC_OMEGA, SC_BRK = 16, SC_STOP = 24, SC_STATUS = 26, SC_XSUMS = 28, SC_SUMS = 30, SC_N = 32 };

__device__ __forceinline__ bool stopped(const double* sc) { return *reinterpret_cast<const int*>(sc + SC_STOP) != 0; }

// The sums of part[0..np) and (two) part[np..2 np), np <= 2 SV, in every
// thread; each of the RT threads stands for SV / RT threads of the one-block
// kernel.
__device__ __forceinline__ void partial_sums(int np, const double* __restrict__ part, bool two, double& d0, double& d1,
                                             double (*red)[SV / 64]) {
  constexpr int NV = SV / RT;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  // every load in flight at once, then the NV (or 2 NV) independent trees
  double a[NV], c[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int b = v * RT + threadIdx.x;
    a[v] = b < np ? part[b] : 0.0;
    c[v] = two && b < np ? part[np + b] : 0.0;
    if (np > SV) {
      a[v] += b + SV < np ? part[b + SV] : 0.0;
      c[v] += two && b + SV < np ? part[np + b + SV] : 0.0;
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (v * RT >= np) break;  // the rest are zeros
    a[v] = wave_sum(a[v]);
    if (two) c[v] = wave_sum(c[v]);
  }
  if (lane == 0)
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      red[0][v * (RT / 64) + wid] = a[v];
      red[1][v * (RT / 64) + wid] = c[v];
    }
  __syncthreads();
  d0 = d1 = 0.0;
  const int nw = min(NV, (np + RT - 1) / RT) * (RT / 64);
  for (int w = 0; w < nw; ++w) {
    d0 += red[0][w];
    if (two) d1 += red[1][w];
  }
}

// partial[j * G + blk] = sum over the block's slice of a_j . b_j, j < nd
__global__ void dots_kernel(long long n, int nd, const double* __restrict__ a0, const double* __restrict__ b0,
                            const double* __restrict__ a1, const double* __restrict__ b1,
                            double* __restrict__ partial) {
  __shared__ double red[RT / 64];
  const int G = gridDim.x;
  double s0 = 0.0, s1 = 0.0;
  for (long long i = (long long)blockIdx.x * RT + threadIdx.x; i < n; i += (long long)G * RT) {
    s0 += a0[i] * b0[i];
    if (nd > 1) s1 += a1[i] * b1[i];
  }
  double t0 = block_sum(s0, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t0;
  if (nd > 1) {
    __syncthreads();
    double t1 = block_sum(s1, red);
    if (threadIdx.x == 0) partial[G + blockIdx.x] = t1;
  }
}

// out[j] = sum of partial row j (np values), j < nd: one workgroup of SV
// threads, several loads in flight per thread
__global__ __launch_bounds__(SV) void reduce_partials_kernel(int np, int nd, const double* __restrict__ partial,
                                                             const double* __restrict__ sc, double* __restrict__ out) {
  __shared__ double red[SV / 64];
  if (stopped(sc)) return;
  for (int j = 0; j < nd; ++j) {
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    const double* pj = partial + (size_t)j * np;
    int b = threadIdx.x;
    for (; b + 3 * SV < np; b += 4 * SV) {
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] += pj[b + u * SV];
    }
    for (; b < np; b += SV) acc[0] += pj[b];
    const double d = block_sum((acc[0] + acc[1]) + (acc[2] + acc[3]), red);
    if (threadIdx.x == 0) out[j] = d;
    __syncthreads();
  }
}

// Rows of one tile of a vector kernel: with face-block Jacobi fused in
// (PC_BJACOBI) a tile holds whole face blocks, so that their values meet in LDS.
template <int PC, int BS>
constexpr int tile_rows() {
  return PC == PC_BJACOBI ? (RT / BS) * BS : RT;
}

// out[t] = (M x)[t] for the tile's value x of row t (in range when on); every
// thread of the block calls it.  PC_NONE copies, PC_JACOBI scales, PC_BJACOBI
// multiplies by the block's inverse; any other kind (a preconditioner that
// runs on its own) leaves out alone.
template <int PC, int BS>
__device__ __forceinline__ void apply_tile(bool on, long long t, double x, const double* __restrict__ dinv,
                                           double* __restrict__ out, double* xs) {
  if constexpr (PC == PC_NONE) {
    if (on) out[t] = x;
  } else if constexpr (PC == PC_JACOBI) {
    if (on) out[t] = dinv[t] * x;
  } else if constexpr (PC == PC_BJACOBI) {
    if (threadIdx.x < tile_rows<PC, BS>()) xs[threadIdx.x] = x;
    __syncthreads();
    if (on) out[t] = bsr_row_dot<BS>(dinv + (size_t)t * BS, xs + (threadIdx.x / BS) * BS);
  }
}

// p = r + beta (p - omega v), beta = (rho / rho_prev) (alpha / omega)
// (first = 1: p = r); p^ = M p.  rho comes from the partials part of
// (rhat, r), (r, r).
template <int PC, int BS>
__global__ __launch_bounds__(RT) void bicg_p_kernel(long long n, int first, int par, int np,
                                                    const double* __restrict__ part, double* __restrict__ sc,
                                                    const double* __restrict__ r, double* __restrict__ p,
                                                    const double* __restrict__ v, const double* __restrict__ dinv,
                                                    double* __restrict__ ph) {
  __shared__ double red[2][SV / 64];
  __shared__ double xs[PC == PC_BJACOBI ? RT : 1];
  if (stopped(sc)) return;
  constexpr int TR = tile_rows<PC, BS>();
  const long long t = (long long)blockIdx.x * TR + threadIdx.x;
  const bool on = threadIdx.x < TR && t < n;
  double x = 0.0, pv = 0.0, vv = 0.0;  // on their way while the partials are added up
  if (on) {
    x = r[t];
    if (!first) {
      pv = p[t];
      vv = v[t];
    }
  }
  const double* old = sc + 8 * (par ^ 1);
  const double rp = old[SC_RHO], al = old[SC_ALPHA], om = old[SC_OMEGA];
  double rho, unused;
  partial_sums(np, part, false, rho, unused, red);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc[8 * par + SC_RHO] = rho;
    if (rho == 0.0) sc[SC_BRK] = 1.0;
  }
  const double beta = (!first && rp != 0.0 && om != 0.0) ? (rho / rp) * (al / om) : 0.0;
  if (!first) x += beta * (pv - om * vv);
  if (on) p[t] = x;
  apply_tile<PC, BS>(on, t, x, dinv, ph, xs);
}

// alpha = rho / (rhat, v); s = r - alpha v; s^ = M s.  (rhat, v) from part.
template <int PC, int BS>
__global__ __launch_bounds__(RT) void bicg_s_kernel(long long n, int par, int np, const double* __restrict__ part,
                                                    double* __restrict__ sc, const double* __restrict__ r,
                                                    const double* __restrict__ v, double* __restrict__ s,
                                                    const double* __restrict__ dinv, double* __restrict__ sh) {
  __shared__ double red[2][SV / 64];
  __shared__ double xs[PC == PC_BJACOBI ? RT : 1];
  if (stopped(sc)) return;
  constexpr int TR = tile_rows<PC, BS>();
  const long long t = (long long)blockIdx.x * TR + threadIdx.x;
  const bool on = threadIdx.x < TR && t < n;
  const double rt = on ? r[t] : 0.0, vt = on ? v[t] : 0.0;
  double rv, unused;
  partial_sums(np, part, false, rv, unused, red);
  const bool bad = rv == 0.0 || !isfinite(rv);
  const double al = bad ? 0.0 : sc[8 * par + SC_RHO] / rv;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc[8 * par + SC_ALPHA] = al;
    if (bad) sc[SC_BRK] = 1.0;
  }
  const double x = rt - al * vt;
  if (on) s[t] = x;
  apply_tile<PC, BS>(on, t, x, dinv, sh, xs);
}

// omega = (t, s) / (t, t) from part; x += alpha p^ + omega s^; r = s - omega t,
// with the block partials of rhat . r and r . r in out
__global__ __launch_bounds__(RT) void bicg_xr_dot_kernel(long long n, int par, int np, const double* __restrict__ part,
                                                         double* __restrict__ sc, const double* __restrict__ ph,
                                                         const double* __restrict__ sh, const double* __restrict__ s,
                                                         const double* __restrict__ tv, const double* __restrict__ rh,
                                                         double* __restrict__ x, double* __restrict__ r,
                                                         double* __restrict__ out) {
  __shared__ double red[2][SV / 64];
  if (stopped(sc)) return;
  const long long t = (long long)blockIdx.x * RT + threadIdx.x;
  const bool on = t < n;
  double xv = 0.0, pv = 0.0, hv = 0.0, sv = 0.0, tt_ = 0.0, rhv = 0.0;
  if (on) {
    xv = x[t];
    pv = ph[t];
    hv = sh[t];
    sv = s[t];
    tt_ = tv[t];
    rhv = rh[t];
  }
  double ts, tt;
  partial_sums(np, part, true, ts, tt, red);
  const bool bad = tt == 0.0 || !isfinite(tt);
  const double al = sc[8 * par + SC_ALPHA], om = bad ? 0.0 : ts / tt;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc[8 * par + SC_OMEGA] = om;
    if (om == 0.0) sc[SC_BRK] = 1.0;
  }
  double a1 = 0.0, a2 = 0.0;
  if (on) {
    x[t] = xv + (al * pv + om * hv);
    const double rv = sv - om * tt_;
    r[t] = rv;
    a1 = rhv * rv;
    a2 = rv * rv;
  }
  __shared__ double red1[RT / 64];
  const double s1 = block_sum(a1, red1);
  if (threadIdx.x == 0) out[blockIdx.x] = s1;
  __syncthreads();
  const double s2 = block_sum(a2, red1);
  if (threadIdx.x == 0) out[gridDim.x + blockIdx.x] = s2;
}

// The recurrence residual after an iteration: (rhat, r) and (r, r) from part;
// sets the stop flag on convergence, a breakdown or a value that is not
// finite, and reports to the host.
__global__ __launch_bounds__(RT) void bicg_check_kernel(int np, const double* __restrict__ part, double target, int seq,
                                                        double* __restrict__ sc, KrylovStatus* __restrict__ st) {
  __shared__ double red[2][SV / 64];
  double rho, rr;
  partial_sums(np, part, true, rho, rr, red);
  if (threadIdx.x != 0) return;
  const int code = !isfinite(rr) ? 2 : (sqrt(fabs(rr)) <= target || rho == 0.0 || sc[SC_BRK] != 0.0) ? 1 : 0;
  *reinterpret_cast<int*>(sc + SC_STOP) = code;
  __hip_atomic_store(&st->code, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&st->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// y = A x (thread per row) with the block partials of w1 . y (and y . y when
// `both`) in partial[blk] (and partial[gridDim.x + blk]): the SpMV of a
// BiCGStab step and its dot products in one pass.
template <int BS>
__global__ __launch_bounds__(RT) void spmv_dot_kernel(int nb, const int* __restrict__ rowptr,
                                                      const int* __restrict__ col, const double* __restrict__ vals,
                                                      const double* __restrict__ x, double* __restrict__ y,
                                                      const double* __restrict__ w1, int both,
                                                      const double* __restrict__ sc, double* __restrict__ partial) {
  __shared__ double red[RT / 64];
  if (stopped(sc)) return;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  double a1 = 0.0, a2 = 0.0;
  if (t < (long long)nb * BS) {
    const int F = (int)(t / BS), r = (int)(t % BS);
    const double acc = bsr_row_sum<BS>(rowptr[F], rowptr[F + 1], r, col, vals, x);
    y[t] = acc;
    a1 = w1[t] * acc;
    a2 = acc * acc;
  }
  const double s1 = block_sum(a1, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = s1;
  if (both) {
    __syncthreads();
    const double s2 = block_sum(a2, red);
    if (threadIdx.x == 0) partial[gridDim.x + blockIdx.x] = s2;
  }
}

__global__ void set_scalars_kernel(double* __restrict__ sc) {
  if (threadIdx.x < SC_N) sc[threadIdx.x] = 0.0;
}

// ------------------------------------------------------------------ GMRES
//
// One Arnoldi step is four launches (and the preconditioner's own, where it is
// not fused): normalise v_j and apply M; w = A z with the products V^T w; one
// pass that subtracts V h and forms V^T w again (the re-orthogonalisation); one
// that subtracts the second h and forms the norm.  V is read three times.  The
// Hessenberg column, its Givens rotations and the stopping test run on the
// device, in a spare block of the next step's product, so the host only limits
// how far it runs ahead.  Once the test has set the done flag every later
// kernel returns at once.  The flag changes while a product kernel runs, so the
// product reads a copy that the v kernel before it makes.
//
// State gs (doubles): cs, sn, g, h1, h2, y (64 or 65 each), R (column c at
// c * 64), the last norm^2 and three ints: done, columns finished, the copy.
enum { GM_CS = 0, GM_SN = 64, GM_G = 128, GM_H1 = 196, GM_H2 = 260, GM_Y = 324, GM_NORM2 = 388, GM_FLAGS = 390,
       GM_R = 392, GM_N = 392 + 64 * 64 };
enum { GM_DONE = 0, GM_COLS = 1, GM_SEEN = 2 };  // ints at gs + GM_FLAGS

__device__ __forceinline__ int gm_flag(const double* gs, int which) {
  return reinterpret_cast<const int*>(gs + GM_FLAGS)[which];
}

// Finish column c of the Hessenberg matrix (h1 + h2 and the norm): apply the
// earlier rotations, make the new one, test for convergence.  One wavefront,
// row i of the column in lane i.
__device__ inline void gm_column(int c, double norm2, double target, int seq, double* gs, KrylovStatus* st) {
  const int lane = threadIdx.x;
  double h = lane <= c ? gs[GM_H1 + lane] + gs[GM_H2 + lane] : 0.0;
  const double cs = gs[GM_CS + lane], sn = gs[GM_SN + lane];
  const double hn = sqrt(norm2);
  double t = lane_value(h, 0);
  for (int i = 0; i < c; ++i) {
    const double a1 = lane_value(h, i + 1), ci = lane_value(cs, i), si = lane_value(sn, i);
    const double ri = ci * t + si * a1;
    t = -si * t + ci * a1;
    if (lane == i) h = ri;
  }
  const double rr = hypot(t, hn);
  const double cc = rr != 0.0 ? t / rr : 1.0, sc = rr != 0.0 ? hn / rr : 0.0;
  if (lane == c) h = rr;
  if (lane <= c) gs[GM_R + c * 64 + lane] = h;
  if (lane == 0) {
    const double g = gs[GM_G + c], g1 = -sc * g;
    gs[GM_CS + c] = cc;
    gs[GM_SN + c] = sc;
    gs[GM_G + c] = cc * g;
    gs[GM_G + c + 1] = g1;
    const int done = !isfinite(g1) || fabs(g1) <= target || hn == 0.0;
    int* f = reinterpret_cast<int*>(gs + GM_FLAGS);
    f[GM_DONE] = done;
    f[GM_COLS] = c + 1;
    __hip_atomic_store(&st->code, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&st->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__global__ void gm_start_kernel(double beta, double* __restrict__ gs) {
  for (int i = threadIdx.x; i < GM_R; i += blockDim.x) gs[i] = i == GM_G ? beta : 0.0;
}

// v_j = w / ||w|| (||w||^2 from part; j = 0: r / beta), z = M v_j
template <int PC, int BS>
__global__ __launch_bounds__(RT) void gm_v_kernel(long long n, int j, double ibeta, int np,
                                                  const double* __restrict__ part, const double* __restrict__ w,
                                                  const double* __restrict__ dinv, double* __restrict__ v,
                                                  double* __restrict__ z, double* __restrict__ gs) {
  __shared__ double red[2][SV / 64];
  __shared__ double xs[PC == PC_BJACOBI ? RT : 1];
  if (gm_flag(gs, GM_DONE)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) reinterpret_cast<int*>(gs + GM_FLAGS)[GM_SEEN] = 1;
    return;
  }
  constexpr int TR = tile_rows<PC, BS>();
  const long long t = (long long)blockIdx.x * TR + threadIdx.x;
  const bool on = threadIdx.x < TR && t < n;
  double x = on ? w[t] : 0.0;
  if (j == 0) {
    x *= ibeta;
  } else {
    double norm2, unused;
    partial_sums(np, part, false, norm2, unused, red);
    const double nv = sqrt(norm2);
    x = nv > 0.0 ? x / nv : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) gs[GM_NORM2] = norm2;
  }
  if (on) v[t] = x;
  apply_tile<PC, BS>(on, t, x, dinv, z, xs);
}

// Sums over the wavefront of KC values per lane at once: each step halves the
// values a lane holds and exchanges the other half (KC - 1 exchanges for all
// of them, against 6 KC for KC separate trees).  The sum of value
// sum_index<KC>(lane) ends in every lane of its group.
template <int KC>
__device__ __forceinline__ double wave_sums(double* v) {
  const int lane = threadIdx.x & 63;
  int m = 32;
#pragma unroll
  for (int K = KC / 2; K >= 1; K >>= 1, m >>= 1) {
    const bool up = (lane & m) != 0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const double keep = up ? v[i + K] : v[i], send = up ? v[i] : v[i + K];
      v[i] = keep + __shfl_xor(send, m, 64);
    }
  }
  double s = v[0];
  for (; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  return s;
}
template <int KC>
__device__ __forceinline__ int sum_index(int lane) {
  int idx = 0, m = 32;
#pragma unroll
  for (int K = KC / 2; K >= 1; K >>= 1, m >>= 1) idx += (lane & m) ? K : 0;
  return idx;
}

// v[i] = V_(c0 + i)[t], 0 from column k on: loads at clamped columns, so that
// they issue back to back without branches
template <int KC>
__device__ __forceinline__ void load_rows(const double* __restrict__ V, long long ldv, int c0, int k, long long t,
                                          double* v) {
#pragma unroll
  for (int i = 0; i < KC; ++i) v[i] = V[(size_t)min(c0 + i, k - 1) * ldv + t];
#pragma unroll
  for (int i = 0; i < KC; ++i) v[i] = c0 + i < k ? v[i] : 0.0;
}

// partial[(c0 + i) nblk + blk] = sum over the block of v[i], c0 + i < k
template <int KC>
__device__ __forceinline__ void block_sums(double* v, int c0, int k, double* __restrict__ partial, int nblk, int blk,
                                           double (*red)[KC]) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const double s = wave_sums<KC>(v);
  __syncthreads();  // red is free
  if ((lane & (64 / KC - 1)) == 0) red[wid][sum_index<KC>(lane)] = s;
  __syncthreads();
  if (threadIdx.x < KC && c0 + threadIdx.x < k) {
    double a = 0.0;
#pragma unroll
    for (int q = 0; q < RT / 64; ++q) a += red[q][threadIdx.x];
    partial[(size_t)(c0 + threadIdx.x) * nblk + blk] = a;
  }
}

// w = A z (thread per row) with the partials of V_i . w, i < k, in
// partial[i nblk + blk]; block nblk finishes Hessenberg column k - 2.
// Chunks of KC basis rows: eight, at every size (see gm_orth_kernel).
template <int BS>
__global__ __launch_bounds__(RT) void gm_product_kernel(int nb, const int* __restrict__ rowptr,
                                                        const int* __restrict__ col, const double* __restrict__ vals,
                                                        const double* __restrict__ z, double* __restrict__ w, int k,
                                                        const double* __restrict__ V, long long ldv, int nblk,
                                                        double* __restrict__ partial, double target, int seq,
                                                        double* gs, KrylovStatus* st) {
  constexpr int KC = 8;
  __shared__ double red[RT / 64][KC];
  if (gm_flag(gs, GM_SEEN)) return;
  if ((int)blockIdx.x == nblk) {
    if (threadIdx.x < 64) gm_column(k - 2, gs[GM_NORM2], target, seq, gs, st);
    return;
  }
  const long long t = (long long)blockIdx.x * RT + threadIdx.x;
  const bool on = t < (long long)nb * BS;
  double acc = 0.0;
  if (on) {
    const int F = (int)(t / BS), r = (int)(t % BS);
    acc = bsr_row_sum<BS>(rowptr[F], rowptr[F + 1], r, col, vals, z);
    w[t] = acc;
  }
  const long long tc = on ? t : 0;
  for (int c0 = 0; c0 < k; c0 += KC) {
    double v[KC];
    load_rows<KC>(V, ldv, c0, k, tc, v);
#pragma unroll
    for (int i = 0; i < KC; ++i) v[i] *= acc;
    block_sums<KC>(v, c0, k, partial, nblk, blockIdx.x, red);
  }
}

// h[i] = sum of the np partials of row i, i < k, in LDS (np = 1: already
// reduced); block 0 keeps them for the Hessenberg column
__device__ __forceinline__ void gather_h(int k, int np, const double* __restrict__ part, double* hs,
                                         double* __restrict__ keep) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (np == 1) {
    if (threadIdx.x < k) hs[threadIdx.x] = part[threadIdx.x];
  } else {
    constexpr int U = 8;  // rows per wavefront at a time, their loads in flight together
    for (int i0 = wid * U; i0 < k; i0 += RT / 64 * U) {
      double a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double* row = part + (size_t)min(i0 + u, k - 1) * np;
        a[u] = row[min(lane, np - 1)];
        a[u] = lane < np ? a[u] : 0.0;
        for (int b = lane + 64; b < np; b += 64) a[u] += row[b];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = wave_sum(a[u]);
      if (lane == 0)
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (i0 + u < k) hs[i0 + u] = a[u];
    }
  }
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x < k) keep[threadIdx.x] = hs[threadIdx.x];
}

// w -= V h, then the partials of V_i . w: the V values of a row stay in
// registers between the two (up to KC of them; from KC on they are read again).
// Few rows in registers, and so more wavefronts, beat one read of the basis:
// with chunks of 8 in the product and 8 (k <= 8) or 16 here, 126 steps take, in
// ms at restart 30 / 63 (in brackets with chunks of 32 from k = 17 on),
//      37 blocks  3.9 / 5.2 (3.9 / 5.4)     340 blocks   4.4 /  6.6 (5.1 /  8.2)
//   1,333 blocks 13.3 / 18.5 (16.0 / 26.1)  3,391 blocks 20.7 / 32.5 (27.7 / 52.1)
// (block sizes 3, 2, 10 and 2, block Jacobi), the larger two 20.7 / 26.8 and
// 23.6 / 36.0 before the four-launch steps.  The order of every sum is the same.
template <int KC>
__global__ __launch_bounds__(RT) void gm_orth_kernel(long long n, int k, const double* __restrict__ V, long long ldv,
                                                     int np, const double* __restrict__ part, double* __restrict__ w,
                                                     int nblk, double* __restrict__ partial, double* gs) {
  __shared__ double hs[64];
  __shared__ double red[RT / 64][KC];
  if (gm_flag(gs, GM_DONE)) return;
  const long long t = (long long)blockIdx.x * RT + threadIdx.x;
  const bool on = t < n;
  double x = on ? w[t] : 0.0;
  const long long tc = on ? t : 0;
  double v[KC];
  load_rows<KC>(V, ldv, 0, k, tc, v);
  gather_h(k, np, part, hs, gs + GM_H1);
#pragma unroll
  for (int i = 0; i < KC; ++i) x -= (i < k ? hs[i] : 0.0) * v[i];
  for (int i = KC; i < k; ++i) x -= hs[i] * V[(size_t)i * ldv + tc];
  if (!on) x = 0.0;
  if (on) w[t] = x;
  for (int c0 = 0; c0 < k; c0 += KC) {
    if (c0 > 0) load_rows<KC>(V, ldv, c0, k, tc, v);
#pragma unroll
    for (int i = 0; i < KC; ++i) v[i] *= x;
    block_sums<KC>(v, c0, k, partial, nblk, blockIdx.x, red);
  }
}

// w -= V h, with the partials of w . w
__global__ __launch_bounds__(RT) void gm_norm_kernel(long long n, int k, const double* __restrict__ V, long long ldv,
                                                     int np, const double* __restrict__ part, double* __restrict__ w,
                                                     double* __restrict__ partial, double* gs) {
  __shared__ double hs[64];
  __shared__ double red[RT / 64];
  if (gm_flag(gs, GM_DONE)) return;
  const long long t = (long long)blockIdx.x * RT + threadIdx.x;
  const bool on = t < n;
  double x = on ? w[t] : 0.0;
  gather_h(k, np, part, hs, gs + GM_H2);
  if (on) {
#pragma unroll 8
    for (int i = 0; i < k; ++i) x -= hs[i] * V[(size_t)i * ldv + t];
    w[t] = x;
  }
  const double s = block_sum(x * x, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// End of a cycle: finish the last column (c, when the done flag has not cut
// the cycle short), then back substitution R y = g
__global__ __launch_bounds__(RT) void gm_finish_kernel(int c, int np, const double* __restrict__ part, double target,
                                                       int seq, double* gs, KrylovStatus* st) {
  __shared__ double red[2][SV / 64];
  double norm2, unused;
  partial_sums(np, part, false, norm2, unused, red);
  if (threadIdx.x >= 64) return;
  if (!gm_flag(gs, GM_DONE)) gm_column(c, norm2, target, seq - 1, gs, st);
  __threadfence_block();
  __builtin_amdgcn_wave_barrier();
  const int lane = threadIdx.x, k = reinterpret_cast<const volatile int*>(gs + GM_FLAGS)[GM_COLS];
  double g = lane < k ? gs[GM_G + lane] : 0.0, y = 0.0;
  for (int i = k - 1; i >= 0; --i) {
    const double ri = lane <= i ? gs[GM_R + i * 64 + lane] : 0.0;
    const double d = lane_value(ri, i), yi = d != 0.0 ? lane_value(g, i) / d : 0.0;
    if (lane == i) y = yi;
    if (lane < i) g -= ri * yi;
  }
  gs[GM_Y + lane] = y;
  if (lane == 0) {
    __hip_atomic_store(&st->code, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&st->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// x += sum_j y_j Z_j over the columns of the cycle
__global__ __launch_bounds__(RT) void gm_combine_kernel(long long n, const double* __restrict__ Z, long long ldz,
                                                        const double* __restrict__ gs, double* __restrict__ x) {
  __shared__ double ys[64];
  const int k = gm_flag(gs, GM_COLS);
  if (threadIdx.x < 64) ys[threadIdx.x] = gs[GM_Y + threadIdx.x];
  __syncthreads();
  const long long t = (long long)blockIdx.x * RT + threadIdx.x;
  if (t >= n) return;
  double acc = x[t];
#pragma unroll 8
  for (int j = 0; j < k; ++j) acc += ys[j] * Z[(size_t)j * ldz + t];
  x[t] = acc;
}

}  // namespace

void bsr_spmv(const BsrDev& A, const double* x, double* y, const double* b, hipStream_t s) {
  const long long n = A.nrows();
  if (n == 0) return;
#define HFX_BS(B)                                                                                         \
  case B:                                                                                                 \
    hipLaunchKernelGGL((spmv_kernel<B>), dim3(ceil_div(n, 256)), dim3(256), 0, s, A.nb, A.rowptr.p, A.col.p, \
                       A.vals.p, x, b, y);                                                                \
    break;
  switch (A.bs) {
    HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
    default: throw std::runtime_error("spmv: unsupported block size");
  }
#undef HFX_BS
  HFX_HIP(hipGetLastError());
}

void bsr_invert_diag(const BsrDev& A, double* dinv, hipStream_t s) {
  if (A.nb == 0) return;
#define HFX_BS(B)                                                                                              \
  case B:                                                                                                      \
    hipLaunchKernelGGL((invert_diag_kernel<B>), dim3(ceil_div(A.nb, IW * (64 / B))), dim3(64 * IW), 0, s, A.nb,  \
                       A.diag.p, A.vals.p, dinv);                                                              \
    break;
  switch (A.bs) {
    HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
    default: throw std::runtime_error("block jacobi: unsupported block size");
  }
#undef HFX_BS
  HFX_HIP(hipGetLastError());
}

void bsr_inv_point_diag(const BsrDev& A, double* dinv, hipStream_t s) {
  const long long n = A.nrows();
  if (n == 0) return;
  hipLaunchKernelGGL(point_diag_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, A.nb, A.bs, A.diag.p, A.vals.p, dinv);
  HFX_HIP(hipGetLastError());
}

void apply_block_diag(int nb, int bs, const double* dinv, const double* x, double* y, hipStream_t s) {
  const long long n = (long long)nb * bs;
  if (n == 0) return;
#define HFX_BS(B)                                                                                              \
  case B:                                                                                                      \
    hipLaunchKernelGGL((block_diag_apply_kernel<B>), dim3(ceil_div(n, 256)), dim3(256), 0, s, nb, dinv, x, y); \
    break;
  switch (bs) {
    HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
    default: throw std::runtime_error("block jacobi: unsupported block size");
  }
#undef HFX_BS
  HFX_HIP(hipGetLastError());
}

void apply_point_diag(long long n, const double* dinv, const double* x, double* y, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(point_diag_apply_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, dinv, x, y);
  HFX_HIP(hipGetLastError());
}

// round a count of doubles up to 256 bytes (caller workspaces are carved in
// 256-byte aligned pieces)
static inline size_t al32(size_t k) { return (k + 31) & ~(size_t)31; }

int Reducer::grid_for(long long n) {
  long long g = (n + RT * 8 - 1) / (RT * 8);
  if (g < 1) g = 1;
  if (g > 1024) g = 1024;
  return (int)g;
}

void Reducer::init(long long n) {
  grid = grid_for(n);
  partial_buf.alloc(grid);
  out_buf.alloc(1);
  partial = partial_buf.p;
  out = out_buf.p;
}

void Reducer::init(long long n, double* mem) {
  grid = grid_for(n);
  partial = mem;
  out = mem + (size_t)grid * 66;
}

double Reducer::norm(long long n, const double* x, hipStream_t s) {
  hipLaunchKernelGGL(norm2_kernel, dim3(grid), dim3(RT), 0, s, n, x, partial);
  HFX_HIP(hipGetLastError());
  hipLaunchKernelGGL(reduce_rows_kernel, dim3(1), dim3(RT), 0, s, grid, partial, out);
  HFX_HIP(hipGetLastError());
  double v = 0.0;
  HFX_HIP(hipMemcpyAsync(&v, out, sizeof(double), hipMemcpyDeviceToHost, s));
  HFX_HIP(hipStreamSynchronize(s));
  return std::sqrt(v);
}

KrylovWs::~KrylovWs() {
  if (status) (void)hipHostFree(status);
}

KrylovStatus* KrylovWs::host() {
  if (!status) {
    void* p = nullptr;
    HFX_HIP(hipHostMalloc(&p, sizeof(KrylovStatus), hipHostMallocCoherent | hipHostMallocMapped));
    status = static_cast<KrylovStatus*>(p);
  }
  status->seq = -1;
  status->code = 0;
  return status;
}

// Wait until the device has reported `seq` (its kernels are queued on s)
void KrylovWs::wait(int seq, hipStream_t s) const {
  for (unsigned spin = 1;; ++spin) {
    if (__atomic_load_n(&status->seq, __ATOMIC_ACQUIRE) >= seq) return;
    if ((spin & 0x3ff) == 0) {  // a stream that ended or failed without reporting
      const hipError_t e = hipStreamQuery(s);
      if (e == hipErrorNotReady) continue;
      HFX_HIP(e);
      if (__atomic_load_n(&status->seq, __ATOMIC_ACQUIRE) >= seq) return;
      throw std::runtime_error("krylov: the stream ended without a status");
    }
#if defined(__x86_64__)
    __builtin_ia32_pause();
#endif
  }
}

// Vectors of up to this many 256-row blocks have their dot products' partials
// added up again by every block of the next kernel; beyond it a one-block
// kernel reduces them first.  At the line each of the (at most 2048) blocks
// reads 32 KB out of L2, about the time of the extra launch it saves
// (3.8 us + 2 us of gap on systems of 40,000 to 300,000 rows, where BiCGStab
// is bound by its launches).
constexpr int INLINE_PARTIALS = 2048;

// Steps whose vectors span at most this many 256-row blocks leave the partials
// of V^T w for every block of the next kernel to add up; longer ones reduce
// them first, one launch more per sum.  126 steps at restart 30, added up in
// place / reduced first: one block 2.8 / 3.5 ms, 4 blocks 3.4 / 3.6, 10 to 60
// level (3.7 to 3.9), 104 blocks 4.7 / 4.1, 127 blocks 4.3 / 3.8, 217 blocks
// 5.8 / 4.2.  Reducing first wins from 65 on already (a second value per lane);
// the line stays because it decides the order of the sums, and so the iterates,
// of systems of 65 to 128 blocks.
constexpr int GM_INLINE = 128;

void fgmres(const BsrDev& A, const double* b, double* x, const PcApply& M, const KrylovOpts& o, KrylovInfo& info,
            hipStream_t s, KrylovWs* kws) {
  const long long n = A.nrows();
  const int m = o.restart;
  if (m < 1 || m > 63) throw std::runtime_error("gmres: restart must be in [1, 63]");
  info = KrylovInfo();
  const int nblk = ceil_div(n, RT);
  // V (m + 1), Z (m), w, r, the partials of two V^T w and of a norm, the state
  DevBuf<double> own;
  const size_t ln = al32((size_t)n);
  const size_t need = al32(Reducer::doubles(n)) + (size_t)(2 * m + 3) * ln + 2 * al32((size_t)64 * nblk) +
                      al32((size_t)nblk) + al32(GM_N) + al32(128);
  KrylovWs local;
  KrylovWs& hw = kws ? *kws : local;
  double* ws = hw.mem_for(need, own);
  Reducer red;
  red.init(n, ws);
  double* q = ws + al32(Reducer::doubles(n));
  auto take = [&q](size_t k) { double* r0 = q; q += al32(k); return r0; };
  double* V = take((size_t)(m + 1) * ln);
  double* Z = take((size_t)m * ln);
  double *w = take(n), *r = take(n);
  double *p1 = take((size_t)64 * nblk), *p2 = take((size_t)64 * nblk), *p3 = take(nblk);
  double* gs = take(GM_N);
  double* hr = take(128);  // reduced h1, h2
  const double bnorm = red.norm(n, b, s);
  if (bnorm == 0.0) {
    HFX_HIP(hipMemsetAsync(x, 0, n * sizeof(double), s));
    HFX_HIP(hipStreamSynchronize(s));
    info.reason = CONVERGED_ATOL;
    return;
  }
  const double target = o.rtol * bnorm;
  KrylovStatus* st = hw.host();
  const bool inl = nblk <= GM_INLINE, inl3 = nblk <= INLINE_PARTIALS;
  const int tiles = M.kind == PC_BJACOBI ? ceil_div(n, (RT / A.bs) * A.bs) : nblk;
  double* sums3 = inl3 ? p3 : gs + GM_NORM2 + 1;  // ||w||^2
  const int np3 = inl3 ? nblk : 1;
  auto vstep = [&](int j, double ibeta) {
    const double* src = j == 0 ? r : w;
    double *v = V + (size_t)j * ln, *z = Z + (size_t)j * ln;
#define HFX_LAUNCH(PC, B)                                                                                          \
  hipLaunchKernelGGL((gm_v_kernel<PC, B>), dim3(tiles), dim3(RT), 0, s, n, j, ibeta, np3, sums3, src, M.dinv, v, z, gs)
#define HFX_BS(B) case B: HFX_LAUNCH(PC_BJACOBI, B); break;
    if (M.kind == PC_NONE) HFX_LAUNCH(PC_NONE, 1);
    else if (M.kind == PC_JACOBI) HFX_LAUNCH(PC_JACOBI, 1);
    else if (M.kind == PC_OTHER) HFX_LAUNCH(PC_OTHER, 1);
    else switch (A.bs) {
      HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
      default: throw std::runtime_error("gmres: unsupported block size");
    }
#undef HFX_BS
#undef HFX_LAUNCH
    HFX_HIP(hipGetLastError());
    if (M.kind == PC_OTHER) M.fn(v, z);
  };
  auto product = [&](int j, int seq) {
    const int k = j + 1, grid = nblk + (j > 0 ? 1 : 0);
    const double* z = Z + (size_t)j * ln;
#define HFX_BS(B)                                                                                                   \
  case B:                                                                                                           \
    hipLaunchKernelGGL((gm_product_kernel<B>), dim3(grid), dim3(RT), 0, s, A.nb, A.rowptr.p, A.col.p, A.vals.p, z,  \
                       w, k, V, (long long)ln, nblk, p1, target, seq, gs, st);                                      \
    break;
    switch (A.bs) {
      HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
      default: throw std::runtime_error("spmv: unsupported block size");
    }
#undef HFX_BS
    HFX_HIP(hipGetLastError());
  };
  // the partials of V^T w, or (long vectors) their sums
  auto rows = [&](int k, const double* part, double* sums) -> const double* {
    if (inl) return part;
    hipLaunchKernelGGL(reduce_rows_kernel, dim3(k), dim3(RT), 0, s, nblk, part, sums);
    HFX_HIP(hipGetLastError());
    return sums;
  };
  const int nph = inl ? nblk : 1;
  int it = 0, base = 0;
  while (true) {
    bsr_spmv(A, x, r, b, s);  // r = b - A x (true FP64 residual)
    const double beta = red.norm(n, r, s);
    info.true_relres = beta / bnorm;
    if (!std::isfinite(beta)) { info.reason = DIVERGED_NANORINF; break; }
    if (beta <= target) { info.reason = CONVERGED_RTOL; break; }
    if (it >= o.maxits) { info.reason = DIVERGED_ITS; break; }
    hipLaunchKernelGGL(gm_start_kernel, dim3(1), dim3(256), 0, s, beta, gs);
    HFX_HIP(hipGetLastError());
    int j = 0;
    for (; j < m && it + j < o.maxits; ++j) {
      // column j - 4 has been tested before step j is queued: at most three
      // steps run past the end of a cycle, as kernels that return at once
      if (j >= 4) {
        hw.wait(base + j - 3, s);
        if (__atomic_load_n(&st->code, __ATOMIC_RELAXED) != 0) break;
      }
      const int k = j + 1;
      vstep(j, 1.0 / beta);
      product(j, base + j);
      const double* h1 = rows(k, p1, hr);
#define HFX_LAUNCH(KC)                                                                                              \
  hipLaunchKernelGGL((gm_orth_kernel<KC>), dim3(nblk), dim3(RT), 0, s, n, k, V, (long long)ln, nph, h1, w, nblk, p2, gs)
      if (k <= 8) HFX_LAUNCH(8);
      else HFX_LAUNCH(16);
#undef HFX_LAUNCH
      HFX_HIP(hipGetLastError());
      const double* h2 = rows(k, p2, hr + 64);
      hipLaunchKernelGGL(gm_norm_kernel, dim3(nblk), dim3(RT), 0, s, n, k, V, (long long)ln, nph, h2, w, p3, gs);
      HFX_HIP(hipGetLastError());
      if (!inl3) {
        hipLaunchKernelGGL(reduce_rows_kernel, dim3(1), dim3(RT), 0, s, nblk, p3, sums3);
        HFX_HIP(hipGetLastError());
      }
    }
    // column j - 1 is still open unless the done flag was set by then
    hipLaunchKernelGGL(gm_finish_kernel, dim3(1), dim3(RT), 0, s, j - 1, np3, sums3, target, base + 100, gs, st);
    HFX_HIP(hipGetLastError());
    hipLaunchKernelGGL(gm_combine_kernel, dim3(nblk), dim3(RT), 0, s, n, Z, (long long)ln, gs, x);
    HFX_HIP(hipGetLastError());
    hw.wait(base + 100, s);
    it += __atomic_load_n(&st->code, __ATOMIC_RELAXED);
    base += 128;
    ++info.restarts;
  }
  info.iters = it;
  HFX_HIP(hipStreamSynchronize(s));
}

}  // namespace hfx

namespace hfx {

// More than the solver carves today (66 G and 2 G values of partials): this size
// decides which systems hfx_hdg_solve_noalloc's fixed workspace takes, so it stays.
size_t bicgstab_ws_doubles(long long n) {
  const size_t G = (size_t)Reducer::grid_for(n), nblk_rows = (size_t)ceil_div(n, RT);
  return al32(Reducer::doubles(n)) + 8 * al32((size_t)n) + al32(SC_N) + al32(2 * G) + al32(2 * nblk_rows);
}

void bicgstab(const BsrDev& A, const double* b, double* x, const PcApply& M, const KrylovOpts& o, KrylovInfo& info,
              hipStream_t s, KrylovWs* kws, double* ws) {
  const long long n = A.nrows();
  info = KrylovInfo();
  if (ws && o.graph) throw std::runtime_error("bicgstab: a caller workspace excludes the graph option");
  const int nblk_rows = ceil_div(n, RT);
  // r, rhat, p, v, p^, s, s^, t, the device scalars and the partials: carved
  // from the caller's memory, the handle's kept workspace or a buffer of this
  // call (systems above the size that is worth keeping)
  DevBuf<double> own;
  const size_t need = bicgstab_ws_doubles(n);
  const bool caller_ws = ws != nullptr;
  if (!ws) ws = kws ? kws->mem_for(need, own) : (own.alloc(need), own.p);
  Reducer red;
  red.init(n, ws);
  double* vec[8];
  double* q = ws + al32(Reducer::doubles(n));
  for (int k = 0; k < 8; ++k, q += al32((size_t)n)) vec[k] = q;
  double* sc = q;
  double* fpart = q + al32(SC_N);
  // the x/r update's partials use the reducer's, which is idle meanwhile, on
  // systems that keep them (2 x 8 G <= 66 G values), and fpart on larger ones,
  // where they are reduced at once
  const bool inl = nblk_rows <= INLINE_PARTIALS;
  double* xpart = inl ? red.partial : fpart;
  double *r = vec[0], *rh = vec[1], *p = vec[2], *v = vec[3], *ph = vec[4], *sv = vec[5], *sh = vec[6], *tv = vec[7];
  const double bnorm = red.norm(n, b, s);
  if (bnorm == 0.0) {
    HFX_HIP(hipMemsetAsync(x, 0, n * sizeof(double), s));
    HFX_HIP(hipStreamSynchronize(s));
    info.reason = CONVERGED_ATOL;
    return;
  }
  const double target = o.rtol * bnorm;
  // the status of the checks: pinned memory that the host polls, or (nothing
  // may be allocated) a word of the workspace that it copies
  KrylovWs local;
  KrylovWs& hw = kws ? *kws : local;
  KrylovStatus* st = caller_ws ? reinterpret_cast<KrylovStatus*>(sc + SC_STATUS) : hw.host();
  int seq = -1;
  auto reduce = [&](int count, int nd, const double* from, double* to) {
    hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(SV), 0, s, count, nd, from, sc, to);
    HFX_HIP(hipGetLastError());
  };
  auto spmv_dot = [&](const double* xin, double* yout, const double* w1, bool both) {
#define HFX_BS(B)                                                                                          \
  case B:                                                                                                  \
    hipLaunchKernelGGL((spmv_dot_kernel<B>), dim3(nblk_rows), dim3(RT), 0, s, A.nb, A.rowptr.p, A.col.p,   \
                       A.vals.p, xin, yout, w1, both ? 1 : 0, sc, fpart);                                 \
    break;
    switch (A.bs) {
      HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
      default: throw std::runtime_error("bicgstab: unsupported block size");
    }
#undef HFX_BS
    HFX_HIP(hipGetLastError());
    if (!inl) reduce(nblk_rows, both ? 2 : 1, fpart, sc + SC_SUMS);
  };
  const int np = inl ? nblk_rows : 1;
  const double* part = inl ? fpart : sc + SC_SUMS;
  const double* xsums = inl ? xpart : sc + SC_XSUMS;  // (rhat, r), (r, r): np values each
  // the vector kernels with the preconditioner fused in (point and block Jacobi) or followed by its own kernels
  const int tiles = M.kind == PC_BJACOBI ? ceil_div(n, (RT / A.bs) * A.bs) : nblk_rows;
  auto pstep = [&](int first, int par) {
    const int fnp = first ? 1 : np;
    const double* fpt = first ? sc + SC_XSUMS : xsums;
#define HFX_LAUNCH(PC, B)                                                                                           \
  hipLaunchKernelGGL((bicg_p_kernel<PC, B>), dim3(tiles), dim3(RT), 0, s, n, first, par, fnp, fpt, sc, r, p, v, \
                     M.dinv, ph)
#define HFX_BS(B) case B: HFX_LAUNCH(PC_BJACOBI, B); break;
    if (M.kind == PC_NONE) HFX_LAUNCH(PC_NONE, 1);
    else if (M.kind == PC_JACOBI) HFX_LAUNCH(PC_JACOBI, 1);
    else if (M.kind != PC_BJACOBI) HFX_LAUNCH(PC_OTHER, 1);
    else switch (A.bs) {
      HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
      default: throw std::runtime_error("bicgstab: unsupported block size");
    }
#undef HFX_BS
#undef HFX_LAUNCH
    HFX_HIP(hipGetLastError());
    if (M.kind == PC_OTHER) M.fn(p, ph);
  };
  auto sstep = [&](int par) {
#define HFX_LAUNCH(PC, B)                                                                                           \
  hipLaunchKernelGGL((bicg_s_kernel<PC, B>), dim3(tiles), dim3(RT), 0, s, n, par, np, part, sc, r, v, sv, M.dinv, sh)
#define HFX_BS(B) case B: HFX_LAUNCH(PC_BJACOBI, B); break;
    if (M.kind == PC_NONE) HFX_LAUNCH(PC_NONE, 1);
    else if (M.kind == PC_JACOBI) HFX_LAUNCH(PC_JACOBI, 1);
    else if (M.kind != PC_BJACOBI) HFX_LAUNCH(PC_OTHER, 1);
    else switch (A.bs) {
      HFX_BS(1) HFX_BS(2) HFX_BS(3) HFX_BS(4) HFX_BS(5) HFX_BS(6) HFX_BS(7) HFX_BS(8) HFX_BS(9) HFX_BS(10) HFX_BS(11) HFX_BS(12) HFX_BS(15) HFX_BS(18) HFX_BS(21) HFX_BS(30)
      default: throw std::runtime_error("bicgstab: unsupported block size");
    }
#undef HFX_BS
#undef HFX_LAUNCH
    HFX_HIP(hipGetLastError());
    if (M.kind == PC_OTHER) M.fn(sv, sh);
  };
  const int check_every = 8;
  // one iteration (first: the one after a restart): p, M p, A p^ with
  // (rhat, v), alpha, s, M s, A s^ with (s, t) and (t, t), omega, x, r with
  // (rhat, r) and (r, r)
  auto iteration = [&](int first, int par) {
    pstep(first, par);
    spmv_dot(ph, v, rh, false);
    sstep(par);
    spmv_dot(sh, tv, sv, true);
    hipLaunchKernelGGL(bicg_xr_dot_kernel, dim3(nblk_rows), dim3(RT), 0, s, n, par, np, part, sc, ph, sh, sv, tv, rh,
                       x, r, xpart);
    HFX_HIP(hipGetLastError());
    if (!inl) reduce(nblk_rows, 2, xpart, sc + SC_XSUMS);
  };
  // check_every steady iterations as one graph, captured at first use; it
  // holds kernels only (no memset or copy nodes), and every buffer it names
  // lives until the end of this call
  struct GraphHold {
    hipGraph_t g = nullptr;
    hipGraphExec_t e = nullptr;
    ~GraphHold() {
      if (e) (void)hipGraphExecDestroy(e);
      if (g) (void)hipGraphDestroy(g);
    }
  } gh;
  const bool use_graph = o.graph && M.kind != PC_NONE;
  auto graph_block = [&]() {
    if (!gh.e) {
      HFX_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      try {
        for (int k = 0; k < check_every; ++k) iteration(0, k & 1);
      } catch (...) {
        hipGraph_t g = nullptr;
        (void)hipStreamEndCapture(s, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
      }
      HFX_HIP(hipStreamEndCapture(s, &gh.g));
      HFX_HIP(hipGraphInstantiate(&gh.e, gh.g, nullptr, nullptr, 0));
    }
    HFX_HIP(hipGraphLaunch(gh.e, s));
  };
  int it = 0;
  while (true) {
    // r = b - A x (true FP64 residual), rhat = r, rho = (r, r)
    bsr_spmv(A, x, r, b, s);
    const double rn = red.norm(n, r, s);
    info.true_relres = rn / bnorm;
    if (!std::isfinite(rn)) { info.reason = DIVERGED_NANORINF; break; }
    if (rn <= target) { info.reason = CONVERGED_RTOL; break; }
    if (it >= o.maxits) { info.reason = DIVERGED_ITS; break; }
    HFX_HIP(hipMemcpyAsync(rh, r, n * sizeof(double), hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(set_scalars_kernel, dim3(1), dim3(64), 0, s, sc);
    HFX_HIP(hipGetLastError());
    hipLaunchKernelGGL(dots_kernel, dim3(red.grid), dim3(RT), 0, s, n, 2, rh, r, r, r, xpart);
    HFX_HIP(hipGetLastError());
    reduce(red.grid, 2, xpart, sc + SC_XSUMS);
    ++info.restarts;
    // Iterations up to the next restart.  The recurrence residual is checked
    // every check_every iterations; one iteration is queued behind each check
    // before its result is awaited (it does nothing once the check has set the
    // stop flag), so the device does not idle meanwhile.
    bool first = true;
    int code = 0, ahead = 0;
    while (true) {
      if (ahead) {
        ahead = 0;  // already queued
        ++it;
      } else if (!first && use_graph && it % check_every == 0 && it + check_every <= o.maxits) {
        graph_block();
        it += check_every;
      } else {
        iteration(first ? 1 : 0, it & 1);
        first = false;
        ++it;
      }
      if (it % check_every != 0 && it < o.maxits) continue;
      hipLaunchKernelGGL(bicg_check_kernel, dim3(1), dim3(RT), 0, s, np, xsums, target, ++seq, sc, st);
      HFX_HIP(hipGetLastError());
      if (caller_ws) {
        HFX_HIP(hipMemcpyAsync(&code, &st->code, sizeof(int), hipMemcpyDeviceToHost, s));
        HFX_HIP(hipStreamSynchronize(s));
      } else {
        if (!use_graph && it < o.maxits) {
          iteration(0, it & 1);
          ahead = 1;
        }
        hw.wait(seq, s);
        code = __atomic_load_n(&st->code, __ATOMIC_RELAXED);
      }
      // converged recurrence, breakdown, or the iteration budget: restart from
      // (and test) the true residual; maxits bounds the number of restarts
      if (code != 0 || it >= o.maxits) break;
    }
    if (code == 2) { info.reason = DIVERGED_NANORINF; break; }
  }
  info.iters = it;
  HFX_HIP(hipStreamSynchronize(s));
}

}  // namespace hfx
