// Gauss-Jordan elimination on an LDS matrix by one workgroup, shared by the
// general element kernel and the Burgers cell kernel.
#pragma once

#include <hip/hip_runtime.h>

#include "wave.h"

namespace hfx {

// largest v of the wavefront, the same value in every lane
__device__ __forceinline__ double gj_wave_max(double v) {
  v = row_max(v);
  return fmax(fmax(lane_value(v, 0), lane_value(v, 16)), fmax(lane_value(v, 32), lane_value(v, 48)));
}

// Gauss-Jordan elimination with partial pivoting, without row swaps, on an
// LDS (or workspace) matrix of NR rows and NC columns (row stride NC,
// NR <= 128).  Step k picks the unused row p of largest |A[p][k]|, the lowest
// row among equals (every wave computes the same pivot with a wave-wide
// maximum over rows lane and lane + 64, so no broadcast barrier is needed) and
// eliminates column k from every other row.  On return row perm[k] holds
// variable k: its right-hand columns (NR..NC-1) are divided by the pivot,
// i.e. X[k][c] = A[perm[k]][c].  One workgroup barrier per step.
//
// Bound by the chain of its NR steps (pivot, reciprocal, update, barrier), so
// each is kept short: the maximum runs on DPP moves, a lane owns a column and
// keeps the pivot row's entry of it, the waves share the rows (the factor of a
// row is one broadcast read), and only the columns right of k are visited.
// Measured with it alone changed, 18,432 2-D p=3 Burgers cells (20 x 45 and
// 10 x 54): 2.09 -> 1.66 ms for the whole cell kernel.
template <int NR, int NC, int NT>
__device__ void gauss_jordan(double* A, int* perm) {
  static_assert(NR <= 128, "gauss_jordan: at most 128 rows");
  constexpr int NW = NT / 64, RB = 8;  // waves; rows in flight per wave
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned long long used = 0ull, used_hi = 0ull;  // rows 0..63, 64..127
  for (int k = 0; k < NR; ++k) {
    double v = -1.0, w = -1.0;
    if (lane < NR && !((used >> lane) & 1ull)) {
      v = fabs(A[lane * NC + k]);
      if (!(v >= 0.0)) v = 0.0;  // NaN: keep the argmax total and uniform
    }
    if constexpr (NR > 64) {
      const int r = lane + 64;
      if (r < NR && !((used_hi >> lane) & 1ull)) {
        w = fabs(A[r * NC + k]);
        if (!(w >= 0.0)) w = 0.0;
      }
    }
    const double top = gj_wave_max(NR > 64 ? fmax(v, w) : v);
    const unsigned long long eq = __ballot(v == top);
    int p;
    if (NR <= 64 || eq) {
      p = __ffsll(eq) - 1;
      used |= 1ull << p;
    } else {
      p = __ffsll(__ballot(w == top)) - 1;
      used_hi |= 1ull << p;
      p += 64;
    }
    if (tid == 0) perm[k] = p;
    const double pinv = 1.0 / A[p * NC + k];
    for (int c = k + 1 + lane; c < NC; c += 64) {
      const double apc = A[p * NC + c];
      for (int r0 = wv; r0 < NR; r0 += NW * RB) {
        double x[RB], f[RB];
#pragma unroll
        for (int u = 0; u < RB; ++u) {
          const int r = r0 + NW * u;
          if (r < NR) {
            x[u] = A[r * NC + c];
            f[u] = A[r * NC + k] * pinv;
          }
        }
#pragma unroll
        for (int u = 0; u < RB; ++u) {
          const int r = r0 + NW * u;
          if (r < NR && r != p) A[r * NC + c] = x[u] - f[u] * apc;
        }
      }
    }
    __syncthreads();
  }
  // normalise the right-hand columns of each pivot row
  constexpr int NRHS = NC - NR;
  for (int t = tid; t < NR * NRHS; t += NT) {
    const int k = t / NRHS, c = NR + t % NRHS;
    const int r = perm[k];
    A[r * NC + c] /= A[r * NC + k];
  }
  __syncthreads();
}

}  // namespace hfx
