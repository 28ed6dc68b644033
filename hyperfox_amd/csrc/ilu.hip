// Block ILU(0): level-scheduled factorisation and triangular sweeps on the
// GPU.  See ilu.h for the algorithm.
#include <stdexcept>
#include <string>

#include "bsr_row.h"
#include "ilu.h"
#include "wave.h"

#include <algorithm>

namespace hfx {

namespace {

constexpr int FT = 64;   // factorisation: one wavefront per block row
constexpr int AT = 256;  // sweeps: one thread per scalar row

// Factor the block rows rows[0..gridDim.x) of one forward level.  Row i is
// staged in LDS (len x bs^2), updated by the already factored rows of earlier
// levels (lu, dinv; each of their blocks staged in LDS with one coalesced load
// before its product), its diagonal block inverted by Gauss-Jordan with
// partial pivoting (the pivot found by a wavefront argmax: the first row of
// largest magnitude, the diagonal's own row when it is NaN), and written to lu
// (earlier blocks L_ik, diagonal A'_ii, later blocks Uhat_ij) and dinv.
// err[0] receives 1 + row on a zero pivot.
//
// Bound by the chain of a row's products and pivot steps.  The block size BS is
// an instance's own: the inner products unroll and an entry's row and column
// need no division by a value known only at run time.  Blocks have at most 12
// rows, so the pivot's maximum stays in a row of 16 lanes (DPP).
// Measured, the five levels of 41,850 block rows of 10 x 10: 0.643 -> 0.478 ms;
// the three of 27,840 rows of 8 x 8: 0.157 -> 0.102 ms.
template <int BS>
__global__ __launch_bounds__(FT) void ilu_factor_kernel(const int* __restrict__ rows,
                                                        const int* __restrict__ rowptr, const double* __restrict__ vals,
                                                        const int* __restrict__ lptr, const int* __restrict__ lpos,
                                                        const int* __restrict__ lcol, const int* __restrict__ pptr,
                                                        const int* __restrict__ pslot, const int* __restrict__ ppos,
                                                        const int* __restrict__ uptr, const int* __restrict__ upos,
                                                        const int* __restrict__ dslot,
                                                        const signed char* __restrict__ kind, double* __restrict__ lu,
                                                        double* __restrict__ dinv, int* __restrict__ err) {
  constexpr int bs = BS;
  extern __shared__ double sm[];
  const int i = rows[blockIdx.x];
  const int r0 = rowptr[i], len = rowptr[i + 1] - r0, B2 = bs * bs, t = threadIdx.x;
  double* R = sm;             // the row's blocks
  double* M = R + len * B2;   // diagonal block being inverted
  double* V = M + B2;         // its inverse
  double* T = V + B2;         // scratch block
  double* W = T + B2;         // staged block of an earlier row (Uhat_kj or Dinv_k)
  for (int e = t; e < len * B2; e += FT) R[e] = vals[(size_t)r0 * B2 + e];
  __syncthreads();
  for (int l = lptr[i]; l < lptr[i + 1]; ++l) {
    const int k = lcol[l], sl = lpos[l] - r0;
    const double* Rk = R + sl * B2;
    // A'_ij -= A'_ik Uhat_kj  (slot j != slot k: no lane reads what another writes)
    for (int q = pptr[l]; q < pptr[l + 1]; ++q) {
      const double* Ug = lu + (size_t)ppos[q] * B2;
      for (int e = t; e < B2; e += FT) W[e] = Ug[e];
      __syncthreads();
      double* Rj = R + pslot[q] * B2;
      for (int e = t; e < B2; e += FT) {
        const int r = e / bs, c = e - r * bs;
        double acc = 0.0;
        for (int m = 0; m < bs; ++m) acc += Rk[r * bs + m] * W[m * bs + c];
        Rj[e] -= acc;
      }
      __syncthreads();  // W is restaged by the next product
    }
    // L_ik = A'_ik Dinv_k
    const double* Dk = dinv + (size_t)k * B2;
    for (int e = t; e < B2; e += FT) W[e] = Dk[e];
    __syncthreads();
    for (int e = t; e < B2; e += FT) {
      const int r = e / bs, c = e - r * bs;
      double acc = 0.0;
      for (int m = 0; m < bs; ++m) acc += Rk[r * bs + m] * W[m * bs + c];
      T[e] = acc;
    }
    __syncthreads();
    for (int e = t; e < B2; e += FT) R[sl * B2 + e] = T[e];
    __syncthreads();
  }
  // Dinv_i = (A'_ii)^-1, Gauss-Jordan with partial pivoting
  const int ds = dslot[i];
  for (int e = t; e < B2; e += FT) {
    const int r = e / bs, c = e - r * bs;
    M[e] = R[ds * B2 + e];
    V[e] = (r == c) ? 1.0 : 0.0;
  }
  __syncthreads();
  for (int c = 0; c < bs; ++c) {
    // pivot: the first row r >= c of largest |M[r][c]| (NaN rows never win);
    // the diagonal's row when |M[c][c]| is NaN
    const double dc = fabs(M[c * bs + c]);
    double v = -1.0;
    if (t >= c && t < bs) {
      v = fabs(M[t * bs + c]);
      if (v != v) v = -1.0;
    }
    const double top = lane_value(row_max(v), 0);
    const int idx = __ffsll(__ballot(v == top)) - 1;
    const int p = (dc != dc) ? c : idx;
    const double best = (dc != dc) ? dc : top;
    if (t == 0 && (!(best > 0.0) || !isfinite(best))) err[0] = i + 1;
    if (p != c && t < bs) {
      double a = M[c * bs + t];
      M[c * bs + t] = M[p * bs + t];
      M[p * bs + t] = a;
      a = V[c * bs + t];
      V[c * bs + t] = V[p * bs + t];
      V[p * bs + t] = a;
    }
    __syncthreads();
    const double inv = 1.0 / M[c * bs + c];
    __syncthreads();
    if (t < bs) {
      M[c * bs + t] *= inv;
      V[c * bs + t] *= inv;
    }
    __syncthreads();
    double f[4];  // bs <= 16: at most 4 entries per lane
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = t + u * FT;
      f[u] = (e < B2 && e / bs != c) ? M[(e / bs) * bs + c] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = t + u * FT;
      if (e < B2 && e / bs != c) {
        const int j = e - (e / bs) * bs;
        M[e] -= f[u] * M[c * bs + j];
        V[e] -= f[u] * V[c * bs + j];
      }
    }
    __syncthreads();
  }
  for (int e = t; e < B2; e += FT) dinv[(size_t)i * B2 + e] = V[e];
  // earlier blocks and the diagonal as they are; later blocks scaled by Dinv_i
  for (int e = t; e < len * B2; e += FT)
    if (kind[r0 + e / B2] <= 0) lu[(size_t)r0 * B2 + e] = R[e];
  for (int u = uptr[i]; u < uptr[i + 1]; ++u) {
    const double* Rj = R + (upos[u] - r0) * B2;
    for (int e = t; e < B2; e += FT) {
      const int r = e / bs, c = e - r * bs;
      double acc = 0.0;
      for (int m = 0; m < bs; ++m) acc += V[r * bs + m] * Rj[m * bs + c];
      lu[(size_t)upos[u] * B2 + e] = acc;
    }
  }
}

// The sweeps.  Level 0 of the forward sweep is y = x, so it is not run: its
// rows are read from x wherever y is meant (FROM_X in an entry's column or a
// slot's row).  The rows without later blocks (backward level 0, the last
// forward level among them) are finished in one launch, which forms y_i and
// z_i = Dinv_i y_i together.  What is left of three colours is four launches
// instead of six, each a few microseconds whatever its size up to some 50,000
// rows: a slot holds its row and its list bounds, an entry its block position
// and column, so that a row's chain is slot, entry, data.  ILU(0) application,
// 49,408 block rows of 5 (three colours): 34 -> 25 us.
constexpr int FROM_X = 1 << 31;

// sum over the entries [l0, l1) of row r of block ent.x times the segment of
// column ent.y of y (or of x); the order of bsr_row_sum
template <int BS, typename V>
__device__ __forceinline__ double entry_sum(int l0, int l1, int r, const int2* __restrict__ ent,
                                            const V* __restrict__ lu, const double* __restrict__ x,
                                            const double* __restrict__ y) {
  double acc = 0.0;
  for (int k = l0; k < l1; ++k) {
    const int2 e = ent[k];
    const V* a = lu + ((size_t)e.x * BS + r) * BS;
    const double* xv = ((e.y & FROM_X) ? x : y) + (size_t)(e.y & ~FROM_X) * BS;
#pragma unroll
    for (int c = 0; c + 1 < BS; c += 2) acc += (double)a[c] * xv[c] + (double)a[c + 1] * xv[c + 1];
    if constexpr (BS % 2 == 1) acc += (double)a[BS - 1] * xv[BS - 1];
  }
  return acc;
}

// Forward sweep over one level: y_i = x_i - sum_k L_ik y_k.
template <int BS, typename V>
__global__ __launch_bounds__(AT) void ilu_fwd_kernel(int n, const int4* __restrict__ slots,
                                                     const int2* __restrict__ ent, const V* __restrict__ lu,
                                                     const double* __restrict__ x, double* __restrict__ y) {
  const int t = blockIdx.x * AT + threadIdx.x;
  if (t >= n * BS) return;
  const int4 s = slots[t / BS];
  const int r = t % BS;
  const size_t o = (size_t)s.x * BS + r;
  const double xi = x[o];
  y[o] = xi - entry_sum<BS, V>(s.y, s.z, r, ent, lu, x, y);
}

// Rows without later blocks: y_i = x_i - sum_k L_ik y_k, z_i = Dinv_i y_i.
template <int BS, typename V>
__global__ __launch_bounds__(AT) void ilu_turn_kernel(int n, const int4* __restrict__ slots,
                                                      const int2* __restrict__ ent, const V* __restrict__ lu,
                                                      const V* __restrict__ dinv, const double* __restrict__ x,
                                                      const double* __restrict__ y, double* __restrict__ z) {
  constexpr int RPB = AT / BS;
  __shared__ double ys[RPB * BS];
  const int b = threadIdx.x / BS, r = threadIdx.x % BS, slot = blockIdx.x * RPB + b;
  const bool on = b < RPB && slot < n;
  int i = 0;
  if (on) {
    const int4 s = slots[slot];
    i = s.x;
    ys[threadIdx.x] = x[(size_t)i * BS + r] - entry_sum<BS, V>(s.y, s.z, r, ent, lu, x, y);
  }
  __syncthreads();
  if (on) z[(size_t)i * BS + r] = bsr_row_dot<BS, V>(dinv + ((size_t)i * BS + r) * BS, ys + b * BS);
}

// Backward sweep over one level: z_i = Dinv_i y_i - sum_j Uhat_ij z_j.
template <int BS, typename V>
__global__ __launch_bounds__(AT) void ilu_bwd_kernel(int n, const int4* __restrict__ slots,
                                                     const int2* __restrict__ ent, const V* __restrict__ lu,
                                                     const V* __restrict__ dinv, const double* __restrict__ x,
                                                     const double* __restrict__ y, double* __restrict__ z) {
  const int t = blockIdx.x * AT + threadIdx.x;
  if (t >= n * BS) return;
  const int4 s = slots[t / BS];
  const int r = t % BS, i = s.x & ~FROM_X;
  const double* ysrc = ((s.x & FROM_X) ? x : y) + (size_t)i * BS;
  z[(size_t)i * BS + r] = bsr_row_dot<BS, V>(dinv + ((size_t)i * BS + r) * BS, ysrc) -
                          entry_sum<BS, V>(s.y, s.z, r, ent, lu, z, z);
}

__global__ void to_float_kernel(size_t n, const double* __restrict__ a, float* __restrict__ b) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    b[i] = (float)a[i];
}

template <int BS, typename V>
void sweeps_v(const Ilu& f, const V* lu, const V* dinv, const double* x, double* y, double* z, hipStream_t s) {
  auto grid = [](int n) { return dim3(ceil_div((long long)n * BS, AT)); };
  for (size_t l = 0; l + 1 < f.fwd_off.size(); ++l) {
    const int o = f.fwd_off[l], n = f.fwd_off[l + 1] - o;
    if (n == 0) continue;
    hipLaunchKernelGGL((ilu_fwd_kernel<BS, V>), grid(n), dim3(AT), 0, s, n, f.fwd_slots.p + o, f.lent.p, lu, x, y);
  }
  for (size_t l = 0; l + 1 < f.bwd_off.size(); ++l) {
    const int o = f.bwd_off[l], n = f.bwd_off[l + 1] - o;
    if (l == 0)
      hipLaunchKernelGGL((ilu_turn_kernel<BS, V>), dim3(ceil_div(n, AT / BS)), dim3(AT), 0, s, n, f.bwd_slots.p,
                         f.lent.p, lu, dinv, x, y, z);
    else
      hipLaunchKernelGGL((ilu_bwd_kernel<BS, V>), grid(n), dim3(AT), 0, s, n, f.bwd_slots.p + o, f.uent.p, lu, dinv, x,
                         y, z);
  }
  HFX_HIP(hipGetLastError());
}

template <int BS>
void sweeps(const Ilu& f, const double* x, double* y, double* z, hipStream_t s) {
  if (f.low) sweeps_v<BS, float>(f, f.lu32.p, f.dinv32.p, x, y, z, s);
  else sweeps_v<BS, double>(f, f.lu.p, f.dinv.p, x, y, z, s);
}

}  // namespace

void Ilu::setup(int nb_, int bs_, const int* rowptr_host, const int* col_host, int ordering_, hipStream_t s) {
  // the block sizes the sweeps of apply() are instantiated for; refused here,
  // before the analysis and factorisation, rather than at the first apply
  if (!(bs_ >= 1 && bs_ <= 12 && bs_ != 7 && bs_ != 11))
    throw std::runtime_error("ILU(0): block size must be one of 1-6, 8, 9, 10, 12");
  plan = ilu_analyse(nb_, rowptr_host, col_host, ordering_);
  nb = nb_;
  bs = bs_;
  ordering = ordering_;
  const size_t lds = ((size_t)plan.maxlen + 4) * bs * bs * sizeof(double);
  if (lds > 65536) throw std::runtime_error("ILU(0): a block row is too long for the factorisation kernel");
  rowptr.upload(rowptr_host, nb + 1, s);
  fwd_rows.upload(plan.fwd_rows, s);
  // the sweeps' slots and entries
  std::vector<int2> le(plan.lpos.size()), ue(plan.upos.size());
  std::vector<char> used(nb, 0);  // rows whose y a later row reads
  for (size_t k = 0; k < le.size(); ++k) {
    const int c = plan.lcol[k];
    used[c] = 1;
    le[k] = make_int2(plan.lpos[k], c | (plan.levf[c] == 0 ? FROM_X : 0));
  }
  for (size_t k = 0; k < ue.size(); ++k) ue[k] = make_int2(plan.upos[k], plan.ucol[k]);
  std::vector<int4> fs, bsl;
  fwd_off.assign(1, 0);
  for (int l = 1; l < plan.nlev_f; ++l) {
    for (int k = plan.fwd_off[l]; k < plan.fwd_off[l + 1]; ++k) {
      const int i = plan.fwd_rows[k];
      if (plan.levb[i] > 0 || used[i]) fs.push_back(make_int4(i, plan.lptr[i], plan.lptr[i + 1], 0));
    }
    fwd_off.push_back((int)fs.size());
  }
  bwd_off.assign(1, 0);
  for (int l = 0; l < plan.nlev_b; ++l) {
    for (int k = plan.bwd_off[l]; k < plan.bwd_off[l + 1]; ++k) {
      const int i = plan.bwd_rows[k];
      if (l == 0) bsl.push_back(make_int4(i, plan.lptr[i], plan.lptr[i + 1], 0));
      else bsl.push_back(make_int4(i | (plan.levf[i] == 0 ? FROM_X : 0), plan.uptr[i], plan.uptr[i + 1], 0));
    }
    bwd_off.push_back((int)bsl.size());
  }
  fwd_slots.upload(fs, s);
  bwd_slots.upload(bsl, s);
  lent.upload(le, s);
  uent.upload(ue, s);
  lptr.upload(plan.lptr, s);
  lpos.upload(plan.lpos, s);
  lcol.upload(plan.lcol, s);
  uptr.upload(plan.uptr, s);
  upos.upload(plan.upos, s);
  dslot.upload(plan.dslot, s);
  pptr.upload(plan.pptr, s);
  pslot.upload(plan.pslot, s);
  ppos.upload(plan.ppos, s);
  kind.upload(plan.kind, s);
  err.alloc(1);
  lu.alloc((size_t)rowptr_host[nb] * bs * bs);
  dinv.alloc((size_t)nb * bs * bs);
  tmp.alloc((size_t)nb * bs);
  HFX_HIP(hipStreamSynchronize(s));
}

void Ilu::factor(const BsrDev& A, hipStream_t s) {
  if (A.nb != nb || A.bs != bs || (size_t)A.nnzb * bs * bs != lu.n)
    throw std::runtime_error("ILU(0): matrix does not match the analysed pattern");
  HFX_HIP(hipMemsetAsync(err.p, 0, sizeof(int), s));
  const size_t lds = ((size_t)plan.maxlen + 4) * bs * bs * sizeof(double);
  for (int l = 0; l < plan.nlev_f; ++l) {
    const int n = plan.fwd_off[l + 1] - plan.fwd_off[l];
#define HFX_FACTOR(B)                                                                                                \
  hipLaunchKernelGGL((ilu_factor_kernel<B>), dim3(n), dim3(FT), lds, s, fwd_rows.p + plan.fwd_off[l], rowptr.p,      \
                     A.vals.p, lptr.p, lpos.p, lcol.p, pptr.p, pslot.p, ppos.p, uptr.p, upos.p, dslot.p, kind.p,     \
                     lu.p, dinv.p, err.p)
    switch (bs) {
      case 1: HFX_FACTOR(1); break;
      case 2: HFX_FACTOR(2); break;
      case 3: HFX_FACTOR(3); break;
      case 4: HFX_FACTOR(4); break;
      case 5: HFX_FACTOR(5); break;
      case 6: HFX_FACTOR(6); break;
      case 8: HFX_FACTOR(8); break;
      case 9: HFX_FACTOR(9); break;
      case 10: HFX_FACTOR(10); break;
      case 12: HFX_FACTOR(12); break;
      default: throw std::runtime_error("ILU(0): unsupported block size");
    }
#undef HFX_FACTOR
  }
  HFX_HIP(hipGetLastError());
  int e = 0;
  HFX_HIP(hipMemcpyAsync(&e, err.p, sizeof(int), hipMemcpyDeviceToHost, s));
  HFX_HIP(hipStreamSynchronize(s));
  if (e) throw std::runtime_error("ILU(0): singular pivot block in block row " + std::to_string(e - 1));
  if (low) {
    lu32.alloc(lu.n);
    dinv32.alloc(dinv.n);
    hipLaunchKernelGGL(to_float_kernel, dim3(std::min<long long>(ceil_div((long long)lu.n, 256), 8192)), dim3(256), 0,
                       s, lu.n, lu.p, lu32.p);
    hipLaunchKernelGGL(to_float_kernel, dim3(std::min<long long>(ceil_div((long long)dinv.n, 256), 8192)), dim3(256),
                       0, s, dinv.n, dinv.p, dinv32.p);
    HFX_HIP(hipGetLastError());
  }
}

void Ilu::apply(const double* x, double* y, hipStream_t s) {
  switch (bs) {
    case 1: sweeps<1>(*this, x, tmp.p, y, s); break;
    case 2: sweeps<2>(*this, x, tmp.p, y, s); break;
    case 3: sweeps<3>(*this, x, tmp.p, y, s); break;
    case 4: sweeps<4>(*this, x, tmp.p, y, s); break;
    case 5: sweeps<5>(*this, x, tmp.p, y, s); break;
    case 6: sweeps<6>(*this, x, tmp.p, y, s); break;
    case 8: sweeps<8>(*this, x, tmp.p, y, s); break;
    case 9: sweeps<9>(*this, x, tmp.p, y, s); break;
    case 10: sweeps<10>(*this, x, tmp.p, y, s); break;
    case 12: sweeps<12>(*this, x, tmp.p, y, s); break;
    default: throw std::runtime_error("ILU(0): unsupported block size for the sweeps");
  }
}

}  // namespace hfx
