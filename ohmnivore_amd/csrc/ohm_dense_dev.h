// ohm_dense_dev.h — dense LU with partial pivoting of a small system inside
// one workgroup, as a device function (kernels in ohm_dense.hip and
// ohm_newton_small.hip).
#pragma once

#include "ohm_reduce.h"

namespace ohm {

// The whole solve in one workgroup with the augmented matrix in LDS. Lane l of
// every wave stands for rows l, l + 64, ...; the waves share out the columns.
// Rows stay where they are: a step marks its pivot row as used, order[] names
// it for the back substitution. Every wave finds the step's pivot by itself
// (its lanes read column k and know which of their rows are used), so a step
// has one barrier, behind its update. Bound by that step's latency: column
// read, wave maximum, reciprocal, multiplier. A quotient is the product with
// the pivot's reciprocal, corrected by its remainder. The back substitution
// runs in one wave without barriers. Kernel time against the two launches per
// column: 24 unknowns 158 -> 23 us, 54 unknowns 395 -> 56 us (a 50-stage
// inverter chain), 140 unknowns about 950 -> 347 us.
constexpr int kDenseLdsRows = 140;

__device__ __forceinline__ double refined_quotient(double a, double piv, double rp) {
  const double q = a * rp;
  return fma(fma(-q, piv, a), rp, q);
}
// 1 / a: the hardware estimate and two Newton-Raphson steps
__device__ __forceinline__ double refined_reciprocal(double a) {
  double r = __builtin_amdgcn_rcp(a);
  r = fma(fma(-a, r, 1.0), r, r);
  return fma(fma(-a, r, 1.0), r, r);
}
__device__ __forceinline__ double lane_of(double v, int l) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, l);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

struct DenseLds {
  uint32_t ptr[kDenseLdsRows + 1];
  double piv[kDenseLdsRows], rpiv[kDenseLdsRows];
  int order[kDenseLdsRows];
};
// Row stride of the augmented matrix: odd, so that a column's entries fall in
// different banks.
__host__ __device__ inline int dense_lds_stride(int n) { return (n + 1) | 1; }

// x = A^-1 rhs by R rows per lane and kWavesLu waves (the whole workgroup);
// aug: n * dense_lds_stride(n) doubles of LDS. False (everywhere) on a zero
// or NaN pivot. x is complete behind the caller's next barrier.
template <int R, int kWavesLu>
__device__ __forceinline__ bool dense_lu_wg(int n, const uint32_t *rowptr, const uint32_t *col,
                                            const double *val, const double *rhs, double *x,
                                            double *aug, DenseLds &sh) {
  uint32_t *ptr = sh.ptr;
  double *piv = sh.piv, *rpiv = sh.rpiv;
  int *order = sh.order;
  const int ld = dense_lds_stride(n);
  constexpr int kThreads = 64 * kWavesLu;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (int i = t; i < n * ld; i += kThreads) aug[i] = 0.0;
  for (int i = t; i <= n; i += kThreads) ptr[i] = rowptr[i];
  __syncthreads();
  // an entry per thread, its row found in ptr; repeated entries add up
  for (uint32_t k = t; k < ptr[n]; k += kThreads) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (ptr[mid] <= k)
        lo = mid;
      else
        hi = mid;
    }
    atomicAdd(&aug[lo * ld + (int)col[k]], val[k]);
  }
  for (int i = t; i < n; i += kThreads) aug[i * ld + n] = rhs[i];
  __syncthreads();
  bool open[R];
#pragma unroll
  for (int c = 0; c < R; c++) open[c] = lane + 64 * c < n;
  for (int k = 0; k < n; k++) {
    double ak[R], best = -1.0;
    int bi = n;
#pragma unroll
    for (int c = 0; c < R; c++) {
      const int i = lane + 64 * c;
      ak[c] = i < n ? aug[i * ld + k] : 0.0;
      const double v = fabs(ak[c]);
      if (open[c] && v > best) {
        best = v;
        bi = c;
      }
    }
    const double top = wave_max(best);
    const unsigned long long tie = __ballot(best == top && bi < n);
    if (!(top > 1e-300) || !tie) {  // a zero or NaN column
      return false;
    }
    const int pl = __builtin_ctzll(tie), pc = __builtin_amdgcn_readlane(bi, pl);
    const int pr = pl + 64 * pc;
    double mine = ak[0];
#pragma unroll
    for (int c = 1; c < R; c++) mine = pc == c ? ak[c] : mine;
    const double pk = lane_of(mine, pl), rp = refined_reciprocal(pk);
    if (t == 0) {
      order[k] = pr;
      piv[k] = pk;
      rpiv[k] = rp;
    }
    double l[R];
#pragma unroll
    for (int c = 0; c < R; c++) {
      if (lane + 64 * c == pr) open[c] = false;
      l[c] = open[c] ? refined_quotient(ak[c], pk, rp) : 0.0;
    }
#pragma unroll 4
    for (int j = k + 1 + wave; j <= n; j += kWavesLu) {
      const double pj = aug[pr * ld + j];
#pragma unroll
      for (int c = 0; c < R; c++)
        if (open[c]) aug[(lane + 64 * c) * ld + j] -= l[c] * pj;
    }
    __syncthreads();
  }
  if (wave) return true;
  double y[R], ac[R];
  int row[R];
#pragma unroll
  for (int c = 0; c < R; c++) {
    const int i = lane + 64 * c;
    row[c] = i < n ? order[i] * ld : 0;
    y[c] = i < n ? aug[row[c] + n] : 0.0;
    ac[c] = aug[row[c] + n - 1];
  }
#pragma unroll
  for (int c = R - 1; c >= 0; c--) {
    const int top = min(n, 64 * (c + 1)) - 1;
    for (int k = top; k >= 64 * c; k--) {
      const double xk = lane_of(refined_quotient(y[c], piv[k], rpiv[k]), k & 63);
      if (lane == 0) x[k] = xk;
#pragma unroll
      for (int q = 0; q <= c; q++) {
        if (lane + 64 * q < k) y[q] -= ac[q] * xk;
        ac[q] = aug[row[q] + max(k - 1, 0)];  // the next column, a step ahead
      }
    }
  }
  return true;
}

}  // namespace ohm
