// ohm_dense.hip — dense LU with partial pivoting on the GPU for small
// systems: the direct solver behind a Newton run whose iterative sub-solve
// cannot converge (the reference falls back to a CPU sparse LU there,
// src/analysis/dc.rs:112-131; NewtonLinearMode::CpuSparseLu,
// src/solver/newton.rs:22-30,286-289).
//
// Layout: the CSR matrix is scattered into a row-major n x n FP64 array in
// HBM (134 MB at the 4096-row limit, kept on the backend for later solves).
// Elimination step k is two launches: a one-workgroup pivot search + row
// swap (matrix and right-hand side), then
// a trailing update over rows k+1..n-1 and columns k+1..n-1 (plus the
// right-hand side as column n) with the multiplier a_ik / a_kk recomputed
// per element, so column k is only read during the update and no multiplier
// array is needed. Back substitution runs in one workgroup.
//
// Systems of up to kDenseLdsRows unknowns (the matrix and right-hand side fit
// a CU's 160 KB of LDS) are solved in one launch of one workgroup instead.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "ohm_internal.h"
#include "ohm_reduce.h"

namespace ohm {

namespace {

constexpr int kDenseWg = 1024;

__global__ void k_dense_zero(int64_t m, double *__restrict__ d) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < m;
       i += (int64_t)gridDim.x * kBlock)
    d[i] = 0.0;
}

__global__ void k_dense_scatter(int n, const uint32_t *__restrict__ rowptr,
                                const uint32_t *__restrict__ col, const double *__restrict__ val,
                                const double *__restrict__ rhs, double *__restrict__ d,
                                double *__restrict__ y) {
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= n) return;
  for (uint32_t k = rowptr[r]; k < rowptr[r + 1]; k++) d[(int64_t)r * n + col[k]] += val[k];
  y[r] = rhs[r];
}

// argmax_{i >= k} |d[i][k]| (lowest index on ties), then swap rows k and p
// of d and y; flag[0] = 1 if the pivot is zero
__global__ __launch_bounds__(kDenseWg) void k_dense_pivot(int n, int k, double *__restrict__ d,
                                                          double *__restrict__ y,
                                                          int *__restrict__ flag) {
  __shared__ double sv[kDenseWg / 64];
  __shared__ int si[kDenseWg / 64];
  __shared__ int s_p;
  double best = -1.0;
  int bi = n;
  for (int i = k + threadIdx.x; i < n; i += kDenseWg) {
    const double a = fabs(d[(int64_t)i * n + k]);
    if (a > best) {
      best = a;
      bi = i;
    }
  }
  // wave64 reduction of (value, index)
  for (int off = 32; off > 0; off >>= 1) {
    const double ov = __shfl_xor(best, off, 64);
    const int oi = __shfl_xor(bi, off, 64);
    if (ov > best || (ov == best && oi < bi)) {
      best = ov;
      bi = oi;
    }
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    sv[w] = best;
    si[w] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double bv = sv[0];
    int bx = si[0];
    for (int q = 1; q < kDenseWg / 64; q++)
      if (sv[q] > bv || (sv[q] == bv && si[q] < bx)) {
        bv = sv[q];
        bx = si[q];
      }
    if (!(bv > 1e-300) || bx >= n) {
      flag[0] = 1;
      bx = k;
    }
    s_p = bx;
  }
  __syncthreads();
  const int p = s_p;
  if (p != k) {
    for (int j = threadIdx.x; j < n; j += kDenseWg) {
      const double t = d[(int64_t)k * n + j];
      d[(int64_t)k * n + j] = d[(int64_t)p * n + j];
      d[(int64_t)p * n + j] = t;
    }
    if (threadIdx.x == 0) {
      const double t = y[k];
      y[k] = y[p];
      y[p] = t;
    }
  }
}

// rows i in (k, n), columns j in (k, n] (j == n: the right-hand side)
__global__ void k_dense_update(int n, int k, double *__restrict__ d, double *__restrict__ y) {
  const int m = n - k - 1;  // rows and matrix columns below / right of the pivot
  const int64_t total = (int64_t)m * (m + 1);
  const double piv = d[(int64_t)k * n + k];
  for (int64_t e = blockIdx.x * (int64_t)kBlock + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * kBlock) {
    const int i = k + 1 + (int)(e / (m + 1));
    const int jj = (int)(e % (m + 1));
    const double l = d[(int64_t)i * n + k] / piv;
    if (jj == m)
      y[i] -= l * y[k];
    else {
      const int j = k + 1 + jj;
      d[(int64_t)i * n + j] -= l * d[(int64_t)k * n + j];
    }
  }
}

__global__ __launch_bounds__(kDenseWg) void k_dense_backsub(int n, const double *__restrict__ d,
                                                            double *__restrict__ y,
                                                            double *__restrict__ x) {
  __shared__ double xk;
  for (int k = n - 1; k >= 0; k--) {
    if (threadIdx.x == 0) {
      xk = y[k] / d[(int64_t)k * n + k];
      x[k] = xk;
    }
    __syncthreads();
    const double v = xk;
    for (int i = threadIdx.x; i < k; i += kDenseWg) y[i] -= d[(int64_t)i * n + k] * v;
    __syncthreads();
  }
}

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

template <int R, int kWavesLu>  // rows per lane, waves
__global__ __launch_bounds__(64 * kWavesLu) void k_dense_lu_wg(
    int n, int ld, const uint32_t *__restrict__ rowptr, const uint32_t *__restrict__ col,
    const double *__restrict__ val, const double *__restrict__ rhs, double *__restrict__ x,
    int *__restrict__ flag) {
  extern __shared__ __align__(16) double aug[];  // [n][ld], column n the right-hand side
  __shared__ uint32_t ptr[kDenseLdsRows + 1];
  __shared__ double piv[kDenseLdsRows], rpiv[kDenseLdsRows];
  __shared__ int order[kDenseLdsRows];
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
      if (t == 0) flag[0] = 1;
      return;
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
  if (wave) return;
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
}

}  // namespace

// Waits for a solve and reports a zero pivot.
static ohm_status dense_result(ohm_backend *b, const int *flag) {
  OHM_HIP(hipGetLastError());
  int h = 0;
  OHM_HIP(hipMemcpyAsync(&h, flag, sizeof(int), hipMemcpyDeviceToHost, b->stream));
  OHM_HIP(hipStreamSynchronize(b->stream));
  b->readbacks++;
  if (h) return fail(OHM_ERR_SOLVE, "Solve error: matrix is singular (zero pivot in dense LU)");
  return OHM_OK;
}

ohm_status dense_lu_solve(ohm_backend *b, const DevCsr &a, const double *rhs, double *x) {
  const int n = a.n;
  if (n <= 0) return OHM_OK;
  if (n > kDenseMaxRows)
    return fail(OHM_ERR_INVALID, "dense LU is limited to %d unknowns (system has %d)",
                kDenseMaxRows, n);
  hipStream_t st = b->stream;
  // workspace kept on the backend between solves (a Newton run in this mode
  // solves once per iteration): n*n matrix, n right-hand side, one flag
  const int64_t nn = (int64_t)n * n;
  const size_t need = sizeof(double) * (size_t)(nn + n) + 256;
  if (b->dense_ws_bytes < need) {
    if (b->dense_ws) OHM_HIP(hipFree(b->dense_ws));
    b->dense_ws = nullptr;
    b->dense_ws_bytes = 0;
    OHM_HIP(hipMalloc(&b->dense_ws, need));
    b->dense_ws_bytes = need;
  }
  double *d = reinterpret_cast<double *>(b->dense_ws), *y = d + nn;
  int *flag = reinterpret_cast<int *>(y + n);
  OHM_HIP(hipMemsetAsync(flag, 0, sizeof(int), st));
  if (n <= kDenseLdsRows) {
    const int ld = (n + 1) | 1;  // odd: a column's entries fall in different banks
    const unsigned lds = (unsigned)(sizeof(double) * n * ld);
    const auto launch = [&](auto kern, int waves) {
      hipLaunchKernelGGL(kern, dim3(1), dim3(64 * waves), lds, st, n, ld, a.rowptr, a.col, a.val,
                         rhs, x, flag);
    };
    if (n <= 64)
      launch(k_dense_lu_wg<1, 4>, 4);
    else if (n <= 128)
      launch(k_dense_lu_wg<2, 8>, 8);
    else
      launch(k_dense_lu_wg<3, 8>, 8);
    b->dispatches++;
    return dense_result(b, flag);
  }
  hipLaunchKernelGGL(k_dense_zero, dim3((unsigned)std::min<int64_t>((nn + kBlock - 1) / kBlock, 8192)),
                     dim3(kBlock), 0, st, nn, d);
  hipLaunchKernelGGL(k_dense_scatter, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, n,
                     a.rowptr, a.col, a.val, rhs, d, y);
  for (int k = 0; k < n; k++) {
    hipLaunchKernelGGL(k_dense_pivot, dim3(1), dim3(kDenseWg), 0, st, n, k, d, y, flag);
    const int64_t m = n - k - 1;
    if (m > 0) {
      const int64_t total = m * (m + 1);
      hipLaunchKernelGGL(k_dense_update,
                         dim3((unsigned)std::min<int64_t>((total + kBlock - 1) / kBlock, 4096)),
                         dim3(kBlock), 0, st, n, k, d, y);
    }
  }
  hipLaunchKernelGGL(k_dense_backsub, dim3(1), dim3(kDenseWg), 0, st, n, d, y, x);
  b->dispatches += 2 * n + 3;
  return dense_result(b, flag);
}

}  // namespace ohm
