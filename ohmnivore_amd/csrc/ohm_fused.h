// ohm_fused.h — the BiCGSTAB solve of a system of at most 64 unknowns in one
// wave, as a device function (ohm_bicgstab.hip launches it alone,
// ohm_newton_small.hip inside a Newton run), and the scalar rules it shares
// with the multi-kernel pipeline.
#pragma once

#include "ohm_precond.h"
#include "ohm_spmv.h"

namespace ohm {

// Breakdown tests: the reference's absolute thresholds, or the same 1e-30
// applied to normalised quantities.
__device__ __forceinline__ bool rho_breakdown(double rho, double hh, double rr, int scaled) {
  return scaled ? fabs(rho) <= 1e-30 * (sqrt(hh) * sqrt(rr)) : fabs(rho) < 1e-30;
}

// Inexact-Newton forcing term for a sub-solve starting at ||F_k|| = f
// (Eisenstat & Walker, SIAM J. Sci. Comput. 17(1), 1996: choice 1 with the
// eta^((1+sqrt 5)/2) safeguard, choice 2 with gamma 0.9, alpha 2), clamped to
// [eta_min, eta_max]; eta_max on the first Newton iteration.
__host__ __device__ inline double forcing_eta(const Forcing &fc, double f) {
  double eta = fc.eta_max;
  if (fc.f_prev > 0.0 && f == f && f < INFINITY) {
    double safe;
    if (fc.kind == OHM_FORCING_EW1) {
      eta = fabs(f - fc.lin_prev) / fc.f_prev;
      safe = pow(fc.eta_prev, 1.6180339887498949);
    } else {
      const double q = f / fc.f_prev;
      eta = 0.9 * q * q;
      safe = 0.9 * fc.eta_prev * fc.eta_prev;
    }
    if (safe > 0.1 || fc.rate_cap) eta = fmax(eta, safe);
    eta = fmin(fc.eta_max, fmax(fc.eta_min, eta));
  }
  return eta;
}

// p_j = r_j + beta (p_j - omega v_j), one rounding sequence for every use.
template <typename T>
__device__ __forceinline__ T p_next(T r, T p, T v, T beta, T omega) {
  return fmac<T>(fmac<T>(-omega, v, p), beta, r);
}

// ------------------------------------------------------ one-wave solve --
// The whole solve of a system of at most 64 unknowns in one 64-lane
// workgroup (the reference's bicgstab_fused, src/solver/ds_shaders.rs:
// 340-728, dispatched for tiny Newton systems at src/solver/newton.rs:
// 216-252): lane r owns row r and keeps its entries of every vector in
// registers; a matrix-vector product gathers from the one vector staged in
// LDS; dot products are DPP wave sums. The recurrences, stopping tests,
// breakdown tests, shadow residual and forcing are those of the multi-kernel
// pipeline above (K1-K5 and k_init), in the same order; the loop is bounded
// by max_iters, so the workgroup always exits.
constexpr int kFusedRows = 64;
constexpr uint32_t kFusedLdsBytes = 60 * 1024;  // staged matrices, beside the vector

// Orders the wave's LDS writes before its later reads: lanes of one wave run
// in step, so no barrier is needed, only that the compiler keeps the order.
__device__ __forceinline__ void fused_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct FusedCsr {
  const uint32_t *rowptr, *col;
  const double *val;
};

// Rows of at most this many entries are walked by their own lanes, four
// entries at a time; one longer row makes the lanes share all products of its
// matrix (a 40-section ladder, 3 entries a row: 64 us walked, 82 shared).
constexpr uint32_t kFusedOwnRow = 8;

// One matrix of the solve: a lane's row bounds in registers, the column
// indices and values in LDS (STAGE) or global memory.
struct FusedRow {
  uint32_t beg, end, nnz;
  bool shared;  // the lanes form the products together (some row is long)
  const uint32_t *col;
  const double *val;
};

// Bytes of LDS the staged column indices and values of a matrix take.
__host__ __device__ inline uint32_t fused_stage_bytes(uint32_t nnz) {
  return 8 * nnz + ((4 * nnz + 7) & ~7u);
}

// Binds lane r to its row of m; with STAGE the whole matrix's columns and
// values are copied into LDS at lds (advanced past them). The caller
// synchronises before the first use.
template <bool STAGE>
__device__ __forceinline__ FusedRow fused_bind(const FusedCsr &m, int r, int n,
                                               unsigned char *&lds) {
  FusedRow f{0, 0, 0, false, m.col, m.val};
  if (STAGE) {  // LDS pointers on every path, so the loads compile to ds_read
    f.col = reinterpret_cast<const uint32_t *>(lds);
    f.val = reinterpret_cast<const double *>(lds);
  }
  if (!m.rowptr) return f;
  if (r < n) {
    f.beg = m.rowptr[r];
    f.end = m.rowptr[r + 1];
  }
  if (STAGE) {
    f.shared = __any(f.end - f.beg > kFusedOwnRow);
    f.nnz = m.rowptr[n];
    double *v = reinterpret_cast<double *>(lds);
    uint32_t *c = reinterpret_cast<uint32_t *>(lds + 8 * f.nnz);
    for (uint32_t k = threadIdx.x & 63; k < f.nnz; k += kFusedRows) {
      v[k] = m.val[k];
      c[k] = m.col[k];
    }
    lds += fused_stage_bytes(f.nnz);
    f.col = c;
    f.val = v;
  }
  return f;
}

// y_r = (A v)_r with v staged in LDS (every lane writes its v_r first). Each
// product is rounded, then a row's products are summed in column order from
// 0, the rounding sequence of the pipeline's row-block SpMV, so the two paths
// agree to the bit. With a long row among them the lanes form all products
// together, wherever their rows lie, and leave them in LDS at sp; a lane then
// adds its row's, eight reads at a time. Lanes that walked their own entries
// one by one waited for two dependent LDS reads per entry, and the whole wave
// for its longest row (a supply node's): 161 -> 84 us per solve of a 50-stage
// inverter chain (54 unknowns), 97 -> 61 us at 24 unknowns.
template <bool STAGE>
__device__ __forceinline__ double fused_spmv(const FusedRow &m, double v, double *sv, double *sp) {
#pragma clang fp contract(off)
  const uint32_t lane = threadIdx.x & 63;
  fused_sync();
  sv[lane] = v;
  fused_sync();
  double acc = 0.0;
  if (!STAGE) {
    for (uint32_t k = m.beg; k < m.end; k++) {
      const double pr = m.val[k] * sv[m.col[k]];
      acc = acc + pr;
    }
    return acc;
  }
  if (!m.shared) {
    for (uint32_t k = m.beg; k < m.end; k += 4) {
      uint32_t c[4];
      double pr[4];
#pragma unroll
      for (int j = 0; j < 4; j++) c[j] = m.col[min(k + j, m.end - 1)];
#pragma unroll
      for (int j = 0; j < 4; j++) pr[j] = m.val[min(k + j, m.end - 1)] * sv[c[j]];
#pragma unroll
      for (int j = 0; j < 4; j++) acc = k + j < m.end ? acc + pr[j] : acc;
    }
    return acc;
  }
  constexpr int kStep = 4;
  for (uint32_t k0 = lane; k0 < m.nnz; k0 += kStep * kFusedRows) {
    uint32_t c[kStep];
    double a[kStep], x[kStep];
#pragma unroll
    for (int j = 0; j < kStep; j++) {
      const uint32_t k = min(k0 + j * kFusedRows, m.nnz - 1);
      c[j] = m.col[k];
      a[j] = m.val[k];
    }
#pragma unroll
    for (int j = 0; j < kStep; j++) x[j] = sv[c[j]];
#pragma unroll
    for (int j = 0; j < kStep; j++)
      if (k0 + j * kFusedRows < m.nnz) sp[k0 + j * kFusedRows] = a[j] * x[j];
  }
  fused_sync();
  if (m.beg >= m.end) return acc;
  double pr[8], ahead[8];
#pragma unroll
  for (int j = 0; j < 8; j++) pr[j] = sp[min(m.beg + j, m.end - 1)];
  for (uint32_t k = m.beg; k < m.end; k += 8) {
#pragma unroll
    for (int j = 0; j < 8; j++) ahead[j] = sp[min(k + 8 + j, m.end - 1)];
#pragma unroll
    for (int j = 0; j < 8; j++) acc = k + j < m.end ? acc + pr[j] : acc;
#pragma unroll
    for (int j = 0; j < 8; j++) pr[j] = ahead[j];
  }
  return acc;
}

template <int PK, bool STAGE>
__device__ __forceinline__ double fused_prec(const FusedRow &ml, const FusedRow &mu, bool two,
                                             double inv, double v, double *sv, double *sp) {
  if (PK == PK_JACOBI) return inv * v;
  if (PK == PK_ISAI) {
    const double y = fused_spmv<STAGE>(ml, v, sv, sp);
    return two ? fused_spmv<STAGE>(mu, y, sv, sp) : y;
  }
  return v;
}

struct FusedOut {
  int status, s_conv, iters;
  double r0, res2, eta, abs_tol;
};

// Runs in one wave (lane = threadIdx.x & 63); sv: kFusedRows doubles of LDS,
// lds: the staged matrices and the products (STAGE). Every lane returns the
// same figures; x is written whatever the status.
template <int PK, bool STAGE>
__device__ __forceinline__ FusedOut fused_solve(
    int n, const FusedCsr &ag, const FusedCsr &mlg, const FusedCsr &mug, int two,
    const double *dinv, const double *b, double *x, int shadow, int warm, double tol,
    double floor_rel, int tol_mode, int max_iters, int scaled, const Forcing &fc, double *sv,
    unsigned char *lds) {
  const int r = threadIdx.x & 63;
  const bool in = r < n;
  const FusedRow a = fused_bind<STAGE>(ag, r, n, lds);
  const FusedRow ml = fused_bind<STAGE>(mlg, r, n, lds);
  const FusedRow mu = fused_bind<STAGE>(mug, r, n, lds);
  double *sp = reinterpret_cast<double *>(lds);  // products of one matrix (STAGE)
  if (STAGE) fused_sync();
  const double inv = (PK == PK_JACOBI && in) ? dinv[r] : 1.0;
  // dot products: lanes past n add +0, as threads without a row do in the
  // pipeline's block sums
  const auto sum = [in](double v) { return wave_sum(in ? v : 0.0); };
  // k_init: r = b - A x0 (warm) or b, r_hat, p = v = 0
  const double bi = in ? b[r] : 0.0;
  double xi = (in && warm) ? x[r] : 0.0;
  double ri = bi;
  if (warm) ri = bi - fused_spmv<STAGE>(a, xi, sv, sp);
  if (!in) ri = 0.0;
  const double rh = in ? (shadow ? shadow_value((uint64_t)r) : ri) : 0.0;
  double p = 0.0, v = 0.0;
  const double bb = sum(bi * bi), hh = sum(rh * rh), hnorm = sqrt(hh);
  double rr = sum(ri * ri), rhr = sum(rh * ri);
  const double r0 = sqrt(rr);
  double eta = 0.0;
  if (fc.kind) {
    tol = forcing_eta(fc, r0);
    eta = tol;
  }
  const double bnorm = sqrt(bb);
  const double abs_tol = tol_mode == OHM_TOL_INITIAL ? fmax(tol * r0, floor_rel * bnorm) : tol * bnorm;
  double rho = 1.0, alpha = 1.0, omega = 1.0, res2 = rr;
  int status = ST_RUNNING, iters = 0, s_conv = 0;
  if (bnorm < 1e-30) {  // b == 0: x = 0 (src/solver/bicgstab.rs:93-97)
    status = ST_CONVERGED;
  } else if (warm && r0 < abs_tol) {
    status = ST_CONVERGED;
  } else if (rho_breakdown(rhr, hh, rr, scaled)) {
    status = ST_BRK_RHO;
  }
  while (status == ST_RUNNING) {
    // K1 head (decide_rho) and p update
    const double rnorm = sqrt(rr);
    if (s_conv) { status = ST_CONVERGED; break; }
    if (std::isnan(rnorm) || std::isinf(rnorm)) { status = ST_NAN; break; }
    if (rnorm < abs_tol) { status = ST_CONVERGED; break; }
    if (fabs(omega) < 1e-30) { status = ST_BRK_OMEGA; break; }
    if (iters >= max_iters) { status = ST_MAXITER; break; }
    if (scaled ? fabs(rhr) <= 1e-30 * (hnorm * rnorm) : fabs(rhr) < 1e-30) {
      status = ST_BRK_RHO;
      break;
    }
    const double beta = (rhr / rho) * (alpha / omega);
    const double rho_new = rhr;
    p = p_next<double>(ri, p, v, beta, omega);
    const double ph = fused_prec<PK, STAGE>(ml, mu, two, inv, p, sv, sp);
    // K2: v = A p_hat; K3 head: alpha
    v = fused_spmv<STAGE>(a, ph, sv, sp);
    if (!in) v = 0.0;
    const double rv = sum(rh * v), vv = sum(v * v);
    const bool brk = scaled ? fabs(rv) <= 1e-30 * (hnorm * sqrt(vv)) : fabs(rv) < 1e-30;
    if (brk) { status = ST_BRK_RV; break; }
    alpha = rho_new / rv;
    rho = rho_new;
    // K3: s = r - alpha v; K4 head: ||s|| exit
    const double s = fma(-alpha, v, ri);
    const double ss = sum(s * s);
    if (sqrt(ss) < abs_tol) {
      xi = xi + alpha * ph;
      iters++;
      s_conv = 1;
      res2 = ss;
      continue;  // the next head turns s_conv into CONVERGED
    }
    const double sh = fused_prec<PK, STAGE>(ml, mu, two, inv, s, sv, sp);
    // K4: t = A s_hat; K5: omega, x and r updates
    double t = fused_spmv<STAGE>(a, sh, sv, sp);
    if (!in) t = 0.0;
    const double ts = sum(t * s), tt = sum(t * t);
    if (scaled ? tt <= 1e-30 * ss : fabs(tt) < 1e-30) { status = ST_BRK_TT; break; }
    omega = ts / tt;
    iters++;
    xi = (xi + alpha * ph) + omega * sh;
    ri = s - omega * t;
    rr = sum(ri * ri);
    rhr = sum(rh * ri);
    res2 = rr;
  }
  if (in) x[r] = xi;
  return FusedOut{status, s_conv, iters, r0, res2, eta, abs_tol};
}

}  // namespace ohm
