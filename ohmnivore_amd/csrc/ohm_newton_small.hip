// ohm_newton_small.hip — whole Newton runs of circuits of at most 64 unknowns
// in one workgroup.
//
// One Newton iteration of the general path is about twenty launches and two
// status readbacks (evaluation, assembly, seven for the ILU(0) / ISAI refresh,
// the one-wave BiCGSTAB or a dense LU, limiting, convergence): on a 20-stage
// inverter chain 140 us of kernels, most of them 2-4 us long, inside 190 us of
// wall time. Here the same steps follow each other behind workgroup barriers,
// and up to kSmallIters iterations run before the host reads one word. The
// arithmetic of every step is the general path's (the same device functions,
// the same order), so iterates and counts are its own to the bit.
//
// Bound by latency in one CU: the sub-solve's wave (7.8 us per BiCGSTAB
// iteration at 54 unknowns) and the chains of the ILU / ISAI sweeps. Up to 64
// unknowns, where the one-wave solve applies (newton_small_fits has the other
// bounds): the rest of the chip would be idle either way. 50-stage inverter
// chain .DC (390 Newton iterations in 39 runs) 75 -> 31 ms, 20-stage .TRAN
// (1,229 iterations) 177 -> 95 ms; 76 us per ISAI iteration, 60 per dense one.
#include <algorithm>

#include "ohm_dense_dev.h"
#include "ohm_fused.h"
#include "ohm_isai_dev.h"
#include "ohm_newton_small.h"

namespace ohm {

constexpr int kSmallThreads = 256;
constexpr int kSmallWaves = kSmallThreads / 64;

struct SmallGather {
  int nt;
  const uint32_t *target, *ptr, *src;
  const double *sign;
};

struct SmallArgs {
  int n, nd, nq, nm;
  const ohm_diode_desc *dd;
  const ohm_bjt_desc *qd;
  const ohm_mosfet_desc *md;
  double *x, *x_old, *S, *rhs;
  const double *base_val, *base_b;
  FusedCsr a, ml, mu;
  double *aval;                 // a.val, writable
  const int32_t *diag_pos;
  double *inv;                  // Jacobi
  float *inv32;
  IsaiView isai;
  SmallGather gm, gb;
  int serial_diode, serial_bjt;
  int dense, first, budget;
  double abs_tol, tol, floor_rel;
  int shadow, max_iters, scaled;
  Forcing fc;
  SmallWord *out;
};

__device__ __forceinline__ bool small_breakdown(int s) {
  return s == ST_BRK_RHO || s == ST_BRK_RV || s == ST_BRK_TT || s == ST_BRK_OMEGA;
}

// every assembled entry a device touches, rewritten from base
__device__ __forceinline__ void small_gather(const SmallGather &g, const double *S,
                                             const double *base, double *out, int *nan) {
  for (int t = threadIdx.x; t < g.nt; t += kSmallThreads) {
    const uint32_t pos = g.target[t];
    const double v = gather_one(base[pos], g.ptr[t], g.ptr[t + 1], g.src, g.sign, S);
    out[pos] = v;
    if (!isfinite(v)) *nan = 1;  // every writer stores the same value
  }
}

// ILU(0) sweeps (warm-started unless `restart`), then both ISAI factors.
__device__ __forceinline__ void small_isai(const IsaiView &v, const double *aval, bool restart) {
  const int t = threadIdx.x;
  if (restart) {
    for (int64_t e = t; e < v.nf; e += kSmallThreads)
      v.f0[e] = ilu_start(e, v.from_a, v.div, aval);
    __syncthreads();
  }
  double *fin = v.f0, *fout = v.f1;
  for (int s = 0; s < v.ilu_sweeps; s++) {
    for (int64_t e = t; e < v.nf; e += kSmallThreads)
      fout[e] = ilu_entry(e, v.from_a, v.div, v.cp_ptr, v.cp_pairs, aval, fin);
    __syncthreads();
    double *h = fin;
    fin = fout;
    fout = h;
  }
  if (fin != v.f0) {  // the factors stay where the plan keeps them
    for (int64_t e = t; e < v.nf; e += kSmallThreads) v.f0[e] = fin[e];
    __syncthreads();
  }
  // the two sides sweep side by side, the shorter one idle at the end
  double *m0[2] = {v.side[0].m0, v.side[1].m0}, *m1[2] = {v.side[0].m1, v.side[1].m1};
  for (int k = 0; k < 2; k++)
    for (int64_t e = t; e < v.side[k].m; e += kSmallThreads) m0[k][e] = 0.0;
  __syncthreads();
  const int most = max(v.side[0].sweeps, v.side[1].sweeps);
  for (int s = 0; s < most; s++) {
    for (int k = 0; k < 2; k++) {
      const IsaiView::Side &d = v.side[k];
      if (s >= d.sweeps) continue;
      for (int64_t e = t; e < d.m; e += kSmallThreads)
        m1[k][e] = isai_entry(e, d.dep_ptr, d.dep, d.diag, d.is_k, v.f0, m0[k]);
      double *h = m0[k];
      m0[k] = m1[k];
      m1[k] = h;
    }
    __syncthreads();
  }
  for (int k = 0; k < 2; k++) {
    const IsaiView::Side &d = v.side[k];
    for (int64_t e = t; e < d.m; e += kSmallThreads) {
      const double w = m0[k][e];
      d.val[d.out_pos[e]] = w;
      if (d.val32) d.val32[d.out_pos[e]] = (float)w;
    }
  }
}

template <int PK>
__global__ __launch_bounds__(kSmallThreads) void k_newton_small(SmallArgs a) {
  extern __shared__ __align__(16) unsigned char small_lds[];
  __shared__ double sv[kFusedRows];
  __shared__ DenseLds dense;
  __shared__ unsigned scale[kFusedRows];
  __shared__ double wave_top[kSmallWaves];
  __shared__ int s_nan, s_limited, s_bad, s_status, s_iters;
  __shared__ double s_r0, s_res, s_eta;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, n = a.n;
  Forcing fc = a.fc;
  int reason = NS_RUNNING, it = 0, status = ST_RUNNING, nan = 0;
  double max_diff = 0.0;
  for (; it < a.budget; it++) {
    for (int i = t; i < n; i += kSmallThreads) {
      a.x_old[i] = a.x[i];
      scale[i] = kScaleOne;
    }
    if (t == 0) s_nan = s_limited = s_bad = 0;
    // evaluation and assembly
    for (int k = t; k < a.nd; k += kSmallThreads) diode_eval_one(k, a.dd, a.x, a.S);
    for (int k = t; k < a.nq; k += kSmallThreads)
      bjt_eval_one(k, a.qd, a.x, a.S + (size_t)kDiodeS * a.nd);
    for (int k = t; k < a.nm; k += kSmallThreads)
      mosfet_eval_one(k, a.md, a.x, a.S + (size_t)kDiodeS * a.nd + (size_t)kBjtS * a.nq);
    __syncthreads();
    small_gather(a.gm, a.S, a.base_val, a.aval, &s_nan);
    small_gather(a.gb, a.S, a.base_b, a.rhs, &s_nan);
    __syncthreads();
    // the linear step
    if (a.dense) {
      const bool ok = dense_lu_wg<1, kSmallWaves>(n, a.a.rowptr, a.a.col, a.aval, a.rhs, a.x,
                                                  reinterpret_cast<double *>(small_lds), dense);
      if (t == 0) {
        s_status = ok ? ST_CONVERGED : ST_BRK_RHO;
        s_iters = 0;
        s_r0 = NAN;
      }
    } else {
      if (PK == PK_ISAI) small_isai(a.isai, a.aval, a.first && it == 0);
      if (PK == PK_JACOBI)
        for (int r = t; r < n; r += kSmallThreads)
          jacobi_row(r, a.a.rowptr, a.a.col, a.aval, a.diag_pos, a.inv, a.inv32);
      __syncthreads();
      if (wave == 0) {
        // a broken-down solve again from its start with the other shadow vector
        int shadow = a.shadow;
        FusedOut o = fused_solve<PK, true>(n, a.a, a.ml, a.mu, PK == PK_ISAI, a.inv, a.rhs, a.x,
                                           shadow, 1, a.tol, a.floor_rel, OHM_TOL_INITIAL,
                                           a.max_iters, a.scaled, fc, sv, small_lds);
        int iters = o.iters;
        const double r0 = o.r0;
        if (small_breakdown(o.status)) {
          if (lane < n) a.x[lane] = a.x_old[lane];
          fused_sync();
          o = fused_solve<PK, true>(n, a.a, a.ml, a.mu, PK == PK_ISAI, a.inv, a.rhs, a.x, !shadow,
                                    1, a.tol, a.floor_rel, OHM_TOL_INITIAL, a.max_iters, a.scaled,
                                    fc, sv, small_lds);
          iters += o.iters;
        }
        if (lane == 0) {
          s_status = o.status;
          s_iters = iters;
          s_r0 = r0;
          s_res = sqrt(o.res2);
          s_eta = o.eta;
        }
      }
    }
    __syncthreads();
    status = s_status;
    nan = s_nan;
    if (t == 0) a.out->iters[it] = s_iters;
    if (fc.kind && isfinite(s_r0)) {
      fc.f_prev = s_r0;
      fc.lin_prev = s_res;
      fc.eta_prev = s_eta;
    }
    if (status != ST_CONVERGED) {
      reason = a.dense ? NS_SINGULAR : NS_SOLVE;
      it++;
      break;
    }
    // limiting: BJT, MOSFET, diode passes in this order
    bool lim = false;
    if (a.nq) {
      if (a.serial_bjt) {
        if (t == 0)
          for (int k = 0; k < a.nq; k++) lim |= bjt_limit_one(a.qd[k], a.x_old, a.x);
      } else {
        for (int k = t; k < a.nq; k += kSmallThreads)
          lim |= bjt_limit_one(a.qd[k], a.x_old, a.x);
      }
      __syncthreads();
    }
    if (a.nm) {
      for (int k = t; k < a.nm; k += kSmallThreads)
        mos_limit_reduce_one(k, a.md, a.x_old, a.x, scale);
      __syncthreads();
      for (int i = t; i < n; i += kSmallThreads) {
        const unsigned s = scale[i];
        if (s < kScaleOne) {
          a.x[i] = a.x_old[i] + (a.x[i] - a.x_old[i]) * ((double)s / (double)kScaleOne);
          lim = true;
        }
      }
      __syncthreads();
    }
    if (a.nd) {
      if (a.serial_diode) {
        if (t == 0)
          for (int k = 0; k < a.nd; k++) lim |= diode_limit_one(a.dd[k], a.x_old, a.x);
      } else {
        for (int k = t; k < a.nd; k += kSmallThreads)
          lim |= diode_limit_one(a.dd[k], a.x_old, a.x);
      }
      __syncthreads();
    }
    if (lim) s_limited = 1;
    // convergence
    double m = 0.0;
    bool bad = false;
    for (int i = t; i < n; i += kSmallThreads) {
      const double v = a.x[i];
      bad |= !isfinite(v);
      m = fmax(m, fabs(v - a.x_old[i]));
    }
    if (bad) s_bad = 1;
    m = wave_max(m);
    if (lane == 0) wave_top[wave] = m;
    __syncthreads();
    max_diff = 0.0;
    for (int w = 0; w < kSmallWaves; w++) max_diff = fmax(max_diff, wave_top[w]);
    nan = s_bad || nan;
    if (fc.kind && s_limited) fc.f_prev = -1.0;
    const bool stop_nan = nan != 0, conv = max_diff < a.abs_tol;
    __syncthreads();  // the flags are reset at the top
    if (stop_nan || conv) {
      reason = stop_nan ? NS_NAN : NS_CONVERGED;
      it++;
      break;
    }
  }
  if (t == 0) {
    a.out->reason = reason;
    a.out->done = it;
    a.out->status = status;
    a.out->nan = nan;
    a.out->max_diff = max_diff;
    a.out->f_prev = fc.f_prev;
    a.out->lin_prev = fc.lin_prev;
    a.out->eta_prev = fc.eta_prev;
  }
}

// LDS of the staged matrices and the products of the largest.
static size_t small_solve_lds(const ohm_newton_ctx *c) {
  size_t lds = fused_stage_bytes((uint32_t)c->A.nnz);
  int64_t most = c->A.nnz;
  if (c->P.kind == PK_ISAI) {
    for (const DevCsr *m : {&c->P.ml, &c->P.mu}) {
      lds += fused_stage_bytes((uint32_t)m->nnz);
      most = std::max(most, m->nnz);
    }
  }
  return lds <= kFusedLdsBytes ? lds + 8 * (size_t)std::max<int64_t>(most, 1) : 0;
}

bool newton_small_fits(const ohm_newton_ctx *c, const ohm_newton_params &prm) {
  // devices: a thread walks at most eight of a kind
  constexpr int kMost = 8 * kSmallThreads;
  if (!fused_small(c->n) || c->n < 1 || c->nd > kMost || c->nq > kMost || c->nm > kMost)
    return false;
  if (prm.linear_solver == OHM_LINEAR_DENSE_LU) return true;
  if (prm.precision != OHM_PRECISION_FP64 || prm.bicgstab_max_iterations <= 0 ||
      !(prm.bicgstab_tolerance > 0.0) || !std::isfinite(prm.bicgstab_tolerance))
    return false;
  // one thread walks devices that share nodes: with 800 of them the general
  // path's saved launches no longer make up for it (14 unknowns, ISAI: 200
  // diodes 2.4 -> 1.8 ms a run, 400 5.6 -> 5.4, 800 8.9 -> 9.5)
  if (c->serial_diode && c->nd > 512) return false;
  // 256 threads sweep the factors where the general path has 1,024: 62
  // unknowns and 460 entries 4.2 -> 3.7 ms, 545 4.9 -> 5.0, 948 11.0 -> 12.2; 52
  // and 422 3.4 -> 3.2, 511 4.2 -> 4.4; 32 and 736 4.6 -> 3.7
  IsaiView v;
  if (c->P.kind == PK_ISAI && (!isai_view(c->P, v) || (c->n > 36 && v.nf > 448))) return false;
  return small_solve_lds(c) > 0;
}

ohm_status newton_small_launch(ohm_newton_ctx *c, const ohm_newton_params &prm, const BicgOpts &o,
                               const Forcing &fc, int budget, bool first, SmallWord &out) {
  ohm_backend *b = c->b;
  if (!c->small) OHM_HIP(hipMalloc(&c->small, sizeof(SmallWord)));
  SmallArgs a{};
  a.n = c->n;
  a.nd = c->nd;
  a.nq = c->nq;
  a.nm = c->nm;
  a.dd = c->dd;
  a.qd = c->qd;
  a.md = c->md;
  a.x = c->x;
  a.x_old = c->x_old;
  a.S = c->S;
  a.rhs = c->rhs;
  a.base_val = c->base_val;
  a.base_b = c->base_b;
  a.a = FusedCsr{c->A.rowptr, c->A.col, c->A.val};
  a.aval = c->A.val;
  a.diag_pos = c->A.diag_pos;
  a.gm = SmallGather{c->nt_m, c->tm, c->pm, c->sm, c->gm};
  a.gb = SmallGather{c->nt_b, c->tb, c->pb, c->sb, c->gb};
  a.serial_diode = c->serial_diode;
  a.serial_bjt = c->serial_bjt;
  a.dense = prm.linear_solver == OHM_LINEAR_DENSE_LU;
  a.first = first;
  a.budget = std::min(budget, kSmallIters);
  a.abs_tol = prm.abs_tol;
  a.tol = prm.bicgstab_tolerance;
  a.floor_rel = o.tol_floor;
  a.shadow = o.shadow == OHM_SHADOW_HASHED ? 1 : 0;
  a.max_iters = (int)std::min<int64_t>(o.max_iters, 0x7fffffff);
  a.scaled = o.scaled_breakdown ? 1 : 0;
  a.fc = fc;
  a.out = static_cast<SmallWord *>(c->small);
  size_t lds = 0;
  int pk = PK_NONE;
  if (a.dense) {
    lds = sizeof(double) * c->n * dense_lds_stride(c->n);
  } else {
    lds = small_solve_lds(c);
    pk = c->P.kind;
    if (pk == PK_ISAI) {
      if (!isai_view(c->P, a.isai)) return fail(OHM_ERR_INVALID, "preconditioner without a plan");
      a.ml = FusedCsr{c->P.ml.rowptr, c->P.ml.col, c->P.ml.val};
      a.mu = FusedCsr{c->P.mu.rowptr, c->P.mu.col, c->P.mu.val};
    } else if (pk == PK_JACOBI) {
      a.inv = c->P.inv;
      a.inv32 = c->P.has_f32 ? c->P.inv32 : nullptr;
    }
  }
  const auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(1), dim3(kSmallThreads), (unsigned)lds, b->stream, a);
  };
  if (pk == PK_ISAI)
    launch(k_newton_small<PK_ISAI>);
  else if (pk == PK_JACOBI)
    launch(k_newton_small<PK_JACOBI>);
  else
    launch(k_newton_small<PK_NONE>);
  OHM_HIP(hipGetLastError());
  b->dispatches++;
  if (pk == PK_ISAI) isai_started(c->P);
  OHM_HIP(hipMemcpyAsync(b->h_pinned, c->small, sizeof(SmallWord), hipMemcpyDeviceToHost,
                         b->stream));
  OHM_HIP(hipStreamSynchronize(b->stream));
  b->readbacks++;
  out = *reinterpret_cast<const SmallWord *>(b->h_pinned);
  return OHM_OK;
}

}  // namespace ohm
