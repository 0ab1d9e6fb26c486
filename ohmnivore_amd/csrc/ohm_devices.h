// ohm_devices.h — diode, BJT and MOSFET evaluation, stamp assembly and step
// limiting of one device or entry, and the Newton context they act on
// (kernels in ohm_newton.hip and ohm_newton_small.hip). Line numbers cite
// src/solver/ds_nonlinear_shaders.rs.
#pragma once

#include <vector>

#include "ohm_precond.h"
#include "ohm_reduce.h"

namespace ohm {

constexpr double kVT = 0.02585;          // MOSFET smoothing voltage (ds_nonlinear_shaders.rs:777)
constexpr unsigned kScaleOne = 1000000u; // MVL_SCALE_ONE (:1027)
constexpr double kStepLimit = 0.5;       // MVL_STEP_LIMIT (:1028)

// stamp value layout per device
constexpr int kDiodeS = 2;   // g, i_eq
constexpr int kBjtS = 12;    // G[9], ieq_c, ieq_b, ieq_e
constexpr int kMosS = 8;     // S[6], ieq_d, ieq_s

__device__ __forceinline__ double xv(const double *x, uint32_t i) {
  return i == OHM_SENTINEL ? 0.0 : x[i];
}
__device__ __forceinline__ double clamp_exp(double a) {  // ds_shaders.rs:96-108
  return exp(fmin(fmax(a, -80.0), 80.0));
}

// diode_eval_ds (:41-76) + Norton current (:212-248) of diode k
__device__ __forceinline__ void diode_eval_one(int k, const ohm_diode_desc *__restrict__ d,
                                               const double *__restrict__ x,
                                               double *__restrict__ S) {
  const ohm_diode_desc q = d[k];
  const double is = q.is_val, nvt = q.n_vt;
  const double vd = xv(x, q.anode_idx) - xv(x, q.cathode_idx);
  const double e = clamp_exp(vd / nvt);
  const double i = is * (e - 1.0), g = is * e / nvt;
  S[kDiodeS * k] = g;
  S[kDiodeS * k + 1] = i - g * vd;
}

// bjt_eval_ds (:281-367) + stamps (:394-573) of transistor k
__device__ __forceinline__ void bjt_eval_one(int k, const ohm_bjt_desc *__restrict__ d,
                                             const double *__restrict__ x,
                                             double *__restrict__ S) {
  const ohm_bjt_desc &q = d[k];
  const double pol = q.polarity, is = q.is_val, bf = q.bf, br = q.br, nf = q.nf_vt,
               nr = q.nr_vt;
  const double vc = xv(x, q.collector_idx), vb = xv(x, q.base_idx), ve = xv(x, q.emitter_idx);
  const double vbe = pol * (vb - ve), vbc = pol * (vb - vc);
  const double ef = clamp_exp(vbe / nf), er = clamp_exp(vbc / nr);
  const double i_f = is * (ef - 1.0), i_r = is * (er - 1.0);
  const double bf_frac = bf / (bf + 1.0);
  const double ic = (bf_frac * i_f - i_r / (br + 1.0)) * pol;
  const double ib = (i_f / (bf + 1.0) + i_r / (br + 1.0)) * pol;
  const double gf = is * ef / nf, gr = is * er / nr;
  const double a = bf_frac * gf, b = -(gr / (br + 1.0)), c = gf / (bf + 1.0), dd = gr / (br + 1.0);
  double G[9] = {-b, a + b, -a, -dd, c + dd, -c, b + dd, -(a + b + c + dd), a + c};
  double *s = S + (size_t)kBjtS * k;
#pragma unroll
  for (int j = 0; j < 9; j++) s[j] = G[j];
  const double ie = -(ic + ib);
  s[9] = ic - (G[0] * vc + G[1] * vb + G[2] * ve);
  s[10] = ib - (G[3] * vc + G[4] * vb + G[5] * ve);
  s[11] = ie - (G[6] * vc + G[7] * vb + G[8] * ve);
}

// Smooth level-1 MOSFET (mosfet_eval_ds :747-849; CPU twin gpu_shaders.rs:1452-1493)
__device__ __forceinline__ void mosfet_core(double vgs, double vds, double vto, double kp,
                                            double lambda, double pol, double &id, double &gm,
                                            double &gds) {
  vgs *= pol;
  vds *= pol;
  const double v_ov = vgs - vto, arg = v_ov / kVT;
  double v_ov_eff, sig;
  if (arg > 20.0) {
    v_ov_eff = v_ov;
    sig = 1.0;
  } else if (arg < -20.0) {
    const double e = exp(arg);
    v_ov_eff = kVT * e;
    sig = e;
  } else {
    v_ov_eff = kVT * log1p(exp(arg));
    sig = 1.0 / (1.0 + exp(-arg));
  }
  const double lam = 1.0 + lambda * vds;
  double i;
  if (vds < v_ov_eff) {
    const double inner = v_ov_eff * vds - vds * vds * 0.5;
    i = kp * inner * lam;
    gm = kp * vds * lam * sig;
    gds = kp * (v_ov_eff - vds) * lam + kp * inner * lambda;
  } else {
    const double sat = 0.5 * kp * v_ov_eff * v_ov_eff;
    i = sat * lam;
    gm = kp * v_ov_eff * lam * sig;
    gds = sat * lambda;
  }
  id = pol * i;
}

__device__ __forceinline__ void mosfet_eval_one(int k, const ohm_mosfet_desc *__restrict__ d,
                                                const double *__restrict__ x,
                                                double *__restrict__ S) {
  const ohm_mosfet_desc &q = d[k];
  const double vd = xv(x, q.drain_idx), vg = xv(x, q.gate_idx), vs = xv(x, q.source_idx);
  double id, gm, gds;
  mosfet_core(vg - vs, vd - vs, q.vto, q.kp, q.lambda, q.polarity, id, gm, gds);
  double *s = S + (size_t)kMosS * k;
  s[0] = gds;
  s[1] = gm;
  s[2] = -(gm + gds);
  s[3] = -gds;
  s[4] = -gm;
  s[5] = gm + gds;
  s[6] = id - (gds * vd + gm * vg - (gm + gds) * vs);
  s[7] = -id - (-gds * vd - gm * vg + (gm + gds) * vs);
}

// One target of the gather assembly: base plus its contributions in device
// order; four are loaded at a time (a supply row's right-hand side gathers
// one from every stage).
__device__ __forceinline__ double gather_one(double v, uint32_t q0, uint32_t q1,
                                             const uint32_t *src, const double *sign,
                                             const double *S) {
  uint32_t q = q0;
  for (; q + 4 <= q1; q += 4) {
    double a[4], g[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      g[j] = sign[q + j];
      a[j] = S[src[q + j]];
    }
#pragma unroll
    for (int j = 0; j < 4; j++) v = fma(g[j], a[j], v);
  }
  for (; q < q1; q++) v = fma(sign[q], S[src[q]], v);
  return v;
}

// ------------------------------------------------------------ limiting ----
__device__ __forceinline__ double pnjlim(double vnew, double vold, double vt, double vcrit) {
  if (vnew > vcrit && fabs(vnew - vold) > vt + vt) {  // :1173-1187 as written
    if (vold > 0.0) {
      const double arg = 1.0 + (vnew - vold) / vt;
      if (arg > 0.0) return vold + vt * (2.0 + log(arg - 2.0));
      return vcrit;
    }
    return vt * log(vnew / vt);
  }
  return vnew;
}

__device__ __forceinline__ void scale_node(const double *xo, double *xn, uint32_t t, double s) {
  if (t != OHM_SENTINEL) xn[t] = xo[t] + (xn[t] - xo[t]) * s;
}

__device__ bool bjt_limit_one(const ohm_bjt_desc &q, const double *xo, double *xn) {
  bool lim = false;
  const double pol = q.polarity, is = q.is_val, nf = q.nf_vt, nr = q.nr_vt;
  const double vcf = nf * log(nf / (M_SQRT2 * is)), vcr = nr * log(nr / (M_SQRT2 * is));
  const uint32_t B = q.base_idx, E = q.emitter_idx, C = q.collector_idx;
  double vo = pol * (xv(xo, B) - xv(xo, E)), vn = pol * (xv(xn, B) - xv(xn, E));
  double vl = pnjlim(vn, vo, nf, vcf);
  if (vl != vn && fabs(vn - vo) > 1e-30) {
    const double s = (vl - vo) / (vn - vo);
    if (!q.node_fixed[1]) scale_node(xo, xn, B, s);
    if (!q.node_fixed[2]) scale_node(xo, xn, E, s);
    lim = true;
  }
  vo = pol * (xv(xo, B) - xv(xo, C));
  vn = pol * (xv(xn, B) - xv(xn, C));
  vl = pnjlim(vn, vo, nr, vcr);
  if (vl != vn && fabs(vn - vo) > 1e-30) {
    const double s = (vl - vo) / (vn - vo);
    if (!q.node_fixed[1]) scale_node(xo, xn, B, s);
    if (!q.node_fixed[0]) scale_node(xo, xn, C, s);
    lim = true;
  }
  return lim;
}

__device__ bool diode_limit_one(const ohm_diode_desc &q, const double *xo, double *xn) {
  const double nvt = q.n_vt, is = q.is_val;
  const double vcrit = nvt * log(nvt / (M_SQRT2 * is));
  const double vo = xv(xo, q.anode_idx) - xv(xo, q.cathode_idx);
  const double vn = xv(xn, q.anode_idx) - xv(xn, q.cathode_idx);
  const double vl = pnjlim(vn, vo, nvt, vcrit);
  if (vl != vn && fabs(vn - vo) > 1e-30) {
    const double s = (vl - vo) / (vn - vo);
    scale_node(xo, xn, q.anode_idx, s);
    scale_node(xo, xn, q.cathode_idx, s);
    return true;
  }
  return false;
}

// mosfet_voltage_limit_reduce_ds (:1052-1103) of transistor k; scale in LDS or
// global memory
__device__ __forceinline__ unsigned encode_scale(double delta) {
  double e = floor(kStepLimit / fabs(delta) * (double)kScaleOne);
  return e < 1.0 ? 1u : (unsigned)e;
}
__device__ __forceinline__ void mos_limit_reduce_one(int k, const ohm_mosfet_desc *__restrict__ d,
                                                     const double *xo, const double *xn,
                                                     unsigned *scale) {
  const ohm_mosfet_desc &q = d[k];
  const uint32_t D = q.drain_idx, G = q.gate_idx, S = q.source_idx, f = q.node_fixed_packed;
  const double dgs = (xv(xn, G) - xv(xn, S)) - (xv(xo, G) - xv(xo, S));
  if (fabs(dgs) > kStepLimit) {
    const unsigned e = encode_scale(dgs);
    if (G != OHM_SENTINEL && !(f & 2u)) atomicMin(&scale[G], e);
    if (S != OHM_SENTINEL && !(f & 4u)) atomicMin(&scale[S], e);
  }
  const double dds = (xv(xn, D) - xv(xn, S)) - (xv(xo, D) - xv(xo, S));
  if (fabs(dds) > kStepLimit) {
    const unsigned e = encode_scale(dds);
    if (D != OHM_SENTINEL && !(f & 1u)) atomicMin(&scale[D], e);
    if (S != OHM_SENTINEL && !(f & 4u)) atomicMin(&scale[S], e);
  }
}

// convergence_check_ds (:1257-1297): max |x - x_old| and a NaN/Inf flag.
struct NewtonWord {
  double max_diff;
  int nan;
  int done;
  int limited;  // a limiter cut this iteration's step
  int pad;
};

}  // namespace ohm

struct ohm_newton_ctx {
  ohm_backend *b = nullptr;
  int n = 0;
  int64_t nnz = 0;
  int nd = 0, nq = 0, nm = 0;
  ohm::DevCsr A;                       // pattern + assembled values
  double *base_val = nullptr, *base_b = nullptr, *rhs = nullptr;
  double *x = nullptr, *x_old = nullptr, *S = nullptr;
  ohm_diode_desc *dd = nullptr;
  ohm_bjt_desc *qd = nullptr;
  ohm_mosfet_desc *md = nullptr;
  unsigned *scale = nullptr;
  int *asm_nan = nullptr;
  void *small = nullptr;  // result word of the one-workgroup run
  ohm::NewtonWord *word = nullptr;
  // gather lists: matrix slots and RHS entries
  int nt_m = 0, nt_b = 0;
  uint32_t *tm = nullptr, *pm = nullptr, *sm = nullptr, *tb = nullptr, *pb = nullptr, *sb = nullptr;
  double *gm = nullptr, *gb = nullptr;
  bool serial_diode = false, serial_bjt = false;
  ohm::PrecondDev P;
  int prec_kind = -1;
  int prec_level = 1;
  double *adj = nullptr;  // adjoint scratch: rhs, lambda, gradients (grown on demand)
  size_t adj_cap = 0;
  int zero_diag = -1;     // base matrix has a zero diagonal (-1: not yet checked)
  // host copies of the descriptors: ohm_newton_update keeps their topology
  std::vector<ohm_diode_desc> h_dd;
  std::vector<ohm_bjt_desc> h_qd;
  std::vector<ohm_mosfet_desc> h_md;
};

