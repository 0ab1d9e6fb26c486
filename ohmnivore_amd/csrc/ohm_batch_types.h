// ohm_batch_types.h — scalars and per-system state of the batched solves
// (ohm_batch.hip, ohm_batch_resident.hip).
#pragma once

#include "ohm_precond.h"
#include "ohm_reduce.h"

namespace ohm {

// Batches whose largest system has at most this many rows may run one
// workgroup per system (k_bpersist).
constexpr int kPersistRows = 4096;

// ------------------------------------------------------------ scalars ----
template <typename R>
struct cx {
  R re, im;
};
template <typename R>
__device__ __forceinline__ cx<R> operator+(cx<R> a, cx<R> b) {
  return {a.re + b.re, a.im + b.im};
}
template <typename R>
__device__ __forceinline__ cx<R> operator-(cx<R> a, cx<R> b) {
  return {a.re - b.re, a.im - b.im};
}
template <typename R>
__device__ __forceinline__ cx<R> operator*(cx<R> a, cx<R> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

template <typename S>
struct Tr;
template <>
struct Tr<double> {
  using R = double;
  static constexpr bool C = false;
};
template <>
struct Tr<float> {
  using R = float;
  static constexpr bool C = false;
};
template <>
struct Tr<cx<double>> {
  using R = double;
  static constexpr bool C = true;
};
template <>
struct Tr<cx<float>> {
  using R = float;
  static constexpr bool C = true;
};

template <typename S>
__device__ __forceinline__ S mk(double re, double im) {
  using R = typename Tr<S>::R;
  if constexpr (Tr<S>::C)
    return S{(R)re, (R)im};
  else
    return (S)re;
}
template <typename S>
__device__ __forceinline__ S zero() {
  return mk<S>(0.0, 0.0);
}
template <typename S>
__device__ __forceinline__ double re_of(S a) {
  if constexpr (Tr<S>::C)
    return (double)a.re;
  else
    return (double)a;
}
template <typename S>
__device__ __forceinline__ double im_of(S a) {
  if constexpr (Tr<S>::C)
    return (double)a.im;
  else
    return 0.0;
}

// a_k = g_k + sigma c_k on the fly
template <typename S>
__device__ __forceinline__ S aval(typename Tr<S>::R g, typename Tr<S>::R c, double sr, double si) {
  using R = typename Tr<S>::R;
  if constexpr (Tr<S>::C)
    return S{g + (R)sr * c, (R)si * c};
  else
    return g + (R)sr * c;
}

// conj(a) . b and ||a||^2 accumulators (compensated in FP32)
template <typename S>
struct DotAcc {
  Acc<typename Tr<S>::R> re, im;
  __device__ __forceinline__ void add(S a, S b) {
    if constexpr (Tr<S>::C) {
      re.add_prod(a.re, b.re);
      re.add_prod(a.im, b.im);
      im.add_prod(a.re, b.im);
      im.add_prod(-a.im, b.re);
    } else {
      re.add_prod(a, b);
    }
  }
};
template <typename S>
struct NrmAcc {
  Acc<typename Tr<S>::R> s;
  __device__ __forceinline__ void add(S a) {
    if constexpr (Tr<S>::C) {
      s.add_prod(a.re, a.re);
      s.add_prod(a.im, a.im);
    } else {
      s.add_prod(a, a);
    }
  }
};

// double-precision complex helpers for the per-system scalar algebra
struct zd {
  double re, im;
};
__device__ __forceinline__ zd zmul(zd a, zd b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ zd zdiv(zd a, zd b) {
  const double d = b.re * b.re + b.im * b.im;
  return {(a.re * b.re + a.im * b.im) / d, (a.im * b.re - a.re * b.im) / d};
}
__device__ __forceinline__ double zabs2(zd a) { return a.re * a.re + a.im * a.im; }

// ---------------------------------------------------------- batch state --
struct BSys {
  double rho[2], alpha[2], omega[2], beta[2];
  double abs_tol, bnorm2, rr, ss, rhrh;
  int status, s_conv, iters, max_iters;
  unsigned counter;
  int scaled;
  int started;  // persistent kernel: scalars below the vectors are live
  int pad;
};

struct BGeo {
  const uint32_t *rowptr, *col;
  const double *g, *c;      // c may be null (then sigma is ignored)
  const float *g32, *c32;
  double sig_re, sig_im;
  int64_t off;              // offset of this system in the concatenated vectors
  int n;
  int first_block, n_blocks;
  int pad;
};

template <typename S>
__device__ __forceinline__ const typename Tr<S>::R *gvals(const BGeo &q) {
  if constexpr (sizeof(typename Tr<S>::R) == 8)
    return q.g;
  else
    return q.g32;
}
template <typename S>
__device__ __forceinline__ const typename Tr<S>::R *cvals(const BGeo &q) {
  if constexpr (sizeof(typename Tr<S>::R) == 8)
    return q.c;
  else
    return q.c32;
}

template <typename S>
__device__ __forceinline__ S load_a(const BGeo &q, const typename Tr<S>::R *g,
                                    const typename Tr<S>::R *c, uint32_t k) {
  using R = typename Tr<S>::R;
  return aval<S>(g[k], c ? c[k] : (R)0, q.sig_re, q.sig_im);
}

__device__ __forceinline__ bool brk_small(double num_abs, double scale, int scaled,
                                          double abs_thresh) {
  return scaled ? num_abs <= 1e-30 * scale : num_abs < abs_thresh;
}

}  // namespace ohm
