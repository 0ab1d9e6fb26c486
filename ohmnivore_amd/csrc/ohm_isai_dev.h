// ohm_isai_dev.h — the ILU(0) / ISAI fixed-point sweeps entry by entry
// (kernels in ohm_isai.hip, the small Newton run in ohm_newton_small.hip).
#pragma once

#include "ohm_precond.h"

namespace ohm {

// Device arrays of one preconditioner's numeric refresh.
struct IsaiView {
  int64_t nf = 0;               // factor entries
  const int32_t *from_a, *div;  // A position / pivot position per factor entry, or -1
  const uint32_t *cp_ptr, *cp_pairs;
  double *f0, *f1;              // factors, and the other buffer of the sweeps
  int ilu_sweeps = 0;
  struct Side {
    int64_t m = 0;
    const uint32_t *dep_ptr, *dep;
    const int32_t *diag;
    const uint8_t *is_k;
    const uint32_t *out_pos;
    double *m0, *m1;
    int sweeps = 0;
    double *val;
    float *val32;
  } side[2];
};
// False when the factors are too large for one workgroup or the product
// M_U M_L is formed.
bool isai_view(const PrecondDev &p, IsaiView &v);

// v - sum over the pairs [q0, q1) of f[first] g[second], in order; four pairs
// are loaded at a time, because a supply node's entry has one for every stage
// and each pair waits for its indices and then for its values.
__device__ __forceinline__ double minus_pairs(double v, uint32_t q0, uint32_t q1,
                                              const uint32_t *pairs, const double *f,
                                              const double *g) {
  uint32_t q = q0;
  for (; q + 4 <= q1; q += 4) {
    uint32_t i[4], k[4];
    double a[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      i[j] = pairs[2 * (q + j)];
      k[j] = pairs[2 * (q + j) + 1];
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] = f[i[j]];
      b[j] = g[k[j]];
    }
#pragma unroll
    for (int j = 0; j < 4; j++) v = fma(-a[j], b[j], v);
  }
  for (; q < q1; q++) v = fma(-f[pairs[2 * q]], g[pairs[2 * q + 1]], v);
  return v;
}

__device__ __forceinline__ double ilu_start(int64_t e, const int32_t *from_a, const int32_t *div,
                                            const double *aval) {
  const int32_t s = from_a[e], d = div[e];
  double v = s >= 0 ? aval[s] : 0.0;
  if (d >= 0) {
    const int32_t ad = from_a[d];
    const double piv = ad >= 0 ? aval[ad] : 0.0;
    v = fabs(piv) < 1e-30 ? 0.0 : v / piv;
  }
  return v;
}
__device__ __forceinline__ double ilu_entry(int64_t e, const int32_t *from_a, const int32_t *div,
                                            const uint32_t *ptr, const uint32_t *pairs,
                                            const double *aval, const double *fin) {
  const int32_t s = from_a[e], d = div[e];
  double v = minus_pairs(s >= 0 ? aval[s] : 0.0, ptr[e], ptr[e + 1], pairs, fin, fin);
  if (d >= 0) {
    const double piv = fin[d];
    v = fabs(piv) < 1e-30 ? 0.0 : v / piv;
  }
  return v;
}
__device__ __forceinline__ double isai_entry(int64_t e, const uint32_t *ptr, const uint32_t *dep,
                                             const int32_t *diag, const uint8_t *is_k,
                                             const double *f, const double *min_) {
  double v = minus_pairs(is_k[e] ? 1.0 : 0.0, ptr[e], ptr[e + 1], dep, f, min_);
  const int32_t d = diag[e];
  if (d >= 0) {
    const double piv = f[d];
    v = fabs(piv) < 1e-30 ? 0.0 : v / piv;
  }
  return v;
}

}  // namespace ohm
