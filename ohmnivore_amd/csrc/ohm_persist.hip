// ohm_persist.hip — BiCGSTAB as one resident launch.
//
// The multi-kernel pipeline (ohm_bicgstab.hip) spends five to seven dependent
// launches per iteration, each of which re-reads the matrix and pays a launch
// and a chain of dependent loads from the Infinity Cache (a kernel starts
// with cold L2s): 21 us per Jacobi iteration at 10,002 rows and 28-45 us per
// ISAI iteration at 16,388 to 129,604 rows, where the bytes of an iteration
// would take 1 to 15 us. Here every workgroup owns at most 512 consecutive
// rows for the whole solve, a thread keeps its row of every matrix and its
// entry of every vector in registers, and the workgroups meet through memory
// without leaving the kernel:
//
// - Vector entries that other rows need (r, q = p - omega v, the first
//   factor's result, p_hat / s_hat, v) go to LDS for the workgroup's own rows
//   and to memory as tagged words: 32 bits of the value beside the 32-bit
//   number of the write. A reader spins on exactly the words it needs, so a
//   matrix-vector product waits for its neighbours' values only and a value's
//   arrival needs no flag, fence or grid barrier. The words are written and
//   read with relaxed agent-scope atomics, which bypass the non-coherent L2s.
// - A dot product is one slot of tagged words per workgroup; every workgroup
//   sums all slots in the same order, so all hold the same bits and take the
//   same decision. Two sets of slots alternate: a workgroup can write a set
//   again only after every other one has written, and therefore read, the
//   other set. The same argument covers the tagged vectors: between a
//   vector's last read and its next write lies a reduction.
//
// Jacobi: 3 reductions per iteration and no other exchange (p_hat and s_hat
// are formed from r, q and v as they are gathered); ISAI: 3 reductions and 4
// exchanges. What bounds it is their latency, about 1.7 us a reduction over
// 20 to 128 workgroups and 1.2 us an exchange, and the 64-bit scalar
// arithmetic between them. Measured per iteration, pipeline -> here: Jacobi
// 15.3 -> 3.8 us (102 rows, one workgroup), 21.2 -> 9.7 (10,002), 21.7 -> 12.8
// (65,540), 24.7 -> 16.6 (129,604); ISAI 29.3 -> 15.1 (2,871), 27.9 -> 15.9
// (16,388), 35.7 -> 20.7 (65,540), 44.7 -> 25.9 (129,604).
//
// All workgroups must run at once: the grid has at most one workgroup per
// compute unit. A wait that lasts longer than kResLimit ends the kernel with
// nothing written (the outcome word says so to the other workgroups) and the
// host continues with the pipeline from the state that k_init left.
#include <algorithm>
#include <mutex>

#include "ohm_persist.h"
#include "ohm_spmv.h"

namespace ohm {

typedef unsigned long long u64;

constexpr u64 kResLimit = 20'000'000;  // 0.2 s of the 100 MHz wall clock
enum : u64 { RES_OPEN = 0, RES_COMMIT = 1, RES_ABORT = 2 };

template <typename T>
struct ResCsr {
  const uint32_t *rowptr, *col;
  const T *val;
};

template <typename T>
struct ResArgs {
  int n, rows;               // unknowns, rows per workgroup
  ResCsr<T> m[3];            // A, M_L, M_U
  const T *inv;              // Jacobi inverse diagonal
  T *x;
  const T *r, *rh;           // from k_init
  SolveState *st;
  u64 *words;                // tagged vectors: r, q, tmp, hat, v
  u64 *slots, *outcome;
};

__device__ __forceinline__ u64 res_load(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void res_store(u64 *p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A value as tagged words: a double's two halves, a float's one.
template <typename T>
struct Tagged;
template <>
struct Tagged<double> {
  static constexpr int kWords = 2;
  u64 lo, hi;
  __device__ __forceinline__ void load(const u64 *p) {
    lo = res_load(p);
    hi = res_load(p + 1);
  }
  __device__ __forceinline__ bool is(uint32_t tag) const {
    return (uint32_t)(lo >> 32) == tag && (uint32_t)(hi >> 32) == tag;
  }
  __device__ __forceinline__ double get() const {
    return __builtin_bit_cast(double, (hi << 32) | (uint32_t)lo);
  }
  static __device__ __forceinline__ void put(u64 *p, double v, uint32_t tag) {
    const u64 b = __builtin_bit_cast(u64, v), t = (u64)tag << 32;
    res_store(p, t | (uint32_t)b);
    res_store(p + 1, t | (b >> 32));
  }
};
template <>
struct Tagged<float> {
  static constexpr int kWords = 1;
  u64 w;
  __device__ __forceinline__ void load(const u64 *p) { w = res_load(p); }
  __device__ __forceinline__ bool is(uint32_t tag) const { return (uint32_t)(w >> 32) == tag; }
  __device__ __forceinline__ float get() const {
    return __builtin_bit_cast(float, (uint32_t)w);
  }
  static __device__ __forceinline__ void put(u64 *p, float v, uint32_t tag) {
    res_store(p, ((u64)tag << 32) | __builtin_bit_cast(uint32_t, v));
  }
};

// A wait's slow path, every 128 failed polls: true when the solve is over
// for this workgroup (another one gave up, or the time limit passed before
// any had committed).
__device__ __forceinline__ bool res_expired(u64 *outcome, volatile int *dead, u64 &t0) {
  if (*dead) return true;
  const u64 o = res_load(outcome);
  if (o == RES_COMMIT) return false;  // everything awaited has been sent
  const u64 now = wall_clock64();
  if (t0 == 0) t0 = now;
  if (o == RES_OPEN && now - t0 > kResLimit) {
    u64 want = RES_OPEN;
    if (__hip_atomic_compare_exchange_strong(outcome, &want, (u64)RES_ABORT, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
        want == RES_ABORT) {
      *dead = 1;
      return true;
    }
    return false;
  }
  if (o == RES_ABORT) {
    *dead = 1;
    return true;
  }
  return false;
}

// A thread's rows of one matrix row each as W entries: `off` is the operand's
// byte offset, into the workgroup's LDS vector or, where its bit of `far` is
// set, into the tagged vector.
template <typename T, int W>
struct RowTile {
  T val[W];
  uint32_t off[W], far;
};

template <typename T, int PK, int W>
struct Resident {
  static constexpr int kMats = PK == PK_ISAI ? 3 : 1;
  static constexpr int kR = 0, kQ = 1, kV = 2, kTmp = 3, kHat = 4;  // vector numbers
  static constexpr int kWaveCap = 16;
  static constexpr uint32_t kWordBytes = 8 * Tagged<T>::kWords;
  static constexpr bool kAhead = PK != PK_ISAI || W <= 6;  // registers left for `ahead`

  struct Shared {
    double sum[2][3][kWaveCap];
    double total[2][3];
    double part[kResMaxLong][kWaveCap];
    int long_row[kMats][kResMaxLong];
    int n_long[kMats];
    int dead, run, given_up[2];
  };

  const ResArgs<T> &a;
  Shared &sh;
  char *lv;  // LDS vectors, `rows` entries each
  int T0, t, lane, wave, waves, g, G, base, cnt;
  uint32_t round;   // reductions so far
  int8_t long_at[kMats];
  RowTile<T, W> tiles[kMats];
  Tagged<T> ahead[2][W];  // words of the foreign operands, requested early

  __device__ __forceinline__ Resident(const ResArgs<T> &a_, Shared &s_, unsigned char *lv_)
      : a(a_), sh(s_), lv(reinterpret_cast<char *>(lv_)) {
    T0 = blockDim.x;
    t = threadIdx.x;
    lane = t & 63;
    wave = t >> 6;
    waves = T0 >> 6;
    g = blockIdx.x;
    G = gridDim.x;
    base = g * a.rows;
    cnt = min(a.rows, a.n - base);
    round = 0;
  }
  __device__ __forceinline__ T near_value(int v, uint32_t off) const {
    return *reinterpret_cast<const T *>(lv + (uint32_t)(v * a.rows) * (uint32_t)sizeof(T) + off);
  }
  // x, its constancy unknown to the compiler: addresses, masks and selected
  // values derived from a row tile are formed at each use (one instruction)
  // instead of being kept in registers through the solve (hundreds)
  static __device__ __forceinline__ uint32_t hidden(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
  }
  // word of a tagged vector: a base common to the workgroup and a 32-bit offset
  __device__ __forceinline__ u64 *word(int v, uint32_t off) const {
    off = hidden(off);
    char *vec = reinterpret_cast<char *>(a.words) + (size_t)v * a.n * kWordBytes;
    return reinterpret_cast<u64 *>(vec + off);
  }
  __device__ __forceinline__ bool mine() const { return t < cnt; }

  // publish this thread's entry of vector v
  __device__ __forceinline__ void put(int v, T x, uint32_t tag) {
    if (!mine()) return;
    reinterpret_cast<T *>(lv)[v * a.rows + t] = x;
    if (G > 1) Tagged<T>::put(word(v, (uint32_t)(base + t) * kWordBytes), x, tag);
  }

  __device__ __forceinline__ uint32_t place(uint32_t col, bool &far) const {
    const uint32_t off = col - (uint32_t)base;
    far = off >= (uint32_t)cnt;
    return far ? col * kWordBytes : off * (uint32_t)sizeof(T);
  }

  // This thread's row of matrix m as a tile padded with zeros. A longer row
  // stays in CSR and is summed by the whole workgroup.
  __device__ __forceinline__ void build(int m) {
    const ResCsr<T> &c = a.m[m];
    const int row = base + (mine() ? t : 0);
    const uint32_t b0 = c.rowptr[row], len = c.rowptr[row + 1] - b0;
    const bool lg = len > (uint32_t)W;
    long_at[m] = -1;
    if (lg && mine()) {
      const int at = atomicAdd(&sh.n_long[m], 1);
      sh.long_row[m][at] = row;
      long_at[m] = (int8_t)at;
    }
    RowTile<T, W> &rt = tiles[m];
    rt.far = 0;
#pragma unroll
    for (int j = 0; j < W; j++) {
      uint32_t col = (uint32_t)row;
      T val = T(0);
      if (mine() && !lg && (uint32_t)j < len) {
        col = c.col[b0 + j];
        val = c.val[b0 + j];
        if (PK == PK_JACOBI && a.inv) val *= a.inv[col];
      }
      bool far;
      rt.off[j] = place(col, far);
      rt.val[j] = val;
      if (far) rt.far |= 1u << j;
    }
  }

  // Requests the foreign operands of one row (entries no lane of the wave
  // needs are skipped as one).
  template <int NV, int E>
  __device__ __forceinline__ void request(const RowTile<T, E> &rt, const int (&vec)[NV],
                                          Tagged<T> (&w)[NV][E]) const {
    const uint32_t far = hidden(rt.far);
    if (!__any(far != 0)) return;
#pragma unroll
    for (int j = 0; j < E; j++)
      if (far >> j & 1) {
#pragma unroll
        for (int v = 0; v < NV; v++) w[v][j].load(word(vec[v], rt.off[j]));
      }
  }

  // acc += val . u over E entries whose foreign words `w` were requested
  // (u = e0, or e0 + coef e1 with two vectors): this workgroup's own entries
  // from LDS, then the foreign ones in order, spinning until their words
  // carry the tag. Entries of the other kind take part with a zero, so that
  // every load is issued before the first is used.
  template <int NV, int E>
  __device__ __forceinline__ T gather(const RowTile<T, E> &rt, const int (&vec)[NV],
                                      const uint32_t (&tag)[NV], Tagged<T> (&w)[NV][E], T coef,
                                      T acc) {
    const uint32_t far = hidden(rt.far);
    T e[NV][E];
#pragma unroll
    for (int j = 0; j < E; j++) {
      const uint32_t off = (far >> j & 1) ? 0u : rt.off[j];
#pragma unroll
      for (int v = 0; v < NV; v++) e[v][j] = near_value(vec[v], off);
    }
#pragma unroll
    for (int j = 0; j < E; j++) {
      T u = e[0][j];
      if constexpr (NV == 2) u = fmac<T>(e[1][j], coef, u);
      acc = fmac<T>((far >> j & 1) ? T(0) : rt.val[j], u, acc);
    }
    if (__any(far != 0)) {
      int tries = 0;
      u64 t0 = 0;
      for (;;) {
        uint32_t bad = 0;
#pragma unroll
        for (int j = 0; j < E; j++) {
          bool ok = true;
#pragma unroll
          for (int v = 0; v < NV; v++) ok = ok && w[v][j].is(tag[v]);
          bad |= ok ? 0u : 1u << j;
        }
        bad &= far;
        if (!__any(bad != 0)) break;
        if ((++tries & 127) == 0 && res_expired(a.outcome, &sh.dead, t0)) break;
#pragma unroll
        for (int j = 0; j < E; j++)
          if (bad >> j & 1) {
#pragma unroll
            for (int v = 0; v < NV; v++) w[v][j].load(word(vec[v], rt.off[j]));
          }
      }
#pragma unroll
      for (int j = 0; j < E; j++) {
        T u = w[0][j].get();
        if constexpr (NV == 2) u = fmac<T>(w[1][j].get(), coef, u);
        acc = fmac<T>((far >> j & 1) ? rt.val[j] : T(0), (far >> j & 1) ? u : T(0), acc);
      }
    }
    return acc;
  }

  // Requests the foreign operands of the product that follows a reduction.
  __device__ __forceinline__ void look_ahead(int m, const int (&vec)[2]) {
    if constexpr (kAhead) request<2, W>(tiles[m], vec, ahead);
  }

  // This thread's entry of M u, u of one or two vectors; a product of two
  // vectors follows look_ahead.
  template <int NV>
  __device__ __forceinline__ T product(int m, const int (&vec)[NV], const uint32_t (&tag)[NV],
                                       T coef) {
    T y;
    if constexpr (NV == 2 && kAhead) {
      y = gather<NV, W>(tiles[m], vec, tag, ahead, coef, T(0));
    } else {
      Tagged<T> w[NV][W];
      request<NV, W>(tiles[m], vec, w);
      y = gather<NV, W>(tiles[m], vec, tag, w, coef, T(0));
    }
    const int nl = sh.n_long[m];
    if (!nl) return y;
    const ResCsr<T> &c = a.m[m];
    for (int i = 0; i < nl; i++) {
      const int row = sh.long_row[m][i];
      const uint32_t b0 = c.rowptr[row], e0 = c.rowptr[row + 1];
      T acc = T(0);
      for (uint32_t k = b0 + t; k < e0; k += 4 * T0) {
        RowTile<T, 4> rt;
        rt.far = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const uint32_t kk = k + u * T0;
          const bool in = kk < e0;
          const uint32_t cc = in ? c.col[kk] : (uint32_t)base;
          rt.val[u] = in ? c.val[kk] : T(0);
          if (PK == PK_JACOBI && a.inv) rt.val[u] *= a.inv[cc];
          bool far;
          rt.off[u] = place(cc, far);
          if (far) rt.far |= 1u << u;
        }
        Tagged<T> w[NV][4];
        request<NV, 4>(rt, vec, w);
        acc = gather<NV, 4>(rt, vec, tag, w, coef, acc);
      }
      const double s = wave_sum((double)acc);
      if (lane == 0) sh.part[i][wave] = s;
    }
    __syncthreads();
    if (long_at[m] >= 0) {
      double s = 0.0;
      for (int w = 0; w < waves; w++) s += sh.part[long_at[m]][w];
      y = (T)s;
    }
    __syncthreads();
    return y;
  }

  static __device__ __forceinline__ double dot(T x, T y) {
    Acc<T> a;
    a.add_prod(x, y);
    return a.get();
  }

  static __device__ __forceinline__ double lane_value(double v, int l) {
    const u64 u = __builtin_bit_cast(u64, v);
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, l);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
    return __builtin_bit_cast(double, ((u64)hi << 32) | lo);
  }

  // First half of a reduction: the workgroup's three sums leave for the other
  // workgroups. Lanes 16k .. 16k+15 return the workgroup's sum k.
  __device__ __forceinline__ double deposit(double (&v)[3]) {
    const int set = round & 1;
    round++;
#pragma unroll
    for (int k = 0; k < 3; k++) v[k] = wave_sum(v[k]);
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < 3; k++) sh.sum[set][k][wave] = v[k];
    }
    __syncthreads();
    double s = 0.0;
    if (G == 1 || wave == 0) {
      const auto add = [](double x, double y) { return x + y; };
      s = lane < 48 ? (&sh.sum[set][0][0])[lane] : 0.0;
      s = dpp_op<0xb1, 0xf>(s, 0.0, add);   // pairs
      s = dpp_op<0x4e, 0xf>(s, 0.0, add);   // quads
      s = dpp_op<0x141, 0xf>(s, 0.0, add);  // eights
      s = dpp_op<0x140, 0xf>(s, 0.0, add);  // sixteens
      if (G > 1 && lane < 48 && (lane & 15) < 2) {
        const u64 b = __builtin_bit_cast(u64, s);
        res_store(a.slots + ((size_t)set * G + g) * kResSlotWords + 2 * (lane >> 4) + (lane & 1),
                  ((u64)round << 32) | ((lane & 1) ? (b >> 32) : (u64)(uint32_t)b));
      }
    }
    return s;
  }

  // Second half: totals over every workgroup, the same bits everywhere; false
  // when the solve was given up.
  __device__ __forceinline__ bool collect(double s, double (&v)[3]) {
    const int set = (round - 1) & 1;
    if (G == 1) {
#pragma unroll
      for (int k = 0; k < 3; k++) v[k] = lane_value(s, 16 * k);
      return true;
    }
    if (wave == 0) {
      const u64 *slot = a.slots + (size_t)set * G * kResSlotWords;
      double tot[3] = {0.0, 0.0, 0.0};
      int tries = 0;
      u64 t0 = 0;
      for (int first = 0; first < G; first += 128) {
        const int i0 = first + lane, i1 = i0 + 64;
        Tagged<double> w[2][3];
        for (;;) {
          const uint32_t at = hidden((uint32_t)i0) * kResSlotWords;
          if (i0 < G) {
#pragma unroll
            for (int k = 0; k < 3; k++) w[0][k].load(slot + at + 2 * k);
          }
          if (i1 < G) {
#pragma unroll
            for (int k = 0; k < 3; k++) w[1][k].load(slot + at + 64 * kResSlotWords + 2 * k);
          }
          bool ok0 = true, ok1 = true;
#pragma unroll
          for (int k = 0; k < 3; k++) {
            ok0 = ok0 && w[0][k].is(round);
            ok1 = ok1 && w[1][k].is(round);
          }
          if (!__any((i0 < G && !ok0) || (i1 < G && !ok1))) break;
          if ((++tries & 127) == 0 && res_expired(a.outcome, &sh.dead, t0)) break;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
          tot[k] += i0 < G ? w[0][k].get() : 0.0;
          tot[k] += i1 < G ? w[1][k].get() : 0.0;
        }
      }
#pragma unroll
      for (int k = 0; k < 3; k++) tot[k] = wave_sum(tot[k]);
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 3; k++) sh.total[set][k] = tot[k];
        sh.given_up[set] = sh.dead;  // one answer for every wave
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; k++) v[k] = sh.total[set][k];
    return sh.given_up[set] == 0;
  }

  __device__ __forceinline__ void solve() {
    if (t == 0) {
      sh.dead = 0;
      sh.run = a.st->status == ST_RUNNING && res_load(a.outcome) == RES_OPEN;
#pragma unroll
      for (int m = 0; m < kMats; m++) sh.n_long[m] = 0;
    }
    for (int i = t; i < 2 * 3 * kWaveCap; i += T0) (&sh.sum[0][0][0])[i] = 0.0;
    __syncthreads();
    if (!sh.run) return;
    const double abs_tol = a.st->abs_tol, hnorm = sqrt(a.st->rhrh);
    const int scaled = a.st->scaled, max_iters = a.st->max_iters;
    // this thread's row: x, r, r_hat, the two halves' u (p, s), hat and
    // product (v, t); zero in threads without one
    T x = T(0), r = T(0), rh = T(0), q = T(0), p = T(0), ph = T(0), v = T(0), u = T(0),
      hat = T(0), out = T(0), inv = T(1);
#pragma unroll
    for (int m = 0; m < kMats; m++) build(m);
    if (mine()) {
      const int row = base + t;
      x = a.x[row];
      r = a.r[row];
      rh = a.rh[row];
      if (PK == PK_JACOBI && a.inv) inv = a.inv[row];
    }
    put(kR, r, 1);
    put(kQ, q, 1);
    double d[3] = {dot(r, r), dot(rh, r), 0.0};
    constexpr int kFirst = PK == PK_ISAI ? 1 : 0;  // the matrix that meets r, q and v
    const int tmpv[1] = {kTmp}, hatv[1] = {kHat};
    int two[2] = {kR, kQ};
    double part = deposit(d);
    look_ahead(kFirst, two);
    if (!collect(part, d)) return;
    double rr = d[0], rhr = d[1], res2 = d[0];
    double rho = 1.0, alpha = 1.0, omega = 1.0;
    int status = ST_RUNNING, iters = 0, s_conv = 0;
    // tags: r and q carry rt; the writes of an iteration's two halves rt + 1
    // and rt + 2, the latter also the next r and q
    uint32_t rt = 1;
    for (;;) {
      const double rnorm = sqrt(rr);
      if (std::isnan(rnorm) || std::isinf(rnorm)) { status = ST_NAN; break; }
      if (rnorm < abs_tol) { status = ST_CONVERGED; break; }
      if (fabs(omega) < 1e-30) { status = ST_BRK_OMEGA; break; }
      if (iters >= max_iters) { status = ST_MAXITER; break; }
      if (scaled ? fabs(rhr) <= 1e-30 * (hnorm * rnorm) : fabs(rhr) < 1e-30) {
        status = ST_BRK_RHO;
        break;
      }
      T coef = (T)((rhr / rho) * (alpha / omega));
      const double rho_new = rhr;
      // half 0: u = p = r + beta q, v = A M^-1 p; half 1: u = s = r - alpha v,
      // t = A M^-1 s
#pragma unroll 1
      for (int half = 0; half < 2; half++) {
        const uint32_t tag2[2] = {rt, half ? rt + 1 : rt}, tag1[1] = {rt + 1 + half};
        u = fmac<T>(half ? v : q, coef, r);
        if constexpr (PK == PK_ISAI) {
          put(kTmp, product<2>(1, two, tag2, coef), tag1[0]);
          __syncthreads();
          hat = product<1>(2, tmpv, tag1, T(0));
          put(kHat, hat, tag1[0]);
          __syncthreads();
          out = product<1>(0, hatv, tag1, T(0));
        } else {
          hat = inv * u;
          out = product<2>(0, two, tag2, coef);
        }
        if (half == 0) put(kV, out, tag1[0]);
        d[0] = half ? dot(u, u) : dot(rh, out);
        d[1] = dot(out, u);
        d[2] = dot(out, out);
        part = deposit(d);
        two[1] = kV;
        if (half == 0) look_ahead(kFirst, two);
        if (!collect(part, d)) return;
        if (half == 0) {
          p = u;
          ph = hat;
          v = out;
          if (scaled ? fabs(d[0]) <= 1e-30 * (hnorm * sqrt(d[2])) : fabs(d[0]) < 1e-30) {
            status = ST_BRK_RV;
            break;
          }
          alpha = rho_new / d[0];
          rho = rho_new;
          coef = -(T)alpha;
        }
      }
      if (status != ST_RUNNING) break;
      const T al = (T)alpha;
      if (sqrt(d[0]) < abs_tol) {  // the ||s|| exit
        x = x + al * ph;
        iters++;
        s_conv = 1;
        res2 = d[0];
        status = ST_CONVERGED;
        break;
      }
      if (scaled ? d[2] <= 1e-30 * d[0] : fabs(d[2]) < 1e-30) {
        status = ST_BRK_TT;
        break;
      }
      omega = d[1] / d[2];
      const T om = (T)omega;
      iters++;
      rt += 2;
      x = (x + al * ph) + om * hat;
      r = u - om * out;
      q = fmac<T>(-om, v, p);
      put(kR, r, rt);
      put(kQ, q, rt);
      d[0] = dot(r, r);
      d[1] = dot(rh, r);
      d[2] = 0.0;
      part = deposit(d);
      two[1] = kQ;
      look_ahead(kFirst, two);
      if (!collect(part, d)) return;
      rr = d[0];
      rhr = d[1];
      res2 = rr;
    }
    // Workgroup 0 decides that the solve stands; nobody writes x before that.
    if (t == 0) {
      u64 o = RES_OPEN;
      if (g == 0) {
        u64 want = RES_OPEN;
        __hip_atomic_compare_exchange_strong(a.outcome, &want, (u64)RES_COMMIT, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        o = want == RES_OPEN ? (u64)RES_COMMIT : want;
      } else {
        u64 t0 = 0;
        int tries = 0;
        while ((o = res_load(a.outcome)) == RES_OPEN)
          if ((++tries & 127) == 0 && res_expired(a.outcome, &sh.dead, t0)) {
            o = RES_ABORT;
            break;
          }
      }
      sh.run = o == RES_COMMIT;
    }
    __syncthreads();
    if (!sh.run) return;
    if (mine()) a.x[base + t] = x;
    if (g == 0 && t == 0) {
      a.st->s_conv = s_conv;
      a.st->iters = iters;
      a.st->res2 = res2;
      a.st->rr = rr;
      a.st->status = status;
    }
  }
};

template <typename T, int PK, int W>
__global__ __launch_bounds__(kResThreads) void k_bicg_resident(ResArgs<T> a) {
  using R = Resident<T, PK, W>;
  __shared__ typename R::Shared sh;
  extern __shared__ __align__(16) unsigned char res_lds[];
  R r(a, sh, res_lds);
  r.solve();
}

// ------------------------------------------------------------ host side --
static std::mutex g_resident_mu;
void resident_lock() { g_resident_mu.lock(); }
void resident_unlock() { g_resident_mu.unlock(); }

// One row per thread: with two or three rows a thread's state leaves the
// registers, and the pipeline, whose launches then carry enough work, is
// faster (ISAI at 160,004 rows: 59 us per iteration against 49, at 262,148 97
// against 62), so the path ends at 512 rows for each compute unit. Tiles of
// 4, 6 or 8 entries; a few longer rows (a supply node's) are summed by their
// whole workgroup, more of them belong to the pipeline's row blocks. Up to 64
// unknowns the one-wave solve needs no workgroup barriers at all.
ResGeo resident_geometry(const ohm_backend *b, const DevCsr &a, const PrecondDev &p, int n) {
  ResGeo g;
  if (n <= 64 || (p.kind == PK_ISAI && p.mm.rowptr)) return g;
  const DevCsr *ms[3] = {&a, &p.ml, &p.mu};
  const int nm = p.kind == PK_ISAI ? 3 : 1;
  static const int kWidths[3] = {4, 6, 8}, kLong[3] = {2, 2, kResMaxLong};
  for (int w = 0; w < 3 && !g.width; w++) {
    bool fits = true;
    for (int m = 0; m < nm; m++)
      fits = fits && ms[m]->long_rows[w] >= 0 && ms[m]->long_rows[w] <= kLong[w];
    if (fits) g.width = kWidths[w];
  }
  if (!g.width) return g;
  const int grid = (n + kResThreads - 1) / kResThreads;
  if (grid > std::min(b->num_cu, kResMaxGrid)) return g;
  g.grid = grid;
  g.rows = (n + grid - 1) / grid;
  g.threads = (g.rows + 63) / 64 * 64;
  return g;
}

ResLayout resident_layout(const ResGeo &g, const PrecondDev &p, int n, bool f32) {
  ResLayout l;
  const size_t vecs = p.kind == PK_ISAI ? 5 : 3;
  l.slots = g.grid > 1 ? vecs * n * (f32 ? 1 : 2) : 0;
  l.outcome = l.slots + (size_t)2 * g.grid * kResSlotWords;
  l.clear_words = l.outcome + 1;
  l.bytes = l.clear_words * 8;
  return l;
}

template <typename T>
ohm_status resident_enqueue(ohm_backend *b, const DevCsr &a, const PrecondDev &p, const ResGeo &g,
                            void *ws, const BicgVecs<T> &v, SolveState *st) {
  constexpr bool f32 = std::is_same<T, float>::value;
  const ResLayout l = resident_layout(g, p, a.n, f32);
  char *base = static_cast<char *>(ws);
  const auto csr = [](const DevCsr &m) {
    ResCsr<T> c{m.rowptr, m.col, nullptr};
    if constexpr (f32)
      c.val = m.val32;
    else
      c.val = m.val;
    return c;
  };
  ResArgs<T> q{};
  q.n = a.n;
  q.rows = g.rows;
  q.m[0] = csr(a);
  if (p.kind == PK_ISAI) {
    q.m[1] = csr(p.ml);
    q.m[2] = csr(p.mu);
  }
  if constexpr (f32)
    q.inv = p.inv32;
  else
    q.inv = p.inv;
  q.x = v.x;
  q.r = v.r;
  q.rh = v.rh;
  q.st = st;
  q.words = reinterpret_cast<u64 *>(base);
  q.slots = q.words + l.slots;
  q.outcome = q.words + l.outcome;
  const unsigned lds = (unsigned)((p.kind == PK_ISAI ? 5 : 3) * (size_t)g.rows * sizeof(T));
  const auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(g.grid), dim3(g.threads), lds, b->stream, q);
  };
  const auto by_width = [&](auto pk) {
    constexpr int PK = decltype(pk)::value;
    if (g.width == 4)
      launch(k_bicg_resident<T, PK, 4>);
    else if (g.width == 6)
      launch(k_bicg_resident<T, PK, 6>);
    else
      launch(k_bicg_resident<T, PK, 8>);
  };
  if (p.kind == PK_ISAI)
    by_width(std::integral_constant<int, PK_ISAI>());
  else  // without a preconditioner inv is null
    by_width(std::integral_constant<int, PK_JACOBI>());
  OHM_HIP(hipGetLastError());
  b->dispatches++;
  return OHM_OK;
}

template ohm_status resident_enqueue<double>(ohm_backend *, const DevCsr &, const PrecondDev &,
                                             const ResGeo &, void *, const BicgVecs<double> &,
                                             SolveState *);
template ohm_status resident_enqueue<float>(ohm_backend *, const DevCsr &, const PrecondDev &,
                                            const ResGeo &, void *, const BicgVecs<float> &,
                                            SolveState *);

}  // namespace ohm
