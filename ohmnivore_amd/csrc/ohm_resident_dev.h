// ohm_resident_dev.h — the resident BiCGSTAB solve of one system by its
// workgroups, as device code (ohm_persist.hip: one system;
// ohm_batch_resident.hip: many, real or complex). ohm_persist.hip describes it.
#pragma once

#include <type_traits>

#include "ohm_batch_types.h"
#include "ohm_persist.h"
#include "ohm_spmv.h"

namespace ohm {

typedef unsigned long long u64;

constexpr u64 kResLimit = 20'000'000;  // 0.2 s of the 100 MHz wall clock
// How a solve ended: it stands, a wait outlasted the limit, or it broke down.
enum : u64 { RES_OPEN = 0, RES_COMMIT = 1, RES_ABORT = 2, RES_BROKE = 3 };

// A matrix G + sigma C (c null: G alone).
template <typename S>
struct ResCsr {
  using R = typename Tr<S>::R;
  const uint32_t *rowptr, *col;
  const R *g, *c;
  double sig_re, sig_im;
  __device__ __forceinline__ S at(uint32_t k) const {
    return aval<S>(g[k], c ? c[k] : (R)0, sig_re, sig_im);
  }
};

// One solve; St is its state word (abs_tol, rhrh, status, iters, ...).
template <typename S, typename St>
struct ResArgs {
  int n, rows;               // unknowns, rows per workgroup
  int first, grid;           // its first workgroup in the launch, and how many
  int halo;                  // ISAI: 1: foreign operands are fetched into LDS; 2: and the
                             // foreign results of the factors formed here
  ResCsr<S> m[3];            // A, M_L, M_U
  const S *inv;              // Jacobi inverse diagonal (null: none)
  S *x;
  const S *r, *rh;           // the solve's start
  St *st;
  u64 *words;                // tagged vectors: r, q, v, tmp, hat
  u64 *slots, *outcome;
  int absent;                // the last workgroup stays away (resident_absent)
};

// Scalar algebra: 64-bit, complex where the vectors are.
template <typename S>
using ResAlg = typename std::conditional<Tr<S>::C, zd, double>::type;
__device__ __forceinline__ double alg_mul(double a, double b) { return a * b; }
__device__ __forceinline__ double alg_div(double a, double b) { return a / b; }
__device__ __forceinline__ double alg_abs(double a) { return fabs(a); }
__device__ __forceinline__ double alg_re(double a) { return a; }
__device__ __forceinline__ double alg_im(double) { return 0.0; }
__device__ __forceinline__ zd alg_mul(zd a, zd b) { return zmul(a, b); }
__device__ __forceinline__ zd alg_div(zd a, zd b) { return zdiv(a, b); }
__device__ __forceinline__ double alg_abs(zd a) { return sqrt(zabs2(a)); }
__device__ __forceinline__ double alg_re(zd a) { return a.re; }
__device__ __forceinline__ double alg_im(zd a) { return a.im; }
template <typename A>
__device__ __forceinline__ A alg_make(double re, double im) {
  if constexpr (std::is_same<A, double>::value)
    return re;
  else
    return zd{re, im};
}
template <typename A, typename S>
__device__ __forceinline__ S alg_to(A a) {
  return mk<S>(alg_re(a), alg_im(a));
}
// a b + c
template <typename S>
__device__ __forceinline__ S res_fma(S a, S b, S c) {
  if constexpr (Tr<S>::C) {
    return S{fma(a.re, b.re, fma(-a.im, b.im, c.re)), fma(a.re, b.im, fma(a.im, b.re, c.im))};
  } else {
    return fmac<S>(a, b, c);
  }
}

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

template <>
struct Tagged<cx<double>> {
  static constexpr int kWords = 4;
  Tagged<double> re, im;
  __device__ __forceinline__ void load(const u64 *p) {
    re.load(p);
    im.load(p + 2);
  }
  __device__ __forceinline__ bool is(uint32_t tag) const { return re.is(tag) && im.is(tag); }
  __device__ __forceinline__ cx<double> get() const { return {re.get(), im.get()}; }
  static __device__ __forceinline__ void put(u64 *p, cx<double> v, uint32_t tag) {
    Tagged<double>::put(p, v.re, tag);
    Tagged<double>::put(p + 2, v.im, tag);
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
  if (o >= RES_ABORT) {
    *dead = 1;
    return true;
  }
  return false;
}

// A thread's row of one matrix as W entries: `off` is the operand's byte
// offset, into the workgroup's LDS vector or, where its bit of `far` is set,
// into the tagged vector. With X set, entry W is the thread's share of a row
// too long for a tile, summed apart.
template <typename T, int W, int X>
struct RowTile {
  T val[W + X];
  uint32_t off[W + X], far;
};

// Row tiles of W entries for A and WF for the factors. kEarly: registers are
// left to request a product's foreign operands before the reduction that
// precedes it is complete.
template <typename T, typename St, int PK, int W, int WF, bool kEarly>
struct Resident {
  using A = ResAlg<T>;
  static constexpr bool kC = Tr<T>::C;
  static constexpr int kN = kC ? 2 : 1;   // words of a dot product
  static constexpr int kSums = kN + 2;    // sums of one reduction
  static constexpr int kMats = PK == PK_ISAI ? 3 : 1;
  static constexpr int kX = PK == PK_ISAI ? 1 : 0;  // long rows' shares in the tiles
  static constexpr int kR = 0, kQ = 1, kV = 2, kTmp = 3, kHat = 4;  // vector numbers
  static constexpr int kWaveCap = 16;
  static constexpr uint32_t kWordBytes = 8 * Tagged<T>::kWords;
  static constexpr int kNoLoads = 0x0f70;  // s_waitcnt: vmcnt 0, the other counters any

  struct Shared {
    double sum[2][kSums][kWaveCap];
    double total[2][kSums];
    double part[kResMaxLong][kN][kWaveCap];
    int long_row[kMats][kResMaxLong];
    int n_long[kMats], kept[kMats];  // kept: the first of them is in the tiles
    int dead, run, given_up[2];
    int n_slots, n_tmp, n_hat, halo_over;
  };
  static constexpr uint32_t kEmpty = ~0u;

  const ResArgs<T, St> &a;
  Shared &sh;
  char *lv;  // LDS vectors, `rows` entries each
  int T0, t, lane, wave, waves, g, G, base, cnt, stride;
  uint32_t round;   // reductions so far
  int8_t long_at[kMats];
  RowTile<T, W, kX> tile_a;
  RowTile<T, WF, kX> tile_f[2];  // M_L, M_U
  Tagged<T> ahead[2][W];  // Jacobi: words of the foreign operands, requested early

  __device__ __forceinline__ Resident(const ResArgs<T, St> &a_, Shared &s_, unsigned char *lv_)
      : a(a_), sh(s_), lv(reinterpret_cast<char *>(lv_)) {
    T0 = blockDim.x;
    t = threadIdx.x;
    lane = t & 63;
    wave = t >> 6;
    waves = T0 >> 6;
    g = blockIdx.x - a.first;
    G = a.grid;
    base = g * a.rows;
    cnt = min(a.rows, a.n - base);
    stride = a.rows + (PK == PK_ISAI ? kResHalo : 0);
    if (PK == PK_ISAI) lv += sizeof(uint32_t) * kResHalo;
    round = 0;
  }
  __device__ __forceinline__ T near_value(int v, uint32_t off) const {
    return *reinterpret_cast<const T *>(lv + (uint32_t)(v * stride) * (uint32_t)sizeof(T) + off);
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

  // publish this thread's entry of vector v (a halo thread's stays here)
  __device__ __forceinline__ void put(int v, T x, uint32_t tag) {
    const int halo = v == kTmp ? sh.n_tmp : v == kHat ? sh.n_hat : 0;
    if (PK == PK_ISAI ? t >= cnt + halo : !mine()) return;
    reinterpret_cast<T *>(lv)[v * stride + t] = x;
    if (mine() && G > 1) Tagged<T>::put(word(v, (uint32_t)(base + t) * kWordBytes), x, tag);
  }

  __device__ __forceinline__ uint32_t place(uint32_t col, bool &far) const {
    const uint32_t off = col - (uint32_t)base;
    far = off >= (uint32_t)cnt;
    return far ? col * kWordBytes : off * (uint32_t)sizeof(T);
  }

  // The halo (ISAI): foreign columns this workgroup reads have a slot in its
  // LDS vectors, behind its own rows. r, q and v are fetched into every slot
  // while a reduction is under way, once for all rows that read them. With
  // a.halo 2 the threads past the own rows also form the foreign entries of
  // the first factor's result (slots below n_tmp) and of hat (below n_hat),
  // thread cnt + s slot s, so that neither is waited for.
  //
  // While the tiles are built the vectors' place holds a hash table of the
  // columns: keys, then slots. Their list stays, in front of the vectors.
  static constexpr int kHash = 2 * kResThreads * 2;
  __device__ __forceinline__ uint32_t *keys() const { return reinterpret_cast<uint32_t *>(lv); }
  __device__ __forceinline__ uint32_t *slot_of() const { return keys() + kHash; }
  __device__ __forceinline__ uint32_t *halo_cols() const { return keys() - kResHalo; }
  static __device__ __forceinline__ uint32_t bucket(uint32_t col) {
    return (col * 2654435761u) >> (32 - __builtin_ctz((uint32_t)kHash));
  }
  __device__ __forceinline__ bool fits_tile(int m, uint32_t row) const {
    return a.m[m].rowptr[row + 1] - a.m[m].rowptr[row] <= (uint32_t)(m == 0 ? W : WF);
  }
  // The foreign columns of row `row` of matrix m join the halo. A result whose
  // own row of a factor is not a tile stays an exchange. Once the halo is too
  // large nothing more joins: it will be dropped, and a full table takes a
  // probe of every bucket per column.
  __device__ __forceinline__ void join(int m, uint32_t row) {
    if (!fits_tile(m, row)) return;
    const ResCsr<T> &c = a.m[m];
    const volatile int *over = &sh.halo_over;
    for (uint32_t k = c.rowptr[row]; k < c.rowptr[row + 1] && !*over; k++) {
      const uint32_t col = c.col[k];
      if (col - (uint32_t)base < (uint32_t)cnt || (m != 1 && !fits_tile(1, col)) ||
          (m == 0 && !fits_tile(2, col)))
        continue;
      uint32_t h = bucket(col);
      for (int tries = 0;; tries++, h = (h + 1) & (kHash - 1)) {
        if (tries == kHash) {
          sh.halo_over = 1;
          break;
        }
        const uint32_t old = atomicCAS(&keys()[h], (unsigned)kEmpty, col);
        if (old == col) break;
        if (old != kEmpty) continue;
        const int s = atomicAdd(&sh.n_slots, 1);
        if (s < kResHalo) {
          slot_of()[h] = s;
          halo_cols()[s] = col;
        } else {
          sh.halo_over = 1;
        }
        break;
      }
    }
  }
  __device__ __forceinline__ void clear_halo() {
    for (int i = t; i < kHash; i += T0) keys()[i] = kEmpty;
    if (t == 0) sh.n_slots = sh.n_tmp = sh.n_hat = sh.halo_over = 0;
    __syncthreads();
  }
  __device__ __forceinline__ void find_halo() {
    clear_halo();
    const int i = t - cnt;
    if (a.halo > 1) {
      if (mine()) join(0, base + t);
      __syncthreads();
      const int n_hat = sh.n_slots;
      __syncthreads();
      if (n_hat <= T0 - cnt) {
        if (mine())
          join(2, base + t);
        else if (i < n_hat)
          join(2, halo_cols()[i]);
      }
      __syncthreads();
      const int n_tmp = sh.n_slots;
      __syncthreads();
      if (n_tmp > T0 - cnt) {
        clear_halo();  // no thread for each: the results are exchanged
      } else if (t == 0) {
        sh.n_hat = n_hat;
        sh.n_tmp = n_tmp;
      }
      __syncthreads();
    }
    if (mine())
      join(1, base + t);
    else if (i < sh.n_tmp)
      join(1, halo_cols()[i]);
    __syncthreads();
    // clear_halo resets the flag: every thread reads it before any goes on
    const int over = sh.halo_over;
    __syncthreads();
    if (over) clear_halo();  // too many: each row reads its own
  }
  // the operand of an entry of matrix m's tile
  __device__ __forceinline__ uint32_t place_halo(int m, uint32_t col, bool &far) const {
    const uint32_t off = place(col, far);
    if (PK != PK_ISAI || !far) return off;
    uint32_t h = bucket(col);
    for (int tries = 0; tries < kHash; tries++, h = (h + 1) & (kHash - 1)) {
      const uint32_t k = keys()[h];
      if (k == kEmpty) break;
      if (k != col) continue;
      const int s = (int)slot_of()[h];
      if (s >= (m == 0 ? sh.n_hat : m == 2 ? sh.n_tmp : sh.n_slots)) break;
      far = false;
      return (uint32_t)(cnt + s) * (uint32_t)sizeof(T);
    }
    return off;
  }
  // The slots' entries of NV vectors, all with the tag `tag`; by the waves
  // that have nothing to do in the reduction under way.
  template <int NV>
  __device__ __forceinline__ void fetch(const int (&vec)[NV], uint32_t tag) {
    const int skip = waves > 1 ? 64 : 0, n = sh.n_slots;
    for (int s = t - skip; s < n; s += T0 - skip) {
      if (s < 0) break;
      const uint32_t at = halo_cols()[s] * kWordBytes;
      Tagged<T> w[NV];
      int tries = 0;
      u64 t0 = 0;
      for (;;) {
        bool ok = true;
#pragma unroll
        for (int v = 0; v < NV; v++) w[v].load(word(vec[v], at));
#pragma unroll
        for (int v = 0; v < NV; v++) ok = ok && w[v].is(tag);
        if (ok || ((++tries & 127) == 0 && res_expired(a.outcome, &sh.dead, t0))) break;
      }
#pragma unroll
      for (int v = 0; v < NV; v++)
        reinterpret_cast<T *>(lv)[vec[v] * stride + cnt + s] = w[v].get();
    }
  }

  // This thread's row of matrix m as a tile padded with zeros. A longer row
  // stays in CSR and is summed by the whole workgroup.
  template <int E>
  __device__ __forceinline__ void build(int m, RowTile<T, E, kX> &rt) {
    const ResCsr<T> &c = a.m[m];
    int row = base + (mine() ? t : 0);
    bool has = mine();
    if (PK == PK_ISAI && !has && m > 0 && t - cnt < (m == 1 ? sh.n_tmp : sh.n_hat)) {
      row = (int)halo_cols()[t - cnt];
      has = true;
    }
    const uint32_t b0 = c.rowptr[row], len = c.rowptr[row + 1] - b0;
    const bool lg = len > (uint32_t)E;
    long_at[m] = -1;
    if (lg && mine()) {
      const int at = atomicAdd(&sh.n_long[m], 1);
      sh.long_row[m][at] = row;
      long_at[m] = (int8_t)at;
    }
    rt.far = 0;
#pragma unroll
    for (int j = 0; j < E; j++) {  // padding: zero times an entry of one's own
      T val = zero<T>();
      uint32_t off = (uint32_t)(mine() ? t : 0) * (uint32_t)sizeof(T);
      bool far = false;
      if (has && !lg && (uint32_t)j < len) {
        const uint32_t col = c.col[b0 + j];
        val = c.at(b0 + j);
        if (PK == PK_JACOBI && a.inv) val = val * a.inv[col];
        off = place_halo(m, col, far);
      }
      rt.off[j] = off;
      rt.val[j] = val;
      if (far) rt.far |= 1u << j;
    }
    if constexpr (kX) {
      rt.off[E] = rt.off[0];
      rt.val[E] = zero<T>();
    }
  }
  // The first row of matrix m too long for a tile, an entry to each thread: a
  // supply node's, read from memory in every product, was a chain of three
  // loads and a second exchange that the whole solve waited for.
  template <int E>
  __device__ __forceinline__ void keep_long(int m, RowTile<T, E, kX> &rt) {
    if (!sh.n_long[m]) return;
    const ResCsr<T> &c = a.m[m];
    const int row = sh.long_row[m][0];
    const uint32_t k = c.rowptr[row] + t, e0 = c.rowptr[row + 1];
    if (e0 - c.rowptr[row] > (uint32_t)T0) return;
    if (t == 0) sh.kept[m] = 1;
    if (k >= e0) return;
    const uint32_t col = c.col[k];
    bool far;
    rt.off[E] = place_halo(m, col, far);
    rt.val[E] = c.at(k);
    if (PK == PK_JACOBI && a.inv) rt.val[E] = rt.val[E] * a.inv[col];
    if (far) rt.far |= 1u << E;
  }

  // Requests the foreign operands of one row (entries no lane of the wave
  // needs are skipped as one).
  template <int NV, int E>
  __device__ __forceinline__ void request(const RowTile<T, E, kX> &rt, const int (&vec)[NV],
                                          Tagged<T> (&w)[NV][E + kX]) const {
    const uint32_t far = hidden(rt.far);
    if (!__any(far != 0)) return;
#pragma unroll
    for (int j = 0; j < E + kX; j++)
      if (far >> j & 1) {
#pragma unroll
        for (int v = 0; v < NV; v++) w[v][j].load(word(vec[v], rt.off[j]));
      }
  }

  // Spins until every foreign word of a row carries its tag. With asked set
  // the words have been requested once.
  template <int NV, int E>
  __device__ __forceinline__ void settle(const RowTile<T, E, kX> &rt, const int (&vec)[NV],
                                         const uint32_t (&tag)[NV], Tagged<T> (&w)[NV][E + kX],
                                         bool asked) {
    const uint32_t far = hidden(rt.far);
    const auto missing = [&]() {
      uint32_t bad = 0;
#pragma unroll
      for (int j = 0; j < E + kX; j++) {
        bool ok = true;
#pragma unroll
        for (int v = 0; v < NV; v++) ok = ok && w[v][j].is(tag[v]);
        bad |= ok ? 0u : 1u << j;
      }
      return bad & far;
    };
    int tries = 0;
    u64 t0 = 0;
    for (uint32_t bad = asked ? missing() : far; __any(bad != 0); bad = missing()) {
      if ((++tries & 127) == 0 && res_expired(a.outcome, &sh.dead, t0)) break;
#pragma unroll
      for (int j = 0; j < E + kX; j++)
        if (bad >> j & 1) {
#pragma unroll
          for (int v = 0; v < NV; v++) w[v][j].load(word(vec[v], rt.off[j]));
        }
    }
  }

  // The near half of a product: acc += val . u over this workgroup's own
  // entries (u = e0, or e0 + coef e1 with two vectors), from LDS. Entries of
  // the other kind take part with a zero, so that every load is issued before
  // the first is used.
  template <int NV, int E>
  __device__ __forceinline__ T near_part(const RowTile<T, E, kX> &rt, const int (&vec)[NV],
                                         uint32_t far, T coef, T acc, T &share) const {
    T e[NV][E + kX];
#pragma unroll
    for (int j = 0; j < E + kX; j++) {
      const uint32_t off = (far >> j & 1) ? 0u : rt.off[j];
#pragma unroll
      for (int v = 0; v < NV; v++) e[v][j] = near_value(vec[v], off);
    }
#pragma unroll
    for (int j = 0; j < E + kX; j++) {
      T u = e[0][j];
      if constexpr (NV == 2) u = res_fma<T>(e[1][j], coef, u);
      T &sum = j < E ? acc : share;
      sum = res_fma<T>((far >> j & 1) ? zero<T>() : rt.val[j], u, sum);
    }
    return acc;
  }

  // acc += val . u over a row's E entries, share += the last one's: this workgroup's own from LDS, then
  // the foreign ones in order, spinning until their words carry the tag. With
  // early set their words `w` have been requested.
  //
  // No path leaves here with a request open: the compiler would have every
  // wave wait for it at its next use of the registers, and as the memory
  // counter is in order, for its own stores of the vector it has just
  // published, about 1 us a product.
  template <int NV, int E>
  __device__ __forceinline__ T gather(const RowTile<T, E, kX> &rt, const int (&vec)[NV],
                                      const uint32_t (&tag)[NV], Tagged<T> (&w)[NV][E + kX],
                                      bool early, T coef, T acc, T &share) {
    const uint32_t far = hidden(rt.far);
    acc = near_part<NV, E>(rt, vec, far, coef, acc, share);
    if (!__any(far != 0)) {
      if (early) __builtin_amdgcn_s_waitcnt(kNoLoads);
      return acc;
    }
    settle<NV, E>(rt, vec, tag, w, early);
#pragma unroll
    for (int j = 0; j < E + kX; j++) {
      T u = w[0][j].get();
      if constexpr (NV == 2) u = res_fma<T>(w[1][j].get(), coef, u);
      T &sum = j < E ? acc : share;
      sum = res_fma<T>((far >> j & 1) ? rt.val[j] : zero<T>(), (far >> j & 1) ? u : zero<T>(), sum);
    }
    return acc;
  }

  template <int M>
  __device__ __forceinline__ auto &tile() {
    if constexpr (M == 0)
      return tile_a;
    else
      return tile_f[M - 1];
  }

  // Requests the foreign operands of the product that follows a reduction.
  // They have been sent before the sums of the reduction, so the waves that
  // have nothing to do in it wait for them here.
  __device__ __forceinline__ void look_ahead(const int (&vec)[2], uint32_t t0, uint32_t t1) {
    if constexpr (PK == PK_ISAI) {
      const int v1[1] = {kV};
      if (G == 1) return;
      if (t0 == t1)
        fetch<2>(vec, t0);
      else  // r is there
        fetch<1>(v1, t1);
    } else if constexpr (kEarly) {
      request<2, W>(tile_a, vec, ahead);
      const uint32_t tag[2] = {t0, t1};
      if (wave != 0) settle<2, W>(tile_a, vec, tag, ahead, true);
    }
  }

  // This thread's share of a long row that is not in the tiles.
  template <int NV>
  __device__ __forceinline__ T long_share(const ResCsr<T> &c, int row, const int (&vec)[NV],
                                          const uint32_t (&tag)[NV], T coef) {
    const uint32_t b0 = c.rowptr[row], e0 = c.rowptr[row + 1];
    T acc = zero<T>(), none = acc;
    for (uint32_t k = b0 + t; k < e0; k += 4 * T0) {
      RowTile<T, 4, kX> rt;
      rt.far = 0;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const uint32_t kk = k + u * T0;
        const bool in = kk < e0;
        const uint32_t cc = in ? c.col[kk] : (uint32_t)base;
        rt.val[u] = in ? c.at(kk) : zero<T>();
        if (PK == PK_JACOBI && a.inv) rt.val[u] = rt.val[u] * a.inv[cc];
        bool far;
        rt.off[u] = place(cc, far);
        if (far) rt.far |= 1u << u;
      }
      if constexpr (kX) {
        rt.val[4] = zero<T>();
        rt.off[4] = 0;
      }
      Tagged<T> w[NV][4 + kX];
      acc = gather<NV, 4>(rt, vec, tag, w, false, coef, acc, none);
    }
    return acc;
  }

  // This thread's entry of M u, u of one or two vectors; a product of two
  // vectors follows look_ahead.
  template <int m, int NV>
  __device__ __forceinline__ T product(const int (&vec)[NV], const uint32_t (&tag)[NV], T coef) {
    constexpr int E = m == 0 ? W : WF;
    T y, share = zero<T>();
    if constexpr (NV == 2 && kEarly && PK != PK_ISAI) {
      y = gather<NV, E>(tile<m>(), vec, tag, ahead, true, coef, zero<T>(), share);
    } else {
      Tagged<T> w[NV][E + kX];
      y = gather<NV, E>(tile<m>(), vec, tag, w, false, coef, zero<T>(), share);
    }
    const int nl = sh.n_long[m];
    if (!nl) return y;
    for (int i = 0; i < nl; i++) {
      T acc = share;
      if (i > 0 || !sh.kept[m]) acc = long_share<NV>(a.m[m], sh.long_row[m][i], vec, tag, coef);
      const double re = wave_sum(re_of(acc)), im = kC ? wave_sum(im_of(acc)) : 0.0;
      if (lane == 0) {
        sh.part[i][0][wave] = re;
        if (kC) sh.part[i][kN - 1][wave] = im;
      }
    }
    __syncthreads();
    if (long_at[m] >= 0) {
      double s[2] = {0.0, 0.0};
      for (int w = 0; w < waves; w++)
        for (int c = 0; c < kN; c++) s[c] += sh.part[long_at[m]][c][w];
      y = mk<T>(s[0], s[1]);
    }
    __syncthreads();
    __builtin_amdgcn_s_waitcnt(kNoLoads);
    return y;
  }

  // conj(x) y at d[0 .. kN), and |x|^2
  static __device__ __forceinline__ void dot(T x, T y, double *d) {
    DotAcc<T> a;
    a.add(x, y);
    d[0] = a.re.get();
    if constexpr (kC) d[1] = a.im.get();
  }
  static __device__ __forceinline__ double norm2(T x) {
    NrmAcc<T> a;
    a.add(x);
    return a.s.get();
  }
  static __device__ __forceinline__ A value(const double *d) {
    return alg_make<A>(d[0], kC ? d[kN - 1] : 0.0);
  }

  static __device__ __forceinline__ double lane_value(double v, int l) {
    const u64 u = __builtin_bit_cast(u64, v);
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, l);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
    return __builtin_bit_cast(double, ((u64)hi << 32) | lo);
  }

  // First half of a reduction: the workgroup's sums leave for the other
  // workgroups. Lanes 16k .. 16k+15 return the workgroup's sum k.
  __device__ __forceinline__ double deposit(double (&v)[kSums]) {
    const int set = round & 1;
    round++;
#pragma unroll
    for (int k = 0; k < kSums; k++) v[k] = wave_sum(v[k]);
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < kSums; k++) sh.sum[set][k][wave] = v[k];
    }
    __syncthreads();
    double s = 0.0;
    if (G == 1 || wave == 0) {
      const auto add = [](double x, double y) { return x + y; };
      s = lane < 16 * kSums ? (&sh.sum[set][0][0])[lane] : 0.0;
      s = dpp_op<0xb1, 0xf>(s, 0.0, add);   // pairs
      s = dpp_op<0x4e, 0xf>(s, 0.0, add);   // quads
      s = dpp_op<0x141, 0xf>(s, 0.0, add);  // eights
      s = dpp_op<0x140, 0xf>(s, 0.0, add);  // sixteens
      if (G > 1 && lane < 16 * kSums && (lane & 15) < 2) {
        const u64 b = __builtin_bit_cast(u64, s);
        res_store(a.slots + ((size_t)set * G + g) * kResSlotWords + 2 * (lane >> 4) + (lane & 1),
                  ((u64)round << 32) | ((lane & 1) ? (b >> 32) : (u64)(uint32_t)b));
      }
    }
    return s;
  }

  // Second half: totals over every workgroup, the same bits everywhere; false
  // when the solve was given up.
  __device__ __forceinline__ bool collect(double s, double (&v)[kSums]) {
    const int set = (round - 1) & 1;
    if (G == 1) {
#pragma unroll
      for (int k = 0; k < kSums; k++) v[k] = lane_value(s, 16 * k);
      return true;
    }
    if (wave == 0) {
      const u64 *slot = a.slots + (size_t)set * G * kResSlotWords;
      double tot[kSums];
#pragma unroll
      for (int k = 0; k < kSums; k++) tot[k] = 0.0;
      int tries = 0;
      u64 t0 = 0;
      for (int first = 0; first < G; first += 128) {
        const int i0 = first + lane, i1 = i0 + 64;
        Tagged<double> w[2][kSums];
        for (;;) {
          const uint32_t at = hidden((uint32_t)i0) * kResSlotWords;
          if (i0 < G) {
#pragma unroll
            for (int k = 0; k < kSums; k++) w[0][k].load(slot + at + 2 * k);
          }
          if (i1 < G) {
#pragma unroll
            for (int k = 0; k < kSums; k++) w[1][k].load(slot + at + 64 * kResSlotWords + 2 * k);
          }
          bool ok0 = true, ok1 = true;
#pragma unroll
          for (int k = 0; k < kSums; k++) {
            ok0 = ok0 && w[0][k].is(round);
            ok1 = ok1 && w[1][k].is(round);
          }
          if (!__any((i0 < G && !ok0) || (i1 < G && !ok1))) break;
          if ((++tries & 127) == 0 && res_expired(a.outcome, &sh.dead, t0)) break;
        }
#pragma unroll
        for (int k = 0; k < kSums; k++) {
          tot[k] += i0 < G ? w[0][k].get() : 0.0;
          tot[k] += i1 < G ? w[1][k].get() : 0.0;
        }
      }
#pragma unroll
      for (int k = 0; k < kSums; k++) tot[k] = wave_sum(tot[k]);
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < kSums; k++) sh.total[set][k] = tot[k];
        sh.given_up[set] = sh.dead;  // one answer for every wave
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSums; k++) v[k] = sh.total[set][k];
    return sh.given_up[set] == 0;
  }

  __device__ __forceinline__ void solve() {
    if (t == 0) {
      sh.dead = 0;
      sh.run = a.st->status == ST_RUNNING && res_load(a.outcome) == RES_OPEN &&
               !(a.absent && G > 1 && g == G - 1);
#pragma unroll
      for (int m = 0; m < kMats; m++) sh.n_long[m] = sh.kept[m] = 0;
    }
    for (int i = t; i < 2 * kSums * kWaveCap; i += T0) (&sh.sum[0][0][0])[i] = 0.0;
    __syncthreads();
    if (!sh.run) return;
    const double abs_tol = a.st->abs_tol, hnorm = sqrt(a.st->rhrh);
    const int scaled = a.st->scaled, max_iters = a.st->max_iters;
    constexpr double kTiny = kC ? 1e-15 : 1e-30;  // unscaled breakdown threshold
    // this thread's row: x, r, r_hat, the two halves' u (p, s), hat and
    // product (v, t); zero in threads without one
    T x = zero<T>(), r = x, rh = x, q = x, p = x, ph = x, v = x, u = x, hat = x, out = x,
      inv = mk<T>(1.0, 0.0);
    if constexpr (PK == PK_ISAI) find_halo();
    build<W>(0, tile_a);
    if constexpr (PK == PK_ISAI) {
      build<WF>(1, tile_f[0]);
      build<WF>(2, tile_f[1]);
    }
    if constexpr (kX) {
      __syncthreads();
      keep_long<W>(0, tile_a);
      keep_long<WF>(1, tile_f[0]);
      keep_long<WF>(2, tile_f[1]);
      __syncthreads();  // the table's place is the vectors' now
    }
    if (mine()) {
      const int row = base + t;
      x = a.x[row];
      r = a.r[row];
      rh = a.rh[row];
      if (PK == PK_JACOBI && a.inv) inv = a.inv[row];
    }
    put(kR, r, 1);
    put(kQ, q, 1);
    double d[kSums];
    dot(rh, r, d);
    d[kN] = norm2(r);
    d[kN + 1] = 0.0;
    const int tmpv[1] = {kTmp}, hatv[1] = {kHat};
    int two[2] = {kR, kQ};
    double part = deposit(d);
    look_ahead(two, 1, 1);
    if (!collect(part, d)) return;
    A rhr = value(d), rho = alg_make<A>(1.0, 0.0), alpha = rho, omega = rho;
    double rr = d[kN], res2 = rr;
    int status = ST_RUNNING, iters = 0, s_conv = 0;
    // tags: r and q carry rt; the writes of an iteration's two halves rt + 1
    // and rt + 2, the latter also the next r and q
    uint32_t rt = 1;
    for (;;) {
      const double rnorm = sqrt(rr), rabs = alg_abs(rhr);
      if (std::isnan(rnorm) || std::isinf(rnorm)) { status = ST_NAN; break; }
      if (rnorm < abs_tol) { status = ST_CONVERGED; break; }
      if (kC ? alg_re(omega) * alg_re(omega) + alg_im(omega) * alg_im(omega) < 1e-30
             : fabs(alg_re(omega)) < 1e-30) {
        status = ST_BRK_OMEGA;
        break;
      }
      if (iters >= max_iters) { status = ST_MAXITER; break; }
      if (scaled ? rabs <= 1e-30 * (hnorm * rnorm) : rabs < kTiny) {
        status = ST_BRK_RHO;
        break;
      }
      T coef = alg_to<A, T>(alg_mul(alg_div(rhr, rho), alg_div(alpha, omega)));
      const A rho_new = rhr;
      // half 0: u = p = r + beta q, v = A M^-1 p; half 1: u = s = r - alpha v,
      // t = A M^-1 s
#pragma unroll 1
      for (int half = 0; half < 2; half++) {
        const uint32_t tag2[2] = {rt, half ? rt + 1 : rt}, tag1[1] = {rt + 1 + half};
        // everything older than the reduction is done: said here, where it costs
        // nothing, so that no later use of a register waits for it
        __builtin_amdgcn_s_waitcnt(kNoLoads);
        u = res_fma<T>(half ? v : q, coef, r);
        if constexpr (PK == PK_ISAI) {
          put(kTmp, product<1, 2>(two, tag2, coef), tag1[0]);
          __syncthreads();
          hat = product<2, 1>(tmpv, tag1, coef);
          put(kHat, hat, tag1[0]);
          __syncthreads();
          out = product<0, 1>(hatv, tag1, coef);
        } else {
          hat = inv * u;
          out = product<0, 2>(two, tag2, coef);
        }
        if (half == 0) put(kV, out, tag1[0]);
        dot(half ? out : rh, half ? u : out, d);
        d[kN] = norm2(out);
        d[kN + 1] = norm2(u);
        part = deposit(d);
        two[1] = kV;
        if (half == 0) look_ahead(two, rt, rt + 1);
        if (!collect(part, d)) return;
        if (half == 0) {
          p = u;
          ph = hat;
          v = out;
          const double rvabs = alg_abs(value(d));
          if (scaled ? rvabs <= 1e-30 * (hnorm * sqrt(d[kN])) : rvabs < kTiny) {
            status = ST_BRK_RV;
            break;
          }
          alpha = alg_div(rho_new, value(d));
          rho = rho_new;
          coef = alg_to<A, T>(alg_make<A>(-alg_re(alpha), -alg_im(alpha)));
        }
      }
      if (status != ST_RUNNING) break;
      const T al = alg_to<A, T>(alpha);
      if (sqrt(d[kN + 1]) < abs_tol) {  // the ||s|| exit
        x = x + al * ph;
        iters++;
        s_conv = 1;
        res2 = d[kN + 1];
        status = ST_CONVERGED;
        break;
      }
      if (scaled ? d[kN] <= 1e-30 * d[kN + 1] : d[kN] < kTiny) {
        status = ST_BRK_TT;
        break;
      }
      omega = alg_make<A>(d[0] / d[kN], kC ? d[kN - 1] / d[kN] : 0.0);
      const T om = alg_to<A, T>(omega);
      iters++;
      rt += 2;
      x = (x + al * ph) + om * hat;
      r = u - om * out;
      q = p - om * v;
      put(kR, r, rt);
      put(kQ, q, rt);
      dot(rh, r, d);
      d[kN] = norm2(r);
      d[kN + 1] = 0.0;
      part = deposit(d);
      two[1] = kQ;
      look_ahead(two, rt, rt);
      if (!collect(part, d)) return;
      rhr = value(d);
      rr = d[kN];
      res2 = rr;
    }
    // Workgroup 0 decides that the solve stands; nobody writes x before that.
    // A breakdown does not stand: it hangs on rounding, so the pipeline, which
    // sums in another order, has the last word on it.
    const bool broke = status == ST_BRK_RHO || status == ST_BRK_RV || status == ST_BRK_TT ||
                       status == ST_BRK_OMEGA;
    if (t == 0) {
      u64 o = RES_OPEN;
      if (g == 0) {
        u64 want = RES_OPEN;
        const u64 end = broke ? RES_BROKE : RES_COMMIT;
        __hip_atomic_compare_exchange_strong(a.outcome, &want, end, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        o = want == RES_OPEN ? end : want;
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
      if constexpr (std::is_same<St, SolveState>::value) a.st->res2 = res2;
      a.st->rr = rr;
      a.st->status = status;
    }
  }
};

}  // namespace ohm
