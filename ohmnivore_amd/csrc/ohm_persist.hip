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
// are formed from r, q and v as they are gathered). ISAI: the foreign entries
// of r, q and v are fetched into LDS, once each, by the waves that a reduction
// leaves idle, so the first product reads LDS alone; the first factor's result
// and p_hat / s_hat are exchanged, or, where a workgroup's threads past its own
// rows suffice, their foreign entries are formed a second time by those
// threads and nothing but the reductions is waited for (2,871 rows: 14.6 us an
// iteration with four exchanges, 12.1 without). A supply node's row, too long
// for a thread, has its entries spread over the workgroup's threads: read from
// memory in every product it cost 1.5 to 3.6 us a product (clock stamps).
// What bounds an iteration is latency: about 1.7 us a reduction over 20 to 128
// workgroups, 1.2 us an exchange, 0.4 us a product from LDS and 0.8 us of
// 64-bit scalar arithmetic. Measured per iteration, pipeline -> here: Jacobi
// 15.3 -> 3.8 us (102 rows, one workgroup), 21.2 -> 9.7 (10,002), 21.7 -> 12.2
// (65,540), 25.3 -> 15.8 (129,604); ISAI 29.3 -> 12.1 (2,871), 27.9 -> 15.1
// (16,388), 29.8 -> 15.9 (32,404), 35.7 -> 19.1 (65,540), 45.4 -> 25.4 (129,604).
// Systems that lose by it are told apart in resident_geometry.
//
// All workgroups must run at once: the grid has at most one workgroup per
// compute unit, and the device's gate lets solves run together only if they fit
// together (ohm_resident_gate.h). A wait that lasts longer than kResLimit ends the
// kernel with nothing written (the outcome word says so to the other workgroups)
// and the host continues with the pipeline from the state that k_init left; so
// does a solve that breaks down.
#include <algorithm>
#include <cstdlib>

#include "ohm_resident_dev.h"

namespace ohm {

template <typename T, int PK, int W, int WF>
__global__ __launch_bounds__(kResThreads) void k_bicg_resident(ResArgs<T, SolveState> a) {
  constexpr bool kEarly = PK != PK_ISAI && (sizeof(T) == 4 || W <= 6);
  using R = Resident<T, SolveState, PK, W, WF, kEarly>;
  __shared__ typename R::Shared sh;
  extern __shared__ __align__(16) unsigned char res_lds[];
  R r(a, sh, res_lds);
  r.solve();
}

// ------------------------------------------------------------ host side --
int resident_absent(const ohm_backend *b) {
  const char *e = getenv("OHM_RESIDENT_ABSENT");
  const int v = e ? atoi(e) : 0;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (v == 2) (void)hipStreamIsCapturing(b->stream, &st);
  return v == 1 || st != hipStreamCaptureStatusNone;
}

ohm_status resident_gave_up(ohm_backend *b, const void *outcome, bool &gave_up) {
  u64 o = RES_OPEN;
  OHM_HIP(hipMemcpyAsync(&o, outcome, sizeof(o), hipMemcpyDeviceToHost, b->stream));
  OHM_HIP(hipStreamSynchronize(b->stream));
  gave_up = o == RES_ABORT;
  return OHM_OK;
}

// One row per thread: with two or three rows a thread's state leaves the
// registers, and the pipeline, whose launches then carry enough work, is
// faster (ISAI at 160,004 rows: 59 us per iteration against 49, at 262,148 97
// against 62), so the path ends at 512 rows for each compute unit. Tiles of
// 4, 6 or 8 entries; kResMaxLong longer rows (a supply node's) are summed by
// their whole workgroup, more of them belong to the pipeline's row blocks. Up to 64
// unknowns the one-wave solve needs no workgroup barriers at all.
//
// A matrix whose rows read far and apart costs a word's round trip for each
// entry, and more workgroups more of them. Per iteration in 64 bits, pipeline
// -> here: Jacobi, a mesh in random order 21.9 -> 21.2 us at 3,969 rows (170
// places), 21.0 -> 22.0 at 5,929 (198), 24.7 -> 27.4 at 60,025 (249); three random
// neighbours a row 26.6 -> 26.2 at 60,000 (186). ISAI, over the three matrices: a
// ladder in random order 28.7 -> 27.4 us at 3,200 rows, 29.2 -> 30.2 at 4,000
// (230), 35.6 -> 45.3 at 60,000 (295); with its own pattern for the factors 28.6 ->
// 13.6 at 6,000 (218; the halo holds), 28.0 -> 29.4 at 9,000 (223). In 32 bits a
// value is one word and the resident solve stays the faster one (1.05 to 2 times).
ResGeo resident_geometry(const ohm_backend *b, const DevCsr &a, const PrecondDev &p, int n,
                         bool f32) {
  ResGeo g;
  if (n <= 64 || (p.kind == PK_ISAI && p.mm.rowptr)) return g;
  const DevCsr *ms[3] = {&a, &p.ml, &p.mu};
  const int nm = p.kind == PK_ISAI ? 3 : 1;
  if (!f32) {
    int places = 0;
    for (int m = 0; m < nm; m++) places += ms[m]->scatter;
    if (places > (nm == 1 ? 185 : 220)) return g;
  }
  static const int kWidths[3] = {4, 6, 8};
  const auto width = [&](int m0, int m1) {
    for (int w = 0; w < 3; w++) {
      bool fits = true;
      for (int m = m0; m < m1; m++)
        fits = fits && ms[m]->long_rows[w] >= 0 && ms[m]->long_rows[w] <= kResMaxLong;
      if (fits) return kWidths[w];
    }
    return 0;
  };
  g.width = width(0, 1);
  g.fwidth = nm > 1 ? width(1, 3) : 4;
  if (!g.width || !g.fwidth) return ResGeo();
  // the factors' rows are about half as long as A's: tiles of 4, or A's width
  if (g.fwidth > 4) g.width = g.fwidth = std::max(g.width, g.fwidth);
  const int grid = (n + kResThreads - 1) / kResThreads;
  if (grid > std::min(b->num_cu, kResMaxGrid)) return g;
  g.grid = grid;
  g.rows = (n + grid - 1) / grid;
  g.threads = (g.rows + 63) / 64 * 64;
  // smaller workgroups, whose spare threads form their halo: more of them make
  // a reduction slower by at most 0.8 us, the four exchanges are worth 2.5
  if (p.kind == PK_ISAI && grid > 1 && p.halo_rows > 0) {
    const int hgrid = (n + p.halo_rows - 1) / p.halo_rows;
    if (hgrid <= std::min(b->num_cu, kResMaxGrid)) {
      g.grid = hgrid;
      g.rows = (n + hgrid - 1) / hgrid;
      g.threads = kResThreads;
      g.halo = 2;
    }
  }
  return g;
}

// Rows per workgroup, the most whose foreign operands of A's and M_U's rows
// all find a thread (the kernel's find_halo, over the patterns).
int resident_halo_rows(const ohm_backend *b, const DevCsr &a, const DevCsr &ml, const DevCsr &mu) {
  const int n = a.n;
  if (n <= kResThreads) return 0;
  const auto tile = [](const DevCsr &m, uint32_t r) {
    return m.h_rowptr[r + 1] - m.h_rowptr[r] <= (uint32_t)kResMaxWidth;
  };
  std::vector<int> seen(n, -1);
  std::vector<uint32_t> list;
  for (int rows = kResThreads - 64; rows >= 128; rows -= 64) {
    const int grid = (n + rows - 1) / rows, even = (n + grid - 1) / grid;
    if (grid > std::min(b->num_cu, kResMaxGrid)) break;
    bool fits = true;
    std::fill(seen.begin(), seen.end(), -1);
    for (int g = 0; g < grid && fits; g++) {
      const uint32_t lo = (uint32_t)g * even, hi = (uint32_t)std::min(n, (g + 1) * even);
      list.clear();
      const auto join = [&](const DevCsr &m, uint32_t r, bool hat) {
        const uint32_t k0 = m.h_rowptr[r], k1 = m.h_rowptr[r + 1];
        if (k0 == k1 || !tile(m, r)) return;
        // columns ascend: most rows are done with their first and last
        if (m.h_col[k0] >= lo && m.h_col[k1 - 1] < hi) return;
        for (uint32_t k = k0; k < k1; k++) {
          const uint32_t c = m.h_col[k];
          if ((c >= lo && c < hi) || seen[c] == g || !tile(ml, c) || (hat && !tile(mu, c))) continue;
          seen[c] = g;
          list.push_back(c);
        }
      };
      const size_t cap = (size_t)(kResThreads - (int)(hi - lo));
      for (uint32_t r = lo; r < hi && list.size() <= cap; r++) join(a, r, true);
      const size_t n_hat = list.size();
      for (uint32_t r = lo; r < hi && list.size() <= cap; r++) join(mu, r, false);
      for (size_t i = 0; i < n_hat && list.size() <= cap; i++) join(mu, list[i], false);
      fits = list.size() <= cap;
    }
    if (fits) return rows;
  }
  return 0;
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
    ResCsr<T> c{m.rowptr, m.col, nullptr, nullptr, 0.0, 0.0};
    if constexpr (f32)
      c.g = m.val32;
    else
      c.g = m.val;
    return c;
  };
  ResArgs<T, SolveState> q{};
  q.n = a.n;
  q.rows = g.rows;
  q.grid = g.grid;
  q.halo = g.halo;
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
  q.absent = resident_absent(b);
  q.words = reinterpret_cast<u64 *>(base);
  q.slots = q.words + l.slots;
  q.outcome = q.words + l.outcome;
  // ISAI: the halo's columns, then the vectors (the hash table before them)
  const unsigned lds = (unsigned)(p.kind == PK_ISAI
                                      ? sizeof(uint32_t) * kResHalo +
                                            std::max(5 * (size_t)(g.rows + kResHalo) * sizeof(T),
                                                     sizeof(uint32_t) * 8 * kResThreads)
                                      : 3 * (size_t)g.rows * sizeof(T));
  const auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(g.grid), dim3(g.threads), lds, b->stream, q);
  };
  const auto by_width = [&](auto pk) {
    constexpr int PK = decltype(pk)::value;
    if (g.width == 4)
      launch(k_bicg_resident<T, PK, 4, 4>);
    else if (g.width == 6)
      launch(k_bicg_resident<T, PK, 6, 4>);
    else
      launch(k_bicg_resident<T, PK, 8, 4>);
  };
  if (p.kind != PK_ISAI)  // without a preconditioner inv is null
    by_width(std::integral_constant<int, PK_JACOBI>());
  else if (g.fwidth == 4)
    by_width(std::integral_constant<int, PK_ISAI>());
  else if (g.fwidth == 6)
    launch(k_bicg_resident<T, PK_ISAI, 6, 6>);
  else
    launch(k_bicg_resident<T, PK_ISAI, 8, 8>);
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
