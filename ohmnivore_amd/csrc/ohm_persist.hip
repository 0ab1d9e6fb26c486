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

#include "ohm_resident_dev.h"

namespace ohm {

template <typename T, int PK, int W>
__global__ __launch_bounds__(kResThreads) void k_bicg_resident(ResArgs<T, SolveState> a) {
  using R = Resident<T, SolveState, PK, W, PK != PK_ISAI || W <= 6>;
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
