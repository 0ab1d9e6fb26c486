// ohm_batch_resident.hip — the batch engine's solves as resident launches.
//
// A batched iteration is nine launches (five kernels and a fold per reduction,
// 30 us at 8 systems of 16,388 rows), and a batch of small systems runs one
// workgroup each with every vector in memory: 21 complex systems of 1,847
// rows took 35 us per iteration on 21 of 256 compute units. Here each
// system has its own workgroups, which keep its rows in registers and meet
// through tagged words as a single resident solve's do (ohm_persist.hip); the
// systems do not wait for each other. Jacobi or no preconditioner, 64-bit,
// real or complex (A = G + sigma C formed as the rows are loaded).
//
// Bound, as there, by the latency of its reductions and by registers (complex
// tiles of six entries spill). Systems that do not fit the chip together go in
// two launches, one after the other; with more the nine launches, or a workgroup
// per system, do as well. Measured, ten
// backward-Euler steps of 8 x 16,388 real rows 39.7 -> 15.0 ms (1,150
// iterations); 21 x 1,847 complex rows 16.6 -> 7.3 ms (375 to 481 iterations).
#include <algorithm>
#include <new>

#include "ohm_batch_resident.h"
#include "ohm_resident_dev.h"

namespace ohm {

// Rows of a workgroup. Real systems: ten waves leave 168 registers a thread,
// enough without requests ahead of a reduction. Complex: eight waves, 256.
template <typename S>
constexpr int kResBatchRows = Tr<S>::C ? 512 : 640;

template <typename S, int W>
__global__ __launch_bounds__(kResBatchRows<S>) void k_batch_resident(
    const ResArgs<S, BSys> *__restrict__ args, const int *__restrict__ owner, int first) {
  using R = Resident<S, BSys, PK_JACOBI, W, 4, false>;
  __shared__ typename R::Shared sh;
  __shared__ ResArgs<S, BSys> a;
  extern __shared__ __align__(16) unsigned char res_lds[];
  if (threadIdx.x == 0) {
    a = args[owner[first + blockIdx.x]];
    a.first -= first;  // within this launch
  }
  __syncthreads();
  R r(a, sh, res_lds);
  r.solve();
}

__global__ void k_clear_words(int64_t n, u64 *w) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    w[i] = 0;
}

namespace {

struct Cut {
  int rows = 0, width = 0;
  std::vector<int> group;  // first system of each launch, then the number of systems
};

// Rows per workgroup, tile width and launches of a list of systems; rows == 0
// when it does not fit, or where the batch engine's own kernels (a workgroup per
// system up to kPersistRows, else nine launches per iteration) are as fast. Those
// cost 7 to 10 us an iteration up to 500 rows, 16 (complex 19) at 1,024, 28 (34)
// at 2,025, 52 (64) at 4,096 and about 37 beyond; here it is, per launch, 5 to 7 us
// with one workgroup a system and 10 to 15 with several, complex 10 to 30.
template <typename S>
Cut cut_batch(const ohm_backend *b, const std::vector<BatchSolve<S>> &sys) {
  Cut c;
  constexpr bool cplx = Tr<S>::C;
  int most = 0, places = 0;
  int64_t total = 0;
  for (const auto &s : sys) {
    most = std::max(most, s.geo->n);
    total += s.geo->n;
    places = std::max(places, s.scatter);
  }
  // whole solves, own kernels -> here: 9 real rows 131 -> 147 us, 25 179 -> 151;
  // complex 256 rows 414 -> 538 us, 1,024 1,281 -> 1,300, 1,225 1,459 -> 1,274
  if (most < (cplx ? 1025 : 24)) return c;
  // in random order, complex: a mesh of 1,225 rows 1,581 -> 1,991 us, 2,025 2,442
  // -> 2,270, 16,384 2,250 -> 2,408; a ladder of 1,100 about even, 1,700 1,900 ->
  // 1,627, 16,384 2,961 -> 1,849, four of 30,000 3,311 -> 3,755
  if (cplx && places > 40 &&
      (most < 1600 || (most > kPersistRows && (places > 185 || total > 50'000))))
    return c;
  static const int kWidths[3] = {4, 6, 8};
  int longs = 0;
  for (int w = 0; w < 3 && !c.width; w++) {
    longs = 0;
    for (const auto &s : sys) longs = std::max(longs, s.long_rows[w]);
    if (longs <= kResMaxLong) c.width = kWidths[w];
  }
  if (!c.width) return c;
  // 3 to 4 us (complex 4 to 5) per long row: real, two of them, 83 rows 328 ->
  // 355 us, 227 474 -> 484, 258 536 -> 443; 678 947 -> 1,108, 786 1,083 -> 1,033
  const bool one_wg = most <= kResBatchRows<S>;
  if (longs && cplx && most < 1400) return c;
  if (longs > 1 && !cplx && (most <= 256 || (!one_wg && most < 768))) return c;
  const int cus = std::min(b->num_cu, kResMaxGrid);
  // Systems of one workgroup each wait for nobody, so any number of them
  // shares a launch; else the smallest workgroups that need the fewest launches.
  for (int rows : {256, 320, 384, 448, 512, 576, 640}) {
    if (rows > kResBatchRows<S>) break;
    if (one_wg && rows < most) continue;
    std::vector<int> group(1, 0);
    int used = 0;
    bool fits = true;
    for (size_t k = 0; most > rows && k < sys.size(); k++) {
      const int wgs = (sys[k].geo->n + rows - 1) / rows;
      fits = fits && wgs <= cus;
      if (used > 0 && used + wgs > cus) {
        group.push_back((int)k);
        used = 0;
      }
      used += wgs;
    }
    group.push_back((int)sys.size());
    if (fits && (c.rows == 0 || group.size() < c.group.size())) {
      c.rows = rows;
      c.group = group;
    }
  }
  // two launches: real, 144 x 1,024 rows 1,208 -> 1,525 us, 163 x 1,225 1,597 ->
  // 1,584, 16 x 12,100 2,656 -> 1,793, 4 x 60,000 with two random neighbours a row
  // 1,466 -> 1,616; complex 68 x 2,116 3,003 -> 3,323, 45 x 3,249 4,281 -> 3,503,
  // 12 x 12,100 2,859 -> 3,676
  const int groups = (int)c.group.size() - 1;
  const bool two = places <= 40 && (cplx ? most > 2600 && most <= kPersistRows : most >= 1200);
  if (groups > (two ? 2 : 1)) c.rows = 0;
  return c;
}

}  // namespace

template <typename S>
int batch_resident_workgroups(const ohm_backend *b, const std::vector<BatchSolve<S>> &sys) {
  if (sys.empty()) return 0;
  const Cut c = cut_batch<S>(b, sys);
  int most = 0;
  for (size_t q = 0; c.rows && q + 1 < c.group.size(); q++) {
    int wgs = 0;
    for (int k = c.group[q]; k < c.group[q + 1]; k++) wgs += (sys[k].geo->n + c.rows - 1) / c.rows;
    most = std::max(most, wgs);
  }
  return most;
}

template <typename S>
ohm_status batch_resident_enqueue(ohm_backend *b, const std::vector<BatchSolve<S>> &sys,
                                  std::vector<char> &tables) {
  const Cut c = cut_batch<S>(b, sys);
  if (!c.rows) return fail(OHM_ERR_INVALID, "batch does not fit the resident solve");
  constexpr int kVecs = 3;
  // words of every system, then the argument and owner tables (one upload)
  size_t words = 0, wgs = 0;
  std::vector<size_t> at(sys.size());
  for (size_t k = 0; k < sys.size(); k++) {
    const int n = sys[k].geo->n, grid = (n + c.rows - 1) / c.rows;
    at[k] = words;
    words += (grid > 1 ? (size_t)kVecs * n * Tagged<S>::kWords : 0) +
             (size_t)2 * grid * kResSlotWords + 1;
    wgs += grid;
  }
  using Args = ResArgs<S, BSys>;
  const auto al = [](size_t v) { return (v + 255) & ~size_t(255); };
  const size_t args_at = al(words * 8), owner_off = al(sizeof(Args) * sys.size());
  tables.resize(owner_off + sizeof(int) * wgs);
  void *ws = nullptr;
  OHM_TRY(resident_ws(b, args_at + tables.size(), &ws));
  u64 *base = static_cast<u64 *>(ws);
  Args *args = reinterpret_cast<Args *>(tables.data());
  int *owner = reinterpret_cast<int *>(tables.data() + owner_off);
  const int absent = resident_absent(b);
  int wg = 0;
  for (size_t k = 0; k < sys.size(); k++) {
    const BGeo &q = *sys[k].geo;
    Args &a = *new (&args[k]) Args{};
    a.n = q.n;
    a.grid = (q.n + c.rows - 1) / c.rows;
    a.rows = (q.n + a.grid - 1) / a.grid;
    a.first = wg;
    std::fill(owner + wg, owner + wg + a.grid, (int)k);
    wg += a.grid;
    a.m[0] = ResCsr<S>{q.rowptr, q.col, q.g, q.c, q.sig_re, q.sig_im};
    a.inv = sys[k].inv;
    a.x = sys[k].x;
    a.r = sys[k].r;
    a.rh = sys[k].rh;
    a.st = sys[k].st;
    a.absent = absent;
    a.words = base + at[k];
    a.slots = a.words + (a.grid > 1 ? (size_t)kVecs * q.n * Tagged<S>::kWords : 0);
    a.outcome = a.slots + (size_t)2 * a.grid * kResSlotWords;
  }
  Args *d_args = reinterpret_cast<Args *>(static_cast<char *>(ws) + args_at);
  int *d_owner = reinterpret_cast<int *>(static_cast<char *>(ws) + args_at + owner_off);
  OHM_HIP(hipMemcpyAsync(d_args, tables.data(), tables.size(), hipMemcpyHostToDevice, b->stream));
  hipLaunchKernelGGL(k_clear_words, dim3(grid_for((int64_t)words)), dim3(kBlock), 0, b->stream,
                     (int64_t)words, base);
  b->dispatches++;
  for (size_t q = 0; q + 1 < c.group.size(); q++) {
    const int k0 = c.group[q], k1 = c.group[q + 1];
    int rows = 0;
    for (int k = k0; k < k1; k++) rows = std::max(rows, args[k].rows);
    const int first = args[k0].first, grid = args[k1 - 1].first + args[k1 - 1].grid - first;
    const unsigned threads = (unsigned)(rows + 63) / 64 * 64;
    const unsigned lds = (unsigned)(kVecs * (size_t)rows * sizeof(S));
    const auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, b->stream, d_args, d_owner, first);
    };
    if (c.width == 4)
      launch(k_batch_resident<S, 4>);
    else if (c.width == 6)
      launch(k_batch_resident<S, 6>);
    else
      launch(k_batch_resident<S, 8>);
    OHM_HIP(hipGetLastError());
    b->dispatches++;
  }
  return OHM_OK;
}

template <typename S>
ohm_status batch_resident_gave_up(ohm_backend *b, int n, const std::vector<char> &tables,
                                  bool &gave_up) {
  const ResArgs<S, BSys> *args = reinterpret_cast<const ResArgs<S, BSys> *>(tables.data());
  gave_up = false;
  for (int k = 0; k < n && !gave_up; k++) OHM_TRY(resident_gave_up(b, args[k].outcome, gave_up));
  return OHM_OK;
}

template int batch_resident_workgroups<double>(const ohm_backend *,
                                               const std::vector<BatchSolve<double>> &);
template int batch_resident_workgroups<cx<double>>(const ohm_backend *,
                                                   const std::vector<BatchSolve<cx<double>>> &);
template ohm_status batch_resident_enqueue<double>(ohm_backend *,
                                                   const std::vector<BatchSolve<double>> &,
                                                   std::vector<char> &);
template ohm_status batch_resident_enqueue<cx<double>>(
    ohm_backend *, const std::vector<BatchSolve<cx<double>>> &, std::vector<char> &);

template ohm_status batch_resident_gave_up<double>(ohm_backend *, int, const std::vector<char> &,
                                                   bool &);
template ohm_status batch_resident_gave_up<cx<double>>(ohm_backend *, int,
                                                       const std::vector<char> &, bool &);

}  // namespace ohm
