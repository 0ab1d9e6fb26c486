// ohm_persist.h — the resident BiCGSTAB solve (ohm_persist.hip): one launch
// iterates to the end, workgroups meeting through tagged words in memory.
#pragma once

#include "ohm_precond.h"
#include "ohm_reduce.h"
#include "ohm_resident_gate.h"

namespace ohm {

constexpr int kResThreads = 512;      // most threads of a workgroup (256 registers each)
constexpr int kResMaxGrid = 256;      // most workgroups (one per CU)
// Rows per matrix beyond the row tile. Each is a product of its own that the
// whole workgroup joins, 2.5 to 6 us an iteration: with two (12 entries each) an
// iteration of 9,027 rows takes 16.5 us against the pipeline's 19.5, with four
// 24.4 against 20.7, with 32 123 against 19.5.
constexpr int kResMaxLong = 2;
constexpr int kResSlotWords = 8;      // 64-bit words of one reduction slot
constexpr int kResMaxWidth = 8;       // widest row tile
constexpr int kResHalo = 768;         // most foreign columns a workgroup keeps in LDS

// How a solve is cut: `grid` workgroups of `threads` threads with `rows`
// consecutive rows each, one per thread, row tiles of `width` entries (the
// ISAI factors' of `fwidth`).
// grid == 0: the system does not fit this path.
struct ResGeo {
  int grid = 0, threads = 0, rows = 0, width = 0, fwidth = 4;
  int halo = 1;  // ISAI: 2: the workgroups' spare threads form their halo
};
// The geometry of a solve of a x = b with p, in 32 bits with f32 set.
ResGeo resident_geometry(const ohm_backend *b, const DevCsr &a, const PrecondDev &p, int n,
                         bool f32);

// Workspace of one solve, cleared before it: tagged vectors, reduction slots
// and the outcome word.
struct ResLayout {
  size_t clear_words = 0, bytes = 0;  // the whole workspace
  size_t slots = 0, outcome = 0;      // word offsets
};
ResLayout resident_layout(const ResGeo &g, const PrecondDev &p, int n, bool f32);

// The backend's workspace for resident solves, at least `bytes` long.
ohm_status resident_ws(ohm_backend *b, size_t bytes, void **ws);

// Enqueues the solve behind k_init: x, r and r_hat as k_init left them, the
// workspace `ws` with its first clear_words words zero. On success the state
// word holds the final status; a solve that could not finish (its workgroups
// did not all run at once within the time limit) leaves every vector and the
// state as k_init did, RUNNING, for the multi-kernel pipeline.
template <typename T>
ohm_status resident_enqueue(ohm_backend *b, const DevCsr &a, const PrecondDev &p, const ResGeo &g,
                            void *ws, const BicgVecs<T> &v, SolveState *st);

// Whether the solve with this outcome word (on the device) ended because a wait
// outlasted its limit; waits for the stream. For solves left RUNNING.
ohm_status resident_gave_up(ohm_backend *b, const void *outcome, bool &gave_up);

// OHM_RESIDENT_ABSENT=1 (tests): the last workgroup of every solve stays away, as
// on a device that does not run it, and the others give up; 2: of captured ones.
int resident_absent(const ohm_backend *b);

}  // namespace ohm
