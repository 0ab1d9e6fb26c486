// ohm_batch_resident.h — resident solves of a batch (ohm_batch_resident.hip).
#pragma once

#include <vector>

#include "ohm_batch_types.h"

namespace ohm {

// One system of a batch as the resident solve needs it; vectors as k_binit
// and k_bfold_init left them.
template <typename S>
struct BatchSolve {
  const BGeo *geo;
  const int *long_rows;   // rows with more than 4, 6 and 8 entries
  int scatter;            // scattered_lines of its pattern
  S *x;
  const S *r, *rh, *inv;  // inv null: no preconditioner
  BSys *st;
};

// The most workgroups of one launch, when these systems take the resident path:
// they run at once in one launch or two, and that is faster than the batch
// engine's own kernels. Else 0.
template <typename S>
int batch_resident_workgroups(const ohm_backend *b, const std::vector<BatchSolve<S>> &sys);

// Enqueues the solves. A system that could not finish stays RUNNING with its
// vectors untouched. The caller holds a ResidentPass for their workgroups until
// the launches are done, and keeps `tables`, which the upload may still be reading, until
// it has waited for the stream.
template <typename S>
ohm_status batch_resident_enqueue(ohm_backend *b, const std::vector<BatchSolve<S>> &sys,
                                  std::vector<char> &tables);

// Whether one of the `n` systems of these tables gave up because a wait outlasted
// its limit.
template <typename S>
ohm_status batch_resident_gave_up(ohm_backend *b, int n, const std::vector<char> &tables,
                                  bool &gave_up);

}  // namespace ohm
