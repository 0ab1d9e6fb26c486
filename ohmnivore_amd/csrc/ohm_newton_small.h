// ohm_newton_small.h — Newton runs of small circuits in one workgroup
// (ohm_newton_small.hip).
#pragma once

#include "ohm_devices.h"

namespace ohm {

constexpr int kSmallIters = 64;  // Newton iterations of one launch

enum { NS_RUNNING = 0, NS_CONVERGED = 1, NS_SOLVE = 2, NS_NAN = 3, NS_SINGULAR = 4 };

// What a launch leaves for the host.
struct SmallWord {
  int reason;      // NS_*: RUNNING means kSmallIters iterations are done
  int done;        // iterations done, a failed one included
  int status;      // SolveStatus of the last sub-solve
  int nan;         // the last assembly held a NaN or an infinity
  double max_diff;
  double f_prev, lin_prev, eta_prev;  // forcing state (Forcing)
  int iters[kSmallIters];             // BiCGSTAB iterations of each sub-solve
};
static_assert(sizeof(SmallWord) <= kPinnedBytes, "the word is read through the backend's staging");

// Whether a run with these settings takes the one-workgroup form.
bool newton_small_fits(const ohm_newton_ctx *c, const ohm_newton_params &prm);

// Enqueues up to `budget` Newton iterations from c->x (base values and
// right-hand side already in c->A.val and c->rhs) and waits for them. `first`:
// the run's first launch, whose ILU(0) restarts from the matrix.
ohm_status newton_small_launch(ohm_newton_ctx *c, const ohm_newton_params &prm, const BicgOpts &o,
                               const Forcing &fc, int budget, bool first, SmallWord &out);

}  // namespace ohm
