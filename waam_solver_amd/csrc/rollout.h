/*
 * rollout.h — what the rollouts' forward (rollout.hip) and backward (adjoint.hip,
 * adjoint_coupled.hip) runs share.
 */
#pragma once

#include "waam_common.h"

namespace waam {

/* the checks of a rollout call; saved: the backward's fields have to be there */
int check_rollout(const char *who, const waam_rollout *r, const double *arc_i, const double *arc_j,
                  int n, bool saved);

/* dL/d(eta, s_h, s_sigma) of a segment: parts holds, per step, kReduceBlocks groups of three
 * compensated pairs; grads += the steps' totals, the last step first (adjoint.hip) */
void launch_rollback_totals(const double *parts, int n, double *step_totals, double *grads,
                            hipStream_t st);

}  // namespace waam
