// local_direct.hpp -- the scalar local kernels for small calls (local_direct.hip).
#pragma once

#include "kf_common.hpp"
#include "local_plan.hpp"

namespace kf {

enum DirectMode { DIRECT_SYMM_RFP = 0, DIRECT_SYMM_DENSE = 1, DIRECT_RECT = 2 };

// K of the planned sets (equal label lists; p2 = p1 and X2 = X1 for the symmetric forms)
// into `out`, with cy the factor from a squared distance to exp_scaled's argument.
int local_direct(int mode, const LocalPlan &p1, const double *X1, const LocalPlan &p2,
                 const double *X2, int rep, double cy, double *out, int timer_id,
                 hipStream_t stream);

}  // namespace kf
