// n-mode product of any mode sizes on the matrix cores (ttm_any.hip).
#pragma once
#include "common.h"
#include "ttm_plan.h"

namespace tla {

// out[a, j, b] = sum_m U[j ldj + m ldm] X[a, m, b], with the plan of these sizes
int ttm_any_launch(bool f64, const TtmPlan& p, const void* X, int64_t Pa, int64_t Im, int64_t Pb, const void* U,
                   int64_t ldj, int64_t ldm, int64_t J, void* out, hipStream_t st);

}  // namespace tla
