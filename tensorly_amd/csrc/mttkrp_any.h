// Matrix-core MTTKRP for shapes the aligned kernels of mttkrp.hip do not take
// (odd mode sizes) and for float64 (mttkrp_any.hip).
#pragma once
#include "common.h"
#include "mttkrp_any_plan.h"

namespace tla {

// Whether the launch takes a side job: its sum of partials is one launch.
inline bool any_takes_job(const AnyPlan& p, int R) { return R <= 64 && p.nblk * p.slices > 1; }

// Runs it: factors and weights in the tensor's dtype, ws of any_plan's size;
// job (nullable): a side job, only where any_takes_job.
int any_launch(bool f64, const AnyPlan& p, const void* X, int ndim, const int64_t* shape, const void* const* factors,
               const void* weights, int R, int mode, void* out, void* ws, const InvJob* job, hipStream_t st);

}  // namespace tla
