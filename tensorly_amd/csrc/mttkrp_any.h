// Matrix-core MTTKRP for shapes the aligned kernels of mttkrp.hip do not take
// (odd mode sizes) and for float64: planning and launch (mttkrp_any.hip).
#pragma once
#include "common.h"

namespace tla {

struct AnyPlan {
  bool last;          // output mode is the contiguous one
  int TN, RT;         // tiles per wave (rows: 16 rows each; last: column tiles) and rank tiles of a slab
  int64_t groups;     // row groups / column groups
  int64_t nblk;       // blocks per group = partial sums per output element
  int64_t A, In, Q;   // X viewed as A x In x Q, mode In kept
  int64_t K, Pb, J;
  int nqc;            // chunks per (A, Q) row
  int64_t nchunks;    // chunks (rows) / row visits (last)
  int64_t g_rows;     // rows of the precomputed scale table (0: none)
  bool build_g;       // the table has to be built (else it is a factor itself, or absent)
  bool direct_g;      // ... but its rows are formed in the kernel
  size_t ws_bytes;
};

// Fills *p and returns true when the kernels take this contraction.
bool any_plan(bool f64, int ndim, const int64_t* shape, int R, int mode, bool weights, AnyPlan* p);

// Whether the launch takes a side job: its sum of partials is one launch.
inline bool any_takes_job(const AnyPlan& p, int R) { return R <= 64 && p.nblk > 1; }

// Runs it: factors and weights in the tensor's dtype, ws of any_plan's size;
// job (nullable): a side job, only where any_takes_job.
int any_launch(bool f64, const AnyPlan& p, const void* X, int ndim, const int64_t* shape, const void* const* factors,
               const void* weights, int R, int mode, void* out, void* ws, const InvJob* job, hipStream_t st);

}  // namespace tla
