// What one launch can hold (host code only).
#pragma once
#include <cstdint>

namespace tla {

// Whether `blocks` workgroups of `threads` threads fit one launch's x
// dimension: it holds fewer than 2^32 threads.
constexpr bool grid_fits(int64_t blocks, int threads) { return blocks <= 0xffffffffll / threads; }

}  // namespace tla
