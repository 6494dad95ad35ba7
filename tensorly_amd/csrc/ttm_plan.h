// How an n-mode product of any mode sizes is cut into workgroups
// (ttm_any.hip); host code only.
#pragma once
#include <algorithm>
#include <cstdint>

#include "grid_limit.h"

namespace tla {

constexpr int kTtmWaves = 4;

struct TtmPlan {
  int JT;         // tiles of 16 rows j per wave
  int TN;         // tiles of b (cols) or of rows of X (rows) per wave
  int64_t tiles;  // cols: wave tiles of b per a
  bool split;     // cols: the block's waves share a tile and split m
  int64_t gx, gy;
  bool vector;    // the vector kernel (one thread per output element) takes less
};

// Whether one thread per output element takes less than the plan's matrix
// tiles: short runs b (a tile is 64 or 32 columns however few there are), few
// rows j (a tile is 16) and short sums m.  Both estimated in ns from sweeps
// over b = 1 ... 4096, m = 2 ... 512, j = 1 ... 64 at 64 and 128 MiB: a wave
// costs a start and its steps over m, an output element a store and its
// products (less where neighbouring lanes share X's lines).  Measured, float32,
// vector / tiles: 2M x 2 x 4, mode 1, 1 row: 24 / 1115 us, 64 rows
// 1490 / 4820; 8192 x 512 x 4, 8 / 16 rows: 91 / 124, 145 / 127; 819 x 5 x
// 4096, 1 / 4 rows: 19 / 41, 58 / 46; 3.4M x 5, mode 1, 1 / 8 rows: 21 / 65,
// 109 / 67.
inline bool ttm_vector_wins(const TtmPlan& p, bool f64, int64_t Pa, int64_t Im, int64_t Pb, int64_t J) {
  const double out = double(Pa) * J * Pb, waves = double(p.gx) * kTtmWaves * p.gy;
  if (out > 4.2e9) return false;  // (past one launch)
  if (Pb == 1) {
    if (Im > 8) return false;
    const double tiles = waves * ((f64 ? 1.1 : 0.85) + 0.1 * Im);
    const double vector = out * (f64 ? 0.0024 + 0.00055 * Im : 0.0013 + 0.00065 * Im);
    return vector + 1000 < tiles;
  }
  const double steps = double((Im + 15) / 16) / (p.split ? kTtmWaves : 1);
  const double start[2][4] = {{0.2, 0.4, 0.75, 1.1}, {0.25, 0.6, 0.85, 1.1}};  // by JT
  const double step[2][4] = {{0.43, 0.63, 0.9, 1.19}, {0.34, 0.66, 1.0, 1.31}};
  const double tiles = waves * (p.TN == 1 ? start[f64][p.JT - 1] + step[f64][p.JT - 1] * steps
                                          : (f64 ? 0.5 : 0.55) * p.JT + (f64 ? 0.7 : 0.72) * p.JT * steps);
  const double vector = out * (f64 ? 0.002 + 0.00075 * Im : 0.0017 + (Pb % 4 == 0 ? 0.00053 : Im <= 8 ? 0.0007 : 0.0012) * Im);
  return std::max(vector, 100.0 * Im) + 1000 < tiles;  // (a chain of Im loads)
}

// Fills *p and returns true when ttm_any_launch takes these sizes.
inline bool ttm_any_plan(bool f64, int64_t Pa, int64_t Im, int64_t Pb, int64_t J, TtmPlan* p) {
  constexpr int64_t kBig = 0x7fffff00;
  const int sz = f64 ? 8 : 4, VL = 16 / sz;
  *p = TtmPlan{};
  if (Pb > 1 && Pb < VL) return false;
  // 32-bit indices: m, the bytes of 16 rows (cols) or 64 rows (rows) of X; the grid's y
  if (Im > kBig / (64 * sz) || Pb > kBig / (16 * sz) || J > 16 * 65535) return false;
  // J > 64: groups of 16 JT rows with the least padding
  p->JT = (int)std::min<int64_t>((J + 15) / 16, 4);
  if (J > 64)
    for (int t = 3; t >= 2; --t)
      if ((J + 16 * t - 1) / (16 * t) * t < (J + 16 * p->JT - 1) / (16 * p->JT) * p->JT) p->JT = t;
  p->gy = (J + 16 * p->JT - 1) / (16 * p->JT);
  if (Pb == 1) {
    if (Pa > kBig * 16) return false;
    const int64_t rows16 = (Pa + 15) / 16;
    // more tiles per wave share the rows of U, fewer fill the GPU
    const int most = p->JT <= 2 ? 4 : 2;
    p->TN = rows16 * p->gy >= most * 4096 ? most : 1;
    p->gx = (rows16 + kTtmWaves * p->TN - 1) / (kTtmWaves * p->TN);
    p->vector = ttm_vector_wins(*p, f64, Pa, Im, Pb, J);
    return grid_fits(p->gx, 64 * kTtmWaves);
  }
  const int most = p->JT <= 2 ? 2 : 1;  // accumulators of 2 tiles fit the register file
  const int64_t narrow = (Pb + 16 * VL - 1) / (16 * VL), wide = (Pb + 16 * VL * most - 1) / (16 * VL * most);
  if (Pa > kBig || narrow > kBig / Pa) return false;
  // (a second tile that is mostly padding costs as much as the first)
  p->TN = Pa * wide * p->gy < 4096 || 4 * wide * most > 5 * narrow ? 1 : most;
  p->tiles = p->TN == 1 ? narrow : wide;
  const int64_t tiles = Pa * p->tiles;
  p->split = tiles * p->gy < 4096 && Im > 32;
  p->gx = p->split ? tiles : (tiles + kTtmWaves - 1) / kTtmWaves;
  p->vector = ttm_vector_wins(*p, f64, Pa, Im, Pb, J);
  return grid_fits(p->gx, 64 * kTtmWaves);
}

}  // namespace tla
