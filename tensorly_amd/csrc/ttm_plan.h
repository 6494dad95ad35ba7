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
};

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
    return grid_fits(p->gx, 64 * kTtmWaves);
  }
  const int most = p->JT <= 2 ? 2 : 1;  // accumulators of 2 tiles fit the register file
  const int64_t narrow = (Pb + 16 * VL - 1) / (16 * VL), wide = (Pb + 16 * VL * most - 1) / (16 * VL * most);
  if (Pa > kBig || narrow > kBig / Pa) return false;
  p->TN = Pa * wide * p->gy < 4096 ? 1 : most;
  p->tiles = p->TN == 1 ? narrow : wide;
  const int64_t tiles = Pa * p->tiles;
  p->split = tiles * p->gy < 4096 && Im > 32;
  p->gx = p->split ? tiles : (tiles + kTtmWaves - 1) / kTtmWaves;
  return grid_fits(p->gx, 64 * kTtmWaves);
}

}  // namespace tla
