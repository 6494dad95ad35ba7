// How a MTTKRP of any mode sizes is cut into workgroups (mttkrp_any.hip); host
// code only but for the two constants that the kernels share.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "grid_limit.h"

namespace tla {

constexpr int kAnyWaves = 4;
constexpr int kAnySlack = 68;  // rows of the table that a slice's ends may add

// rows per lane of one visit of any_last_kernel
constexpr int any_last_rows(int TN, int RT) { return TN > 1 || RT > 1 ? 4 : 8; }
// Waves per SIMD that a kernel's registers are cut for: two sets of loaded
// values, the factor rows, the accumulators and some 40 for addresses.
constexpr int any_occ(int TN, int RT, bool last, bool f64) {
  const int d = f64 ? 2 : 1;
  const int nr = any_last_rows(TN, RT);
  const int regs = last ? 8 * TN * nr + 16 * TN * RT + d * RT * (nr + 2) + (RT == 4 ? 56 : 40)
                        : 16 * TN + 4 * d * TN * RT + (8 + 2 * d) * RT + (f64 ? 54 : 40);
  return regs <= 128 ? 4 : regs <= 168 ? 3 : 2;
}

struct AnyPlan {
  bool last;          // output mode is the contiguous one
  int TN, RT;         // tiles per wave (rows: 16 rows each; last: column tiles) and rank tiles of a slab
  int64_t groups;     // row groups / column groups
  int64_t slices;     // the chunks in this many launches, each with its part of the table,
  int64_t per;        // and chunks of one launch
  int64_t nblk;       // blocks per group and slice; partial sums per output element = nblk slices
  int64_t A, In, Q;   // X viewed as A x In x Q, mode In kept
  int64_t K, Pb, J;
  int nqc;            // chunks per (A, Q) row
  int64_t nchunks;    // chunks (rows) / row visits (last)
  int64_t g_rows;     // rows of the precomputed scale table (0: none)
  int64_t g_slice;    // ... of one slice, at most
  bool build_g;       // the table has to be built (else it is a factor itself, or absent)
  bool direct_g;      // ... but its rows are formed in the kernel
  size_t ws_bytes;
  bool vector;        // the vector kernel (a workgroup per output row and 16 ranks) takes less
};

// Whether the vector kernel takes less, which needs no table, no sum of partials
// and no second slab: few contracted indices q per output row, many short modes,
// ranks above 64.  Both estimated in us from 954 calls of 2^4 to 2^19 entries,
// orders 2 to 6, ranks 1 to 130 (the median of either within a tenth): the
// vector kernel's passes of 256 q, times order and ranks, in rounds of 512
// workgroups (256 where that is all a matrix product); launches, chunks per wave, and a chunk's scale rows (formed in the
// kernel, GD, or read; one by one where the inner mode is shorter than a lane's
// values).  Measured, vector / matrix, GPU time: 4 x 2 x 2 x 2 x 2 x 7, rank 100, mode 3: 14 / 133
// us; 16 x 50 x 3, rank 65, mode 1: 11 / 53; 26 x 24 x 8, rank 3, mode 1: 8 / 6;
// 14 x 27 x 5 x 5, rank 64, mode 2: 55 / 20.
inline bool any_vector_wins(const AnyPlan& p, bool f64, int ndim, int R, bool weights) {
  const int Rs = R < 64 ? R : 64, slabs = (R + 63) / 64;
  const double passes = double((p.A * p.Q + 255) / 256), blocks = double(p.In) * ((R + 15) / 16);
  const double vector = 6 + passes * ndim * (0.3 + 0.065 * std::min(R, 16)) * std::max(1.0, blocks / (ndim == 2 ? 256 : 512));
  const int NR = p.last ? any_last_rows(p.TN, p.RT) : f64 ? 4 : 8;
  const bool table = p.build_g && !p.direct_g;
  const int64_t sets = p.nblk * p.slices;
  const double launches = (!table ? 0 : p.slices == 1 ? 1 : p.slices * slabs) + slabs * (p.slices + (sets > 1 || R > 64 ? 1 : 0));
  const double visits = double((p.per + kAnyWaves * p.nblk - 1) / (kAnyWaves * p.nblk)) * p.slices * slabs;
  const double scales = double((Rs + 15) / 16) * ((p.last ? p.J : p.K) < NR ? NR : 2);
  const double matrix = 3.1 * launches + visits * (0.93 + 0.0165 * p.RT * NR +
                        (p.direct_g ? 0.099 * scales * (ndim - 2 + weights) : p.g_rows > 0 ? 0.041 * scales : 0.0));
  return vector < 0.95 * matrix;
}

inline size_t any_align(size_t b) { return (b + 255) & ~size_t(255); }

// Fills *p and returns true when the kernels take this contraction.
inline bool any_plan(bool f64, int ndim, const int64_t* shape, int R, int mode, bool weights, AnyPlan* p) {
  *p = AnyPlan{};
  const int V = f64 ? 2 : 4, sz = f64 ? 8 : 4;
  int64_t total = 1;  // (no product below overflows)
  for (int m = 0; m < ndim; ++m) {
    if (shape[m] > (int64_t(1) << 40) / total) return false;
    total *= shape[m];
  }
  const int Rs = std::min(R, 64);
  p->RT = (Rs + 15) / 16;
  p->last = mode == ndim - 1;
  p->K = shape[ndim - 1];
  p->In = shape[mode];
  p->A = 1;
  p->Q = 1;
  for (int m = 0; m < mode; ++m) p->A *= shape[m];
  for (int m = mode + 1; m < ndim; ++m) p->Q *= shape[m];
  // the kernels' 32-bit indices: q or p, an element of a factor or of the
  // scale rows of one a, a byte within the rows of a wave's tiles
  constexpr int64_t kBig = 0x7fffff00;
  for (int m = 0; m < ndim; ++m)
    if (shape[m] > kBig / (R * sz)) return false;
  int64_t tiles;
  int most;  // tiles per wave that the registers hold
  if (p->last) {
    if (p->K < V) return false;
    p->J = shape[ndim - 2];
    p->g_rows = p->A / p->J;
    if (p->A > kBig || p->g_rows > kBig / (R * sz) || p->K > kBig / (32 * sz)) return false;
    tiles = (p->K + 16 * V - 1) / (16 * V);
    most = p->RT == 1 ? 3 : 1;  // (two tiles of two rank tiles halve the waves: never less)
  } else {
    p->Pb = p->Q / p->K;
    if (p->Q > kBig / (32 * sz) || p->Pb > kBig / (R * sz)) return false;
    p->g_rows = p->A * p->Pb;
    p->nqc = (int)((p->Q + 8 * V - 1) / (8 * V));
    tiles = (p->In + 15) / 16;
    most = !f64 || p->RT <= 2 ? 4 : p->RT == 3 ? 3 : 2;
  }
  if (ndim == 2) p->g_rows = 0;
  // Tiles per wave: every wave forms its part of B once for all its tiles
  // (about the cost of one more tile), and the chunks are dealt to the waves
  // that fit the GPU at once in equal numbers, at least the four of one
  // workgroup per group: the least sum over a wave's chunks, times the rounds
  // that the groups of a long mode take, wins.  Tiles per wave against one,
  // long mode: 200000 x 30 x 41, float32, rank 32 / 64: 253 / 389 us with
  // several, 286 / 456 with one; 100000 x 33 x 35, rank 20: 125, 139, and float64
  // 252, 307; 5 x 9 x 500001, rank 8: 34, 42.
  int64_t best = -1;
  for (int tn = most; tn >= 1; --tn) {
    const int64_t groups = (tiles + tn - 1) / tn;
    const int TN = (int)((tiles + groups - 1) / groups);
    const int RV = 4 * any_last_rows(TN, p->RT);
    const int64_t chunks = p->last ? (p->A + RV - 1) / RV : p->A * p->nqc;
    const int64_t slots = 256 * 4 * any_occ(TN, p->RT, p->last, f64);
    const int64_t waves = std::max<int64_t>(kAnyWaves, slots / groups);
    const int64_t per = (chunks + waves - 1) / waves;
    const int64_t rounds = (groups * waves + slots - 1) / slots;
    const int64_t cost = per * rounds * (TN + 1) * (p->last ? RV : 16);
    // (over several rounds the sharing of two and more rank tiles gives a
    // little more than this counts: fewer tiles have to win by a seventh)
    if (best >= 0 && cost >= (rounds > 1 && p->RT > 1 ? best - best / 7 : best)) continue;
    best = cost;
    p->TN = TN;
    p->groups = groups;
    p->nchunks = chunks;
    p->nblk = (chunks + kAnyWaves * per - 1) / (kAnyWaves * per);
  }
  // the table is a factor as it is when it covers one mode and no weights
  p->build_g = p->g_rows > 0 && !(ndim == 3 && !weights);
  // Small problems are short of launches, not of work: up to 24 chunks, a few
  // per wave, one workgroup per group writes the output itself (5 us, where
  // the sum of partials is another launch of 3 us on the host and 2.5 us on
  // the GPU); up to 1024 chunks, a fraction of the GPU's waves, the scale
  // rows are formed in place of a table (one launch of 3 us).
  p->direct_g = p->build_g && p->TN == 1 && p->nchunks * p->groups <= 1024 && p->g_rows <= kBig;
  if (p->nchunks <= 24) p->nblk = 1;
  // The table holds at most 256 MiB, so that the scratch does not grow with
  // the tensor (where output and contiguous mode are both short a whole table
  // would be larger than the tensor): the chunks are taken in slices, each
  // with its own rows of the table.  4096 x 1024 x 4 x 6 (384 MiB), rank 64,
  // modes 2 / 3: 6.40 / 2.12 ms in four slices, 6.32 / 2.06 with the whole
  // table of 1 GiB; the rows formed in every wave instead 17.2 / 3.02 ms.
  p->slices = 1;
  p->per = p->nchunks;
  p->g_slice = p->g_rows;
  const int64_t most_rows = (int64_t(256) << 20) / (R * sz);
  if (p->build_g && !p->direct_g && p->g_rows > most_rows) {
    const int64_t span = p->last ? 4 * any_last_rows(p->TN, p->RT) : 8 * V;  // p or q of a chunk
    const int64_t inner = p->last ? p->J : p->K;                            // ... that share a row
    if (!p->last && p->Pb < most_rows) {  // whole a
      const int64_t as = most_rows / p->Pb;
      p->slices = (p->A + as - 1) / as;
      const int64_t even = (p->A + p->slices - 1) / p->slices;
      p->per = even * p->nqc;
      p->g_slice = even * p->Pb;
    } else {
      const int64_t cs = std::max<int64_t>(1, (most_rows - kAnySlack) * inner / span);
      p->slices = (p->nchunks + cs - 1) / cs;
      p->per = (p->nchunks + p->slices - 1) / p->slices;
      p->g_slice = p->per * span / inner + kAnySlack;
    }
    p->nblk = std::min(p->nblk, (p->per + kAnyWaves - 1) / kAnyWaves);
  }
  // at most 32 MiB of partial sums beside it (one set: written to the output)
  const int64_t set = p->In * Rs * sz;
  p->nblk = std::max<int64_t>(1, std::min<int64_t>(p->nblk, (int64_t(32) << 20) / set / p->slices));
  const int64_t sets = p->nblk * p->slices;
  if (!grid_fits(p->groups * p->nblk, 64 * kAnyWaves) || !grid_fits((p->In * Rs + 31) / 32 + 1, 256)) return false;
  p->ws_bytes = (p->build_g && !p->direct_g ? any_align(size_t(p->g_slice) * R * sz) : 0) +
                (sets > 1 || R > 64 ? any_align(size_t(sets) * set) : 0);
  p->vector = any_vector_wins(*p, f64, ndim, R, weights);
  return true;
}

}  // namespace tla
