// Mode Gram: G[i, j] = sum_{a,b} X[a, i, b] X[a, j, b], the rows' Gram matrix
// of unfold(X, mode) in float64 without forming the unfolding.
//
// A block computes one 32 x 32 tile (ti <= tj) of G for one chunk of the
// columns (a, b), the partial tiles are summed in chunk order.  The blocks of
// one chunk run on one XCD (chunks vary fastest in the grid, a multiple of
// eight of them where there are that many), so its L2 holds what they share.
//
//  * mode_gram_rows_kernel (b of 14 or more): each of the four waves takes a
//    quarter of the chunk's 16-column pieces and loads the tile's rows as
//    they lie, 16 bytes per lane, straight into the operands of 2 x 2 matrix
//    tiles; the two operands order the columns alike, so any order will do.
//  * mode_gram_last_kernel (the contiguous mode): two consecutive rows i per
//    lane and column, so a column's 32 rows are one piece of memory.
//  * mode_gram_short_kernel (runs of 2 to 13 and 17 to 24 columns b, where the pieces would
//    be padding; 512 x 512 x 8, mode 1: 66 us against 108 of the pieces, x 12:
//    90 against 97, x 15: 117 against 103): column by column through LDS, one
//    matrix tile per wave.
//
// Bound: the float64 matrix rate (products of float32 are exact there).
// Measured, 256^3 float32, modes 0 / 1 / 2: 112 / 114 / 107 us (43 TFLOP/s of the 72 that a
// large product reaches, the upper triangle's tiles counted); all through LDS, a matrix
// tile per two operand reads and 32 or 4 contiguous bytes per load, 224 / 224 /
// 512 us.
#include <algorithm>

#include "mma_any.h"

namespace tla {

constexpr int kGramWaves = 4;

// Tile (ti, tj), ti <= tj, of an index counted row by row of the upper triangle.
__device__ __forceinline__ void gram_tile(int t, int nt, int& ti, int& tj) {
  ti = 0;
  for (; t >= nt - ti; ++ti) t -= nt - ti;
  tj = ti + t;
}

// The waves' sums of a tile to its place and its mirror's; element (r, c) of
// the tile is G[row(r)][col(c)].
template <typename Row, typename Col>
__device__ __forceinline__ void gram_store(doublex4 (&acc)[4], double* red, double* out, int64_t In, int64_t i1,
                                           int64_t j1, int wave, int lane, Row row, Col col) {
  any_block_sum<double, 4, kGramWaves>(acc, red, wave, lane);
  // wave w: matrix tile (w / 2, w % 2)
  const int lr = lane & 15, lk = lane >> 4, ta = wave >> 1, tb = wave & 1;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t i = row(lk + 4 * e, ta), j = col(lr, tb);
    if (i < i1 && j < j1) {
      const double v = red[((ta * 2 + tb) * 4 + e) * 64 + lane];
      out[i * In + j] = v;
      out[j * In + i] = v;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(64 * kGramWaves, sizeof(T) == 4 ? 4 : 3) void mode_gram_rows_kernel(const T* __restrict__ X, int64_t Pa,
                                                                            int64_t In, int64_t Pb, int64_t chunk,
                                                                            double* __restrict__ partial) {
  using V = typename AnyT<T>::vec;
  constexpr int VL = AnyT<T>::V, NL = 4 / VL;
  __shared__ double red[4 * 256];
  int ti, tj;
  gram_tile(blockIdx.y, (int)((In + 31) / 32), ti, tj);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t i0 = (int64_t)ti * 32, j0 = (int64_t)tj * 32;
  // columns 4 g, ... of the piece, rows c and 16 + c of the tile (the last row
  // again past the end)
  uint32_t off[4];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    off[t] = (uint32_t)((min(i0 + 16 * t + c, In - 1) * Pb - i0 * Pb + 4 * g) * sizeof(T));
    off[2 + t] = (uint32_t)((min(j0 + 16 * t + c, In - 1) * Pb - j0 * Pb + 4 * g) * sizeof(T));
  }
  const int64_t nb = (Pb + 15) / 16, pieces = Pa * nb;
  const int64_t p1 = min(pieces, ((int64_t)blockIdx.x + 1) * chunk);
  int64_t p = (int64_t)blockIdx.x * chunk + wave;
  int64_t a = p / nb, ib = p - a * nb;
  doublex4 acc[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) acc[n] = doublex4{0, 0, 0, 0};
  // loads piece (a, ib) and steps to the wave's next
  auto load = [&](T (&x)[4][4]) {
    const T* xa = X + (a * In + i0) * Pb + 16 * ib;
    const T* xb = X + (a * In + j0) * Pb + 16 * ib;
    if (16 * ib + 16 <= Pb) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int h = 0; h < NL; ++h) {
          const V v = at<V>((t < 2 ? xa : xb) + h * VL, off[t]);
#pragma unroll
          for (int u = 0; u < VL; ++u) x[t][h * VL + u] = v[u];
        }
    } else {
      const int left = (int)(Pb - 16 * ib) - 4 * g;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) x[t][u] = u < left ? at<T>((t < 2 ? xa : xb) + u, off[t]) : (T)0;
    }
    ib += kGramWaves;
    while (ib >= nb) { ib -= nb; ++a; }
  };
  auto visit = [&](T (&x)[4][4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[2 * s + t] = AnyT<double>::mma((double)x[s][u], (double)x[2 + t][u], acc[2 * s + t]);
  };
  T x0[4][4], x1[4][4];
  if (p < p1) load(x0);
  while (p < p1) {
    p += kGramWaves;
    if (p < p1) load(x1);
    visit(x0);
    if (p >= p1) break;
    p += kGramWaves;
    if (p < p1) load(x0);
    visit(x1);
  }
  gram_store(acc, red, partial + (int64_t)blockIdx.x * In * In, In, In, In, wave, lane,
             [=](int r, int t) { return i0 + 16 * t + r; }, [=](int r, int t) { return j0 + 16 * t + r; });
}

template <typename T>
__global__ __launch_bounds__(64 * kGramWaves, 3) void mode_gram_last_kernel(const T* __restrict__ X, int64_t Q,
                                                                            int64_t In, int64_t chunk,
                                                                            double* __restrict__ partial) {
  typedef T V __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  __shared__ double red[4 * 256];
  int ti, tj;
  gram_tile(blockIdx.y, (int)((In + 31) / 32), ti, tj);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  // rows 2 c and 2 c + 1 of the tile (the last two again past the end),
  // column g of four
  auto row = [=](int r, int t) { return min((int64_t)ti * 32 + 2 * r, In - 2) + t; };
  auto col = [=](int r, int t) { return min((int64_t)tj * 32 + 2 * r, In - 2) + t; };
  const uint32_t offa = (uint32_t)((g * In + row(c, 0)) * sizeof(T)), offb = (uint32_t)((g * In + col(c, 0)) * sizeof(T));
  const int64_t p1 = min((Q + 15) / 16, ((int64_t)blockIdx.x + 1) * chunk);
  int64_t p = (int64_t)blockIdx.x * chunk + wave;
  doublex4 acc[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) acc[n] = doublex4{0, 0, 0, 0};
  auto load = [&](int64_t at_piece, V (&x)[4], V (&y)[4]) {
    const T* xb = X + at_piece * 16 * In;
    if (at_piece * 16 + 16 <= Q) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[u] = at<V>(xb + 4 * u * In, offa);
        y[u] = at<V>(xb + 4 * u * In, offb);
      }
    } else {
      const int left = (int)(Q - at_piece * 16) - g;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[u] = y[u] = V{0, 0};
        if (4 * u < left) {
          x[u] = at<V>(xb + 4 * u * In, offa);
          y[u] = at<V>(xb + 4 * u * In, offb);
        }
      }
    }
  };
  auto visit = [&](V (&x)[4], V (&y)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[2 * s + t] = AnyT<double>::mma((double)x[u][s], (double)y[u][t], acc[2 * s + t]);
  };
  V x0[4], x1[4], y0[4], y1[4];
  if (p < p1) load(p, x0, y0);
  while (p < p1) {
    p += kGramWaves;
    if (p < p1) load(p, x1, y1);
    visit(x0, y0);
    if (p >= p1) break;
    p += kGramWaves;
    if (p < p1) load(p, x0, y0);
    visit(x1, y1);
  }
  gram_store(acc, red, partial + (int64_t)blockIdx.x * In * In, In, In, In, wave, lane, row, col);
}

// Tile (blockIdx.x, blockIdx.y) of one chunk: four waves, one 16 x 16 matrix
// tile each, 64 columns at a time.
template <typename T>
__global__ __launch_bounds__(256) void mode_gram_short_kernel(const T* __restrict__ X, int64_t Pa, int64_t In, int64_t Pb,
                                                        int64_t chunk, double* __restrict__ partial) {
  __shared__ double Ti[32][65];
  __shared__ double Tj[32][65];
  const int ti = blockIdx.x, tj = blockIdx.y;
  if (tj < ti) return;
  const int tid = threadIdx.x;
  const int64_t q0 = (int64_t)blockIdx.z * chunk;
  const int64_t Q = Pa * Pb;
  const int64_t q1 = min(Q, q0 + chunk);
  const int wave = tid >> 6, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int mi = (wave >> 1) * 16, nj = (wave & 1) * 16;
  doublex4 acc = doublex4{0.0, 0.0, 0.0, 0.0};
  // thread: column qq of the 64-wide chunk, rows r0, r0 + 4, ..., r0 + 28 of
  // both 32-row blocks; the chunk after the current one is loaded into
  // registers while the current one is multiplied
  const int qq = tid & 63, r0 = tid >> 6;
  T ci[8], cj[8];
  auto fetch = [&](int64_t qb) {
    const int64_t q = qb + qq;
    int64_t base = -1;
    if (q < q1) {
      const int64_t aa = q / Pb;
      base = aa * In * Pb + (q - aa * Pb);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t gi = (int64_t)ti * 32 + r0 + 4 * u, gj = (int64_t)tj * 32 + r0 + 4 * u;
      ci[u] = (base >= 0 && gi < In) ? X[base + gi * Pb] : (T)0;
      cj[u] = (base >= 0 && gj < In) ? X[base + gj * Pb] : (T)0;
    }
  };
  if (q0 < q1) fetch(q0);
  for (int64_t qb = q0; qb < q1; qb += 64) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      Ti[r0 + 4 * u][qq] = (double)ci[u];
      Tj[r0 + 4 * u][qq] = (double)cj[u];
    }
    __syncthreads();
    if (qb + 64 < q1) fetch(qb + 64);
    // wave w: the 16 x 16 output tile (w / 2, w % 2) of the 32 x 32 block on
    // FP64 MFMA (products of the float inputs are exact in FP64)
#pragma unroll
    for (int k0 = 0; k0 < 64; k0 += 4)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(Ti[mi + lr][k0 + lk], Tj[nj + lr][k0 + lk], acc, 0, 0, 0);
    __syncthreads();
  }
  double* out = partial + (int64_t)blockIdx.z * In * In;
  // lane holds D[lk + 4 e][lr]
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t i = (int64_t)ti * 32 + mi + lk + 4 * e, j = (int64_t)tj * 32 + nj + lr;
    if (i < In && j < In) {
      out[i * In + j] = acc[e];
      out[j * In + i] = acc[e];
    }
  }
}

// Partial sums of 32 elements per block: eight threads each take every eighth
// chunk, and their sums are added in order.
__global__ __launch_bounds__(256) void sum_gram_partials_kernel(const double* __restrict__ partial, int64_t nn,
                                                                int splits, double* __restrict__ G) {
  __shared__ double part[8][32];
  const int col = threadIdx.x & 31, row = threadIdx.x >> 5;
  const int64_t e = (int64_t)blockIdx.x * 32 + col;
  double s = 0.0;
  if (e < nn)
    for (int k = row; k < splits; k += 8) s += partial[(int64_t)k * nn + e];
  part[row][col] = s;
  __syncthreads();
  if (row == 0 && e < nn) {
#pragma unroll
    for (int r = 1; r < 8; ++r) s += part[r][col];
    G[e] = s;
  }
}

// How the work of a mode is split: which kernel, the chunks, and the columns
// (short) or 16-column pieces (the others) of a chunk.
struct GramPlan {
  enum Kind { Short, Rows, Last } kind;
  int64_t chunk;
  int splits;
};

static GramPlan gram_plan(bool f64, int64_t Pa, int64_t In, int64_t Pb) {
  const int64_t Q = Pa * Pb, nt = (In + 31) / 32, tiles = nt * (nt + 1) / 2;
  GramPlan p;
  // 32-bit offsets: the bytes of a tile's 32 rows, or of four columns
  constexpr int64_t kBig = 0x7fffff00;
  // Runs of 17 to 24 columns leave a second piece that is mostly padding (300 rows,
  // float32, 17 / 20 / 24 columns: 42 / 39 / 36 us, short 34 / 32 / 33; from 25 on,
  // float64 from 22, and for 64 rows the pieces win).  Float64 rows that begin off the 16-byte grid: past some 90 MB
  // the pieces' loads fetch too many lines twice (3000 x 4001 / 3 x 3000 x 2049:
  // 1118 / 2222 us, short 996 / 1568; 2048 x 4001: 543, short 594).
  const bool padded = In >= 200 && Pb >= 17 && Pb <= (f64 ? 21 : 24);
  const bool astray = f64 && Pb % 2 != 0 && tiles >= 2048 && Q > (int64_t(90) << 20) / 8 / In;
  if (Pb == 1 && In >= 2 && In <= kBig / 64 && tiles <= 65535) p.kind = GramPlan::Last;
  else if (!padded && !astray && Pb >= 14 && Pb <= kBig / (33 * 8) && tiles <= 65535) p.kind = GramPlan::Rows;
  else p.kind = GramPlan::Short;
  if (p.kind == GramPlan::Short) {
    int64_t s = std::max<int64_t>(1, 1024 / std::max<int64_t>(tiles, 1));
    s = std::min<int64_t>(s, (Q + 63) / 64);
    p.splits = (int)std::max<int64_t>(1, std::min<int64_t>(s, 64));
    p.chunk = ((Q + p.splits - 1) / p.splits + 63) / 64 * 64;
    return p;
  }
  // blocks of at least eight pieces (two per wave), in eights where there are
  // that many.  About two per CU, as each adds a partial tile to write and
  // sum (1000 x 1000: 36 us, with eight per CU 46), but eight where that
  // leaves a block 64 pieces, for an even finish (256^3 123-133 -> 107-114 us,
  // 512^3 1.9 -> 1.5 ms), or three (what float64 keeps in flight) where it leaves
  // 60 (3 x 600 x 2049: 90 -> 66 us, float32 76 -> 62; with 48, 120 x 512 x 26: 50 ->
  // 56), but in the contiguous mode (157 x 60 x 514 float64: 80 -> 90).  At most
  // 128: their sum is a serial chain.
  const int64_t pieces = p.kind == GramPlan::Last ? (Q + 15) / 16 : Pa * ((Pb + 15) / 16);
  const int64_t nt1 = std::max<int64_t>(tiles, 1);
  const int64_t blocks = pieces / 64 >= 2048 / nt1 ? 2048
                         : p.kind == GramPlan::Rows && pieces / 60 >= 768 / nt1 ? 768 : 576;
  int64_t s = std::min<int64_t>({(pieces + 7) / 8, std::max<int64_t>(1, blocks / nt1), 128});
  if (s > 8) s = s / 8 * 8;
  p.splits = (int)std::max<int64_t>(1, s);
  p.chunk = (pieces + p.splits - 1) / p.splits;
  return p;
}

static void gram_sizes(int ndim, const int64_t* shape, int mode, int64_t& Pa, int64_t& In, int64_t& Pb) {
  Pa = Pb = 1;
  for (int m = 0; m < mode; ++m) Pa *= shape[m];
  for (int m = mode + 1; m < ndim; ++m) Pb *= shape[m];
  In = shape[mode];
}

template <typename T>
static void gram_run(const GramPlan& p, const T* X, int64_t Pa, int64_t In, int64_t Pb, double* out, hipStream_t st) {
  const int nt = (int)ceil_div(In, 32);
  const dim3 grid(p.splits, nt * (nt + 1) / 2);
  if (p.kind == GramPlan::Rows)
    mode_gram_rows_kernel<T><<<grid, 64 * kGramWaves, 0, st>>>(X, Pa, In, Pb, p.chunk, out);
  else if (p.kind == GramPlan::Last)
    mode_gram_last_kernel<T><<<grid, 64 * kGramWaves, 0, st>>>(X, Pa, In, p.chunk, out);
  else
    mode_gram_short_kernel<T><<<dim3(nt, nt, p.splits), 256, 0, st>>>(X, Pa, In, Pb, p.chunk, out);
}

}  // namespace tla

using namespace tla;

extern "C" size_t tla_mode_gram64_workspace_size(int ndim, const int64_t* shape, int mode) {
  if (mode < 0 || mode >= ndim) return 0;
  int64_t Pa, In, Pb;
  gram_sizes(ndim, shape, mode, Pa, In, Pb);
  const int splits = std::max(gram_plan(false, Pa, In, Pb).splits, gram_plan(true, Pa, In, Pb).splits);
  return (size_t(splits) * In * In * 8 + 255) & ~size_t(255);
}

extern "C" int tla_mode_gram64(int dtype, const void* X, int ndim, const int64_t* shape, int mode, double* G,
                               void* ws, size_t ws_bytes, void* stream) {
  TLA_REQUIRE(dtype == TLA_F32 || dtype == TLA_F64, "mode_gram64: bad dtype %d", dtype);
  TLA_REQUIRE(ndim >= 1 && ndim <= kMaxOrder && mode >= 0 && mode < ndim, "mode_gram64: bad mode");
  TLA_REQUIRE(ws_bytes >= tla_mode_gram64_workspace_size(ndim, shape, mode), "mode_gram64: workspace too small");
  int64_t Pa, In, Pb;
  gram_sizes(ndim, shape, mode, Pa, In, Pb);
  const GramPlan p = gram_plan(dtype == TLA_F64, Pa, In, Pb);
  hipStream_t st = (hipStream_t)stream;
  // one chunk is the result itself
  double* out = p.splits == 1 ? G : (double*)ws;
  if (dtype == TLA_F32) gram_run(p, (const float*)X, Pa, In, Pb, out, st);
  else gram_run(p, (const double*)X, Pa, In, Pb, out, st);
  TLA_LAUNCH_CHECK();
  if (p.splits > 1) {
    const int64_t nn = In * In;
    sum_gram_partials_kernel<<<ceil_div(nn, 32), 256, 0, st>>>((double*)ws, nn, p.splits, G);
    TLA_LAUNCH_CHECK();
  }
  return TLA_OK;
}
