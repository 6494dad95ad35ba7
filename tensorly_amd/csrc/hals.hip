// HALS non-negative least squares of one CP factor.
#include <math.h>

#include <algorithm>

#include "common.h"
#include "inverse.h"

namespace tla {

// ---------------------------------------------------------------------------
// HALS non-negative least squares for one CP factor (tensorly/solvers/
// nnls.py:5-173 as called by non_negative_parafac_hals, _nn_cp.py:300-311):
// UtU = (Hadamard of the other modes' Grams) * w w^T, UtM = M^T, V = A^T.
// Each iteration updates the rows k = 0..R-1 of V in order (Gauss-Seidel),
//   V[k,:] <- max((UtM[k,:] - UtU[k,:] V + UtU[k,k] V[k,:] - s) / UtU[k,k], 0)
// and stops when the iteration's error sum is below tol times the first
// iteration's; as in the reference (nnls.py:147, ||V - newV||^2 with the new
// row broadcast against all of V) each row update adds
// sum_{j < R} (V[j, i] - newV[i])^2 over the columns i.  The columns of V
// (rows of A) are independent within an iteration.  Long runs (exact mode) and
// callers without a workspace use one workgroup, each thread keeping its
// rows' values in registers for the R updates; the squared update is summed
// in a fixed order.
// ---------------------------------------------------------------------------
struct HalsArgs {
  const double* grams[kMaxOrder];
  int ndim, mode, R;
  const void* weights;
  int wdt;
  const void* M;
  void* A;
  int64_t rows;
  double sparsity;
  int has_sparsity;
  int n_iter_max;
  double tol;
  int* iters_out;
};

constexpr int kHalsThreads = 512;

template <typename T, int RT>
__global__ __launch_bounds__(kHalsThreads) void hals_nnls_kernel(HalsArgs a) {
  __shared__ double utu[RT * RT];
  __shared__ double acc[kMaxRank * kMaxRank];
  __shared__ double red[kHalsThreads / 64];
  __shared__ int stop;
  const int R = a.R, tid = threadIdx.x;
  build_v(a, a.ndim, a.mode, -1, nullptr, a.weights, a.wdt, 0.0, R, acc);
  for (int e = tid; e < RT * RT; e += blockDim.x) {
    const int k = e / RT, l = e % RT;
    utu[e] = (k < R && l < R) ? acc[k * R + l] : 0.0;
  }
  __syncthreads();
  T* A = (T*)a.A;
  const T* M = (const T*)a.M;
  double err0 = 0.0;
  int it = 0;
  for (; it < a.n_iter_max; ++it) {
    double err = 0.0;
    for (int64_t i = tid; i < a.rows; i += blockDim.x) {
      // UtU is loop-invariant; an opaque copy of its address per row keeps
      // the compiler from holding all RT * RT values in registers
      const double* U = utu;
      asm volatile("" : "+v"(U));
      // at RT = 64 the MTTKRP row is read per update (v and m together would
      // need every register)
      constexpr bool kMRegs = RT <= 48;
      double v[RT], m[kMRegs ? RT : 1];
#pragma unroll
      for (int l = 0; l < RT; ++l) {
        v[l] = l < R ? (double)A[i * R + l] : 0.0;
        if constexpr (kMRegs) m[l] = l < R ? (double)M[i * R + l] : 0.0;
      }
#pragma unroll
      for (int k = 0; k < RT; ++k) {
        const double d = U[k * RT + k];
        if (d != 0.0) {
          double dot = 0.0;
#pragma unroll
          for (int l = 0; l < RT; ++l) dot = fma(U[k * RT + l], v[l], dot);
          double mk;
          if constexpr (kMRegs) mk = m[k];
          else mk = (double)M[i * R + k];  // d != 0 only for k < R
          double num = mk - dot + d * v[k];
          if (a.has_sparsity) num -= a.sparsity;
          const double nv = fmax(num / d, 0.0);
          // the stopping sum subtracts the new value from every entry of
          // this column of V (the reference's broadcast ||V - newV||^2)
#pragma unroll
          for (int l = 0; l < RT; ++l)
            if (l < R) {
              const double df = v[l] - nv;
              err = fma(df, df, err);
            }
          v[k] = nv;
        }
      }
#pragma unroll
      for (int l = 0; l < RT; ++l)
        if (l < R) A[i * R + l] = (T)v[l];
    }
    err = wave_sum(err);
    if ((tid & 63) == 0) red[tid >> 6] = err;
    __syncthreads();
    if (tid == 0) {
      double s = 0.0;
      for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
      if (it == 0) red[0] = s, err0 = s;
      stop = (s < a.tol * (it == 0 ? s : err0)) ? 1 : 0;
    }
    __syncthreads();
    const bool done = stop != 0;
    __syncthreads();
    if (done) {
      ++it;
      break;
    }
  }
  if (tid == 0 && a.iters_out) *a.iters_out = it;
}


// HALS over the whole GPU.  The rows of A do not depend on one another but
// for the stopping rule, so every row runs a chunk of iterations in one
// launch without looking at the others and leaves each iteration's error sum
// behind; one workgroup then finds the iteration at which the rule fires, if
// any, and the last launch replays the chunk up to it from the values the
// chunk began with.
//
// Four lanes share a row, lane q holding columns q E .. q E + E - 1 of V and
// of the gradient U V - M in registers.  An update then is a chain of one
// multiply-add, one maximum, a broadcast among the four lanes and one
// multiply-add into the next column's gradient, where a dot product per
// update is a chain of R multiply-adds.  The gradient is formed afresh every
// kHalsRefresh iterations, and in each of the first four: from a start far
// above the solution it falls by orders of magnitude there, and would keep
// the rounding of its first size (a start 200 times too large, rank 64, two
// iterations: 6e-12 of the largest entry, now below 1e-12).  Bound: with few rows on the GPU an
// update costs its chain of dependent FP64 operations, some 25 ns, and the issue
// of the lane's E columns, some 8 ns each (57 ns at rank 16, 155 at rank 64).
// 256 rows, rank 16, 100 iterations take 92 us and 96 us with the decision and
// the last launch (one launch per iteration, a thread per row and a dot
// product per update: 1362 us); 512 rows, rank 64: 1011 us in two chunks
// (16.2 ms).
constexpr int kHalsRows = 16;     // rows per workgroup of one wave
constexpr int kHalsChunk = 128;   // iterations per launch, at most
constexpr int kHalsBlocks = 65536;  // workgroups, at most: more rows take turns
constexpr int kHalsSums = 256;      // sets that more than 1024 workgroups' error sums are added up to
constexpr int kHalsRefresh = 8;

// state: [0] the rule fired, [1] iterations run, [2] chunk in which it fired,
// [3] iterations of that chunk.
struct HalsRun {
  HalsArgs a;
  double* vbuf[2];   // rows x R FP64: V after the odd / even chunks
  double* partial;   // [workgroup][iteration of the chunk]
  double* sums;      // [kHalsSums][iteration of the chunk]
  int* state;
  double* err0;
  int chunk, iters;  // this chunk and its iterations
  int begin;         // iterations before it
  int final, only;   // the last launch; the only one (one iteration)
  int nblk;          // workgroups, each every nblk-th group of rows
};

template <int Q>
__device__ __forceinline__ double quad_bcast(double v) {
  constexpr int ctrl = Q * 0x55;  // quad_perm [Q, Q, Q, Q]
  const int2 w = *(const int2*)&v;
  int2 r;
  r.x = __builtin_amdgcn_mov_dpp(w.x, ctrl, 0xf, 0xf, true);
  r.y = __builtin_amdgcn_mov_dpp(w.y, ctrl, 0xf, 0xf, true);
  return *(const double*)&r;
}
__device__ __forceinline__ double quad_get(double v, int q) {
  return q == 0 ? quad_bcast<0>(v) : q == 1 ? quad_bcast<1>(v) : q == 2 ? quad_bcast<2>(v) : quad_bcast<3>(v);
}

// h.final: replays the chunk in which the rule fired (state), or takes the
// last chunk's values, and writes the factor.
// FULL: R == RT.  LOOP: more groups of rows than workgroups.
template <typename T, int RT, bool FULL, bool LOOP>
__global__ __launch_bounds__(64) void hals_run_kernel(HalsRun h) {
  constexpr int E = RT / 4;
  __shared__ double U[RT * RT];  // zero outside R x R
  __shared__ double rd[RT];      // 1 / U[k][k], 0 where the column is skipped
  __shared__ double errs[16 * 65];
  const HalsArgs& a = h.a;
  const int lane = threadIdx.x, q = lane & 3, R = a.R;
  int chunk = h.chunk, iters = h.iters;
  if (h.final) {
    if (h.only) {  // one iteration: it runs whatever the rule says
      if (blockIdx.x == 0 && lane == 0) h.state[1] = iters;
    } else if (h.state[0]) {
      chunk = h.state[2];
      iters = h.state[3];
    } else {
      ++chunk;  // the values after the last chunk
      iters = 0;
    }
  } else if (h.state[0] && chunk > 0) {
    return;
  }
  T* A = (T*)a.A;
  const T* M = (const T*)a.M;
  const double* src = h.vbuf[chunk & 1];
  if (iters > 0) {
    // (16 loads of a Gram in flight)
    constexpr int NU = RT * RT / 64 > 0 ? RT * RT / 64 : 1, NB = NU < 16 ? NU : 16;
#pragma unroll 1
    for (int b = 0; b < (RT * RT + 64 * NB - 1) / (64 * NB); ++b) {
      double u[NB], w[NB];
      int at[NB];
#pragma unroll
      for (int x = 0; x < NB; ++x) {
        const int e = (b * NB + x) * 64 + lane, k = e / RT, l = e % RT;
        at[x] = k < R && l < R ? k * R + l : -1;
        u[x] = at[x] >= 0 ? 1.0 : 0.0;
      }
      for (int n = 0; n < a.ndim; ++n)
        if (n != a.mode) {
          const double* G = a.grams[n];
#pragma unroll
          for (int x = 0; x < NB; ++x) w[x] = at[x] >= 0 ? G[at[x]] : 0.0;
#pragma unroll
          for (int x = 0; x < NB; ++x) u[x] *= w[x];
        }
#pragma unroll
      for (int x = 0; x < NB; ++x) {
        const int e = (b * NB + x) * 64 + lane;
        if (a.weights && at[x] >= 0) u[x] *= weight_at(a.weights, a.wdt, e / RT) * weight_at(a.weights, a.wdt, e % RT);
        if (e < RT * RT) U[e] = u[x];
      }
    }
    __syncthreads();
    for (int k = lane; k < RT; k += 64) rd[k] = U[k * RT + k] != 0.0 ? 1.0 / U[k * RT + k] : 0.0;
    __syncthreads();
  }
  // this lane's part of U stays in registers up to rank 16; above, the part
  // for the next column is read while the present one is updated
  constexpr bool kReg = RT <= 16;
  double ur[kReg ? RT : 2][E], rr[kReg ? RT : 2];
  auto read_u = [&](int k, int slot) {
#pragma unroll
    for (int e = 0; e < E; ++e) ur[slot][e] = U[k * RT + q * E + e];
    rr[slot] = rd[k];
  };
  if constexpr (kReg)
    if (iters > 0) {
#pragma unroll
      for (int k = 0; k < RT; ++k) read_u(k, k);
    }
#pragma unroll 1
  for (int64_t i0 = (int64_t)blockIdx.x * kHalsRows; !LOOP || i0 < a.rows; i0 += (int64_t)h.nblk * kHalsRows) {
    const int64_t i = i0 + (lane >> 2);
    const bool live = i < a.rows;
    double v[E], m[E], g[E];
    const int64_t base = live ? i * R : 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int l = q * E + e;
      const bool on = live && l < R;
      v[e] = !on ? 0.0 : chunk == 0 ? (double)A[base + l] : src[base + l];
      m[e] = on ? (double)M[base + l] - (a.has_sparsity ? a.sparsity : 0.0) : 0.0;
    }
    int fresh = 0;  // the next iteration with a gradient formed afresh
#pragma unroll 1
    for (int it = 0; it < iters; ++it) {
      if (it == fresh) {
        fresh = chunk == 0 && it < 3 ? it + 1 : (it | (kHalsRefresh - 1)) + 1;
#pragma unroll
        for (int e = 0; e < E; ++e) g[e] = -m[e];
        if constexpr (!kReg) read_u(0, 0);
#pragma unroll
        for (int l = 0; l < RT; ++l) {
          if constexpr (!kReg) read_u((l + 1) % RT, (l + 1) & 1);
          const double vl = quad_get(v[l % E], l / E);
#pragma unroll
          for (int e = 0; e < E; ++e) g[e] = fma(ur[kReg ? l : l & 1][e], vl, g[e]);
        }
      } else if constexpr (!kReg) {
        read_u(0, 0);
      }
      double err = 0.0;
#pragma unroll
      for (int k = 0; k < RT; ++k) {
        // no branches: the whole iteration is one run of instructions.  A
        // skipped column (and the padding past R) has rr = 0.
        if constexpr (!kReg) read_u((k + 1) % RT, (k + 1) & 1);
        const double r = rr[kReg ? k : k & 1];
        const double mine = r != 0.0 ? fmax(fma(-g[k % E], r, v[k % E]), 0.0) : v[k % E];
        const double nv = quad_get(mine, k / E), dv = quad_get(mine - v[k % E], k / E);
        // the stopping sum subtracts the new value from every entry of this
        // row of A as it is before the update (the reference's broadcast
        // ||V - newV||^2)
        double s = 0.0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const double df = FULL || q * E + e < R ? v[e] - nv : 0.0;
          s = fma(df, df, s);
        }
        err += r != 0.0 ? s : 0.0;
        v[k % E] = q == k / E ? nv : v[k % E];
#pragma unroll
        for (int e = 0; e < E; ++e) g[e] = fma(ur[kReg ? k : k & 1][e], dv, g[e]);
      }
      // sixteen iterations' lane sums at a time, added up in lane order
      errs[(it & 15) * 65 + lane] = live ? err : 0.0;
      if ((it & 15) == 15 || it + 1 == iters) {
        __syncthreads();
        if (!h.final && lane <= (it & 15)) {
          double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
          for (int t = 0; t < 64; t += 4) {
            s0 += errs[lane * 65 + t];
            s1 += errs[lane * 65 + t + 1];
            s2 += errs[lane * 65 + t + 2];
            s3 += errs[lane * 65 + t + 3];
          }
          double* p = h.partial + (int64_t)blockIdx.x * kHalsChunk + (it & ~15) + lane;
          double sum = (s0 + s1) + (s2 + s3);
          if (LOOP && i0 >= (int64_t)h.nblk * kHalsRows) sum += *p;  // this workgroup's earlier rows
          *p = sum;
        }
        __syncthreads();
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int l = q * E + e;
      if (live && l < R) {
        if (h.final) A[base + l] = (T)v[e];
        else h.vbuf[(chunk + 1) & 1][base + l] = v[e];
      }
    }
    if constexpr (!LOOP) break;
  }
}

// Many workgroups' error sums: kHalsSums of every so many each, in order.
__global__ __launch_bounds__(kHalsChunk) void hals_sum_kernel(HalsRun h) {
  if (h.chunk > 0 && h.state[0]) return;
  const int it = threadIdx.x;
  if (it >= h.iters) return;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  const double* p = h.partial + it;
  int b = blockIdx.x;
  for (; b + 3 * kHalsSums < h.nblk; b += 4 * kHalsSums) {
    s0 += p[(int64_t)b * kHalsChunk];
    s1 += p[(int64_t)(b + kHalsSums) * kHalsChunk];
    s2 += p[(int64_t)(b + 2 * kHalsSums) * kHalsChunk];
    s3 += p[(int64_t)(b + 3 * kHalsSums) * kHalsChunk];
  }
  for (; b < h.nblk; b += kHalsSums) s0 += p[(int64_t)b * kHalsChunk];
  h.sums[blockIdx.x * kHalsChunk + it] = (s0 + s1) + (s2 + s3);
}

// Every iteration's error sum over n sets of them (interleaved sums per
// iteration, 8 and more, added up in order), then the first iteration at which
// the rule fires.
__global__ __launch_bounds__(8 * kHalsChunk) void hals_decide_kernel(HalsRun h, const double* sets, int n) {
  __shared__ double part[8 * kHalsChunk];
  __shared__ int first;
  if (h.chunk > 0 && h.state[0]) return;
  int W = kHalsChunk;  // threads beside each other: the iterations, rounded up
  while (W > 8 && W / 2 >= h.iters) W /= 2;
  const int it = threadIdx.x % W, lane = threadIdx.x / W, lanes = 8 * kHalsChunk / W;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  if (it < h.iters) {
    const double* p = sets + it;
    int b = lane;
    for (; b + 3 * lanes < n; b += 4 * lanes) {
      s0 += p[(int64_t)b * kHalsChunk];
      s1 += p[(int64_t)(b + lanes) * kHalsChunk];
      s2 += p[(int64_t)(b + 2 * lanes) * kHalsChunk];
      s3 += p[(int64_t)(b + 3 * lanes) * kHalsChunk];
    }
    for (; b < n; b += lanes) s0 += p[(int64_t)b * kHalsChunk];
  }
  part[threadIdx.x] = (s0 + s1) + (s2 + s3);
  if (threadIdx.x == 0) first = h.iters;
  __syncthreads();
  double sum = 0.0;
  if (lane == 0) {
    for (int l = 0; l < lanes; l += 8)
#pragma unroll
      for (int x = 0; x < 8; ++x) sum += part[(l + x) * W + it];
    part[it] = sum;
  }
  __syncthreads();
  const double err0 = h.chunk == 0 ? part[0] : *h.err0;
  if (lane == 0 && it < h.iters && sum < h.a.tol * err0) atomicMin(&first, it);
  __syncthreads();
  if (threadIdx.x != 0) return;
  const bool done = first < h.iters;
  if (h.chunk == 0) *h.err0 = err0;
  h.state[0] = done;
  h.state[1] = h.begin + (done ? first + 1 : h.iters);
  h.state[2] = h.chunk;
  h.state[3] = first + 1;
}

// The first chunk has 16 iterations where one iteration of all rows takes more
// than some 4 us (by R^2 and the rounds of workgroups on the GPU): there a rule
// that fires early would leave most of a long chunk for nothing.  100
// iterations, a rule that fires at the second / never, one chunk before: 512
// rows, rank 64: 1036 -> 234 / 986 -> 1011 us; 20000 rows, rank 64: 2270 ->
// 508 / 2171 -> 2209; 1M rows, rank 16: 5835 -> 1013 / 5706 -> 4618.  (Chunks
// of 16, 64 and 20 took 1048 us for the 512 rows.)
template <typename T, int RT, bool FULL, bool LOOP>
static void hals_run(HalsRun h, int n_iter_max, hipStream_t st) {
  const bool heavy = (int64_t)RT * RT * std::max<int64_t>(1024, (h.a.rows + kHalsRows - 1) / kHalsRows) > 1700000;
  const bool sum = h.nblk > 1024;
  int chunk = heavy ? 16 : kHalsChunk;
  h.only = n_iter_max == 1;
  for (h.begin = 0; h.begin < n_iter_max && !h.only; h.begin += h.iters, ++h.chunk) {
    h.iters = std::min(chunk, n_iter_max - h.begin);
    chunk = kHalsChunk;
    hals_run_kernel<T, RT, FULL, LOOP><<<(unsigned)h.nblk, 64, 0, st>>>(h);
    if (sum) hals_sum_kernel<<<kHalsSums, kHalsChunk, 0, st>>>(h);
    hals_decide_kernel<<<1, 8 * kHalsChunk, 0, st>>>(h, sum ? h.sums : h.partial, sum ? kHalsSums : h.nblk);
  }
  if (h.only) h.iters = 1;
  else --h.chunk;
  h.final = 1;
  hals_run_kernel<T, RT, FULL, LOOP><<<(unsigned)h.nblk, 64, 0, st>>>(h);
}

template <typename T, int RT>
static bool hals_try(const HalsRun& h, int n_iter_max, hipStream_t st) {
  if (h.a.R > RT) return false;
  if (h.a.rows > (int64_t)kHalsBlocks * kHalsRows) hals_run<T, RT, false, true>(h, n_iter_max, st);
  else if (h.a.R == RT) hals_run<T, RT, true, false>(h, n_iter_max, st);
  else hals_run<T, RT, false, false>(h, n_iter_max, st);
  return true;
}

// the rank padded to a multiple of 4, of 8 from 32 and of 16 from 48 on
template <typename T>
static void hals_run_rank(const HalsRun& h, int n, hipStream_t st) {
  (void)(hals_try<T, 4>(h, n, st) || hals_try<T, 8>(h, n, st) || hals_try<T, 12>(h, n, st) ||
         hals_try<T, 16>(h, n, st) || hals_try<T, 20>(h, n, st) || hals_try<T, 24>(h, n, st) ||
         hals_try<T, 32>(h, n, st) || hals_try<T, 40>(h, n, st) || hals_try<T, 48>(h, n, st) ||
         hals_try<T, 64>(h, n, st));
}

}  // namespace tla

using namespace tla;

static size_t hals_align(size_t b) { return (b + 255) & ~size_t(255); }

// Iteration counts up to this run over the grid in chunks of kHalsChunk;
// longer runs (exact mode) stay in one workgroup.
constexpr int kHalsMaxIters = 1000;

extern "C" size_t tla_hals_nnls_workspace_size(int64_t rows, int rank) {
  const int64_t r = rows > 0 ? rows : 1, nb = std::min<int64_t>((r + kHalsRows - 1) / kHalsRows, kHalsBlocks);
  return 2 * hals_align(size_t(r) * rank * 8) + hals_align(size_t(nb) * kHalsChunk * 8) +
         hals_align(size_t(kHalsSums) * kHalsChunk * 8) + hals_align(16) + hals_align(8);
}

extern "C" int tla_hals_nnls(int dtype, void* factor, const void* mttkrp, int64_t rows, int rank,
                             const double* const* grams, int ndim, int mode, const void* weights, int wdtype,
                             double sparsity, int has_sparsity, int n_iter_max, double tol, int* iters_out,
                             void* workspace, size_t workspace_bytes, void* stream) {
  TLA_REQUIRE(dtype == TLA_F32 || dtype == TLA_F64, "hals_nnls: bad dtype %d", dtype);
  TLA_REQUIRE(ndim >= 2 && ndim <= kMaxOrder, "hals_nnls: order %d", ndim);
  TLA_REQUIRE(mode >= 0 && mode < ndim, "hals_nnls: mode %d", mode);
  TLA_REQUIRE(rank >= 1 && rank <= kMaxRank, "hals_nnls: rank %d not in [1, %d]", rank, kMaxRank);
  TLA_REQUIRE(rows >= 0, "hals_nnls: rows = %lld", (long long)rows);
  TLA_REQUIRE(n_iter_max >= 0, "hals_nnls: n_iter_max = %d", n_iter_max);
  TLA_REQUIRE(factor && mttkrp, "hals_nnls: NULL pointer");
  TLA_REQUIRE(!weights || wdtype == TLA_F32 || wdtype == TLA_F64, "hals_nnls: bad weight dtype %d", wdtype);
  if (rows == 0 || n_iter_max == 0) return TLA_OK;
  HalsArgs a{};
  for (int m = 0; m < ndim; ++m) {
    TLA_REQUIRE(m == mode || grams[m] != nullptr, "hals_nnls: gram %d is NULL", m);
    a.grams[m] = grams[m];
  }
  a.ndim = ndim; a.mode = mode; a.R = rank;
  a.weights = weights; a.wdt = wdtype;
  a.M = mttkrp; a.A = factor; a.rows = rows;
  a.sparsity = sparsity; a.has_sparsity = has_sparsity;
  a.n_iter_max = n_iter_max; a.tol = tol; a.iters_out = iters_out;
  hipStream_t st = (hipStream_t)stream;
  const int rt = rank <= 16 ? 16 : rank <= 32 ? 32 : rank <= 48 ? 48 : 64;
  if (workspace && n_iter_max <= kHalsMaxIters) {
    TLA_REQUIRE(workspace_bytes >= tla_hals_nnls_workspace_size(rows, rank), "hals_nnls: workspace too small");
    const int64_t nb = std::min<int64_t>((rows + kHalsRows - 1) / kHalsRows, kHalsBlocks);
    HalsRun h{};
    h.a = a;
    h.nblk = (int)nb;
    char* w = (char*)workspace;
    const size_t vb = hals_align(size_t(rows) * rank * 8);
    h.vbuf[0] = (double*)w;
    h.vbuf[1] = (double*)(w + vb);
    h.partial = (double*)(w + 2 * vb);
    h.sums = (double*)(w + 2 * vb + hals_align(size_t(nb) * kHalsChunk * 8));
    h.state = (int*)((char*)h.sums + hals_align(size_t(kHalsSums) * kHalsChunk * 8));
    h.err0 = (double*)((char*)h.state + hals_align(16));
    if (dtype == TLA_F32) hals_run_rank<float>(h, n_iter_max, st);
    else hals_run_rank<double>(h, n_iter_max, st);
    TLA_LAUNCH_CHECK();
    if (iters_out) {
      TLA_HIP(hipMemcpyAsync(iters_out, h.state + 1, sizeof(int), hipMemcpyDeviceToDevice, st));
    }
    return TLA_OK;
  }
#define TLA_HALS(T_)                                                                  \
  switch (rt) {                                                                       \
    case 16: hals_nnls_kernel<T_, 16><<<1, kHalsThreads, 0, st>>>(a); break;          \
    case 32: hals_nnls_kernel<T_, 32><<<1, kHalsThreads, 0, st>>>(a); break;          \
    case 48: hals_nnls_kernel<T_, 48><<<1, kHalsThreads, 0, st>>>(a); break;          \
    default: hals_nnls_kernel<T_, 64><<<1, kHalsThreads, 0, st>>>(a); break;          \
  }
  if (dtype == TLA_F32) {
    TLA_HALS(float)
  } else {
    TLA_HALS(double)
  }
#undef TLA_HALS
  TLA_LAUNCH_CHECK();
  return TLA_OK;
}
