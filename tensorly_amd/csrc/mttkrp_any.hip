// MTTKRP of any mode sizes on the matrix cores, float32 and float64 (but for a
// contiguous output mode shorter than a 16-byte load).
//
// The tensor is viewed as X[a, i, q] (i = output mode) and the output is
// out[i, r] = sum_{a, q} X[a, i, q] B[(a, q), r], where B holds the rows of
// the Khatri-Rao product of the other modes.  B is never stored: every wave
// forms the part it needs in the registers that the matrix instructions read.
//
//  * any_rows_kernel (output mode is not the contiguous one): a wave takes
//    chunks of 128 contiguous bytes of q for TN tiles of 16 rows i.  Lane
//    (c, g) reads 32 consecutive bytes of row c of each tile, as they lie
//    (dword aligned 16-byte loads), and forms B[(a, q), r] = G[(a, b), r]
//    F_k[k, r] for its own q = (b, k) once for all TN tiles; G is the product
//    of the weights and the factors of every mode but the output and the
//    contiguous one.
//  * any_last_kernel (output mode contiguous): a wave takes blocks of rows p
//    (all the other modes, flattened) for TN tiles of 256 contiguous bytes of
//    columns; the matrix instruction contracts over p.
//
// Bound: memory for ranks up to 32, the FP32 matrix rate above.  One set of
// B rows serves all TN tiles of a wave; two sets of loaded values take turns,
// so that a chunk is in flight while the one before is multiplied; a wave's
// loads are all independent, so 16 waves per compute unit keep 100 KB in
// flight.  Before, these shapes ran one block per output row on the vector
// ALU, which read the tensor once per 16 rank columns with a 64-bit division
// per element.  Measured, call by call with the reduction, mode 0 / 1 / 2:
//   257 x 301 x 203, R = 20, float32: 1333 (mean) -> 27 / 29 / 28 us (2.3 TB/s)
//   761 x 380 x 283, R = 16, float32: 77 / 98 / 73 us (4.3 / 3.3 / 4.5 TB/s)
//   201 x 179 x 160, R = 16, float64: 621 (mean) -> 18 / 17 / 16 us (2.7 TB/s)
//   149 x 120 x 90,  R = 10, float32: 172 (mean) -> 8 / 8 / 11 us
#include <algorithm>

#include "inverse.h"
#include "mma_any.h"
#include "mttkrp_any.h"

namespace tla {

// G[q, r] = w[r] * product over the listed modes' factor rows (q row-major
// over those modes).
template <typename T>
struct AnyGArgs {
  int n, R;
  int64_t sz[kMaxOrder];
  const T* fac[kMaxOrder];
  const T* weights;
  int64_t rows;
};

// The entry of row q and byte column rb of the table G, formed from the
// factors.
template <typename T>
__device__ __forceinline__ T g_entry(const AnyGArgs<T>& a, uint32_t q, uint32_t rb, uint32_t ldb) {
  T v = a.weights ? at<T>(a.weights, rb) : (T)1;
#pragma unroll
  for (int m = kMaxOrder - 1; m >= 0; --m)
    if (m < a.n) {
      const uint32_t sz = (uint32_t)a.sz[m], i = q % sz;
      q /= sz;
      v *= at<T>(a.fac[m], i * ldb + rb);
    }
  return v;
}

template <typename T>
struct AnyRowsArgs {
  const T* X;
  int64_t In, Q;
  int K, Pb;
  int R, ldr;       // columns of this slab, row stride of the factors
  const T* G;       // (A Pb) x ldr scale rows (a slice of them, from where row 0 would be), nullable
  AnyGArgs<T> ga;   // GD: the factors of G instead
  const T* Fk;      // K x ldr
  T* partial;       // [nblk][In][R]
  int nqc;
  int64_t first, nchunks, nblk;  // chunks [first, nchunks)
};

// GD: every wave forms its scale rows from the factors (small problems, where
// a launch for the table G costs more).
template <typename T, int TN, int RT, bool GD = false>
__global__ __launch_bounds__(64 * kAnyWaves, any_occ(TN, RT, false, sizeof(T) == 8)) void any_rows_kernel(AnyRowsArgs<T> a) {
  using V = typename AnyT<T>::vec;
  using Acc = typename AnyT<T>::acc;
  constexpr int VL = AnyT<T>::V, NV = 2 * VL, CH = 4 * NV;
  __shared__ T red[TN * RT * 256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t grp = blockIdx.x / a.nblk, blk = blockIdx.x - grp * a.nblk;
  const int K = a.K, R = a.R;
  const int64_t Q = a.Q, In = a.In, i0 = grp * (16 * TN);
  // rows past the mode's end read its last row; their results are dropped
  uint32_t roff[TN];  // bytes
#pragma unroll
  for (int t = 0; t < TN; ++t) 
    roff[t] = (uint32_t)((min((int64_t)(16 * t + c), In - 1 - i0) * Q + NV * g) * sizeof(T));
  uint32_t rr[RT];  // rank columns, in bytes; those past the slab read its last one
#pragma unroll
  for (int n = 0; n < RT; ++n) rr[n] = min(n * 16 + c, R - 1) * sizeof(T);
  const uint32_t ldb = a.ldr * sizeof(T);
  Acc acc[TN * RT];
#pragma unroll
  for (int n = 0; n < TN * RT; ++n) acc[n] = Acc{0, 0, 0, 0};

  const int64_t step = a.nblk * kAnyWaves;
  auto load = [&](int64_t ch, T (&x)[TN][NV]) {
    const int64_t ia = ch / a.nqc;
    const int q0 = (int)(ch - ia * a.nqc) * CH;
    const T* xb = a.X + (ia * In + i0) * Q + q0;
    if (q0 + CH <= (int)Q) {
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const V v0 = at<V>(xb, roff[t]), v1 = at<V>(xb + VL, roff[t]);
#pragma unroll
        for (int v = 0; v < VL; ++v) { x[t][v] = v0[v]; x[t][VL + v] = v1[v]; }
      }
    } else {
      const int left = (int)Q - (q0 + NV * g);  // values of this lane inside the row
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int v = 0; v < NV; ++v) x[t][v] = v < left ? at<T>(xb + v, roff[t]) : (T)0;
    }
  };
  // Multiplies the chunk in x while the next one is loaded into xn (loads
  // return in order, so the chunk's own factor rows are requested first).
  auto visit = [&](int64_t ch, T (&x)[TN][NV], T (&xn)[TN][NV]) {
    const int64_t ia = ch / a.nqc;
    const int q0 = (int)(ch - ia * a.nqc) * CH;
    const int left = (int)Q - (q0 + NV * g);
    // this lane's rows of B: q = b K + k, and the next NV - 1 values of q
    // may run into b + 1 (K >= NV), or are divided one by one
    T f[RT][NV], g0[RT], g1[RT];
    const int q = left > 0 ? q0 + NV * g : (int)Q - 1;
    const int b0 = q / K;
    int k0 = q - b0 * K;
    const T* Gb = !GD && a.G ? a.G + ia * a.Pb * a.ldr : nullptr;
    auto scale = [&](int b, uint32_t rb) -> T {
      if constexpr (GD) return g_entry(a.ga, (uint32_t)ia * a.Pb + b, rb, ldb);
      else return Gb ? at<T>(Gb, b * ldb + rb) : (T)1;
    };
    if (K >= NV) {
      const int b1 = min(b0 + 1, a.Pb - 1);
#pragma unroll
      for (int n = 0; n < RT; ++n) {
        g0[n] = scale(b0, rr[n]);
        g1[n] = scale(b1, rr[n]);
#pragma unroll
        for (int v = 0; v < NV; ++v) f[n][v] = at<T>(a.Fk, (k0 + v - (k0 + v >= K ? K : 0)) * ldb + rr[n]);
      }
    } else {
#pragma unroll
      for (int n = 0; n < RT; ++n) {
        g0[n] = g1[n] = (T)1;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const int qv = min(q + v, (int)Q - 1), b = qv / K;
          f[n][v] = at<T>(a.Fk, (qv - b * K) * ldb + rr[n]) * scale(b, rr[n]);
        }
      }
      k0 = -NV;  // the products are complete
    }
    if (ch + step < a.nchunks) load(ch + step, xn);
#pragma unroll
    for (int n = 0; n < RT; ++n)
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        f[n][v] *= k0 + v >= K ? g1[n] : g0[n];
        f[n][v] = v < left ? f[n][v] : (T)0;  // past the row's end both sides are zero
      }
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int n = 0; n < RT; ++n) acc[t * RT + n] = AnyT<T>::mma(x[t][v], f[n][v], acc[t * RT + n]);
  };
  int64_t ch = a.first + blk * kAnyWaves + wave;
  T x0[TN][NV], x1[TN][NV];
  if (ch < a.nchunks) load(ch, x0);
  while (ch < a.nchunks) {
    visit(ch, x0, x1);
    ch += step;
    if (ch >= a.nchunks) break;
    visit(ch, x1, x0);
    ch += step;
  }
  any_block_sum<T, TN * RT, kAnyWaves>(acc, red, wave, lane);
  // red[(t RT + n) 4 + e][lane] = out[i0 + 16 t + row(g, e)][16 n + c]
  T* dst = a.partial + blk * In * R;
  for (int idx = tid; idx < TN * RT * 256; idx += 64 * kAnyWaves) {
    const int col = idx % (16 * RT), row = idx / (16 * RT);
    const int t = row >> 4, ri = row & 15, n = col >> 4, cc = col & 15;
    const int gg = sizeof(T) == 4 ? ri >> 2 : ri & 3, e = sizeof(T) == 4 ? ri & 3 : ri >> 2;
    const int64_t i = i0 + row;
    if (i < In && col < R) dst[i * R + col] = red[((t * RT + n) * 4 + e) * 64 + gg * 16 + cc];
  }
}

template <typename T>
struct AnyLastArgs {
  const T* X;
  int64_t P, K;
  int J, nG;    // P = nG J
  int R, ldr;
  const T* G;   // (P / J) x ldr scale rows (a slice of them, from where row 0 would be), nullable
  AnyGArgs<T> ga;  // GD: the factors of G instead
  const T* Fj;  // J x ldr
  T* partial;   // [nblk][K][R]
  int64_t first, nvisits, nblk;  // visits [first, nvisits)
};

template <typename T, int TN, int RT, bool GD = false>
__global__ __launch_bounds__(64 * kAnyWaves, any_occ(TN, RT, true, sizeof(T) == 8)) void any_last_kernel(AnyLastArgs<T> a) {
  using V = typename AnyT<T>::vec;
  using Acc = typename AnyT<T>::acc;
  constexpr int VL = AnyT<T>::V;
  constexpr int NR = any_last_rows(TN, RT);
  constexpr int RV = 4 * NR;
  __shared__ T red[TN * VL * RT * 256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t grp = blockIdx.x / a.nblk, blk = blockIdx.x - grp * a.nblk;
  const int R = a.R, J = a.J;
  const int64_t K = a.K, k0 = grp * (16 * VL * TN);
  // lanes that would read past the row's end read its last 16 bytes (and
  // write those columns, with the same values as the lane they belong to)
  uint32_t col[TN];  // bytes, with the lane's first row
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    const int64_t k = k0 + (16 * t + c) * VL;
    col[t] = (uint32_t)((NR * g * K + min(k, K - VL)) * sizeof(T));
  }
  uint32_t rr[RT];  // rank columns, in bytes; those past the slab read its last one
#pragma unroll
  for (int n = 0; n < RT; ++n) rr[n] = min(n * 16 + c, R - 1) * sizeof(T);
  const uint32_t ldb = a.ldr * sizeof(T);
  Acc acc[TN * VL * RT];
#pragma unroll
  for (int n = 0; n < TN * VL * RT; ++n) acc[n] = Acc{0, 0, 0, 0};

  const int step = (int)a.nblk * kAnyWaves, nv = (int)a.nvisits, P = (int)a.P;
  auto load = [&](int v, V (&x)[NR][TN]) {
    const T* xb = a.X + (int64_t)v * RV * K;
    const int left = P - (v * RV + NR * g);
    if (v * RV + RV <= P) {
#pragma unroll
      for (int u = 0; u < NR; ++u)
#pragma unroll
        for (int t = 0; t < TN; ++t) x[u][t] = at<V>(xb + u * K, col[t]);
    } else {
#pragma unroll
      for (int u = 0; u < NR; ++u)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          x[u][t] = V{};
          if (u < left) x[u][t] = at<V>(xb + u * K, col[t]);
        }
    }
  };
  // Multiplies the visit in x while the next one is loaded into xn.
  auto visit = [&](int v, V (&x)[NR][TN], V (&xn)[NR][TN]) {
    const int p0 = v * RV + NR * g;
    const int left = P - p0;
    // rows p0 + u of the Khatri-Rao product of the other modes
    T f[RT][NR], g0[RT], g1[RT];
    const uint32_t p = left > 0 ? p0 : P - 1;
    const int a0 = (int)(p / (uint32_t)J);
    int j0 = (int)(p - (uint32_t)a0 * J);
    auto scale = [&](int i, uint32_t rb) -> T {
      if constexpr (GD) return g_entry(a.ga, (uint32_t)i, rb, ldb);
      else return a.G ? at<T>(a.G, i * ldb + rb) : (T)1;
    };
    if (J >= NR) {
      const int a1 = min(a0 + 1, a.nG - 1);
#pragma unroll
      for (int n = 0; n < RT; ++n) {
        g0[n] = scale(a0, rr[n]);
        g1[n] = scale(a1, rr[n]);
#pragma unroll
        for (int u = 0; u < NR; ++u) f[n][u] = at<T>(a.Fj, (j0 + u - (j0 + u >= J ? J : 0)) * ldb + rr[n]);
      }
    } else {
#pragma unroll
      for (int n = 0; n < RT; ++n) {
        g0[n] = g1[n] = (T)1;
#pragma unroll
        for (int u = 0; u < NR; ++u) {
          const uint32_t pu = min(p + u, (uint32_t)P - 1), au = pu / (uint32_t)J;
          f[n][u] = at<T>(a.Fj, (pu - au * J) * ldb + rr[n]) * scale(au, rr[n]);
        }
      }
      j0 = -NR;  // the products are complete
    }
    if (v + step < nv) load(v + step, xn);
#pragma unroll
    for (int n = 0; n < RT; ++n)
#pragma unroll
      for (int u = 0; u < NR; ++u) {
        f[n][u] *= j0 + u >= J ? g1[n] : g0[n];
        f[n][u] = u < left ? f[n][u] : (T)0;
      }
#pragma unroll
    for (int u = 0; u < NR; ++u)
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int e = 0; e < VL; ++e)
#pragma unroll
          for (int n = 0; n < RT; ++n) {
            Acc& d = acc[(t * VL + e) * RT + n];
            d = AnyT<T>::mma(f[n][u], x[u][t][e], d);
          }
  };
  int v = (int)(a.first + blk * kAnyWaves) + wave;
  V x0[NR][TN], x1[NR][TN];
  if (v < nv) load(v, x0);
  while (v < nv) {
    visit(v, x0, x1);
    v += step;
    if (v >= nv) break;
    visit(v, x1, x0);
    v += step;
  }
  any_block_sum<T, TN * VL * RT, kAnyWaves>(acc, red, wave, lane);
  // red[((t VL + s) RT + n) 4 + e][lane] = out[col[t] + s][16 n + row(g, e)]
  T* dst = a.partial + blk * K * R;
  for (int idx = tid; idx < TN * VL * RT * 256; idx += 64 * kAnyWaves) {
    const int r = idx % (16 * RT), kc = idx / (16 * RT);  // kc: column within the group
    const int t = kc / (16 * VL), cc = (kc / VL) % 16, s = kc % VL;
    const int n = r >> 4, ri = r & 15;
    const int gg = sizeof(T) == 4 ? ri >> 2 : ri & 3, e = sizeof(T) == 4 ? ri & 3 : ri >> 2;
    const int64_t k = k0 + (16 * t + cc) * VL;
    if (k < K && r < R) dst[(min(k, K - VL) + s) * R + r] = red[(((t * VL + s) * RT + n) * 4 + e) * 64 + gg * 16 + cc];
  }
}

// out[i ldo + r] = sum_{b < nblk} partial[b][i][r] in a fixed order: 32
// elements x 8 lanes of b per block.  In float64: the sums of a hundred
// float32 partials would round more than all that came before (149 x 120 x 90,
// positive data: relative error 5.2e-8 against 2.6e-8).
// JOB: the grid's last block inverts the normal-equations matrix of the solve
// that follows (inverse.h) instead, so that the solve need not (rank 10, 150
// rows, sum and solve: 4.4 + 11.8 -> 6.4 + 7.9 us).
template <typename T, bool JOB>
__global__ __launch_bounds__(256) void any_reduce_kernel(const T* __restrict__ partial, int64_t n, int64_t nblk, int R,
                                                         int64_t ldo, T* __restrict__ out, InvJob job) {
  if constexpr (JOB) {
    extern __shared__ char job_lds[];
    if (take_inv_job<256>(job, job_lds)) return;
  }
  __shared__ double red[8][32];
  const int el = threadIdx.x & 31, bl = threadIdx.x >> 5;
  const int64_t e = (int64_t)blockIdx.x * 32 + el;
  double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
  if (e < n) {
    const T* p = partial + e;
    int64_t b = bl;
    for (; b + 24 < nblk; b += 32) {
      s0 += p[b * n];
      s1 += p[(b + 8) * n];
      s2 += p[(b + 16) * n];
      s3 += p[(b + 24) * n];
    }
    for (; b < nblk; b += 8) s0 += p[b * n];
  }
  red[bl][el] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (bl == 0 && e < n) {
    double s = red[0][el];
#pragma unroll
    for (int k = 1; k < 8; ++k) s += red[k][el];
    out[(e / R) * ldo + e % R] = (T)s;
  }
}

// Rows g0, ... of the table, `cols` of its R columns.
template <typename T>
__global__ void any_g_kernel(AnyGArgs<T> a, int64_t g0, int cols, T* __restrict__ out) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= a.rows * cols) return;
  const int r = (int)(e % cols);
  const int64_t row = e / cols;
  int64_t q = g0 + row;
  T v = a.weights ? a.weights[r] : (T)1;
#pragma unroll
  for (int m = kMaxOrder - 1; m >= 0; --m)
    if (m < a.n) {
      const int64_t i = q % a.sz[m];
      q /= a.sz[m];
      v *= a.fac[m][i * a.R + r];
    }
  out[row * a.R + r] = v;
}

template <typename T, int RT>
static void any_run_rows(int TN, unsigned grid, const AnyRowsArgs<T>& a, hipStream_t st) {
  if (TN == 1 && a.ga.R) any_rows_kernel<T, 1, RT, true><<<grid, 64 * kAnyWaves, 0, st>>>(a);
  else if (TN == 1) any_rows_kernel<T, 1, RT><<<grid, 64 * kAnyWaves, 0, st>>>(a);
  if (TN == 2) any_rows_kernel<T, 2, RT><<<grid, 64 * kAnyWaves, 0, st>>>(a);
  if constexpr (RT <= 3 || sizeof(T) == 4)
    if (TN == 3) any_rows_kernel<T, 3, RT><<<grid, 64 * kAnyWaves, 0, st>>>(a);
  if constexpr (RT <= 2 || sizeof(T) == 4)
    if (TN == 4) any_rows_kernel<T, 4, RT><<<grid, 64 * kAnyWaves, 0, st>>>(a);
}

template <typename T, int RT>
static void any_run_last(int TN, unsigned grid, const AnyLastArgs<T>& a, hipStream_t st) {
  // (a slab of ranks past 64 may have fewer rank tiles than the plan's)
  if constexpr (RT == 1) {
    if (TN == 3) any_last_kernel<T, 3, RT><<<grid, 64 * kAnyWaves, 0, st>>>(a);
    if (TN == 2) any_last_kernel<T, 2, RT><<<grid, 64 * kAnyWaves, 0, st>>>(a);
  }
  if (TN == 1 && a.ga.R) any_last_kernel<T, 1, RT, true><<<grid, 64 * kAnyWaves, 0, st>>>(a);
  else if (TN == 1) any_last_kernel<T, 1, RT><<<grid, 64 * kAnyWaves, 0, st>>>(a);
}

template <typename T>
static int any_launch_t(const AnyPlan& p, const T* X, int ndim, const int64_t* shape, const void* const* factors,
                        const T* weights, int R, int mode, T* out, void* ws, const InvJob* job, hipStream_t st) {
  for (int m = 0; m < ndim; ++m) TLA_REQUIRE(m == mode || factors[m] != nullptr, "factor %d is NULL", m);
  // modes of the table: all but the output mode and the one the kernel reads itself
  const int own = p.last ? ndim - 2 : ndim - 1;
  AnyGArgs<T> ga{};
  if (p.g_rows > 0) {
    ga.R = R;
    ga.weights = weights;
    for (int m = 0; m < ndim; ++m)
      if (m != mode && m != own) {
        ga.sz[ga.n] = shape[m];
        ga.fac[ga.n++] = (const T*)factors[m];
      }
  }
  const bool table = p.build_g && !p.direct_g;
  const int64_t sets = p.nblk * p.slices;
  const unsigned grid = (unsigned)(p.groups * p.nblk);
  for (int r0 = 0; r0 < R; r0 += 64) {
    const int Rs = std::min(64, R - r0), RT = (Rs + 15) / 16;
    const bool direct = sets == 1 && Rs == R;
    T* const sums = direct ? out : (T*)((char*)ws + (table ? any_align(size_t(p.g_slice) * R * sizeof(T)) : 0));
    AnyGArgs<T> gs = ga;  // of this slab's columns
    if (gs.weights) gs.weights += r0;
    for (int m = 0; m < gs.n; ++m) gs.fac[m] += r0;
    const int RV = 4 * any_last_rows(p.TN, RT);
    const int64_t chunks = p.last ? (p.A + RV - 1) / RV : p.nchunks;
    const int64_t per = chunks == p.nchunks ? p.per : (chunks + p.slices - 1) / p.slices;
    for (int64_t s = 0; s < p.slices; ++s) {
      const int64_t c0 = std::min(chunks, s * per), c1 = std::min(chunks, c0 + per);
      T* part = sums + s * p.nblk * p.In * Rs;
      const T* G = nullptr;
      int64_t g0 = 0;
      if (table) {
        // the rows of chunks c0, ..., c1 - 1 and the one after
        int64_t g1 = p.g_rows;
        if (p.slices > 1 && c0 < c1) {
          if (p.last) {
            g0 = c0 * RV / p.J;
            g1 = std::min(p.g_rows, (c1 * RV - 1) / p.J + 2);
          } else {
            constexpr int CH = 8 * AnyT<T>::V;
            g0 = c0 / p.nqc * p.Pb + c0 % p.nqc * CH / p.K;
            g1 = (c1 - 1) / p.nqc * p.Pb + std::min(((c1 - 1) % p.nqc + 1) * CH / p.K + 2, p.Pb);
          }
        }
        TLA_REQUIRE(g1 - g0 <= p.g_slice, "scale table of %lld rows", (long long)(g1 - g0));
        // one slice holds every slab's columns; of several, each is made again
        // for a slab
        const bool whole = p.slices == 1;
        if (!whole || r0 == 0) {
          AnyGArgs<T> gt = whole ? ga : gs;
          const int cols = whole ? R : Rs;
          gt.rows = g1 - g0;
          const int64_t ne = gt.rows * cols;
          any_g_kernel<T><<<(unsigned)((ne + 255) / 256), 256, 0, st>>>(gt, g0, cols, (T*)ws + (whole ? 0 : r0));
          TLA_LAUNCH_CHECK();
        }
        // (row 0 lies before the buffer where the slice begins later)
        G = (const T*)((uintptr_t)ws + uintptr_t(r0 - g0 * R) * sizeof(T));
      } else if (p.g_rows > 0 && !p.direct_g) {
        G = gs.fac[0];
      }
      const AnyGArgs<T> gd = p.direct_g ? gs : AnyGArgs<T>{};  // R = 0: not used
      if (p.last) {
        AnyLastArgs<T> a{X,  p.A, p.K,  (int)p.J, (int)(p.A / p.J), Rs, R, G, gd,
                         (const T*)factors[own] + r0, part, c0, c1, p.nblk};
        switch (RT) {
          case 1: any_run_last<T, 1>(p.TN, grid, a, st); break;
          case 2: any_run_last<T, 2>(p.TN, grid, a, st); break;
          case 3: any_run_last<T, 3>(p.TN, grid, a, st); break;
          default: any_run_last<T, 4>(p.TN, grid, a, st); break;
        }
      } else {
        AnyRowsArgs<T> a{X, p.In, p.Q, (int)p.K, (int)p.Pb, Rs, R, G, gd, (const T*)factors[own] + r0, part,
                         p.nqc, c0, c1, p.nblk};
        switch (RT) {
          case 1: any_run_rows<T, 1>(p.TN, grid, a, st); break;
          case 2: any_run_rows<T, 2>(p.TN, grid, a, st); break;
          case 3: any_run_rows<T, 3>(p.TN, grid, a, st); break;
          default: any_run_rows<T, 4>(p.TN, grid, a, st); break;
        }
      }
      TLA_LAUNCH_CHECK();
    }
    if (!direct) {
      const int64_t n = p.In * Rs;
      const unsigned blocks = (unsigned)((n + 31) / 32);
      if (job) {
        const size_t lds = inv_job_lds_bytes(job->R);
        const auto kernel = any_reduce_kernel<T, true>;
        if (lds > 64 * 1024)
          TLA_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        kernel<<<blocks + 1, 256, lds, st>>>(sums, n, sets, Rs, R, out + r0, *job);
      } else {
        any_reduce_kernel<T, false><<<blocks, 256, 0, st>>>(sums, n, sets, Rs, R, out + r0, InvJob{});
      }
      TLA_LAUNCH_CHECK();
    }
  }
  return TLA_OK;
}

int any_launch(bool f64, const AnyPlan& p, const void* X, int ndim, const int64_t* shape, const void* const* factors,
               const void* weights, int R, int mode, void* out, void* ws, const InvJob* job, hipStream_t st) {
  return f64 ? any_launch_t<double>(p, (const double*)X, ndim, shape, factors, (const double*)weights, R, mode,
                                    (double*)out, ws, job, st)
             : any_launch_t<float>(p, (const float*)X, ndim, shape, factors, (const float*)weights, R, mode,
                                   (float*)out, ws, job, st);
}

}  // namespace tla
