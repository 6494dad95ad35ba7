// FP64 symmetric eigensolver for the leading eigenpairs of a Gram matrix.
//
// These replace the LAPACK SVDs of tensorly/tenalg/svd.py:211-235
// (truncated_svd) on the Tucker / CP-init path: the left singular vectors of
// A are the eigenvectors of A A^T and the singular values the square roots
// of its eigenvalues.
//
//  * n <= 128: tridiagonalisation, Sturm counts and twisted factorisations
//    (direct_eig); where eigenvalues cluster, cyclic Jacobi on the whole
//    matrix (round-robin pair ordering, all n/2 rotations of a round applied
//    in parallel).
//  * n  > 128: block subspace iteration with Rayleigh-Ritz, block b = 48 for
//    k <= 40, 64 for k <= 56 or 128 for k <= 120.  Each step: Z = G V, H = V^T Z on FP64
//    MFMA, H = W diag(t) W^T (perturbation theory where the previous Ritz
//    basis nearly diagonalises H, else the direct solver for block 48, else
//    Jacobi), Ritz vectors Y = V W and U = Z W = G Y, residuals of the k
//    leading pairs, V <- orth(U) by one Cholesky-QR pass or a shifted and a
//    plain one (S = M^T M on MFMA, forward elimination of [S | I] in
//    registers).  Converged when every leading residual is below tol * t_1.
// One workgroup per problem; the padded np x b blocks live in the caller's
// workspace (L2-resident).
#include <math.h>

#include <algorithm>

#include "common.h"
#include "mma_any.h"

namespace tla {

constexpr int kEigThreads = 512;
constexpr int kEigWaves = kEigThreads / 64;
constexpr int kJac = 64;           // n <= kJac: Jacobi with A and W in LDS
constexpr int kJacLarge = 128;     // n <= kJacLarge: Jacobi with A in LDS, W in the workspace
constexpr int kEigCapLarge = 128;  // larger subspace block

// C (M x N, ldc) = op(A) B over K, op(A)[m][k] = TA ? A[k * lda + m] : A[m * lda + k],
// B[k][n] = B[k * ldb + n]; M, N multiples of 16, K a multiple of 8.  The
// block's waves take 16 x 16 output tiles in turn; operands may be in LDS or
// global memory (L2-resident here).  Ends with a barrier.
template <bool TA>
__device__ void block_gemm_f64(const double* A, int lda, const double* B, int ldb, double* C, int ldc, int M, int N,
                               int K) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int tn = N / 16, ntile = (M / 16) * tn;
  for (int t = wave; t < ntile; t += blockDim.x >> 6) {
    const int mi = (t / tn) * 16, nj = (t % tn) * 16;
    doublex4 acc = doublex4{0.0, 0.0, 0.0, 0.0};
    // eight k-steps' operands requested before their MFMAs (k-ascending
    // accumulation either way)
    int k0 = 0;
    for (; k0 + 32 <= K; k0 += 32) {
      double a[8], b[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int kk = k0 + 4 * s + lk;
        a[s] = TA ? A[kk * lda + mi + lr] : A[(mi + lr) * lda + kk];
        b[s] = B[kk * ldb + nj + lr];
      }
#pragma unroll
      for (int s = 0; s < 8; ++s) acc = mfma_f64(a[s], b[s], acc);
    }
    for (; k0 < K; k0 += 4) {
      const int kk = k0 + lk;
      const double a0 = TA ? A[kk * lda + mi + lr] : A[(mi + lr) * lda + kk];
      acc = mfma_f64(a0, B[kk * ldb + nj + lr], acc);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) C[(mi + lk + 4 * e) * ldc + nj + lr] = acc[e];
  }
  __syncthreads();
}

// C (N x N) = A^T B for a product known to be symmetric (A^T A, or V^T G V
// with G symmetric): only the tiles on and above the diagonal are formed
// (16 k-steps' operands in flight) and each off-diagonal one is written to
// both places (a diagonal tile holds whatever rounding its own sums give).
// N a multiple of 16, K a multiple of 4.  Ends with a barrier.
__device__ void block_gemm_sym_f64(const double* A, int lda, const double* B, int ldb, double* C, int ldc, int N,
                                   int K) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int tn = N / 16, ntile = tn * (tn + 1) / 2;
  for (int t = wave; t < ntile; t += blockDim.x >> 6) {
    int ti = 0, rem = t;  // t -> (ti <= tj), row by row of the upper triangle
    while (rem >= tn - ti) {
      rem -= tn - ti;
      ++ti;
    }
    const int tj = ti + rem, mi = ti * 16, nj = tj * 16;
    doublex4 acc = doublex4{0.0, 0.0, 0.0, 0.0};
    int k0 = 0;
    for (; k0 + 64 <= K; k0 += 64) {
      double a[16], b[16];
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const int kk = k0 + 4 * s + lk;
        a[s] = A[kk * lda + mi + lr];
        b[s] = B[kk * ldb + nj + lr];
      }
#pragma unroll
      for (int s = 0; s < 16; ++s) acc = mfma_f64(a[s], b[s], acc);
    }
    for (; k0 < K; k0 += 4) {
      const int kk = k0 + lk;
      acc = mfma_f64(A[kk * lda + mi + lr], B[kk * ldb + nj + lr], acc);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      C[(mi + lk + 4 * e) * ldc + nj + lr] = acc[e];
      if (ti != tj) C[(nj + lr) * ldc + mi + lk + 4 * e] = acc[e];
    }
  }
  __syncthreads();
}

// C (M x N) = A B for a row-major A in global memory with lda == K == KB:
// each wave stages one 16-row panel of A (16 * KB contiguous doubles, read
// with coalesced loads) in LDS and uses it for all N / 16 column tiles.
// Read straight from memory, an MFMA A operand is 16 rows x 32 bytes per
// load, which measured ~2.3x slower than contiguous pieces.  B (ldb) in LDS
// or global; the same k-ascending MFMA sequence as block_gemm_f64.  stage
// holds 16 * (KB + 1) doubles per wave.  Ends with a barrier.
template <int KB>
__device__ void block_gemm_f64_panel(const double* A, const double* B, int ldb, double* C, int ldc, int M, int N,
                                     double* stage) {
  constexpr int LDP = KB + 1;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  double* P = stage + wave * 16 * LDP;
  const int tn = N / 16;
  for (int pnl = wave; pnl < M / 16; pnl += blockDim.x >> 6) {
    const double* Ap = A + (size_t)pnl * 16 * KB;
#pragma unroll
    for (int e = lane; e < 16 * KB; e += 64) P[(e / KB) * LDP + (e % KB)] = Ap[e];
    // the wave's LDS writes reach LDS before its later reads (in-order LDS
    // queue per wave); this keeps the compiler from reordering across
    __builtin_amdgcn_wave_barrier();
    for (int nb = 0; nb < tn; ++nb) {
      doublex4 acc = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k0 = 0; k0 < KB; k0 += 4) {
        const int kk = k0 + lk;
        acc = mfma_f64(P[lr * LDP + kk], B[kk * ldb + nb * 16 + lr], acc);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) C[(pnl * 16 + lk + 4 * e) * ldc + nb * 16 + lr] = acc[e];
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
}

// Z = G V for the zero-padded symmetric np x np G and the np x B block V
// (both in global memory, ld np and B), read as G^T V so that each A-operand
// load takes 4 rows x 128 contiguous bytes of G.  V goes through LDS (vs,
// KC x B doubles) in KC-row chunks; each wave keeps two 16-row strips of Z
// with all B / 16 column tiles in registers, so one pass reads every element
// of G once and every V operand comes from LDS.  Same k-ascending MFMA
// sequence per output tile as block_gemm_f64.  Ends with a barrier.
template <int B, int KC>
__device__ void gv_product(const double* __restrict__ G, int np, const double* __restrict__ V, double* Z,
                           double* vs) {
  constexpr int TN = B / 16, SPW = 2;
  static_assert(B % 16 == 0 && KC % 32 == 0, "tile shape");
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int nw = blockDim.x >> 6, nstrip = np / 16;
  for (int g0 = 0; g0 < nstrip; g0 += nw * SPW) {
    const int s0 = g0 + wave * SPW;
    const bool live0 = s0 < nstrip, live1 = s0 + 1 < nstrip;  // wave-uniform
    doublex4 acc[SPW][TN];
#pragma unroll
    for (int s = 0; s < SPW; ++s)
#pragma unroll
      for (int t = 0; t < TN; ++t) acc[s][t] = doublex4{0.0, 0.0, 0.0, 0.0};
    for (int kc = 0; kc < np; kc += KC) {
      const int kn = min(KC, np - kc);  // a multiple of 16
      __syncthreads();                  // the previous chunk is consumed
      for (int e = threadIdx.x; e < kn * B; e += blockDim.x) vs[e] = V[(int64_t)kc * B + e];
      __syncthreads();
      if (live0) {
        const double* g0p = G + (int64_t)kc * np + s0 * 16 + lr;
        int k0 = 0;
        for (; k0 + 16 <= kn; k0 += 16) {
          double a0[4], a1[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int kk = k0 + 4 * q + lk;
            a0[q] = g0p[(int64_t)kk * np];
            a1[q] = live1 ? g0p[(int64_t)kk * np + 16] : 0.0;
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int kk = k0 + 4 * q + lk;
#pragma unroll
            for (int t = 0; t < TN; ++t) {
              const double bv = vs[kk * B + t * 16 + lr];
              acc[0][t] = mfma_f64(a0[q], bv, acc[0][t]);
              acc[1][t] = mfma_f64(a1[q], bv, acc[1][t]);
            }
          }
        }
      }
    }
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      const int strip = s0 + s;
      if (strip < nstrip) {
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) Z[(int64_t)(strip * 16 + lk + 4 * e) * B + t * 16 + lr] = acc[s][t][e];
      }
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// Jacobi on an m x m symmetric matrix A (LDS, leading dimension LDA: odd, so
// that the column walks of a rotation hit distinct banks), accumulating the
// rotations into W (leading dimension LDW, in LDS or global memory,
// initialised by the caller).  Returns the number of sweeps.
// ---------------------------------------------------------------------------
// 1 / x and 1 / sqrt(x) for finite x > 0 (here x > 1e-300): the hardware
// estimates refined by two Newton steps each, to full double precision.
__device__ __forceinline__ double jac_recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
}
// 1 / x of either sign, x != 0
__device__ __forceinline__ double jac_recip_signed(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
}
// the exponent field of x, unbiased (very small for zero and denormals)
__device__ __forceinline__ int ilogb_fast(double x) { return ((__double2hiint(x) >> 20) & 0x7ff) - 1023; }
__device__ __forceinline__ double jac_rsqrt(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  y = y * fma(-hx * y, y, 1.5);
  return y * fma(-hx * y, y, 1.5);
}

// Slot a's pair (p < q) in round `round` of the round-robin ordering of me
// (even) slots: slot 0 stays, the others rotate.
__device__ __forceinline__ void jac_pair(int a, int round, int me, int& p, int& q) {
  const int L = me - 1;
  int x = (a == 0 ? me - 2 : a - 1) + round;
  if (x >= L) x -= L;
  int y = me - 2 - a + round;
  if (y >= L) y -= L;
  p = a == 0 ? 0 : 1 + x;
  q = a == 0 ? 1 + x : 1 + y;
  if (p > q) {
    const int t = p;
    p = q;
    q = t;
  }
}

// Items e = first, first + step, ... < count of an (outer, inner) grid with
// `inner` columns, walked without divisions: (o, i) advances by (dq, dr).
struct JacIter {
  int o, i, dq, dr, inner;
  __device__ JacIter(int first, int step, int inner_) : inner(inner_) {
    o = first / inner_;
    i = first - o * inner_;
    dq = step / inner_;
    dr = step - dq * inner_;
  }
  __device__ __forceinline__ void next() {
    o += dq;
    i += dr;
    if (i >= inner) {
      i -= inner;
      ++o;
    }
  }
};

// W <- W J for one round (cr: (c, s) per slot, pr: p | q << 16 per slot; a
// column index >= ma is the dummy slot): items (row < rows, slot) from
// `first` by `step` (it: the walk from `first`), four in flight.
template <int LDW>
__device__ __forceinline__ void jac_apply_w(double* W, const double2* cr, const int* pr, int rows, int ma, int npairs,
                                            int first, int step, JacIter it) {
  const int items = npairs * rows;
  for (int e0 = first; e0 < items; e0 += 4 * step) {
    double x[4], y[4];
    double2 cs[4];
    int p[4], q[4], row[4];
    bool on[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      on[u] = e0 + u * step < items;
      row[u] = it.o;
      const int pq = on[u] ? pr[it.i] : 0;
      p[u] = pq & 0xffff;
      q[u] = pq >> 16;
      on[u] = on[u] && q[u] < ma;  // the dummy slot has no column
      if (on[u]) {
        cs[u] = cr[it.i];
        x[u] = W[row[u] * LDW + p[u]];
        y[u] = W[row[u] * LDW + q[u]];
      }
      it.next();
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (on[u]) {
        W[row[u] * LDW + p[u]] = cs[u].x * x[u] - cs[u].y * y[u];
        W[row[u] * LDW + q[u]] = cs[u].y * x[u] + cs[u].x * y[u];
      }
  }
}

// True when the `lead` largest eigenvalues of the symmetric A (m x m, LDS)
// belong to its leading rows: the Gershgorin discs of rows < lead lie above
// those of the other rows, and the coupling between the two sets is at most
// rel_off2 of ||A||_F^2 (uniform across the block; scratch[0..34]).
template <int LDA>
__device__ bool lead_block_separated(const double* A, int m, int lead, double rel_off2, double* scratch) {
  const int tid = threadIdx.x, nt = blockDim.x;
  // per row: Gershgorin radius, squared coupling to the other set, squares
  double lo = INFINITY, hi = -INFINITY, cpl = 0.0, tot = 0.0;
  if (tid < m) {
    double rad = 0.0;
    for (int j = 0; j < m; ++j) {
      const double v = A[tid * LDA + j];
      tot += v * v;
      if (j != tid) rad += fabs(v);
      if ((j < lead) != (tid < lead)) cpl += v * v;
    }
    const double d = A[tid * LDA + tid];
    if (tid < lead) lo = d - rad;
    else hi = d + rad;
  }
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off, 64));
    hi = fmax(hi, __shfl_xor(hi, off, 64));
  }
  cpl = wave_sum(cpl);
  tot = wave_sum(tot);
  if ((tid & 63) == 0) {
    const int w = tid >> 6;
    scratch[w] = lo; scratch[8 + w] = hi; scratch[16 + w] = cpl; scratch[24 + w] = tot;
  }
  __syncthreads();
  if (tid == 0) {
    double l = INFINITY, h = -INFINITY, c = 0.0, t = 0.0;
    for (int w = 0; w < nt / 64 && w < 8; ++w) {
      l = fmin(l, scratch[w]); h = fmax(h, scratch[8 + w]); c += scratch[16 + w]; t += scratch[24 + w];
    }
    scratch[34] = (l > h && c <= rel_off2 * t) ? 1.0 : 0.0;
  }
  __syncthreads();
  const bool ok = scratch[34] != 0.0;
  __syncthreads();
  return ok;
}

// The leading ma eigenvectors of a symmetric m x m A that is nearly diagonal
// but for its trailing block, A = D + E (D its diagonal), by second-order
// perturbation theory: with M[l][i] = E[l][i] / (d_i - d_l) (l != i < ma),
//   v_i = e_i + M e_i + sum_l e_l (E M)[l][i] / (d_i - d_l) - e_i sum_l M[l][i]^2 / 2,
//   lambda_i = d_i + sum_l E[l][i] M[l][i].
// With mu = max |M|, g the same over the trailing rows l >= ma, and rho the
// largest ratio of a trailing row's absolute sum within the trailing block to
// its distance from the leading diagonal entries, the neglected terms are sums
// of up to ma^2 products of three entries of M, and rho^2 g: taken when the
// trailing diagonal lies below the leading one, mu <= mu_max, rho <= 0.05 and
// rho^2 g <= 1e-13.  Returns 2 when mu <= 1e-5 (vectors good to ~1e-12), 1
// otherwise (~1e-7: enough to go on with the iteration, not to end it), 0,
// with nothing but scratch written, when not taken.  Writes columns < ma of W
// (the identity on entry) and A's leading diagonal = the eigenvalues (its
// other entries are left as they were).  Mbuf, Pbuf: m x ma LDS scratch
// (stride ma).  Replaces the direct solver in a converging warm solve (n = 256,
// k = 32, block 48): 125 -> 18 us.
template <int LDA, int LDW>
__device__ int perturb_eigvecs(double* A, double* W, int m, int ma, double* Mbuf, double* Pbuf, double* scratch,
                               double mu_max) {
  const int tid = threadIdx.x, nt = blockDim.x;
  double mu = 0.0, g = 0.0;
  for (int e = tid; e < m * ma; e += nt) {
    const int l = e / ma, i = e - l * ma;
    double mv = 0.0;
    if (l != i) mv = A[l * LDA + i] / (A[i * LDA + i] - A[l * LDA + l]);
    Mbuf[e] = mv;
    const double mag = isfinite(mv) ? fabs(mv) : INFINITY;
    mu = fmax(mu, mag);
    if (l >= ma) g = fmax(g, mag);
  }
  // trailing row tid: its sum, and its distance from the leading entries
  double rho = 0.0;
  if (tid >= ma && tid < m) {
    double rad = 0.0, lo = INFINITY;
#pragma unroll 4
    for (int j = ma; j < m; ++j) rad += j == tid ? 0.0 : fabs(A[tid * LDA + j]);
#pragma unroll 4
    for (int i = 0; i < ma; ++i) lo = fmin(lo, A[i * LDA + i]);
    const double gap = lo - A[tid * LDA + tid];
    rho = gap > 0.0 && isfinite(rad) ? rad / gap : INFINITY;
  }
  for (int off = 32; off > 0; off >>= 1) {
    mu = fmax(mu, __shfl_xor(mu, off, 64));
    g = fmax(g, __shfl_xor(g, off, 64));
    rho = fmax(rho, __shfl_xor(rho, off, 64));
  }
  if ((tid & 63) == 0) {
    const int w = tid >> 6;
    scratch[w] = mu; scratch[8 + w] = g; scratch[16 + w] = rho;
  }
  __syncthreads();
  for (int w = 0; w < nt / 64; ++w) {
    mu = fmax(mu, scratch[w]); g = fmax(g, scratch[8 + w]); rho = fmax(rho, scratch[16 + w]);
  }
  __syncthreads();
  if (!(mu <= mu_max && rho <= 0.05 && rho * rho * g <= 1e-13)) return 0;
  // P = E M (E: A without its diagonal)
  for (int e = tid; e < m * ma; e += nt) {
    const int l = e / ma, i = e - l * ma;
    double pv = 0.0;
#pragma unroll 8
    for (int q = 0; q < m; ++q) pv = fma(q == l ? 0.0 : A[l * LDA + q], Mbuf[q * ma + i], pv);
    Pbuf[e] = pv;
  }
  __syncthreads();
  for (int e = tid; e < m * ma; e += nt) {
    const int l = e / ma, i = e - l * ma;
    double wv;
    if (l != i) {
      wv = Mbuf[e] + Pbuf[e] / (A[i * LDA + i] - A[l * LDA + l]);
    } else {
      double n2 = 0.0;
#pragma unroll 4
      for (int q = 0; q < m; ++q) n2 = fma(Mbuf[q * ma + i], Mbuf[q * ma + i], n2);
      wv = 1.0 - 0.5 * n2;
    }
    W[l * LDW + i] = wv;
  }
  // eigenvalues after every thread has read the diagonal above
  double lam = 0.0;
  if (tid < ma) {
    lam = A[tid * LDA + tid];
#pragma unroll 4
    for (int l = 0; l < m; ++l) lam = fma(l == tid ? 0.0 : A[l * LDA + tid], Mbuf[l * ma + tid], lam);
  }
  __syncthreads();
  if (tid < ma) A[tid * LDA + tid] = lam;
  __syncthreads();
  return mu <= 1e-5 ? 2 : 1;
}

// One sweep is me - 1 rounds of me / 2 disjoint rotations.  Per round: wave 0
// computes the round's rotations (c, s and the pair p | q << 16 per slot, in
// cs / pr, two rounds' worth each) while the other waves apply the previous
// round's to W; after a barrier every thread applies A <- J^T A J to whole
// 2 x 2 blocks (two in flight).  Every thread's items are fixed for the call
// and walked without divisions.
//
// lead > 0: only the eigenpairs of the `lead` largest eigenvalues are wanted.
// If the Gershgorin discs of rows < lead lie above those of the other rows
// (so the lead largest eigenvalues belong to the leading rows) and the
// coupling between the two sets is below the threshold
// (lead_block_separated; lead_known: its answer if already known, -1 not),
// the sweeps rotate the leading lead x lead block only; the coupling and the
// trailing block are left as they are (W must be the identity on entry; its
// trailing columns stay so).  Returns the number of sweeps.
template <int LDA, int LDW>
__device__ int lds_jacobi(double* A, double* W, int m, int max_sweeps, double2* cs, int* pr, double* scratch,
                          double rel_off2 = 1e-30, int lead = 0, int lead_known = -1) {
  const int tid = threadIdx.x, nt = blockDim.x;
  int ma = m;  // the rows and columns the sweeps rotate
  if (lead > 0 && lead < m && (lead_known == 1 || (lead_known < 0 && lead_block_separated<LDA>(A, m, lead, rel_off2, scratch))))
    ma = lead;
  const int me = ma + (ma & 1);  // even number of slots (one dummy)
  const int npairs = me / 2, nblk = npairs * npairs;
  const JacIter blk0(tid, nt, npairs);                         // A blocks (pa, pb)
  const JacIter wside(tid < 64 ? 0 : tid - 64, nt - 64, npairs);  // W (row, slot), waves 1..
  const JacIter wall(tid, nt, npairs);                         // W (row, slot), every thread
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    // off-diagonal and total Frobenius norms of the rotated block
    double off = 0.0, tot = 0.0;
    for (int e = tid; e < ma * ma; e += nt) {
      const int i = e / ma, j = e % ma;
      const double v = A[i * LDA + j];
      tot += v * v;
      if (i != j) off += v * v;
    }
    off = wave_sum(off);
    tot = wave_sum(tot);
    if ((tid & 63) == 0) { scratch[tid >> 6] = off; scratch[16 + (tid >> 6)] = tot; }
    __syncthreads();
    if (tid == 0) {
      double o = 0.0, t = 0.0;
      for (int w = 0; w < nt / 64; ++w) { o += scratch[w]; t += scratch[16 + w]; }
      scratch[32] = o;
      scratch[33] = t;
    }
    __syncthreads();
    if (!(scratch[32] > rel_off2 * scratch[33]) || scratch[33] == 0.0) break;
    for (int round = 0; round < me - 1; ++round) {
      double2* cr = cs + (round & 1) * npairs;
      int* prr = pr + (round & 1) * npairs;
      if (tid < 64) {
        if (tid < npairs) {
          int p, q;
          jac_pair(tid, round, me, p, q);
          double c = 1.0, s = 0.0;
          if (q < ma) {
            const double apq = A[p * LDA + q], app = A[p * LDA + p], aqq = A[q * LDA + q];
            if (fabs(apq) > 1e-300) {
              // tan of the rotation angle t = sgn(tau) / (|tau| + sqrt(1 + tau^2)),
              // c = 1 / sqrt(1 + t^2); reciprocals and reciprocal square roots
              // from the hardware estimates refined by Newton steps (this
              // is on the critical path of every round)
              const double tau = (aqq - app) * jac_recip(2.0 * apq);
              const double at = fabs(tau);
              double t;
              if (at > 1e100) {
                t = 0.5 / at;
              } else {
                const double u = 1.0 + tau * tau;
                t = jac_recip(at + u * jac_rsqrt(u));
              }
              t = tau >= 0.0 ? t : -t;
              c = jac_rsqrt(1.0 + t * t);
              s = t * c;
            }
          }
          cr[tid] = double2{c, s};
          prr[tid] = p | (q << 16);
        }
      } else if (round > 0) {
        jac_apply_w<LDW>(W, cs + ((round - 1) & 1) * npairs, pr + ((round - 1) & 1) * npairs, ma, ma, npairs,
                         tid - 64, nt - 64, wside);
      }
      __syncthreads();
      // A <- J^T A J: each thread owns whole 2 x 2 blocks (rows of pair pa,
      // columns of pair pb), so no entry is touched twice
      JacIter it = blk0;
      for (int e0 = tid; e0 < nblk; e0 += 2 * nt) {
        double v[2][4];
        double2 ca[2], cb[2];
        int p0[2], q0[2], p1[2], q1[2];
        bool on[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          on[u] = e0 + u * nt < nblk;
          if (on[u]) {
            const int pqa = prr[it.o], pqb = prr[it.i];
            ca[u] = cr[it.o];
            cb[u] = cr[it.i];
            p0[u] = pqa & 0xffff; q0[u] = pqa >> 16;
            p1[u] = pqb & 0xffff; q1[u] = pqb >> 16;
            const bool r1 = q0[u] < ma, c1 = q1[u] < ma;  // the dummy slot has no row / column
            v[u][0] = A[p0[u] * LDA + p1[u]];
            v[u][1] = c1 ? A[p0[u] * LDA + q1[u]] : 0.0;
            v[u][2] = r1 ? A[q0[u] * LDA + p1[u]] : 0.0;
            v[u][3] = (r1 && c1) ? A[q0[u] * LDA + q1[u]] : 0.0;
          }
          it.next();
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          if (!on[u]) continue;
          const bool r1 = q0[u] < ma, c1 = q1[u] < ma;
          const double sa = ca[u].y, cc = ca[u].x, sb = cb[u].y, cd = cb[u].x;
          const double u00 = cc * v[u][0] - sa * v[u][2], u01 = cc * v[u][1] - sa * v[u][3];
          const double u10 = sa * v[u][0] + cc * v[u][2], u11 = sa * v[u][1] + cc * v[u][3];
          A[p0[u] * LDA + p1[u]] = cd * u00 - sb * u01;
          if (c1) A[p0[u] * LDA + q1[u]] = sb * u00 + cd * u01;
          if (r1) A[q0[u] * LDA + p1[u]] = cd * u10 - sb * u11;
          if (r1 && c1) A[q0[u] * LDA + q1[u]] = sb * u10 + cd * u11;
        }
      }
      __syncthreads();
    }
    // the last round's rotations into W
    jac_apply_w<LDW>(W, cs + ((me - 2) & 1) * npairs, pr + ((me - 2) & 1) * npairs, ma, ma, npairs, tid, nt, wall);
    __syncthreads();
  }
  return sweep;
}

// order[r] = index of the r-th largest diagonal entry of A (ties by index,
// NaN last: order is a permutation whatever A holds, as it indexes memory)
template <int LDA>
__device__ void sort_desc(const double* A, int m, int* order) {
  const int tid = threadIdx.x;
  if (tid < m) {
    auto key = [=](int i) {
      const double v = A[i * LDA + i];
      return v == v ? v : -INFINITY;
    };
    const double v = key(tid);
    int rank = 0;
    for (int j = 0; j < m; ++j) {
      const double u = key(j);
      if (u > v || (u == v && j < tid)) ++rank;
    }
    order[rank] = tid;
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// Direct solver: the leading ne eigenpairs of an n x n symmetric matrix,
// n <= 64 NB, by one workgroup.
//
//  1. Householder tridiagonalisation with the matrix in registers: four
//     lanes share a row.  Every wave forms the reflector redundantly from the
//     published column, so a step has two barriers: around the sum of the
//     four partial products per row and before the next column is read.
//  2. Eigenvalues by Sturm counts (signs of the leading principal minors),
//     512 / ne points of each one's interval at a time.
//  3. Eigenvectors of the tridiagonal matrix from its twisted factorisation:
//     one thread eliminates from the top, one from the bottom, and the twist
//     is where the two meet with the least remainder gamma; gamma / ||z|| is
//     the residual.
//  4. Back transformation, eight lanes per column.
//  5. One Newton step towards orthonormal columns, Z <- Z (3 I - Z^T Z) / 2.
//
// Returns false, with nothing but scratch written, when two eigenvalues after
// step 2 are within 1e-14 of the norm, a residual exceeds 1e-13 of it or the
// vectors before step 5 are not orthogonal to 1e-8 (clusters of eigenvalues,
// where the vectors of one are not determined by their own value), for NaN and
// for norms outside [1e-200, 1e150]: the caller then takes the Jacobi sweeps,
// which need no separation.  (Implicit QR steps from the same tridiagonal form
// took a sixth of the sweeps' time, but give another basis of a null space, which
// factors of more columns than the rank then show.)  The FP64 instructions that
// one workgroup issues bound it, most of all in 1 (1.1 us a step up to 64 rows,
// 1.7 above).  Measured, one call:
// n = 120, k = 10: 317 us against 9.4 ms of Jacobi sweeps; n = 128, k = 128:
// 605 us against 11.0 ms; n = 48, k = 10: 90 us against 825; a 48 x 48 Ritz
// matrix: 103 us against 94 per sweep.
// ---------------------------------------------------------------------------
template <int NB>
struct DirectLds {
  static constexpr int N = 64 * NB;
  double d[N], e[N], e2[N], tau[N], col[N];
  double vbuf[kEigWaves][N];  // per wave; then the intervals of the eigenvalues
  double wbuf[kEigWaves][N];  // per wave; then gamma and norms
  double pbuf[4][N];          // then the Sturm counts
  int ok;                     // 2: the matrix is diagonal
};

template <>
struct DirectLds<0> {};  // (a block that does not use it)

// Sum over the wave, the same value in every lane (row shifts and row
// broadcasts; no LDS).
__device__ __forceinline__ double dpp_wave_sum(double v) {
#define TLA_DPP_ADD(CTRL, ROWS)                                                \
  {                                                                            \
    const int2 w = *(const int2*)&v;                                           \
    int2 r;                                                                    \
    r.x = __builtin_amdgcn_update_dpp(0, w.x, CTRL, ROWS, 0xf, true);          \
    r.y = __builtin_amdgcn_update_dpp(0, w.y, CTRL, ROWS, 0xf, true);          \
    v += *(const double*)&r;                                                   \
  }
  TLA_DPP_ADD(0x111, 0xf)  // row_shr:1
  TLA_DPP_ADD(0x112, 0xf)
  TLA_DPP_ADD(0x114, 0xf)
  TLA_DPP_ADD(0x118, 0xf)
  TLA_DPP_ADD(0x142, 0xa)  // row_bcast:15 into rows 1 and 3
  TLA_DPP_ADD(0x143, 0xc)  // row_bcast:31 into rows 2 and 3
#undef TLA_DPP_ADD
  const int2 w = *(const int2*)&v;
  int2 r;
  r.x = __builtin_amdgcn_readlane(w.x, 63);
  r.y = __builtin_amdgcn_readlane(w.y, 63);
  return *(const double*)&r;
}

// v + v of the lane that CTRL (quad permutation, half-row mirror) names
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const int2 w = *(const int2*)&v;
  int2 r;
  r.x = __builtin_amdgcn_update_dpp(0, w.x, CTRL, 0xf, 0xf, true);
  r.y = __builtin_amdgcn_update_dpp(0, w.y, CTRL, 0xf, 0xf, true);
  return v + *(const double*)&r;
}

// Z <- H_0 H_1 ... Z: eight columns of a wave at a time, eight lanes per
// column, each with 8 NB consecutive rows in registers.
template <int NB>
__device__ __forceinline__ void direct_back(const double* Vh, double* Z, int ldZ, int n, int ne, DirectLds<NB>& L) {
  constexpr int N = 64 * NB, M = 8 * NB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = (lane & 7) * M;
  for (int c0 = 8 * wave; c0 < ne; c0 += 8 * kEigWaves) {
    const int c = c0 + (lane >> 3);
    double z[M];
#pragma unroll
    for (int i = 0; i < M; ++i) z[i] = r0 + i < n && c < ne ? Z[(r0 + i) * ldZ + c] : 0.0;
    for (int j = n - 3; j >= 0; --j) {
      double v[M], s[2] = {0.0, 0.0};
#pragma unroll
      for (int i = 0; i < M; ++i) v[i] = Vh[j * N + r0 + i];
#pragma unroll
      for (int i = 0; i < M; ++i) s[i & 1] = fma(z[i], v[i], s[i & 1]);
      double t = s[0] + s[1];
      t = dpp_add<0xb1>(t);   // lanes 0-1, 2-3, ...
      t = dpp_add<0x4e>(t);   // quads
      t = dpp_add<0x141>(t);  // the mirrored quad of the eight lanes
      t *= -L.tau[j];
#pragma unroll
      for (int i = 0; i < M; ++i) z[i] = fma(t, v[i], z[i]);
    }
#pragma unroll
    for (int i = 0; i < M; ++i)
      if (r0 + i < n && c < ne) Z[(r0 + i) * ldZ + c] = z[i];
  }
}

// place[i] = the place of d[i] in descending order (of equal ones, the first
// first).  Begins and ends with a barrier.
__device__ __forceinline__ void descending(const double* d, int n, int* place) {
  __syncthreads();
  const int tid = threadIdx.x;
  if (tid < n) {
    const double t = d[tid];
    int rank = 0;
    for (int i = 0; i < n; ++i) rank += d[i] > t || (d[i] == t && i < tid);
    place[tid] = rank;
  }
  __syncthreads();
}

// get(i, c): the matrix.  Vh: n x 64 NB (the reflectors, then the corrected
// vectors), S: ldS >= round16(ne), round16(n) rows; Z: likewise, the vectors
// on return (columns in descending order of theta).  theta: ne.  WHOLE: a matrix
// of the caller's; diagonal ones and clusters are seen early.  (A Ritz matrix is
// next to diagonal as a rule, its null space in no order, and graded: vectors
// of eigenvalues close to one another may hold all the same.)
template <int NB, bool WHOLE, typename Get>
__device__ bool direct_eig(Get get, int n, int ne, double* Vh, double* S, int ldS, double* Z, int ldZ, double* theta,
                           DirectLds<NB>& L) {
  constexpr int N = 64 * NB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // thread (row, lk): columns 64 b + 16 s + 4 lk + u of its row
  const int lr = lane & 15, lk = lane >> 4, row = 16 * wave + lr;
  const bool works = wave < 4 * NB, rowok = works && row < n;
  double x[NB][4][4];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = b * 64 + s * 16 + lk * 4 + u;
        x[b][s][u] = rowok && c < n ? get(row, c) : 0.0;
      }
  if (rowok && lk == 0) L.col[row] = x[0][0][0];
  // a matrix that is diagonal already, by the measure of the Jacobi sweeps, has
  // its entries and unit vectors (n = 128: 590 us -> 28)
  if constexpr (WHOLE) {
    double off = 0.0, diag = 0.0;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const double sq = x[b][s][u] * x[b][s][u];
          if (b * 64 + s * 16 + lk * 4 + u == row) {
            diag += sq;
            if (rowok) L.d[row] = x[b][s][u];
          } else {
            off += sq;
          }
        }
    off = dpp_wave_sum(off);
    diag = dpp_wave_sum(diag);
    if (lane == 0) L.wbuf[0][2 * wave] = off, L.wbuf[0][2 * wave + 1] = diag;
    __syncthreads();
    off = 0.0, diag = 0.0;
    for (int w = 0; w < 4 * NB; ++w) off += L.wbuf[0][2 * w], diag += L.wbuf[0][2 * w + 1];
    if (off <= 1e-30 * (off + diag)) {  // (the same for every thread)
      int* place = (int*)L.pbuf;
      for (int e = tid; e < n * ne; e += kEigThreads) Z[(e / ne) * ldZ + e % ne] = 0.0;
      descending(L.d, n, place);
      if (tid < n && place[tid] < ne) {
        theta[place[tid]] = L.d[tid];
        Z[tid * ldZ + place[tid]] = 1.0;
      }
      if (tid == 0) L.ok = 2;
      __syncthreads();
      return true;
    }
  }
  __syncthreads();
  double* vb = L.vbuf[wave];
  double* wb = L.wbuf[wave];
#pragma unroll 1
  for (int j = 0; j + 2 < n; ++j) {
    double v[NB], tau = 0.0;
    const bool busy = works && 16 * wave + 15 > j;  // rows past j among this wave's
    if (works) {
      double xs = 0.0;
      const double alpha = L.col[j + 1], dj = L.col[j];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int i = lane + 64 * b;
        v[b] = i > j && i < n ? L.col[i] : 0.0;
        xs += i > j + 1 ? v[b] * v[b] : 0.0;
      }
      const double sigma = dpp_wave_sum(xs);
      double beta = alpha, inv = 0.0;
      if (sigma > 1e-300) {
        const double s2 = fma(alpha, alpha, sigma), rn = jac_rsqrt(s2);
        beta = -copysign(s2 * rn, alpha);
        tau = fma(fabs(alpha), rn, 1.0);  // (beta - alpha) / beta
        inv = jac_recip_signed(alpha - beta);
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int i = lane + 64 * b;
        v[b] = i == j + 1 ? (tau != 0.0 ? 1.0 : 0.0) : v[b] * inv;
        vb[i] = v[b];
        if (wave == 0) Vh[j * N + i] = v[b];
      }
      if (tid == 0) {
        L.d[j] = dj;
        L.e[j] = beta;
        L.tau[j] = tau;
      }
      __builtin_amdgcn_wave_barrier();
      if (busy) {
        double p[4] = {0.0, 0.0, 0.0, 0.0};  // four short chains
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int s = 0; s < 4; ++s)
            if (b * 64 + s * 16 + 15 > j) {  // (columns up to j are done)
#pragma unroll
              for (int u = 0; u < 4; ++u) p[u] = fma(x[b][s][u], vb[b * 64 + s * 16 + lk * 4 + u], p[u]);
            }
        L.pbuf[lk][row] = (p[0] + p[1]) + (p[2] + p[3]);
      }
    }
    __syncthreads();
    if (busy) {
      double p[NB], pv = 0.0;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int i = lane + 64 * b;
        p[b] = i > j && i < n ? (L.pbuf[0][i] + L.pbuf[1][i]) + (L.pbuf[2][i] + L.pbuf[3][i]) : 0.0;
        pv = fma(p[b], v[b], pv);
      }
      const double kk = 0.5 * tau * tau * dpp_wave_sum(pv);
#pragma unroll
      for (int b = 0; b < NB; ++b) wb[lane + 64 * b] = tau * p[b] - kk * v[b];
      __builtin_amdgcn_wave_barrier();
      const double vr = -vb[row], wr = -wb[row];
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          if (b * 64 + s * 16 + 15 > j) {
            const int c = b * 64 + s * 16 + lk * 4;
#pragma unroll
            for (int u = 0; u < 4; ++u) x[b][s][u] = fma(wr, vb[c + u], fma(vr, wb[c + u], x[b][s][u]));
            // publish column j + 1
            if ((j + 1) >> 4 == b * 4 + s && rowok && lk == (((j + 1) >> 2) & 3)) {
              const int u = (j + 1) & 3;
              L.col[row] = u == 0 ? x[b][s][0] : u == 1 ? x[b][s][1] : u == 2 ? x[b][s][2] : x[b][s][3];
            }
          }
    }
    __syncthreads();
  }
  // the last two rows
  if (tid == 0 && n >= 2) {
    L.d[n - 2] = L.col[n - 2];
    L.e[n - 2] = L.col[n - 1];
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (rowok && row == n - 1 && b * 64 + s * 16 + lk * 4 + u == n - 1) L.d[n - 1] = x[b][s][u];
  __syncthreads();
  // Gershgorin bounds of the spectrum (every wave the same)
  double gl = INFINITY, gu = -INFINITY;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int i = lane + 64 * b;
    if (i < n) {
      const double r = (i > 0 ? fabs(L.e[i - 1]) : 0.0) + (i + 1 < n ? fabs(L.e[i]) : 0.0);
      gl = fmin(gl, L.d[i] - r);
      gu = fmax(gu, L.d[i] + r);
    }
    if (wave == 0) L.e2[i] = i + 1 < n ? L.e[i] * L.e[i] : 0.0;
  }
  for (int off = 32; off > 0; off >>= 1) {
    gl = fmin(gl, __shfl_xor(gl, off, 64));
    gu = fmax(gu, __shfl_xor(gu, off, 64));
  }
  const double tn = fmax(fabs(gl), fabs(gu));
  if (!(tn > 1e-200 && tn < 1e150)) return false;  // (the same for every thread)
  const double pivmin = 1e-46 * tn, eps = 2.3e-16;
  // the scaled matrix as (d_i, -e_{i-1}^2); past its end entries above every
  // x, which change no sign
  const double sc = ldexp(1.0, -ilogb(tn));
  double2* tri = (double2*)L.vbuf[2];
  if (tid < N + 8) {
    const double es = tid > 0 && tid < n ? L.e[tid - 1] * sc : 0.0;
    tri[tid] = double2{tid < n ? L.d[tid] * sc : 8.0, -es * es};
  }
  double* lo = L.vbuf[0];
  double* hi = L.vbuf[1];
  int* cnt = (int*)L.pbuf;
  if (tid < ne) {
    lo[tid] = gl - 4 * eps * tn;
    hi[tid] = gu + 4 * eps * tn;
  }
  if (tid == 0) L.ok = 1;
  __syncthreads();
  {
    const int npt = kEigThreads / ne, r = tid / npt, pt = tid - r * npt;
    const int want = n - 1 - r;  // eigenvalues below the r-th largest
    const bool on = r < ne;
    int passes = 1;
    for (double w = npt + 1.0; w < 1.2e17; w *= npt + 1.0) ++passes;
    for (int pass = 0; pass < passes; ++pass) {
      double a = 0.0, w = 0.0, xv = 0.0;
      int c = 0;
      if (on) {
        a = fmin(lo[r], hi[r]);
        w = (fmax(lo[r], hi[r]) - a) / (npt + 1);
        xv = a + w * (pt + 1);
        // signs of the leading principal minors of (T - x I) / sc, two
        // multiply-adds per step; every eight steps the last two are scaled
        // back (a step grows them at most tenfold, and shrinks them no
        // further than 1e-17 of the norm at a time)
        double m0 = 1.0, m1 = 0.0;  // the minors of orders i and i - 1
        const double xs = xv * sc;
        for (int i0 = 0; i0 < n; i0 += 8) {
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const double2 de = tri[i0 + u];
            const double t = fma(de.x - xs, m0, de.y * m1);
            c += (uint32_t)(__double2hiint(t) ^ __double2hiint(m0)) >> 31;
            m1 = m0;
            m0 = t;
          }
          const int ex = -max(ilogb_fast(m0), ilogb_fast(m1));
          m0 = ldexp(m0, ex);
          m1 = ldexp(m1, ex);
        }
        cnt[tid] = c;
      }
      __syncthreads();
      if (on) {
        const bool over = c > want, before = pt > 0 && cnt[tid - 1] > want;
        if (over && !before) {
          lo[r] = xv - w;
          hi[r] = xv;
        } else if (!over && pt == npt - 1) {
          lo[r] = xv;
          hi[r] = xv + w;
        }
      }
      __syncthreads();
    }
  }
  // eigenvalues this close give one vector twice, orthogonal to 1e-2 at best:
  // what follows would be in vain (n = 128, clusters of four: 0.39 ms before the
  // sweeps' 15.4, 0.63 with the whole attempt; n = 16: 26 and 31 us before 192)
  if constexpr (WHOLE) {
    if (tid + 1 < ne && lo[tid] + hi[tid] - (lo[tid + 1] + hi[tid + 1]) < 2e-14 * tn) L.ok = 0;
    __syncthreads();
    if (!L.ok) return false;
  }
  // twisted factorisations: thread r from the top, thread 256 + r from the bottom
  const int r = tid & 255;
  const bool down = tid < 256, on = r < ne;
  const double lam = on ? 0.5 * (lo[r] + hi[r]) : 0.0;
  double* gam = L.wbuf[0];
  double* nrm = L.wbuf[1];  // [0, N) top, [N, 2 N) bottom
  int* twist = (int*)L.wbuf[3];
  if (on) {
    double q = down ? L.d[0] - lam : L.d[n - 1] - lam;
    if (fabs(q) < pivmin) q = -pivmin;
    if (down) {
      S[r] = q;
      for (int i = 1; i < n; ++i) {
        q = (L.d[i] - lam) - L.e2[i - 1] * jac_recip_signed(q);
        if (fabs(q) < pivmin) q = -pivmin;
        S[i * ldS + r] = q;
      }
    } else {
      Z[(n - 1) * ldZ + r] = q;
      for (int i = n - 2; i >= 0; --i) {
        q = (L.d[i] - lam) - L.e2[i] * jac_recip_signed(q);
        if (fabs(q) < pivmin) q = -pivmin;
        Z[i * ldZ + r] = q;
      }
    }
  }
  __syncthreads();
  if (on && down) {
    double best = INFINITY, g = 0.0;
    int at = 0;
    for (int i = 0; i < n; ++i) {
      const double gi = S[i * ldS + r] + Z[i * ldZ + r] - (L.d[i] - lam);
      if (fabs(gi) < best) {
        best = fabs(gi);
        g = gi;
        at = i;
      }
    }
    gam[r] = g;
    twist[r] = at;
  }
  __syncthreads();
  if (on) {
    const int at = twist[r];
    double z = 1.0, s2 = 0.0;
    if (down) {  // upwards from the twist, over S
      for (int i = at - 1; i >= 0; --i) {
        z = -z * L.e[i] * jac_recip_signed(S[i * ldS + r]);
        S[i * ldS + r] = z;
        s2 = fma(z, z, s2);
      }
    } else {  // downwards, over Z
      for (int i = at + 1; i < n; ++i) {
        z = -z * L.e[i - 1] * jac_recip_signed(Z[i * ldZ + r]);
        Z[i * ldZ + r] = z;
        s2 = fma(z, z, s2);
      }
    }
    nrm[(down ? 0 : N) + r] = s2;
  }
  __syncthreads();
  const int n16 = (n + 15) & ~15, ne16 = (ne + 15) & ~15;
  if (tid < ne) {
    const double s2 = 1.0 + nrm[tid] + nrm[N + tid], g = gam[tid];
    theta[tid] = lam + g / s2;
    if (!(fabs(g) <= 1e-13 * tn * sqrt(s2))) L.ok = 0;  // (NaN included)
  }
  // unit columns into Z, zero columns and rows up to the matrix tiles
  for (int e = tid; e < n16 * ne16; e += kEigThreads) {
    const int i = e / ne16, c = e - i * ne16;
    double z = 0.0;
    if (i < n && c < ne) {
      const int at = twist[c];
      z = (i == at ? 1.0 : i < at ? S[i * ldS + c] : Z[i * ldZ + c]) / sqrt(1.0 + nrm[c] + nrm[N + c]);
    }
    Z[i * ldZ + c] = z;
  }
  __syncthreads();
  if (!L.ok) return false;
  direct_back<NB>(Vh, Z, ldZ, n, ne, L);
  __syncthreads();
  block_gemm_sym_f64(Z, ldZ, Z, ldZ, S, ldS, ne16, n16);
  double worst = 0.0;
  for (int e = tid; e < ne16 * ne16; e += kEigThreads) {
    const int i = e / ne16, c = e - i * ne16;
    const double v = S[i * ldS + c], id = i == c ? 1.0 : 0.0;
    if (i < ne && c < ne) worst = fmax(worst, isfinite(v) ? fabs(v - id) : INFINITY);
    S[i * ldS + c] = 1.5 * id - 0.5 * v;
  }
  if (!(worst <= 1e-8)) L.ok = 0;
  __syncthreads();
  if (!L.ok) return false;
  block_gemm_f64<false>(Z, ldZ, S, ldS, Vh, N, n16, ne16, ne16);
  for (int e = tid; e < n * ne; e += kEigThreads) {
    const int i = e / ne, c = e - i * ne;
    Z[i * ldZ + c] = Vh[i * N + c];
  }
  __syncthreads();
  return true;
}

// ---------------------------------------------------------------------------
struct EigArgs {
  const double* G;
  int n, k;
  const double* Q0;  // warm start (row-major, ld q0_ld) or nullptr; its first k0 columns are used
  int k0, q0_ld;
  double* evals;     // k
  double* evecs;     // n x k row-major
  double tol;
  int max_iter;
  int* iters;
  int np;     // n rounded up to a multiple of 16 (subspace kernel)
  double* Gp;  // np x np zero-padded copy of G (subspace kernel)
  double* V;   // np x capacity, likewise Z, Y, U
  double* Z;
  double* Y;
  double* U;
  double* W;  // rotations when they do not fit LDS
  double* T;  // orthonormalising factor when it does not fit LDS
  // singular-vector outputs (tla_gram_left_singular; zero / NULL otherwise)
  int flip;        // apply the u-based sign rule to the k leading vectors
  int out_dtype;   // TLA_F32 / TLA_F64 for u_out and s_out
  void* u_out;     // n x k sign-corrected vectors in out_dtype
  void* s_out;     // k square roots of max(eigenvalue, 0) in out_dtype
  double* wblk;    // n x b: the whole final block (subspace kernel)
  int wblock;      // Q0 is a whole block (k0 == b) used without orthonormalising
};

// Output of one problem: the k leading eigenpairs are column colmap[r] (r
// without a map) of Ysrc (ld ldy) and theta[r].  evals / evecs as
// tla_sym_eig writes them (when non-NULL); with a.flip the reference's
// u-based sign rule first (each column multiplied by the sign of its entry
// of largest magnitude, as rounded to the output's type, the first such row
// on ties: entries that are equal but for the last bits of the solve do not
// decide by those; sgn: k doubles of LDS);
// u_out / s_out in a.out_dtype; with a.wblk the first nb columns of Ysrc.
__device__ void eig_emit(const EigArgs& a, const double* Ysrc, int ldy, const int* colmap, const double* theta,
                         double* sgn, int nb) {
  const int tid = threadIdx.x, nt = blockDim.x, n = a.n, k = a.k;
  if (a.flip) {
    for (int r = tid >> 6; r < k; r += nt >> 6) {
      const int c = colmap ? colmap[r] : r;
      double best = -1.0;
      int bi = 0;
      for (int i = tid & 63; i < n; i += 64) {
        double v = fabs(Ysrc[i * ldy + c]);
        if (a.out_dtype == TLA_F32) v = (float)v;
        if (v > best) {
          best = v;
          bi = i;
        }
      }
      for (int off = 32; off > 0; off >>= 1) {
        const double ob = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if ((tid & 63) == 0) {
        const double y = Ysrc[bi * ldy + c];
        sgn[r] = y > 0.0 ? 1.0 : (y < 0.0 ? -1.0 : 0.0);
      }
    }
    __syncthreads();
  }
  for (int e = tid; e < n * k; e += nt) {
    const int i = e / k, r = e - (e / k) * k;
    double v = Ysrc[i * ldy + (colmap ? colmap[r] : r)];
    if (a.flip) v *= sgn[r];
    if (a.evecs) a.evecs[e] = v;
    if (a.u_out) {
      if (a.out_dtype == TLA_F32) ((float*)a.u_out)[e] = (float)v;
      else ((double*)a.u_out)[e] = v;
    }
  }
  for (int r = tid; r < k; r += nt) {
    if (a.evals) a.evals[r] = theta[r];
    if (a.s_out) {
      const double sv = sqrt(fmax(theta[r], 0.0));
      if (a.out_dtype == TLA_F32) ((float*)a.s_out)[r] = (float)sv;
      else ((double*)a.s_out)[r] = sv;
    }
  }
  if (a.wblk)
    for (int e = tid; e < n * nb; e += nt) a.wblk[e] = Ysrc[(e / nb) * ldy + e % nb];
}

// Problems solved by one launch, one workgroup each (blockIdx.x selects).
constexpr int kEigMaxBatch = 8;
struct EigBatch {
  EigArgs a[kEigMaxBatch];
};

__device__ __forceinline__ double hash_unit(uint32_t i, uint32_t j) {
  uint32_t h = i * 0x9E3779B1u ^ (j + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 15; h *= 0x2C1B3C6Du; h ^= h >> 12; h *= 0x297A2D39u; h ^= h >> 15;
  return (double)h * (1.0 / 4294967296.0) - 0.5;
}

// Set-up of the subspace problems of one launch (blockIdx.y selects), spread
// over many workgroups: the zero-padded symmetric copy Gp = (G + G^T) / 2 in
// 32 x 32 tiles (the transposed tile of G read row by row through LDS), then
// the starting block Y (np x B): warm-start columns, then pseudo-random ones.
template <int B>
__global__ __launch_bounds__(256) void eig_prep_kernel(EigBatch batch, int gtiles) {
  const EigArgs a = batch.a[blockIdx.y];
  const int n = a.n, np = a.np, tid = threadIdx.x;
  if ((int)blockIdx.x < gtiles) {
    __shared__ double Tt[32][33];
    const int nt = (np + 31) / 32;
    if ((int)blockIdx.x >= nt * nt) return;
    const int ti = blockIdx.x / nt, tj = blockIdx.x % nt;
    for (int e = tid; e < 1024; e += 256) {  // Tt[r][c] = G[tj * 32 + r][ti * 32 + c]
      const int r = e >> 5, c = e & 31, gi = tj * 32 + r, gj = ti * 32 + c;
      Tt[r][c] = (gi < n && gj < n) ? a.G[(int64_t)gi * n + gj] : 0.0;
    }
    __syncthreads();
    for (int e = tid; e < 1024; e += 256) {
      const int r = e >> 5, c = e & 31, i = ti * 32 + r, j = tj * 32 + c;
      if (i < np && j < np) a.Gp[(int64_t)i * np + j] = (i < n && j < n) ? 0.5 * (a.G[(int64_t)i * n + j] + Tt[c][r]) : 0.0;
    }
    return;
  }
  const int64_t e = (int64_t)(blockIdx.x - gtiles) * 256 + tid;
  if (e >= (int64_t)np * B) return;
  const int i = (int)(e / B), j = (int)(e % B);
  a.Y[e] = i >= n ? 0.0 : ((a.Q0 && j < a.k0) ? a.Q0[(int64_t)i * a.q0_ld + j] : hash_unit(i, j));
}

// The whole matrix, n <= CAP: the direct solver, and Jacobi sweeps where it
// gives up.  CAP 64 keeps everything in LDS; CAP 128 keeps the reflectors (or
// the Jacobi's matrix) in LDS and the vectors in the workspace (a.W and a.Z,
// ld 128).
template <int CAP>
__global__ __launch_bounds__(kEigThreads) void sym_eig_small_kernel(EigBatch batch) {
  const EigArgs a = batch.a[blockIdx.x];
  constexpr int LDA = CAP + 1;
  constexpr bool LOCAL = CAP == kJac;
  __shared__ double A[CAP * LDA];
  __shared__ double Wl[LOCAL ? CAP * LDA : 1];
  __shared__ double Vl[LOCAL ? CAP * CAP : 1];
  __shared__ DirectLds<CAP / 64> dl;
  __shared__ double scratch[64];
  __shared__ int order[CAP];
  __shared__ double theta[CAP];
  __shared__ double sgn[CAP];
  constexpr int LDW = LOCAL ? LDA : CAP;
  double* W = LOCAL ? Wl : a.W;
  const int n = a.n, tid = threadIdx.x;
  {
    const double* G = a.G;
    auto get = [=](int i, int c) { return 0.5 * (G[i * n + c] + G[c * n + i]); };
    if (direct_eig<CAP / 64, true>(get, n, a.k, LOCAL ? Vl : A, LOCAL ? A : a.Z, LOCAL ? LDA : CAP, W, LDW, theta, dl)) {
      eig_emit(a, W, LDW, nullptr, theta, sgn, 0);
      if (tid == 0 && a.iters) *a.iters = dl.ok == 2 ? 0 : 1;
      return;
    }
    __syncthreads();
  }
  for (int e = tid; e < n * n; e += blockDim.x) {
    const int i = e / n, j = e % n;
    A[i * LDA + j] = 0.5 * (a.G[i * n + j] + a.G[j * n + i]);
    W[i * LDW + j] = (i == j) ? 1.0 : 0.0;
  }
  __syncthreads();
  // (the rotations of a round where the direct solver's buffers were)
  double2* cs = (double2*)dl.vbuf;
  int* pr = (int*)dl.wbuf;
  const int sweeps = lds_jacobi<LDA, LDW>(A, W, n, 60, cs, pr, scratch);
  sort_desc<LDA>(A, n, order);
  for (int r = tid; r < a.k; r += blockDim.x) theta[r] = A[order[r] * LDA + order[r]];
  __syncthreads();
  eig_emit(a, W, LDW, order, theta, sgn, 0);
  if (tid == 0 && a.iters) *a.iters = sweeps;
}

// Out = M T with T = L^-T D^-1/2 from S + shift I = L D L^T, S = M^T M: the
// Cholesky-QR orthonormalisation of the np x b block M (global, ld CAP),
// through a forward elimination of [S | I] held in registers by the block
// (TPR threads per row; per pivot its row and column go through LDS, one
// barrier).  S and the factor live in Sbuf (LDS, ld b + 1) and Tbuf (ld ldt).
//
// equil (dsc: B doubles of LDS): orthonormalise M D instead, D = diag(S)^-1/2
// (the same span; columns of very different lengths no longer spoil the
// conditioning), and report whether one pass suffices: true when every
// pivot of the equilibrated S is >= 1e-3 (cond(S) ~ 1e3 at most, so the
// columns come out orthonormal to ~1e-13).
//
// A column whose pivot is lost to rounding (below 1e-15 of its own diagonal
// entry: M has fewer than b independent columns) has no direction of its own;
// eliminating with such a pivot overflows after a few of them.  It is left
// out and comes out zero, with dpiv = infinity.  Without equil the return
// value says whether there was none.
template <int B>
__device__ bool block_orth(const double* M, double* Out, int np, double* Sbuf, double* Tbuf, int ldt, bool shift,
                           double* pbuf, double* dpiv, double* scratch, double* stage, bool equil = false,
                           double* dsc = nullptr) {
  constexpr int LDS_S = B + 1, CAP = B;
  // TPR threads per row of [S | I] (rows past B idle), CPT columns each
  constexpr int TPR = B > 64 ? 4 : 8, CPT = 2 * B / TPR;
  static_assert(TPR * B <= kEigThreads && CPT * TPR == 2 * B && TPR % 2 == 0, "thread layout");
  block_gemm_sym_f64(M, CAP, M, CAP, Sbuf, LDS_S, B, np);
  const int tid = threadIdx.x;
  if (equil) {
    if (tid < B) dsc[tid] = 1.0 / sqrt(fmax(Sbuf[tid * LDS_S + tid], 1e-300));
    __syncthreads();
    for (int e = tid; e < B * B; e += blockDim.x) {
      const int r = e / B, c = e % B;
      Sbuf[r * LDS_S + c] *= dsc[r] * dsc[c];
    }
    __syncthreads();
  }
  if (tid == 0) {
    double mx = 0.0;
    for (int i = 0; i < B; ++i) mx = fmax(mx, Sbuf[i * LDS_S + i]);
    scratch[40] = mx;
    scratch[42] = 1.0;
  }
  __syncthreads();
  const double mx = scratch[40];
  const double sh = shift ? 1e-13 * mx * (double)np : 0.0;
  const double floor = 1e-300 + 1e-30 * mx;
  const int i = tid / TPR, seg = tid % TPR, c0 = seg * CPT;
  const bool live = i < B;
  double x[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int c = c0 + j;
    x[j] = !live ? 0.0 : (c < B ? Sbuf[i * LDS_S + c] + (c == i ? sh : 0.0) : ((c - B == i) ? 1.0 : 0.0));
  }
  for (int kb = 0; kb < TPR / 2; ++kb) {
#pragma unroll
    for (int kk = 0; kk < CPT; ++kk) {
      const int k = kb * CPT + kk;
      double* row = pbuf + (k & 1) * (3 * B);
      double* col = row + 2 * B;
      if (i == k) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) row[c0 + j] = x[j];
      }
      if (live && seg == kb) col[i] = x[kk];
      __syncthreads();
      const double q = col[k];
      const bool lost = !(q > fmax(floor, 1e-15 * Sbuf[k * LDS_S + k]));
      const double p = lost ? INFINITY : q;
      if (i == k && seg == 0) {
        dpiv[k] = p;
        if (lost) scratch[42] = 0.0;
      }
      if (live && i > k) {
        const double f = col[i] / p;
#pragma unroll
        for (int j = 0; j < CPT; ++j) x[j] = fma(-f, row[c0 + j], x[j]);
      }
    }
  }
  if (equil && tid == 0) {
    double mn = INFINITY;
    for (int k = 0; k < B; ++k) mn = fmin(mn, dpiv[k]);
    scratch[41] = (mn >= 1e-3) ? 1.0 : 0.0;
  }
  __syncthreads();
  // x now holds row i of [D L^T | L^-1]; T[r][i] = L^-1[i][r] / sqrt(D[i])
  // (times dsc[r] when equilibrated)
  const double ds = live ? 1.0 / sqrt(dpiv[i]) : 0.0;
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int c = c0 + j;
    if (live && c >= B) Tbuf[(c - B) * ldt + i] = x[j] * ds * (equil ? dsc[c - B] : 1.0);
  }
  const bool well = scratch[42] != 0.0 && (!equil || scratch[41] != 0.0);
  __syncthreads();
  if constexpr (B == 48) block_gemm_f64_panel<B>(M, Tbuf, ldt, Out, CAP, np, B, stage);
  else block_gemm_f64<false>(M, CAP, Tbuf, ldt, Out, CAP, np, B, B);
  return well;
}

// Out <- orth(M): one equilibrated Cholesky-QR pass when that leaves S well
// conditioned, else two passes, shifted and plain, through `spare` (M itself
// is kept).  Columns that the plain pass left out are filled with
// pseudo-random ones and two more passes make the whole block orthonormal, so
// that a matrix of rank below b keeps a whole block.
template <int B>
__device__ void orth_step(const double* M, double* spare, double* Out, int n, int np, double* H, double* T, int ldt,
                          double* pbuf, double* dpiv, double* scratch, double* stage, double* resid) {
#pragma unroll 1
  for (int pass = 0; pass < 5; ++pass) {
    const double* from = pass < 2 ? M : pass == 3 ? Out : spare;
    double* to = pass == 1 || pass == 3 ? spare : Out;
    const bool whole =
        block_orth<B>(from, to, np, H, T, ldt, pass == 1, pbuf, dpiv, scratch, stage, pass == 0, resid);
    if (whole && (pass == 0 || pass == 2)) return;
    if (pass == 2) {
      for (int e = threadIdx.x; e < n * B; e += blockDim.x)
        if (isinf(dpiv[e % B])) Out[e] = hash_unit(e / B, B + e % B);
      __syncthreads();
    }
  }
}

// Z = G V of the warm-block path spread over the GPU: one wave per 16 x 16
// tile of Z (blockIdx.x: tile, blockIdx.y: problem), V = Y (the warm block,
// src 0) or V (src 1).  G read as G^T, the same k-ascending MFMA sequence per
// tile as gv_product, so Z is the same to the bit.
template <int B>
__global__ __launch_bounds__(64) void eig_gv_kernel(EigBatch batch, int src) {
  const EigArgs a = batch.a[blockIdx.y];
  constexpr int TN = B / 16;
  const int np = a.np;
  if ((int)blockIdx.x >= (np / 16) * TN) return;
  const int mi = (blockIdx.x / TN) * 16, nj = (blockIdx.x % TN) * 16;
  const double* V = src ? a.V : a.Y;
  const int lane = threadIdx.x, lr = lane & 15, lk = lane >> 4;
  const double* gp = a.Gp + mi + lr;
  doublex4 acc = doublex4{0.0, 0.0, 0.0, 0.0};
  int k0 = 0;
  for (; k0 + 64 <= np; k0 += 64) {
    double x[16], y[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int kk = k0 + 4 * s + lk;
      x[s] = gp[(int64_t)kk * np];
      y[s] = V[kk * B + nj + lr];
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) acc = mfma_f64(x[s], y[s], acc);
  }
  for (; k0 < np; k0 += 4) {
    const int kk = k0 + lk;
    acc = mfma_f64(gp[(int64_t)kk * np], V[kk * B + nj + lr], acc);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) a.Z[(int64_t)(mi + lk + 4 * e) * B + nj + lr] = acc[e];
}

// Block subspace iteration with Rayleigh-Ritz for n > kJacLarge.  B is the
// block: 48 and 64 keep H, W and T in LDS; 128 keeps H in LDS and W, T in the
// workspace.  All products are FP64 MFMA on zero-padded np-row blocks.
// phase 0: the whole solve.  A warm block (a.wblock) instead runs as
// eig_gv_kernel (Z = G Y), phase 1 (V <- orth(Z)), eig_gv_kernel (Z = G V),
// phase 2 (the solve from its first Rayleigh-Ritz step), so that both
// products spread over the GPU.
template <int B>
__global__ __launch_bounds__(kEigThreads) void sym_eig_subspace_kernel(EigBatch batch, int phase) {
  const EigArgs a = batch.a[blockIdx.x];
  constexpr int LDH = B + 1, CAP = B;
  constexpr bool SMALL = B <= 64;
  __shared__ double H[B * LDH];  // Ritz matrix; also S of the orthonormalisation; then sorted rotations
  __shared__ double Wl[SMALL ? B * LDH : 1];
  __shared__ double Tl[SMALL ? B * LDH : 1];
  __shared__ double2 cs[B + 2];
  __shared__ int pr[B + 2];
  __shared__ double scratch[64];
  __shared__ double resid[B];
  __shared__ int order[B];
  __shared__ double theta[B];
  __shared__ double pbuf[6 * B];
  __shared__ double dpiv[B];
  // 16-row panels of the np x B blocks for the products with B x B factors
  __shared__ double stage[B == 48 ? kEigWaves * 16 * (B + 1) : 1];
  __shared__ DirectLds<B == 48 ? 1 : 0> dl;
  constexpr int LDW = SMALL ? LDH : CAP;
  double* W = SMALL ? Wl : a.W;
  double* T = SMALL ? Tl : a.T;
  const int ldt = SMALL ? LDH : CAP;
  const int n = a.n, np = a.np, k = a.k, tid = threadIdx.x, nt = blockDim.x;
  double* V = a.V;
  double* Z = a.Z;
  double* Y = a.Y;
  double* U = a.U;
  // Gp (zero-padded symmetric G) and the starting block Y come from
  // eig_prep_kernel, launched just before on the same stream
  if (phase == 1) {
    orth_step<B>(Z, U, V, n, np, H, T, ldt, pbuf, dpiv, scratch, stage, resid);
    return;
  }
  const double jfloor = fmax(1e-30, 1e-2 * a.tol * a.tol);
  double jthr = 1e-10;
  int it = 0;
  bool have_z = false;  // phase 2: Z = G V is there already
  bool direct = false;  // the Ritz matrix went through the direct solver
  int pert = 0;         // or through perturb_eigvecs (its return value)
  if (phase == 2) {
    jthr = jfloor;
    it = 1;
    have_z = true;
  } else if (a.Q0 && a.k0 > 0 && a.wblock) {
    // a whole block from an earlier solve: the plain subspace step below
    // orthonormalises G V, so V itself is used as it is
    double* t = V;
    V = Y;
    Y = t;
  } else if (a.Q0 && a.k0 > 0) {
    // orthonormal warm-start columns and B - k0 pseudo-random ones: the
    // block is well conditioned (cond(S) ~ 1e2), one unshifted Cholesky-QR
    // pass leaves V orthonormal to ~1e-13
    block_orth<B>(Y, V, np, H, T, ldt, false, pbuf, dpiv, scratch, stage);
  } else {
    block_orth<B>(Y, V, np, H, T, ldt, true, pbuf, dpiv, scratch, stage);
    block_orth<B>(V, Y, np, H, T, ldt, false, pbuf, dpiv, scratch, stage);
    double* t = V;
    V = Y;
    Y = t;
  }
  if (phase == 0 && a.Q0 && a.k0 > 0 && a.max_iter >= 2) {
    // warm start: its first Ritz test fails whenever the matrix has moved by
    // more than the tolerance, so the first step is a plain subspace step,
    // V <- orth(G V) (the span a Rayleigh-Ritz step would leave), and the
    // next Rayleigh-Ritz step rotates to the final threshold
    if constexpr (B == 48) gv_product<B, 128>(a.Gp, np, V, Z, stage);
    else block_gemm_f64<true>(a.Gp, np, V, CAP, Z, CAP, np, B, np);
    // G V's columns are close to multiples of the warm columns: once
    // equilibrated, one unshifted Cholesky-QR pass usually suffices
    orth_step<B>(Z, U, V, n, np, H, T, ldt, pbuf, dpiv, scratch, stage, resid);
    jthr = jfloor;
    it = 1;
  } else if (phase == 0 && !(a.Q0 && a.k0 > 0)) {
    // cold start: two plain subspace steps V <- orth(G V) before the first
    // Rayleigh-Ritz step (whose Ritz matrix on a random block is dense and
    // costs full Jacobi sweeps); a plain step is a fraction of a Ritz step
    for (int p = 0; p < 2 && it + 2 < a.max_iter; ++p, ++it) {
      if constexpr (B == 48) gv_product<B, 128>(a.Gp, np, V, Z, stage);
      else block_gemm_f64<true>(a.Gp, np, V, CAP, Z, CAP, np, B, np);
      orth_step<B>(Z, U, V, n, np, H, T, ldt, pbuf, dpiv, scratch, stage, resid);
    }
  }
  for (; it < a.max_iter; ++it) {
    // Z = G V, read as G^T V (Gp is exactly symmetric): each load then takes
    // 4 rows x 128 contiguous bytes of G instead of 16 rows x 32 bytes, which
    // measured 2.3x faster
    if (!have_z) {
      if constexpr (B == 48) gv_product<B, 128>(a.Gp, np, V, Z, stage);
      else block_gemm_f64<true>(a.Gp, np, V, CAP, Z, CAP, np, B, np);
    }
    have_z = false;
    block_gemm_sym_f64(V, CAP, Z, CAP, H, LDH, B, np);           // H = V^T Z = V^T G V
    for (int e = tid; e < B * B; e += nt) {
      const int i = e / B, j = e % B;
      if (i < j) H[i * LDH + j] = H[j * LDH + i] = 0.5 * (H[i * LDH + j] + H[j * LDH + i]);
      W[i * LDW + j] = (i == j) ? 1.0 : 0.0;
    }
    __syncthreads();
    // the Ritz rotations only need the accuracy of the current subspace:
    // off-diagonal mass down to (residual / t_1)^2 / 100 of the total,
    // tightening to tol^2 / 100 as the residuals fall
    {
      // a nearly diagonal leading part (a converging warm start): second-
      // order perturbation (block 48: its two B x k scratch matrices use the
      // panel staging area); else the direct solver (block 48, its scratch in
      // the staging area too); else Jacobi sweeps
      direct = false;
      // (not twice in a row with what cannot end the iteration, nor in the
      // last step allowed, whose vectors are returned whatever they are)
      if constexpr (B == 48)
        pert = perturb_eigvecs<LDH, LDW>(H, W, B, k, stage, stage + B * k, scratch,
                                         pert == 1 || it + 1 == a.max_iter ? 1e-5 : 1e-3);
      const bool sep = pert == 0 && k < B && lead_block_separated<LDH>(H, B, k, jthr, scratch);
      if constexpr (B == 48) {
        // (a separated leading block of few columns sweeps in less)
        if (pert == 0 && (!sep || k >= 24)) {
          direct = direct_eig<1, false>([=](int i, int c) { return H[i * LDH + c]; }, B, B, stage, stage + B * 64, B, W, LDW,
                                 theta, dl);
          if (!direct) {
            __syncthreads();
            for (int e = tid; e < B * B; e += nt) W[(e / B) * LDW + e % B] = (e / B == e % B) ? 1.0 : 0.0;
            __syncthreads();
          }
        }
      }
      if (pert == 0 && !direct) lds_jacobi<LDH, LDW>(H, W, B, 30, cs, pr, scratch, jthr, k, sep ? 1 : 0);
    }
    if (direct) {
      if (tid < B) order[tid] = tid;
    } else {
      sort_desc<LDH>(H, B, order);
      if (tid < B) theta[tid] = H[order[tid] * LDH + order[tid]];
    }
    __syncthreads();
    for (int e = tid; e < B * B; e += nt) {  // rotations in Ritz-value order
      const int l = e / B, j = e % B;
      H[l * LDH + j] = W[l * LDW + order[j]];
    }
    __syncthreads();
    if constexpr (B == 48) {
      block_gemm_f64_panel<B>(V, H, LDH, Y, CAP, np, B, stage);  // Y = V W (Ritz vectors)
      block_gemm_f64_panel<B>(Z, H, LDH, U, CAP, np, B, stage);  // U = Z W = G Y
    } else {
      block_gemm_f64<false>(V, CAP, H, LDH, Y, CAP, np, B, B);
      block_gemm_f64<false>(Z, CAP, H, LDH, U, CAP, np, B, B);
    }
    // residual norms of the leading k pairs: thread (g, r) sums column r
    // over rows g, g + ng, ... (row-wise, coalesced), partials through H
    {
      const int ng = nt / k;
      if (tid < ng * k) {
        const int g = tid / k, r = tid - g * k;
        const double th = theta[r];
        double r2 = 0.0;
        for (int i = g; i < n; i += ng) {
          const double d = U[i * CAP + r] - th * Y[i * CAP + r];
          r2 += d * d;
        }
        H[tid] = r2;
      }
      __syncthreads();
      if (tid < k) {
        double r2 = 0.0;
        for (int g = 0; g < ng; ++g) r2 += H[g * k + tid];
        resid[tid] = sqrt(r2);
      }
    }
    __syncthreads();
    if (tid == 0) {
      double worst = 0.0;
      for (int r = 0; r < k; ++r) worst = fmax(worst, resid[r]);
      const double t1 = fmax(fabs(theta[0]), 1e-300);
      scratch[63] = (worst <= a.tol * t1 && pert != 1) ? 1.0 : 0.0;
      const double rr = worst / t1;
      scratch[62] = fmin(1e-10, fmax(jfloor, 1e-2 * rr * rr));
      // A subspace step takes the residuals down by about the ratio of the
      // block's last Ritz value to the k-th.  The steps that are still needed
      // but the last are plain ones, V <- orth(G V), without the Ritz
      // problem (n = 256, block 48: 125 us of a step's 220).
      const double rate = fabs(theta[B - 1]) / fmax(fabs(theta[k - 1]), 1e-300);
      const double need = rate < 0.98 ? log(a.tol / rr) / log(rate) : 8.0;
      scratch[61] = fmin(fmax(ceil(need) - 1.0, 0.0), 8.0);
    }
    __syncthreads();
    const bool done = scratch[63] != 0.0;
    jthr = scratch[62];
    int plain = scratch[61] >= 1.0 ? (int)scratch[61] : 0;  // (0 for NaN)
    __syncthreads();
    if (done || it + 1 == a.max_iter) break;
    // V <- orth(U): the columns of U = G Y scale with the Ritz values
    orth_step<B>(U, Z, V, n, np, H, T, ldt, pbuf, dpiv, scratch, stage, resid);
    for (; plain > 0 && it + 2 < a.max_iter; --plain, ++it) {
      if constexpr (B == 48) gv_product<B, 128>(a.Gp, np, V, Z, stage);
      else block_gemm_f64<true>(a.Gp, np, V, CAP, Z, CAP, np, B, np);
      orth_step<B>(Z, U, V, n, np, H, T, ldt, pbuf, dpiv, scratch, stage, resid);
    }
  }
  eig_emit(a, Y, CAP, nullptr, theta, resid, B);
  if (tid == 0 && a.iters) *a.iters = it + 1;
}

static size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace tla

using namespace tla;

static int64_t eig_np(int n) { return (int64_t)(n + 15) / 16 * 16; }

extern "C" size_t tla_sym_eig_workspace_size(int n) {
  if (n <= kJac) return 0;
  const size_t rot = align256(size_t(kEigCapLarge) * kEigCapLarge * 8);
  if (n <= kJacLarge) return 2 * rot;  // the vectors and the direct solver's factors
  // padded G, four np x 128 blocks, rotations and the orthonormalising factor
  const size_t np = (size_t)eig_np(n);
  return align256(np * np * 8) + 4 * align256(np * kEigCapLarge * 8) + 2 * rot;
}

// Arguments of one problem (workspace carved as the kernel kind needs);
// *kind: 0 Jacobi in LDS, 1 Jacobi with rotations in the workspace, 2/3/4
// subspace iteration with block 48 / 64 / 128.
static int eig_args(const double* G, int n, int k, const double* Q0, int k0, double* evals, double* evecs, double tol,
                    int max_iter, int* iters_out, void* ws, size_t ws_bytes, EigArgs* out, int* kind) {
  TLA_REQUIRE(n >= 1, "sym_eig: n = %d", n);
  TLA_REQUIRE(k >= 1 && k <= n, "sym_eig: k = %d not in [1, n = %d]", k, n);
  TLA_REQUIRE(G, "sym_eig: NULL pointer");
  TLA_REQUIRE(!Q0 || k0 >= 1, "sym_eig: warm start with k0 = %d columns", k0);
  TLA_REQUIRE(ws_bytes >= tla_sym_eig_workspace_size(n), "sym_eig: workspace too small");
  TLA_REQUIRE(n <= kJacLarge || ws, "sym_eig: NULL workspace");
  EigArgs a{};
  a.G = G; a.n = n; a.k = k; a.Q0 = Q0; a.q0_ld = k0;
  a.evals = evals; a.evecs = evecs; a.tol = tol > 0 ? tol : 1e-11; a.max_iter = max_iter > 0 ? max_iter : 200;
  a.iters = iters_out;
  if (n <= kJac) {
    *out = a;
    *kind = 0;
    return TLA_OK;
  }
  if (n <= kJacLarge) {
    a.W = (double*)ws;
    a.Z = a.W + kEigCapLarge * kEigCapLarge;
    *out = a;
    *kind = 1;
    return TLA_OK;
  }
  // block: 48 for k <= 40 (cheaper Jacobi sweeps), 64 for k <= 56, 128 for k <= 120
  const bool small_block = k <= 56;
  if (!small_block && k > kEigCapLarge - 8) {
    set_error("sym_eig: k = %d > %d leading eigenpairs of an n = %d > %d matrix is not supported", k,
              kEigCapLarge - 8, n, kJacLarge);
    return TLA_ERR_UNSUPPORTED;
  }
  const int b = k <= 40 ? 48 : (small_block ? 64 : kEigCapLarge);
  a.np = (int)eig_np(n);
  const size_t np = (size_t)a.np;
  const size_t blk = align256(np * kEigCapLarge * 8);
  const size_t rot = align256(size_t(kEigCapLarge) * kEigCapLarge * 8);
  char* base = (char*)ws;
  a.Gp = (double*)base;
  base += align256(np * np * 8);
  a.V = (double*)base;
  a.Z = (double*)(base + blk);
  a.Y = (double*)(base + 2 * blk);
  a.U = (double*)(base + 3 * blk);
  a.W = (double*)(base + 4 * blk);
  a.T = (double*)(base + 4 * blk + rot);
  a.k0 = Q0 ? std::min(k0, b) : 0;
  *out = a;
  *kind = b == 48 ? 2 : (b == 64 ? 3 : 4);
  return TLA_OK;
}

// The warm-block sequence of sym_eig_subspace_kernel (m problems).
template <int B>
static void launch_split(const EigBatch& b, int m, hipStream_t st) {
  int tiles = 0;
  for (int i = 0; i < m; ++i) tiles = std::max(tiles, (b.a[i].np / 16) * (B / 16));
  const dim3 g((unsigned)tiles, (unsigned)m);
  eig_gv_kernel<B><<<g, 64, 0, st>>>(b, 0);
  sym_eig_subspace_kernel<B><<<m, kEigThreads, 0, st>>>(b, 1);
  eig_gv_kernel<B><<<g, 64, 0, st>>>(b, 1);
  sym_eig_subspace_kernel<B><<<m, kEigThreads, 0, st>>>(b, 2);
}

// One launch per kernel kind present, one workgroup per problem.
static int eig_launch(const EigArgs* args, const int* kinds, int count, hipStream_t st) {
  for (int kind = 0; kind < 5; ++kind) {
    EigBatch b{};
    int m = 0;
    for (int i = 0; i < count; ++i)
      if (kinds[i] == kind) b.a[m++] = args[i];
    if (m == 0) continue;
    if (kind >= 2) {
      int gt = 0, yt = 0;
      const int bk = kind == 2 ? 48 : (kind == 3 ? 64 : kEigCapLarge);
      for (int i = 0; i < m; ++i) {
        const int nt = (b.a[i].np + 31) / 32;
        gt = std::max(gt, nt * nt);
        yt = std::max(yt, (int)ceil_div((int64_t)b.a[i].np * bk, 256));
      }
      dim3 grid(gt + yt, m);
      switch (kind) {
        case 2: eig_prep_kernel<48><<<grid, 256, 0, st>>>(b, gt); break;
        case 3: eig_prep_kernel<64><<<grid, 256, 0, st>>>(b, gt); break;
        default: eig_prep_kernel<kEigCapLarge><<<grid, 256, 0, st>>>(b, gt); break;
      }
      TLA_LAUNCH_CHECK();
    }
    bool split = kind >= 2;  // every problem a warm block
    for (int i = 0; i < m; ++i) split = split && b.a[i].wblock;
    switch (kind) {
      case 0: sym_eig_small_kernel<kJac><<<m, kEigThreads, 0, st>>>(b); break;
      case 1: sym_eig_small_kernel<kJacLarge><<<m, kEigThreads, 0, st>>>(b); break;
      case 2: split ? launch_split<48>(b, m, st) : sym_eig_subspace_kernel<48><<<m, kEigThreads, 0, st>>>(b, 0); break;
      case 3: split ? launch_split<64>(b, m, st) : sym_eig_subspace_kernel<64><<<m, kEigThreads, 0, st>>>(b, 0); break;
      default: sym_eig_subspace_kernel<kEigCapLarge><<<m, kEigThreads, 0, st>>>(b, 0); break;
    }
    TLA_LAUNCH_CHECK();
  }
  return TLA_OK;
}

extern "C" int tla_sym_eig(const double* G, int n, int k, const double* Q0, int k0, double* evals, double* evecs,
                           double tol, int max_iter, int* iters_out, void* ws, size_t ws_bytes, void* stream) {
  TLA_REQUIRE(evals && evecs, "sym_eig: NULL pointer");
  EigArgs a;
  int kind = 0;
  const int rc = eig_args(G, n, k, Q0, k0, evals, evecs, tol, max_iter, iters_out, ws, ws_bytes, &a, &kind);
  if (rc != TLA_OK) return rc;
  return eig_launch(&a, &kind, 1, (hipStream_t)stream);
}

extern "C" int tla_gram_svd_block(int n, int k) {
  if (n <= kJacLarge || k < 1 || k > n || k > kEigCapLarge - 8) return 0;
  return k <= 40 ? 48 : (k <= 56 ? 64 : kEigCapLarge);
}

static int svd_args(const double* G, int n, int k, const double* W0, int k0, int dtype, void* U, void* s, double* U64,
                    double* W_out, double tol, int max_iter, int* iters_out, void* ws, size_t ws_bytes, EigArgs* a,
                    int* kind) {
  TLA_REQUIRE(dtype == TLA_F32 || dtype == TLA_F64, "gram_left_singular: bad dtype %d", dtype);
  TLA_REQUIRE(U, "gram_left_singular: NULL U");
  const int rc = eig_args(G, n, k, W0, W0 ? k0 : 0, nullptr, U64, tol, max_iter, iters_out, ws, ws_bytes, a, kind);
  if (rc != TLA_OK) return rc;
  const int b = tla_gram_svd_block(n, k);
  a->flip = 1;
  a->out_dtype = dtype;
  a->u_out = U;
  a->s_out = s;
  a->wblk = b > 0 ? W_out : nullptr;
  a->wblock = (b > 0 && W0 && k0 == b && a->max_iter >= 2) ? 1 : 0;
  return TLA_OK;
}

extern "C" int tla_gram_left_singular(const double* G, int n, int k, const double* W0, int k0, int dtype, void* U,
                                      void* s, double* U64, double* W_out, double tol, int max_iter, int* iters_out,
                                      void* ws, size_t ws_bytes, void* stream) {
  EigArgs a;
  int kind = 0;
  const int rc = svd_args(G, n, k, W0, k0, dtype, U, s, U64, W_out, tol, max_iter, iters_out, ws, ws_bytes, &a, &kind);
  if (rc != TLA_OK) return rc;
  return eig_launch(&a, &kind, 1, (hipStream_t)stream);
}

extern "C" int tla_gram_left_singular_batch(int count, const double* const* G, const int* n, const int* k, int dtype,
                                            void* const* U, void* const* s, double* const* W_out, double tol,
                                            int max_iter, void* const* workspace, const size_t* workspace_bytes,
                                            void* stream) {
  TLA_REQUIRE(count >= 1 && count <= kEigMaxBatch, "gram_left_singular_batch: count %d not in [1, %d]", count,
              kEigMaxBatch);
  TLA_REQUIRE(G && n && k && U && s && W_out && workspace && workspace_bytes, "gram_left_singular_batch: NULL array");
  EigArgs args[kEigMaxBatch];
  int kinds[kEigMaxBatch];
  for (int i = 0; i < count; ++i) {
    const int rc = svd_args(G[i], n[i], k[i], nullptr, 0, dtype, U[i], s[i], nullptr, W_out[i], tol, max_iter, nullptr,
                            workspace[i], workspace_bytes[i], &args[i], &kinds[i]);
    if (rc != TLA_OK) return rc;
  }
  return eig_launch(args, kinds, count, (hipStream_t)stream);
}

extern "C" int tla_sym_eig_batch(int count, const double* const* G, const int* n, const int* k,
                                 const double* const* Q0, const int* k0, double* const* evals, double* const* evecs,
                                 double tol, int max_iter, void* const* workspace, const size_t* workspace_bytes,
                                 void* stream) {
  TLA_REQUIRE(count >= 1 && count <= kEigMaxBatch, "sym_eig_batch: count %d not in [1, %d]", count, kEigMaxBatch);
  TLA_REQUIRE(G && n && k && evals && evecs && workspace && workspace_bytes, "sym_eig_batch: NULL array");
  EigArgs args[kEigMaxBatch];
  int kinds[kEigMaxBatch];
  for (int i = 0; i < count; ++i) {
    TLA_REQUIRE(evals[i] && evecs[i], "sym_eig_batch: NULL pointer");
    const int rc = eig_args(G[i], n[i], k[i], Q0 ? Q0[i] : nullptr, k0 ? k0[i] : 0, evals[i], evecs[i], tol,
                            max_iter, nullptr, workspace[i], workspace_bytes[i], &args[i], &kinds[i]);
    if (rc != TLA_OK) return rc;
  }
  return eig_launch(args, kinds, count, (hipStream_t)stream);
}
