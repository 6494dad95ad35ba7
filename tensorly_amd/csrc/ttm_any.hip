// n-mode product on the matrix cores, float32 and float64, any mode sizes but
// contiguous runs shorter than a 16-byte load:
// out[a, j, b] = sum_m U'(j, m) X[a, m, b], U'(j, m) = U[j ldj + m ldm].
//
//  * ttm_any_cols_kernel (b not empty): U' is the first operand and 16-byte
//    pieces of X's rows m, as they lie, the second; a wave takes TN tiles of
//    256 bytes of b for JT tiles of 16 rows j and walks m, two sets of loaded
//    rows taking turns.  Where the tiles alone leave the GPU idle the four
//    waves of a block share one tile and a quarter of m each.
//  * ttm_any_rows_kernel (contiguous mode contracted): a wave takes TN tiles
//    of 16 rows of X, 128 contiguous bytes of each at a time.
// More than 64 rows j are further blocks, which read X again.
//
// Bound: memory, X read and out written once; the FP32 matrix rate from about
// 48 rows j on.  Measured per call, float32, modes 0 / 1 / 2:
//   256^3 -> 32:  21 / 21 / 25 us (3.5 TB/s); the aligned kernel this replaced,
//     one 16-byte load per lane and step with no load ahead, 26 / 26 / 26
//   512^3 -> 64:  200 / 198 / 264 us (86 TFLOP/s); before 312 / 298 / 299
//   512^3 -> 16:  100 / 99 / 113 us (5.5 TB/s); before 113 / 104 / 119
// Odd sizes, more than 64 rows j and float64 ran one thread per output
// element, which read X once per row j: 250 x 331 x 190 to 25 x 30 x 20 and
// back 772 -> 89 us.
#include "mma_any.h"
#include "ttm_any.h"

namespace tla {

template <typename T>
struct TtmAnyArgs {
  const T* X;
  int64_t Pa, Im, Pb;  // rows: P = Pa, K = Im
  const T* U;
  int64_t ldj, ldm;
  int64_t J;
  T* out;
  int64_t tiles;  // wave tiles of b per a (cols)
  int split;      // cols: the block's waves share a tile and split m
};

// N consecutive m of row j of U' from m on (those past the end are zero).
template <typename T, int N>
__device__ __forceinline__ void ttm_load_u(const T* __restrict__ uj, int64_t ldm, int m, int left, T (&u)[N]) {
  using V = typename AnyT<T>::vec;
  constexpr int VL = AnyT<T>::V;
  if (ldm == 1 && left >= N) {
#pragma unroll
    for (int h = 0; h < N / VL; ++h) {
      const V w = *(const V*)(uj + m + h * VL);
#pragma unroll
      for (int v = 0; v < VL; ++v) u[h * VL + v] = w[v];
    }
  } else {
#pragma unroll
    for (int v = 0; v < N; ++v) u[v] = v < left ? uj[(m + v) * ldm] : (T)0;
  }
}

template <typename T, int TN, int JT>
__global__ __launch_bounds__(64 * kTtmWaves, 2) void ttm_any_cols_kernel(TtmAnyArgs<T> a) {
  using V = typename AnyT<T>::vec;
  using Acc = typename AnyT<T>::acc;
  constexpr int VL = AnyT<T>::V, NR = 4, RV = 4 * NR;
  __shared__ T red[TN * VL * JT * 256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t tile = a.split ? blockIdx.x : (int64_t)blockIdx.x * kTtmWaves + wave;
  if (tile >= a.Pa * a.tiles) return;  // (whole waves; never with split)
  const int64_t ia = tile / a.tiles, b0 = (tile - ia * a.tiles) * (16 * VL * TN);
  const int64_t j0 = (int64_t)blockIdx.y * (16 * JT);
  const int Im = (int)a.Im;
  const int64_t Pb = a.Pb;
  // lanes past the end of b read (and write) its last 16 bytes
  uint32_t col[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t)
    col[t] = (uint32_t)((NR * g * Pb + min(b0 + (16 * t + c) * VL, Pb - VL)) * sizeof(T));
  const T* uj[JT];
#pragma unroll
  for (int n = 0; n < JT; ++n) uj[n] = a.U + min(j0 + 16 * n + c, a.J - 1) * a.ldj;
  Acc acc[TN * VL * JT];
#pragma unroll
  for (int n = 0; n < TN * VL * JT; ++n) acc[n] = Acc{0, 0, 0, 0};
  const T* Xa = a.X + ia * Im * Pb;
  auto load = [&](int m0, V (&x)[NR][TN]) {
    const T* xb = Xa + (int64_t)m0 * Pb;
    if (m0 + RV <= Im) {
#pragma unroll
      for (int u = 0; u < NR; ++u)
#pragma unroll
        for (int t = 0; t < TN; ++t) x[u][t] = at<V>(xb + u * Pb, col[t]);
    } else {
      const int left = Im - (m0 + NR * g);
#pragma unroll
      for (int u = 0; u < NR; ++u)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          x[u][t] = V{};
          if (u < left) x[u][t] = at<V>(xb + u * Pb, col[t]);
        }
    }
  };
  const int step = a.split ? RV * kTtmWaves : RV;
  auto visit = [&](int m0, V (&x)[NR][TN], V (&xn)[NR][TN]) {
    T u[JT][NR];
    const int m = m0 + NR * g;
#pragma unroll
    for (int n = 0; n < JT; ++n) ttm_load_u<T, NR>(uj[n], a.ldm, m, Im - m, u[n]);
    if (m0 + step < Im) load(m0 + step, xn);
#pragma unroll
    for (int v = 0; v < NR; ++v)
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int s = 0; s < VL; ++s)
#pragma unroll
          for (int n = 0; n < JT; ++n) {
            Acc& d = acc[(t * VL + s) * JT + n];
            d = AnyT<T>::mma(u[n][v], x[v][t][s], d);
          }
  };
  int m0 = a.split ? RV * wave : 0;
  V x0[NR][TN], x1[NR][TN];
  if (m0 < Im) load(m0, x0);
  while (m0 < Im) {
    visit(m0, x0, x1);
    m0 += step;
    if (m0 >= Im) break;
    visit(m0, x1, x0);
    m0 += step;
  }
  // acc[(t VL + s) JT + n][e] = out[a][j0 + 16 n + row(g, e)][column of (t, c), + s]
  if (a.split) {
    any_block_sum<T, TN * VL * JT, kTtmWaves>(acc, red, wave, lane);
    if (wave != 0) return;
#pragma unroll
    for (int n = 0; n < TN * VL * JT; ++n)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[n][e] = red[(n * 4 + e) * 64 + lane];
  }
  T* oa = a.out + ia * a.J * Pb;
#pragma unroll
  for (int n = 0; n < JT; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t j = j0 + 16 * n + AnyT<T>::row(g, e);
      if (j < a.J)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          const int64_t b = b0 + (16 * t + c) * VL;
          V o;
#pragma unroll
          for (int s = 0; s < VL; ++s) o[s] = acc[(t * VL + s) * JT + n][e];
          if (b < Pb) *(V*)(oa + j * Pb + min(b, Pb - VL)) = o;
        }
    }
}

template <typename T, int TN, int JT>
__global__ __launch_bounds__(64 * kTtmWaves, 2) void ttm_any_rows_kernel(TtmAnyArgs<T> a) {
  using V = typename AnyT<T>::vec;
  using Acc = typename AnyT<T>::acc;
  constexpr int VL = AnyT<T>::V, NV = 2 * VL, CH = 4 * NV;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t p0 = ((int64_t)blockIdx.x * kTtmWaves + wave) * (16 * TN);
  if (p0 >= a.Pa) return;
  const int64_t j0 = (int64_t)blockIdx.y * (16 * JT);
  const int K = (int)a.Im;
  uint32_t roff[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) roff[t] = (uint32_t)((min((int64_t)(16 * t + c), a.Pa - 1 - p0) * K + NV * g) * sizeof(T));
  const T* uj[JT];
#pragma unroll
  for (int n = 0; n < JT; ++n) uj[n] = a.U + min(j0 + 16 * n + c, a.J - 1) * a.ldj;
  Acc acc[TN * JT];
#pragma unroll
  for (int n = 0; n < TN * JT; ++n) acc[n] = Acc{0, 0, 0, 0};
  const T* Xp = a.X + p0 * K;
  auto load = [&](int k0, T (&x)[TN][NV]) {
    const T* xb = Xp + k0;
    if (k0 + CH <= K) {
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const V v0 = at<V>(xb, roff[t]), v1 = at<V>(xb + VL, roff[t]);
#pragma unroll
        for (int v = 0; v < VL; ++v) { x[t][v] = v0[v]; x[t][VL + v] = v1[v]; }
      }
    } else {
      const int left = K - (k0 + NV * g);
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int v = 0; v < NV; ++v) x[t][v] = v < left ? at<T>(xb + v, roff[t]) : (T)0;
    }
  };
  auto visit = [&](int k0, T (&x)[TN][NV], T (&xn)[TN][NV]) {
    T u[JT][NV];
    const int k = k0 + NV * g;
#pragma unroll
    for (int n = 0; n < JT; ++n) ttm_load_u<T, NV>(uj[n], a.ldm, k, K - k, u[n]);
    if (k0 + CH < K) load(k0 + CH, xn);
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int n = 0; n < JT; ++n) acc[t * JT + n] = AnyT<T>::mma(x[t][v], u[n][v], acc[t * JT + n]);
  };
  T x0[TN][NV], x1[TN][NV];
  load(0, x0);
  for (int k0 = 0; k0 < K;) {
    visit(k0, x0, x1);
    k0 += CH;
    if (k0 >= K) break;
    visit(k0, x1, x0);
    k0 += CH;
  }
  // acc[t JT + n][e] = out[p0 + 16 t + row(g, e)][j0 + 16 n + c]
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t p = p0 + 16 * t + AnyT<T>::row(g, e);
      if (p < a.Pa)
#pragma unroll
        for (int n = 0; n < JT; ++n) {
          const int64_t j = j0 + 16 * n + c;
          if (j < a.J) a.out[p * a.J + j] = acc[t * JT + n][e];
        }
    }
}

template <typename T, int JT>
static void ttm_any_run(const TtmPlan& p, const TtmAnyArgs<T>& a, hipStream_t st) {
  const dim3 grid((unsigned)p.gx, (unsigned)p.gy);
  constexpr int TNR = JT <= 2 ? 4 : 2, TNC = JT <= 2 ? 2 : 1;
  if (a.Pb == 1) {
    if (p.TN == 1) ttm_any_rows_kernel<T, 1, JT><<<grid, 64 * kTtmWaves, 0, st>>>(a);
    else ttm_any_rows_kernel<T, TNR, JT><<<grid, 64 * kTtmWaves, 0, st>>>(a);
  } else {
    if (p.TN == 1) ttm_any_cols_kernel<T, 1, JT><<<grid, 64 * kTtmWaves, 0, st>>>(a);
    else ttm_any_cols_kernel<T, TNC, JT><<<grid, 64 * kTtmWaves, 0, st>>>(a);
  }
}

template <typename T>
static int ttm_any_t(const TtmPlan& p, TtmAnyArgs<T> a, hipStream_t st) {
  a.tiles = p.tiles;
  a.split = p.split;
  switch (p.JT) {
    case 1: ttm_any_run<T, 1>(p, a, st); break;
    case 2: ttm_any_run<T, 2>(p, a, st); break;
    case 3: ttm_any_run<T, 3>(p, a, st); break;
    default: ttm_any_run<T, 4>(p, a, st); break;
  }
  TLA_LAUNCH_CHECK();
  return TLA_OK;
}

int ttm_any_launch(bool f64, const TtmPlan& p, const void* X, int64_t Pa, int64_t Im, int64_t Pb, const void* U,
                   int64_t ldj, int64_t ldm, int64_t J, void* out, hipStream_t st) {
  if (f64)
    return ttm_any_t<double>(p, {(const double*)X, Pa, Im, Pb, (const double*)U, ldj, ldm, J, (double*)out, 0, 0}, st);
  return ttm_any_t<float>(p, {(const float*)X, Pa, Im, Pb, (const float*)U, ldj, ldm, J, (float*)out, 0, 0}, st);
}

}  // namespace tla
