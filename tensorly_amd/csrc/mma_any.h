// 16 x 16 x 4 matrix instructions of float32 and float64, and the loads and
// sums that the kernels for any mode sizes share.
#pragma once
#include "common.h"

namespace tla {

typedef double doublex4 __attribute__((ext_vector_type(4)));

// D = A B + C on FP64 MFMA (16 x 4 by 4 x 16): lane l supplies A[l % 16][l / 16]
// and B[l / 16][l % 16] and holds D[l / 16 + 4 e][l % 16], e < 4 (rows
// interleaved by 4, unlike the FP32 16x16x4 form).
__device__ __forceinline__ doublex4 mfma_f64(double a, double b, doublex4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Vector types of the tensor's loads: 16 bytes, aligned to one element.
template <typename T> struct AnyT;
template <> struct AnyT<float> {
  typedef float vec __attribute__((ext_vector_type(4), aligned(4)));
  typedef floatx4 acc;
  static constexpr int V = 4;
  // row of element e of a lane's accumulator (lane group g)
  static __device__ __forceinline__ int row(int g, int e) { return 4 * g + e; }
  static __device__ __forceinline__ acc mma(float a, float b, acc c) { return mfma_f32_16x16x4(a, b, c); }
};
template <> struct AnyT<double> {
  typedef double vec __attribute__((ext_vector_type(2), aligned(8)));
  typedef doublex4 acc;
  static constexpr int V = 2;
  static __device__ __forceinline__ int row(int g, int e) { return g + 4 * e; }
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return mfma_f64(a, b, c);
  }
};

// *(p + off bytes): a wave-uniform base with a 32-bit lane offset
template <typename U, typename T>
__device__ __forceinline__ U at(const T* p, uint32_t off) {
  return *(const U*)((const char*)p + off);
}

// Sum the waves' accumulators in wave order through LDS.
template <typename T, int N, int WAVES>
__device__ __forceinline__ void any_block_sum(typename AnyT<T>::acc (&acc)[N], T* red, int wave, int lane) {
  for (int w = 0; w < WAVES; ++w) {
    if (wave == w) {
#pragma unroll
      for (int n = 0; n < N; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          T* p = red + (n * 4 + e) * 64 + lane;
          *p = w == 0 ? acc[n][e] : *p + acc[n][e];
        }
    }
    __syncthreads();
  }
}

}  // namespace tla
