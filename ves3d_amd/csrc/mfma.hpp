// mfma.hpp -- the FP64 and FP32 16x16x4 matrix instructions.
#pragma once
#include "common.hpp"

namespace v3d {

// MFMA operand layout.  For both v_mfma_f64_16x16x4f64 and
// v_mfma_f32_16x16x4f32 lane l supplies A(l%16, l/16) and B(l/16, l%16) of a
// 16x4 / 4x16 step and holds 4 results of column l%16; their rows differ:
// l/16 + 4r (f64) and 4(l/16) + r (f32) for result register r (the
// accumulator layouts composable_kernel's xdlops_gemm.hpp records as
// group_size 1 / 4).
template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 step(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
};
template <>
struct Mfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 step(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

}  // namespace v3d
