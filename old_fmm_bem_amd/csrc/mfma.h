// mfma.h -- v_mfma 16x16x4 in FP32 and FP64, and the zeros its sums start from.
#pragma once

#include <hip/hip_runtime.h>

namespace fmmx {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
  using v4 = f32x4;
  static __device__ __forceinline__ v4 zero() { return v4{0.f, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ v4 fma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<double> {
  using v4 = f64x4;
  // in registers: with a constant zero for its accumulator the compiler may give
  // an FP64 MFMA an output that overlaps its own operands
  static __device__ __forceinline__ v4 zero() {
    v4 z = {0., 0., 0., 0.};
    asm volatile("" : "+v"(z));
    return z;
  }
  static __device__ __forceinline__ v4 fma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};

}  // namespace

}  // namespace fmmx
