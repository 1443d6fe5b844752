// orbit.h -- device helpers of the reflection-orbit M2L kernels (m2l_orbit.hip,
// m2l_orbit_gen.hip, m2l_orbit_fp64.hip).
#pragma once

#include <type_traits>

#include "m2l.h"
#include "tree_util.h"

namespace fmmx {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// e of the power of two that brings a level's (or group's) largest magnitude just
// below 2^ORB_TOP, or half of it where sums of 4 would round beyond FP16's 65,504.  Applied with ldexpf, here and when it is undone: 2^e itself is
// no FP32 number for magnitudes near the ends of FP32's range.
__device__ __forceinline__ int orbit_exp(const unsigned* mmax) {
  const float m = __uint_as_float(*mmax);
  if (!(m > 0.f) || !(m < __builtin_inff())) return 0;
  int e;
  const float f = frexpf(m, &e);
  return (f <= 65504.f / 65536.f ? ORB_TOP : ORB_TOP - 1) - e;
}

// bits of v (0..3) at positions 0 and 3 (one axis of a Morton key)
__device__ __forceinline__ uint32_t dil3(int v) { return (uint32_t)(v & 1) | ((uint32_t)(v & 2) << 2); }

// rank of a submask of D among the submasks (pext)
constexpr __host__ __device__ int sub_rank(int D, int r) {
  int s = 0, j = 0;
  for (int a = 0; a < 3; a++)
    if ((D >> a) & 1) s |= ((r >> a) & 1) << j++;
  return s;
}
constexpr __host__ __device__ int bits3(int D) { return (D & 1) + ((D >> 1) & 1) + ((D >> 2) & 1); }
// in-place Walsh-Hadamard transform over the 2^J sources of one word
template <int J>
__device__ __forceinline__ void wht(float (&raw)[1 << J][4], int t) {
#pragma unroll
  for (int b = 0; b < J; b++)
#pragma unroll
    for (int s = 0; s < (1 << J); s++)
      if (!(s & (1 << b))) {
        const float u = raw[s][t], v = raw[s | (1 << b)][t];
        raw[s][t] = u + v;
        raw[s | (1 << b)][t] = u - v;
      }
}

__device__ __forceinline__ uint32_t hi_pair(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, h2));
}
// the residuals of a pair against its rounded halves h (exact in FP32:
// a - h in one mixed fused multiply-add)
__device__ __forceinline__ uint32_t lo_pair(float a, float b, uint32_t h) {
  float ra, rb;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(ra) : "v"(h), "v"(a));
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(rb) : "v"(h), "v"(b));
  return hi_pair(ra, rb);
}

// 16 bytes per lane from global memory to LDS, the wave's 1,024 bytes at dst,
// without registers.  Written out so that the compiler does not hold every LDS
// read behind it back until the copy has landed; the caller waits for it.  The
// scalar write of M0 and the copy that reads it need a wait state between them,
// which the compiler puts into its own code but not into this.
__device__ __forceinline__ void lds_copy16(uint32_t dst, const u32x4* from) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(from) : "memory", "m0");
}

}  // namespace

}  // namespace fmmx
