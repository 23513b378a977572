// Device-side pieces shared by the pair kernels (nbody_kernels.hip,
// wide_kernels.hip): position records and overlap tests.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pair_math.hpp"

namespace lm {

template <class R>
struct Rec;
template <>
struct Rec<float> {
  using T = float4;
};
template <>
struct Rec<double> {
  using T = double4;
};

// A record far from everything: padding sources (zero force) and idle target
// lanes evaluate finite arithmetic against it and contribute nothing.
template <class R4>
__device__ inline R4 far_record() {
  R4 r;
  r.x = 1.0e6f;
  r.y = 1.0e6f;
  r.z = 1.0e6f;
  r.w = 1.0f;
  return r;
}

// Overlap test of a group of pairs: is any r^2 below 4 (radius units)?
// NearTestCmp compares every r^2 (the mask lives in scalar registers).
// NearTest in FP32 keeps the smallest r^2 by its bit pattern, which orders
// like the value for r^2 >= 0 (NaN sorts above 4 and stays on the far
// formula), so a group costs one unsigned min per pair (the compiler forms
// v_min3_u32) and a single compare; it takes a vector register, which the
// ordered kernel's 4-target tiling cannot spare without losing a wave per
// SIMD, so that kernel keeps the compares.
template <class R>
struct NearTestCmp {
  bool any = false;
  __device__ void add(R r2) { any |= r2 < R(4); }
  __device__ bool hit() const { return any; }
};
template <class R>
struct NearTest : NearTestCmp<R> {};
// FP64: the high words of non-negative doubles order like the values, and
// every double whose high word is that of 4.0 (0x40100000) is >= 4.0, so
// r^2 < 4 exactly when its high word is below 0x40100000.
template <>
struct NearTest<double> {
  uint32_t m = 0xffffffffu;
  __device__ void add(double r2) {
    const uint32_t h = (uint32_t)(__builtin_bit_cast(uint64_t, r2) >> 32);
    m = h < m ? h : m;
  }
  __device__ bool hit() const { return m < 0x40100000u; }
};
template <>
struct NearTest<float> {
  uint32_t m = 0xffffffffu;
  __device__ void add(float r2) {
    const uint32_t b = __builtin_bit_cast(uint32_t, r2);
    m = b < m ? b : m;
  }
  __device__ bool hit() const { return m < 0x40800000u; }  // the bits of 4.0f
};

}  // namespace lm
