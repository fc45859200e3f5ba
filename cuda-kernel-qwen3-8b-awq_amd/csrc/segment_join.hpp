// Segments of a pass that go side by side: a state behind a segment from the one ahead of it (linear_attention.hip, gated_state.hip).
#pragma once
#include "common.hpp"

namespace {

// A decay's power over a segment, in 64 bits, which hold it where binary32 would not: 0.86^640 is 1e-42.  A smaller one than 2^-500 brings nothing
// finite of binary32 with it; it stays a number above zero, as every step of the recurrence has one.
__device__ __forceinline__ double segment_power(float decay, int tokens) {
  double x = 1.0, y = (double)decay;
  for (int e = tokens; e; e >>= 1, y *= y)
    if (e & 1) x *= y;
  return x < 0x1p-500 ? 0x1p-500 : x;
}

// Rounded once; a state of zero brings nothing, whatever the power (of a decay above 1 it may be infinite), and an infinite one stays so.
__device__ __forceinline__ float behind_segment(float ahead, double power, float add) {
  return ahead != 0.0f ? (float)__builtin_fma((double)ahead, power, (double)add) : add;
}

// Where every channel has a decay of its own a segment leaves a product of them, kept as its root (with the product's sign): the smallest root,
// 2^-126, is that of a factor that brings nothing finite with it, and products stay above it as powers do.
template <typename R>
__device__ __forceinline__ R times_decay(R left, R by, R smallest) {
  const R x = left * by;
  return __builtin_elementwise_abs(x) < smallest && left != (R)0 && by != (R)0 ? __builtin_elementwise_copysign(smallest, x) : x;
}
__device__ __forceinline__ double of_root(float r) { return (double)r * __builtin_fabs((double)r); }

}  // namespace
