// Sums and maxima over the lanes of a wavefront without a trip through LDS: a shuffle between any two lanes takes that trip, about
// 50 cycles of latency each; exchanges within 16 lanes are operands of the addition itself (DPP), and gfx950 swaps rows of 16
// and of 32 lanes between two registers.
#pragma once
#include "common.hpp"

namespace lanes {

template <int CTRL>
__device__ __forceinline__ float from(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
struct Add {
  __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct Max {
  __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};

// over groups of N lanes next to each other, in every lane: lane ^ 1, lane ^ 2, then the mirror images within 8 and 16 lanes (whose
// groups of 4 and 8 hold one value by then), then rows of 16 and 32
template <int N, typename F>
__device__ __forceinline__ float over(float v, F f) {
  static_assert(N >= 2 && N <= 64 && (N & (N - 1)) == 0, "a power of two");
  v = f(v, from<0xB1>(v));
  if constexpr (N >= 4) v = f(v, from<0x4E>(v));
  if constexpr (N >= 8) v = f(v, from<0x141>(v));
  if constexpr (N >= 16) v = f(v, from<0x140>(v));
  if constexpr (N >= 32) {  // (the waits are the data hazard slots the compiler would insert if it saw the instruction)
    float a = v, b = v;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    v = f(a, b);
  }
  if constexpr (N >= 64) {
    float a = v, b = v;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    v = f(a, b);
  }
  return v;
}
template <int N = 64>
__device__ __forceinline__ float sum(float v) {
  return over<N>(v, Add());
}
template <int N = 64>
__device__ __forceinline__ float maximum(float v) {
  return over<N>(v, Max());
}

// n lanes next to each other (8, 16, 32 or 64, the same in the whole wavefront), in every lane
__device__ __forceinline__ float sum_of(float v, int n) {
  v = sum<8>(v);
  if (n > 8) v += from<0x140>(v);
  if (n > 16) {
    float a = v, b = v;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    v = a + b;
  }
  if (n > 32) {
    float a = v, b = v;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    v = a + b;
  }
  return v;
}
// the lanes n, 2 n, .. apart (n: 8, 16 or 32), in every lane
__device__ __forceinline__ float sum_apart(float v, int n) {
  if (n <= 8) v += from<0x128>(v);  // rotated by 8 within 16
  float a = v, b = v;
  if (n <= 16) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    v = a + b;
    a = b = v;
  }
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return a + b;
}

}  // namespace lanes
