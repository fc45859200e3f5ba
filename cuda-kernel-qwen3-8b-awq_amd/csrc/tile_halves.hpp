// Tiles of queries whose keys two sets of four wavefronts share: a maximum that moves when it must, and what their halves of a softmax come to
// (window_attention.hip, latent_attention.hip, prefill.hip).
#pragma once
#include "common.hpp"

namespace {

// the values of lane % 32 and lane % 32 + 32
struct HalfPair {
  float low, high;
};
__device__ __forceinline__ HalfPair half_pair(float x) {
  typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
  const u32x2_t p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return {__uint_as_float(p[0]), __uint_as_float(p[1])};
}

// The maximum m that a query's weights are relative to moves to mx, the largest score of a tile: always, or (LAGS) only once it is 2^kSlack behind
// it: sums grow by as much and no more (the conditional rescaling of FlashAttention-4).  Every query decides for itself, so that its
// bits do not depend on those that share its wavefront; what the wavefront decides is whether any has to.
// A maximum that lags saves the rescaling of most tiles: latents of 192 + 64, 1,024 tokens of 16 heads 98 -> 84 us, int4 256 tokens 9.8 -> 9.2; windows 0 to 1 %.
constexpr float kSlack = 8.0f;
template <bool LAGS, int BLOCKS, typename V>
__device__ __forceinline__ void move_maximum(float mx, float& m, float& l, V (&o)[BLOCKS]) {
  const bool moves = mx > (LAGS ? m + kSlack : m);
  if (__builtin_amdgcn_ballot_w64(moves) == 0) return;
  const float to = moves ? mx : m, alpha = moves ? __builtin_amdgcn_exp2f(m - to) : 1.0f;
  l *= alpha;
  m = to;
#pragma unroll
  for (int d = 0; d < BLOCKS; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
}

// A wavefront's o[d][i] are sums of weights and values for one query a lane (two lanes share a query), m its maximum (binary logarithm), l the sum of
// the weights.  Behind this a wavefront of half h has the sums of both halves of the blocks from h DV / 64 on, and l is the whole sum.
// `mine` and `other`: 16 KB of the halves' tiles, ml [2][2][256].
template <int DV, typename V>
__device__ __forceinline__ void merge_halves(const V (&o)[DV / 32], float m, float& l, float* mine, const float* other, float* ml, int tid, int half,
                                             V (&out)[DV / 64]) {
  constexpr int H = DV / 64;
  float f = 0.0f, f_other = 0.0f;
  __syncthreads();  // the last tiles' readers are done
  ml[half * 512 + tid] = m;
  ml[half * 512 + 256 + tid] = l;
#pragma unroll
  for (int d = 0; d < H; ++d) {
#pragma unroll
    for (int i = 0; i < 16; ++i) mine[i * 256 + tid] = half ? o[d][i] : o[H + d][i];
    __syncthreads();
    if (d == 0) {
      const float m_other = ml[(half ^ 1) * 512 + tid], l_other = ml[(half ^ 1) * 512 + 256 + tid], both = fmaxf(m, m_other);
      f = __builtin_amdgcn_exp2f(m - both);
      f_other = __builtin_amdgcn_exp2f(m_other - both);
      l = l * f + l_other * f_other;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) out[d][i] = (half ? o[H + d][i] : o[d][i]) * f + other[i * 256 + tid] * f_other;
    if (d + 1 < H) __syncthreads();
  }
}

}  // namespace
