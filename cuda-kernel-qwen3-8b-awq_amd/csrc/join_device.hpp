// The end of a sublayer for a row that a workgroup holds in registers (JoinArgs): a launch of its own (sublayer_ops.hip), or part of
// the one-token product that reads its result (dense.hip, dense_f32.hip).
#pragma once
#include "lane_sums.hpp"
#include "layers.hpp"

namespace {

template <typename T, int V>
struct Vec {
  typedef T type __attribute__((ext_vector_type(V)));
};
template <typename T, int V>
__device__ __forceinline__ void read(const T* p, float (&v)[V]) {
  if constexpr (V == 1) {
    v[0] = (float)*p;
  } else {
    const typename Vec<T, V>::type r = *reinterpret_cast<const typename Vec<T, V>::type*>(p);
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = (float)r[i];
  }
}
template <typename T, int V>
__device__ __forceinline__ void write(T* p, const float (&v)[V]) {
  if constexpr (V == 1) {
    *p = (T)v[0];
  } else {
    typename Vec<T, V>::type r;
#pragma unroll
    for (int i = 0; i < V; ++i) r[i] = (T)v[i];
    *reinterpret_cast<typename Vec<T, V>::type*>(p) = r;
  }
}

__device__ __forceinline__ float wave_sum(float v) { return lanes::sum(v); }
// sum over the workgroup; `sums` has a place per wavefront and is free again behind the next barrier
__device__ __forceinline__ float group_sum(float v, float* sums) {
  v = lanes::sum(v);
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  if (lane == 0) sums[threadIdx.x >> 6] = v;
  __syncthreads();
  return lanes::sum<16>((lane & 15) < waves ? sums[lane & 15] : 0.0f);
}

// y of token t from column c on, its shares in order, four requested at a time
template <int V>
__device__ __forceinline__ void read_y(const JoinArgs& a, int64_t t, int c, float (&v)[V]) {
  if (a.y_shares == 1) {
    read<float, V>(a.y + t * a.width + c, v);
    return;
  }
  const float* const y = a.y + t * a.ldy + c;
  for (int s = 0; s < a.y_shares; s += 4) {
    float u[4][V];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s + i < a.y_shares) read<float, V>(y + (s + i) * a.y_share, u[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s + i < a.y_shares) {
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = s + i == 0 ? u[i][e] : v[e] + u[i][e];
      }
  }
}

// Choices of a token that wait in registers.
constexpr int kJoinTop = 8;

// Q turns of V values per thread of a workgroup of `threads` threads.  Bound by trips to memory: everything is requested at once (an
// identity output's row of `pairs` too, which is then not used), the rows ahead of the weights of the norms.
template <typename T, int V, int Q>
struct JoinRow {
  const JoinArgs& a;
  const int64_t t;
  const int W, threads;
  float v[Q][V], g[Q][V], r[Q][V], w_post[Q][V], w_next[Q][V], h[Q][V], u[kJoinTop][Q][V], w[kJoinTop], y_gate;
  int ids[kJoinTop];
  __device__ __forceinline__ JoinRow(const JoinArgs& j, int64_t token, int n) : a(j), t(token), W((int)j.width), threads(n) {}
  __device__ __forceinline__ int column(int q) const { return ((int)threadIdx.x + q * threads) * V; }
  __device__ __forceinline__ void request_rows() {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int c = column(q);
#pragma unroll
      for (int i = 0; i < V; ++i) v[q][i] = g[q][i] = r[q][i] = h[q][i] = 0.0f;
      if (c >= W) continue;
      if (a.y) read_y<V>(a, t, c, v[q]);
      if (a.gate) read<T, V>(reinterpret_cast<const T*>(a.gate) + t * a.ldg + c, g[q]);
      read<float, V>(a.x + t * W + c, r[q]);
      if (a.top > 0) read<T, V>(reinterpret_cast<const T*>(a.h) + t * a.ldh + c, h[q]);
    }
#pragma unroll
    for (int j = 0; j < kJoinTop; ++j)
      if (j < a.top) {
        ids[j] = a.ids[t * a.top + j];
        w[j] = a.weights[t * a.top + j];
#pragma unroll
        for (int q = 0; q < Q; ++q)
          if (column(q) < W) read<float, V>(a.pairs + (t * a.top + j) * W + column(q), u[j][q]);
      }
    y_gate = a.y_gate ? a.y_gate[t] : 0.0f;
  }
  __device__ __forceinline__ void request_weights() {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (column(q) >= W) continue;
      read<float, V>(a.w_post + column(q), w_post[q]);
      if (a.w_next) read<float, V>(a.w_next + column(q), w_next[q]);
    }
  }
  // r: the new residual, then what the next sublayer reads; `sums`: two places per wavefront.  store(column, residual) in between
  template <typename S>
  __device__ __forceinline__ void finish(float (&sums)[2][16], S store) {
    const float y_mul = a.y_gate ? 1.0f / (1.0f + expf(-y_gate)) : 1.0f;
    float sq = 0.0f;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (column(q) >= W) continue;
      if (a.y) {
#pragma unroll
        for (int i = 0; i < V; ++i) v[q][i] *= y_mul;
      }
#pragma unroll
      for (int j = 0; j < kJoinTop; ++j)
        if (j < a.top) {
#pragma unroll
          for (int i = 0; i < V; ++i) v[q][i] = __builtin_fmaf(w[j], ids[j] < a.experts ? u[j][q][i] : h[q][i], v[q][i]);
        }
      if (a.gate) {
#pragma unroll
        for (int i = 0; i < V; ++i) v[q][i] *= g[q][i];
      }
#pragma unroll
      for (int i = 0; i < V; ++i) sq = __builtin_fmaf(v[q][i], v[q][i], sq);
    }
    const float inv = 1.0f / sqrtf(group_sum(sq, sums[0]) / (float)W + a.eps);
    sq = 0.0f;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (column(q) >= W) continue;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        r[q][i] = r[q][i] + v[q][i] * inv * w_post[q][i];
        sq = __builtin_fmaf(r[q][i], r[q][i], sq);
      }
      store(column(q), r[q]);
    }
    if (!a.out || !a.w_next) return;
    const float next = 1.0f / sqrtf(group_sum(sq, sums[1]) / (float)W + a.eps);
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int i = 0; i < V; ++i) r[q][i] = r[q][i] * next * w_next[q][i];
  }
};

// ... whose result the workgroup's own product reads: into LDS, zeros to the k-th input; `keeps`: this workgroup writes the residual
// and the result for the launches that follow
template <typename T, int Q, typename B>
__device__ __forceinline__ void joined_input(const JoinArgs& a, bool keeps, int k, T* in, float (&sums)[2][16], B between) {
  const int threads = (int)blockDim.x;
  JoinRow<T, 4, Q> row(a, 0, threads);
  row.request_rows();
  __builtin_amdgcn_sched_barrier(0);
  between();
  __builtin_amdgcn_sched_barrier(0);
  row.request_weights();
  row.finish(sums, [&](int c, const float (&r)[4]) {
    if (keeps) write<float, 4>(a.x_out + c, r);
  });
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int c = row.column(q);
    if (c >= row.W) continue;
    write<T, 4>(in + c, row.r[q]);
    if (keeps) write<T, 4>(reinterpret_cast<T*>(a.out) + c, row.r[q]);
  }
  for (int c = row.W + (int)threadIdx.x; c < k; c += threads) in[c] = (T)0.0f;
  __syncthreads();
}

}  // namespace
