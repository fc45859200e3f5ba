// Attention of a few queries of one head against cache rows, any sizes: what window_query_kernel and latent_query_kernel share
// (the binary32 forms, and rows that the tiled kernels have no instance for).
#pragma once
#include "layers.hpp"

namespace {

typedef float q4_t __attribute__((ext_vector_type(4)));
// four values of a row, aligned like one
template <typename T>
struct Four {
  typedef T type __attribute__((ext_vector_type(4), aligned(sizeof(T))));
};

// Queries that share a workgroup.  A workgroup's time grows with them (one, two and four: 9, 11 and 15 us for 4 queries against their own
// keys, 122, 143 and 218 for 64 queries of 8 heads of 128 behind 3,000), so they share one only where single ones would be
// several per compute unit, and then for the rows that are read once: 200 queries of 8 heads of 128 behind 3,000 259, 213 and
// 247 us, of 32 heads 850, 630 and 560.  The lines lie between what was slower and what was faster there at 0, 60, 400 and 3,000 keys
// ahead of 2 to 512 queries (heads of 64 to 512, latents of 160 to 1,064).  Without a window a query's sums are the same in all three.
inline int queries_together(int64_t heads, int64_t queries) {
  const int64_t alone = heads * queries;  // workgroups
  return alone <= 1024 ? 1 : alone <= 2560 ? 2 : 4;
}

inline size_t query_lds(int row, int queries) { return sizeof(float) * (size_t)(queries * (row + 256 + 4 + 1024)); }

// A workgroup of 256 threads takes QN queries next to each other, `q` [QN][row] in LDS, query i the keys lo[i] .. hi[i] (both
// ascending in i), in blocks of 256 with a running maximum.  Scores: sixteen lanes per key, four values each, so that a row is read in whole lines and
// by all queries at once; softmax: a thread per key; values: a thread per four columns and share of the block's keys.
// key_row(key), value_row(key): rows (row and cols values, row a multiple of 4; the columns behind
// the last to the next multiple of 4 are read too); score(i, key, dot): query i's score of a key that
// it sees (one of the first block among them).  m, l: where a query's maximum and sum start; they and the columns come out
// through store(i, column, four sums, l), for columns below `cols`.  A row that a query does not see is not in its
// sums, whatever the row holds.
// Bound by the reads out of the L2 and, for few queries, by the trips to it.  8 heads of 128, binary32: 333 queries 42 us (a thread per
// key and query that read its row value by value: 103), 16 queries 9.4 (11.5) and behind 3,000 keys 102 (361).  One query of
// 8 heads against 3,001 latents of 1,064 in bfloat16: 505 (735; 815 while the loop over value rows had a branch for the last columns
// in it, which waits for each row).  (The few keys that only some of the queries see have loops of their own: 0.2 us.)
template <typename T, int QN, typename K, typename V, typename S, typename O>
__device__ __forceinline__ void attend_queries(float* lds, int row, int cols, const int (&lo)[QN], const int (&hi)[QN], K key_row,
                                               V value_row, S score, float (&m)[QN], float (&l)[QN], O store) {
  typedef typename Four<T>::type four_t;
  float* const q = lds;               // [QN][row]
  float* const p = q + QN * row;      // [QN][256]
  float* const red = p + QN * 256;    // [QN][4]
  float* const part = red + QN * 4;   // [256][QN][4]
  const int tid = threadIdx.x, sub = tid & 15, group = tid >> 4;
  const int quads = (cols + 3) / 4, shares = max(1, 256 / quads), share = tid / quads, quad = tid % quads;
  q4_t acc[QN];
#pragma unroll
  for (int i = 0; i < QN; ++i) acc[i] = q4_t{0.0f, 0.0f, 0.0f, 0.0f};
  __syncthreads();  // q is written
  for (int k0 = lo[0]; k0 <= hi[QN - 1]; k0 += 256) {
    const int n = min(256, hi[QN - 1] + 1 - k0);
    for (int j0 = 0; j0 < n; j0 += 64) {  // four keys of a group at a time: j0 + 16 u + group
      float dot[4][QN] = {};
      const T* rows[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) rows[u] = key_row(k0 + min(j0 + 16 * u + group, n - 1));
#pragma unroll 2
      for (int c = 4 * sub; c < row; c += 64) {
        four_t k4[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) k4[u] = *reinterpret_cast<const four_t*>(rows[u] + c);
#pragma unroll
        for (int i = 0; i < QN; ++i) {
          const q4_t q4 = *reinterpret_cast<const q4_t*>(q + i * row + c);
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) dot[u][i] = __builtin_fmaf(q4[e], (float)k4[u][e], dot[u][i]);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < QN; ++i) {
          float d = dot[u][i];
#pragma unroll
          for (int off = 8; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
          if (sub == 0) p[i * 256 + j0 + 16 * u + group] = d;
        }
    }
    __syncthreads();
    float alpha[QN];
#pragma unroll
    for (int i = 0; i < QN; ++i) {
      const int key = k0 + tid;
      const float s = key >= lo[i] && key <= hi[i] ? score(i, key, p[i * 256 + tid]) : -INFINITY;
      float mx = s;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
      if ((tid & 63) == 0) red[i * 4 + (tid >> 6)] = mx;
      p[i * 256 + tid] = s;
    }
    __syncthreads();
    float sum[QN];
#pragma unroll
    for (int i = 0; i < QN; ++i) {
      const float m_new = fmaxf(m[i], fmaxf(fmaxf(red[i * 4], red[i * 4 + 1]), fmaxf(red[i * 4 + 2], red[i * 4 + 3])));
      const float e = expf(p[i * 256 + tid] - m_new);
      alpha[i] = expf(m[i] - m_new);
      m[i] = m_new;
      p[i * 256 + tid] = e;
      sum[i] = e;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) sum[i] += __shfl_xor(sum[i], off, 64);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < QN; ++i)
      if ((tid & 63) == 0) red[i * 4 + (tid >> 6)] = sum[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < QN; ++i) {
      l[i] = l[i] * alpha[i] + ((red[i * 4] + red[i * 4 + 1]) + (red[i * 4 + 2] + red[i * 4 + 3]));
      acc[i] = acc[i] * alpha[i];
    }
    if (share < shares) {
      auto add = [&](int j, bool all) __attribute__((always_inline)) {
        // (columns behind the last, which are there, are not stored: a branch for them would wait for each key's row)
        const four_t v = *reinterpret_cast<const four_t*>(value_row(k0 + j) + 4 * quad);
#pragma unroll
        for (int i = 0; i < QN; ++i) {
          if (!all && (k0 + j < lo[i] || k0 + j > hi[i])) continue;
          const float w = p[i * 256 + j];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(w, (float)v[e], acc[i][e]);
        }
      };
      // the keys ahead of the last query's first and behind the first query's last are not seen by all
      const int from = min(lo[QN - 1] - k0, n), to = min(hi[0] + 1 - k0, n);
      int j = share;
      if constexpr (QN > 1)
        for (; j < from; j += shares) add(j, false);
#pragma unroll 4
      for (; j < (QN > 1 ? to : n); j += shares) add(j, true);
      if constexpr (QN > 1)
        for (; j < n; j += shares) add(j, false);
    }
    __syncthreads();  // the block's weights are read
  }
  if (shares > 1) {
#pragma unroll
    for (int i = 0; i < QN; ++i) *reinterpret_cast<q4_t*>(part + (tid * QN + i) * 4) = acc[i];
    __syncthreads();
    const int used = min(shares, hi[QN - 1] + 1 - lo[0]);  // shares that had a key
    if (share == 0)
#pragma unroll 4
      for (int o = 1; o < used; ++o)
#pragma unroll
        for (int i = 0; i < QN; ++i) acc[i] = acc[i] + *reinterpret_cast<const q4_t*>(part + ((o * quads + quad) * QN + i) * 4);
  }
  if (share == 0)
#pragma unroll
    for (int i = 0; i < QN; ++i) store(i, 4 * quad, acc[i], l[i]);
}

}  // namespace
