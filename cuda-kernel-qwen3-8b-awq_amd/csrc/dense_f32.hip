// Dense products of binary32 weights with one token or many (layers.hpp).
#include "dense_device.hpp"

namespace {

// --- one token -----------------------------------------------------------------------------------------------
// Bound by the weights' bytes.  A wavefront takes R rows (R = 2, 4: among them both rows of a gated pair) against one
// reading of the input, a workgroup of four wavefronts 4 R rows; a lane's sum of a row takes every 64th piece of four
// inputs whatever R is.  Rows of 1,024 inputs: 32,768 of them (a vocabulary's logits, R = 4) 29 us, 4.6 TB/s; four blocks of
// 1,536 gated rows (R = 2) 6.8 us, where a wavefront that took the two rows of a pair one after the other, beside one
// that had none, took 9.8; below 8,192 rows one each, so that 1,024 rows still make 256 workgroups.
template <int OUT, int R>
__global__ __launch_bounds__(256) void dense_one_f32_kernel(DenseArgs a) {
  __shared__ unsigned long long candidates[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // rows of the wavefront: row(0), and with R = 2 row(0) + 8, with R = 4 row(0) + 1, + 8, + 9
  const int base = R == 1 ? blockIdx.x * 4 : R == 2 ? (blockIdx.x >> 1) * 16 + (blockIdx.x & 1) * 4 : blockIdx.x * 16;
  const int row0 = base + wave * (R == 4 ? 2 : 1);
  auto row_of = [&](int i) { return row0 + (R == 4 ? (i & 1) + 8 * (i >> 1) : 8 * i); };
  const DenseSegment& s = segment_of(a, base);
  const int local0 = base - s.row0;
  if (local0 >= s.rows) return;
  int group = blockIdx.y;
  if (a.ids) {
    group = a.ids[blockIdx.y];
    if (group >= a.n_groups) return;
  }
  const f32x4u_t* x = reinterpret_cast<const f32x4u_t*>(reinterpret_cast<const float*>(s.x) + blockIdx.y * a.x_batch);
  const f32x4_t* w = reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(a.w) + group * a.w_batch);
  const int64_t k4 = a.k >> 2;
  float acc[R] = {};
  auto add = [&](const f32x4_t (&wv)[R], f32x4_t xv) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i] = __builtin_fmaf(wv[i][j], xv[j], acc[i]);
  };
  constexpr int U = R == 4 ? 4 : 8;
  int at = lane;
  for (; at + 64 * (U - 1) < (int)k4; at += 64 * U) {
    f32x4_t wv[U][R], xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < R; ++i) wv[u][i] = __builtin_nontemporal_load(w + row_of(i) * k4 + at + 64 * u);
      xv[u] = x[at + 64 * u];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) add(wv[u], xv[u]);
  }
  for (; at < (int)k4; at += 64) {
    f32x4_t wv[R];
#pragma unroll
    for (int i = 0; i < R; ++i) wv[i] = __builtin_nontemporal_load(w + row_of(i) * k4 + at);
    add(wv, x[at]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < R; ++i) acc[i] += __shfl_xor(acc[i], off, 64);
  // lane i ends row i
  float sum = acc[0];
  int row = row_of(0);
#pragma unroll
  for (int i = 1; i < R; ++i)
    if (lane == i) sum = acc[i], row = row_of(i);
  const int local = row - s.row0;
  const int64_t y0 = blockIdx.y * a.y_batch;
  if constexpr (OUT == DENSE_STORE && R > 1) {
    if (s.act == DENSE_GLU) {
      const int r = (local >> 4) * 8 + (local & 7);
      const float up = R == 4 && lane == 1 ? acc[R - 1] : acc[R / 2];
      if (lane < R / 2 && r < s.glu_rows) store_one<float>(s, y0, 0, r, glu<true>(sum, up));
      return;
    }
  }
  const bool mine = lane < R && local < s.rows;
  if (mine) finish_one<float, OUT>(a, s, 0, local, sum, y0);
  if constexpr (OUT == DENSE_ARGMAX) {
    if (s.act == DENSE_SOFTCAP) sum = softcap(s, sum);
    unsigned long long b = mine ? awq_pack_candidate(f32_key(sum), (uint32_t)local) : 0ull;
#pragma unroll
    for (int off = 1; off < R; off <<= 1) {
      const unsigned long long o = __shfl_xor(b, off, 64);
      b = o > b ? o : b;
    }
    if (lane == 0) candidates[wave] = b;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int v = 1; v < 4; ++v) b = candidates[v] > b ? candidates[v] : b;
      a.best[blockIdx.x] = b;
    }
  }
}

// --- many tokens ---------------------------------------------------------------------------------------------
// 64 rows x 64 tokens per workgroup, 4 x 4 per thread, through LDS.  A thread's rows are two of an eight and the same two of
// the eight behind it: a gate and its up row meet.
template <int OUT, bool LISTED = false>
__global__ __launch_bounds__(256) void dense_many_f32_kernel(DenseArgs a) {
  __shared__ float ws[16][68], xs[16][68];
  const int tid = threadIdx.x;
  const int row0 = blockIdx.x * 64;
  const int64_t tok0 = LISTED ? 0 : (int64_t)blockIdx.y * 64;
  const DenseSegment& s = segment_of(a, row0);
  if (row0 >= a.seg[a.n_seg - 1].row0 + a.seg[a.n_seg - 1].rows) return;
  int64_t group = blockIdx.z, n_tok = a.M;
  const int32_t* list = nullptr;
  if constexpr (LISTED) {
    const DenseTile run = a.tiles[blockIdx.y];
    if (run.count == 0) return;
    group = run.group;
    n_tok = run.count;
    list = a.list + run.first;
  }
  const int lr = tid >> 2, lk = (tid & 3) * 4;
  const float* w = reinterpret_cast<const float*>(a.w) + group * a.w_batch + (int64_t)(row0 + lr) * a.k + lk;
  int64_t tok = min(tok0 + lr, n_tok - 1);
  if constexpr (LISTED) tok = list[tok] / a.list_div;
  const float* x = reinterpret_cast<const float*>(s.x) + blockIdx.z * a.x_batch + tok * s.ldx + lk;
  const int tc = (tid >> 4) * 4;
  int tr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) tr[i] = 16 * ((tid & 15) >> 2) + 2 * (tid & 3) + (i & 1) + 8 * (i >> 1);
  float acc[4][4] = {};
  for (int k0 = 0; k0 < (int)a.k; k0 += 16) {
    const f32x4_t wv = *reinterpret_cast<const f32x4_t*>(w + k0);
    f32x4_t xv;
#pragma unroll
    for (int j = 0; j < 4; ++j) xv[j] = x[k0 + j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) ws[lk + j][lr] = wv[j], xs[lk + j][lr] = xv[j];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(ws[k][tr[i]], xs[k][tc + j], acc[i][j]);
  }
  const int64_t y0 = blockIdx.z * a.y_batch;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (tok0 + tc + j >= n_tok) continue;
    int64_t t = tok0 + tc + j;
    if constexpr (LISTED) t = list[t];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const DenseSegment& out = segment_of(a, row0 + tr[i]);
      const int row = row0 + tr[i] - out.row0;
      if (row >= out.rows) continue;
      if constexpr (OUT == DENSE_STORE) {
        if (out.act == DENSE_GLU) {
          const int r = (row >> 4) * 8 + (row & 7);
          if (i < 2 && r < out.glu_rows) store_one<float>(out, y0, t, r, glu<true>(acc[i][j], acc[i | 2][j]));
          continue;
        }
      }
      finish_one<float, OUT>(a, out, t, row, acc[i][j], y0);
    }
  }
}

template <int OUT>
int launch_one(const DenseArgs& a, int64_t rows, hipStream_t st) {
  bool pairs = false;
  for (int i = 0; i < a.n_seg; ++i) pairs |= a.seg[i].act == DENSE_GLU;
  const int64_t all = rows * a.batch;
  if (OUT == DENSE_ARGMAX || all >= 16384)
    hipLaunchKernelGGL((dense_one_f32_kernel<OUT, 4>), dim3((unsigned)(rows / 16), (unsigned)a.batch), dim3(256), 0, st, a);
  else if (pairs || all >= 8192)
    hipLaunchKernelGGL((dense_one_f32_kernel<OUT, 2>), dim3((unsigned)(rows / 8), (unsigned)a.batch), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((dense_one_f32_kernel<OUT, 1>), dim3((unsigned)(rows / 4), (unsigned)a.batch), dim3(256), 0, st, a);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

template <int OUT>
int launch_many(const DenseArgs& a, int64_t rows, hipStream_t st) {
  hipLaunchKernelGGL(dense_many_f32_kernel<OUT>, dim3((unsigned)(rows / 64), (unsigned)((a.M + 63) / 64), (unsigned)a.batch),
                     dim3(256), 0, st, a);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

}  // namespace

int launch_dense_one_f32(const DenseArgs& a, int64_t rows, hipStream_t st) {
  switch (a.out) {
    case DENSE_STORE: return launch_one<DENSE_STORE>(a, rows, st);
    case DENSE_RESIDUAL: return launch_one<DENSE_RESIDUAL>(a, rows, st);
    case DENSE_F32: return launch_one<DENSE_F32>(a, rows, st);
    default: return launch_one<DENSE_ARGMAX>(a, rows, st);
  }
}

int launch_dense_many_f32(const DenseArgs& a, int64_t rows, hipStream_t st) {
  if (a.tiles) {
    hipLaunchKernelGGL((dense_many_f32_kernel<DENSE_STORE, true>), dim3((unsigned)(rows / 64), (unsigned)a.max_tiles), dim3(256), 0,
                       st, a);
    AWQ_HIP_TRY(hipGetLastError());
    return AWQ_OK;
  }
  switch (a.out) {
    case DENSE_STORE: return launch_many<DENSE_STORE>(a, rows, st);
    case DENSE_RESIDUAL: return launch_many<DENSE_RESIDUAL>(a, rows, st);
    default: return launch_many<DENSE_F32>(a, rows, st);
  }
}
