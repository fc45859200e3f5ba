// Attention over a sliding window with a distance bias (layers.hpp).
#include "dense_one_device.hpp"
#include "query_attention.hpp"
#include "tile_halves.hpp"

namespace {

__device__ __forceinline__ float temperature(const WindowAttnArgs& a, int p) {
  if (a.temp_coef == 0.0f) return 1.0f;
  return 1.0f + a.temp_coef * logf((float)floor((double)(p + 1) / a.temp_every) + 1.0f);
}

// One wavefront per (token, head of q, k or v): q normalised in place, k normalised into its cache row, v copied
// into its cache row.
template <typename T>
__global__ __launch_bounds__(256) void window_append_kernel(WindowAttnArgs a) {
  const int lane = threadIdx.x & 63, item = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int t = blockIdx.y;
  if (item >= a.heads + 2 * a.kv_heads) return;
  T* row = reinterpret_cast<T*>(a.proj) + (int64_t)t * a.ldp;
  const int pos = a.pos.position() + t;
  if (item >= a.heads + a.kv_heads) {
    const int g = item - a.heads - a.kv_heads;
    const T* v = row + (int64_t)(a.heads + a.kv_heads) * a.dim + (int64_t)g * a.vdim;
    T* dst = reinterpret_cast<T*>(a.v_cache) + ring_row(a.vl, g, pos % a.vl.slots);
    for (int d = lane; d < a.vl.row; d += 64) dst[d] = d < a.vdim ? v[d] : (T)0.0f;
    return;
  }
  T* x = row + (int64_t)item * a.dim;
  float acc = 0.0f;
  for (int d = lane; d < a.dim; d += 64) acc = __builtin_fmaf((float)x[d], (float)x[d], acc);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  const float inv = 1.0f / sqrtf(acc / (float)a.dim + a.eps);
  if (item < a.heads) {
    for (int d = lane; d < a.dim; d += 64) x[d] = (T)((float)x[d] * inv);
  } else {
    T* dst = reinterpret_cast<T*>(a.k_cache) + ring_row(a.kl, item - a.heads, pos % a.kl.slots);
    for (int d = lane; d < a.kl.row; d += 64) dst[d] = d < a.dim ? (T)((float)x[d] * inv) : (T)0.0f;
  }
}

// The same for head sizes that are whole 16-byte pieces: a group of lanes per row, 8 elements each.
__global__ __launch_bounds__(256) void window_append8_kernel(WindowAttnArgs a, int lanes) {
  const int items = a.heads + 2 * a.kv_heads;
  const int64_t at = (int64_t)blockIdx.x * (256 / lanes) + threadIdx.x / lanes;
  const int t = (int)(at / items), item = (int)(at - (int64_t)t * items), d0 = (threadIdx.x % lanes) * 8;
  if (t >= (int)a.M) return;
  bf16_t* row = reinterpret_cast<bf16_t*>(a.proj) + (int64_t)t * a.ldp;
  const int pos = a.pos.position() + t;
  const bool value = item >= a.heads + a.kv_heads;
  bf16_t* src = value ? row + (int64_t)(a.heads + a.kv_heads) * a.dim + (int64_t)(item - a.heads - a.kv_heads) * a.vdim
                      : row + (int64_t)item * a.dim;
  const int n = value ? a.vdim : a.dim;
  bf16x8_t x;
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = (bf16_t)0.0f;
  if (d0 < n) x = *reinterpret_cast<const bf16x8_t*>(src + d0);
  float acc = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) acc = __builtin_fmaf((float)x[i], (float)x[i], acc);
  for (int off = lanes >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (value) {
    if (d0 < a.vl.row)
      *reinterpret_cast<bf16x8_t*>(reinterpret_cast<bf16_t*>(a.v_cache) +
                                   ring_row(a.vl, item - a.heads - a.kv_heads, pos % a.vl.slots) + d0) = x;
    return;
  }
  const float inv = 1.0f / sqrtf(acc / (float)a.dim + a.eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = (bf16_t)((float)x[i] * inv);
  if (item < a.heads) {
    if (d0 < a.dim) *reinterpret_cast<bf16x8_t*>(src + d0) = x;
  } else if (d0 < a.kl.row) {
    *reinterpret_cast<bf16x8_t*>(reinterpret_cast<bf16_t*>(a.k_cache) + ring_row(a.kl, item - a.heads, pos % a.kl.slots) + d0) = x;
  }
}

// A few queries of a head at a time (query_attention.hpp); the binary32 form and what the tiled kernel has no instance for.
constexpr int kMaxCols = 1024;
template <typename T, int QN>
__global__ __launch_bounds__(256) void window_query_kernel(WindowAttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];  // query_lds(kl.row, QN)
  const int h = blockIdx.x, t0 = blockIdx.y * QN, tid = threadIdx.x, row = a.kl.row, M = (int)a.M;
  const int g = h / (a.heads / a.kv_heads);
  const int pos0 = a.pos.position();
  const float slope = a.slope[h];
  int pos[QN], lo[QN];
  float mul[QN], m[QN], l[QN];
#pragma unroll
  for (int i = 0; i < QN; ++i) {
    const int t = min(t0 + i, M - 1);
    const T* const q = reinterpret_cast<const T*>(a.proj) + (int64_t)t * a.ldp + (int64_t)h * a.dim;
    for (int d = tid; d < row; d += 256) lds[i * row + d] = d < a.dim ? (float)q[d] : 0.0f;
    pos[i] = pos0 + t;
    lo[i] = a.window > 0 ? max(0, pos[i] - a.window + 1) : 0;
    mul[i] = a.scale * temperature(a, pos[i]);
    m[i] = -INFINITY;
    l[i] = 0.0f;
  }
  const T* const kc = reinterpret_cast<const T*>(a.k_cache);
  const T* const vc = reinterpret_cast<const T*>(a.v_cache);
  attend_queries<T, QN>(
      lds, row, a.vdim, lo, pos, [&](int key) { return kc + ring_row(a.kl, g, key % a.kl.slots); },
      [&](int key) { return vc + ring_row(a.vl, g, key % a.vl.slots); },
      [&](int i, int key, float dot) { return dot * mul[i] - slope * (float)(pos[i] - key); }, m, l,
      [&](int i, int col, q4_t sum, float total) {
        if (t0 + i >= M) return;
        T* const out = reinterpret_cast<T*>(a.ctx) + (int64_t)(t0 + i) * a.ldc + (int64_t)h * a.vdim + col;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < a.vdim) out[e] = (T)(sum[e] / total);
      });
}

// One token.  blockIdx.x: kv head and up to R of its query heads, blockIdx.y: 64 of the visible keys.  The rows a
// workgroup needs are requested before anything else; every lane group normalises the queries for itself, and the
// workgroup of the newest position takes its key and value from the projections and appends them.  A wavefront's
// lane holds the weight of one key.  Sums over lanes go without LDS: 8 heads of 128 and one part 8.2 us with trips through it, 6.5 without.
// Several parts are added up by a second launch, a workgroup per head, or where window_counted_parts says so by the workgroup that
// counts itself in last.
constexpr int kPartKeys = 64;

__host__ __device__ inline int window_parts(int64_t window, int64_t max_pos) {
  const int64_t n = window > 0 && window < max_pos ? window : max_pos;
  return (int)((n + kPartKeys - 1) / kPartKeys);
}

template <typename T>
struct Vec8;
template <>
struct Vec8<bf16_t> {
  bf16x8_t v;
};
template <>
struct Vec8<float> {
  typedef float f8 __attribute__((ext_vector_type(8)));
  f8 v;
};
// elements at .. at + 7 of a row of n, zeros behind it
template <typename T>
__device__ __forceinline__ void row_piece(const T* row, int at, int n, bool aligned, float (&x)[8]) {
  if (aligned && at + 8 <= n) {
    const Vec8<T> v = *reinterpret_cast<const Vec8<T>*>(row + at);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = (float)v.v[i];
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = at + i < n ? (float)row[at + i] : 0.0f;
  }
}

// SAME: the parts are added up in the launch that forms them.  They then leave the die as they are stored and are read past its
// caches, since another die's workgroup may be the one that adds them.
template <bool SAME>
__device__ __forceinline__ void put_part(float* p, float v) {
  if constexpr (SAME) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}
template <bool SAME>
__device__ __forceinline__ float get_part(const float* p) {
  if constexpr (SAME) return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return *p;
}

// One head's parts, [maximum, sum, context] each, by a workgroup of 256; red: 256 floats of LDS
template <typename T, bool SAME>
__device__ __forceinline__ void combine_parts(const WindowAttnArgs& a, int h, int n_parts, int parts, float* red) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t ps = 2 + a.vdim;
  const float* p = a.parts + (int64_t)h * n_parts * ps;
  // columns, and as many runs of parts next to each other as there are threads left
  const int cols = min(256, a.vdim), runs = 256 / cols, run = tid / cols;
  float m = -INFINITY, l = 0.0f;
  for (int s = lane; s < parts; s += 64) m = fmaxf(m, get_part<SAME>(p + s * ps));
  m = lanes::maximum(m);
  for (int s = lane; s < parts; s += 64) l = __builtin_fmaf(expf(get_part<SAME>(p + s * ps) - m), get_part<SAME>(p + s * ps + 1), l);
  l = lanes::sum(l);
  for (int c = tid % cols; c < (a.vdim + cols - 1) / cols * cols; c += cols) {
    float x = 0.0f;
    if (run < runs && c < a.vdim)
#pragma unroll 4
      for (int s = run; s < parts; s += runs) x = __builtin_fmaf(expf(get_part<SAME>(p + s * ps) - m), get_part<SAME>(p + s * ps + 2 + c), x);
    red[tid] = x;
    __syncthreads();
    if (run == 0 && c < a.vdim) {
      for (int i = 1; i < runs; ++i) x += red[tid + i * cols];
      reinterpret_cast<T*>(a.ctx)[(int64_t)h * a.vdim + c] = (T)(x / l);
    }
    __syncthreads();
  }
}

// U: cache rows of a lane, row length / 32
template <typename T, int R, int U, bool SAME>
__device__ __forceinline__ void decode_part(const WindowAttnArgs& a, const int chunks, const int block, const int part, const int n_parts) {
  extern __shared__ float red[];      // [4][R][vw]
  __shared__ float sc[R][kPartKeys];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = block / chunks, rz = (block - g * chunks) * R;
  const int per_group = a.heads / a.kv_heads;
  const int nr = min(R, per_group - rz), h0 = g * per_group + rz;
  const int pos = a.pos.position();
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int parts = (pos + 1 - lo + kPartKeys - 1) / kPartKeys;
  if (part >= parts) return;
  const int b = lo + part * kPartKeys, nk = min(kPartKeys, pos + 1 - b);
  const bool newest = part == parts - 1;
  const int kw = a.kl.row, vw = a.vl.row;
  // lanes of a key and of a value row: 8 elements each
  const int lpk = kw >> 3, sub = lane / lpk, d0 = (lane - sub * lpk) * 8, kpw = 64 / lpk, uk = kw >> 5;
  const int tpv = vw >> 3, c0 = (tid % tpv) * 8, first = tid / tpv, step = 256 / tpv, uv = vw >> 5;
  const T* const kc = reinterpret_cast<const T*>(a.k_cache);
  const T* const vc = reinterpret_cast<const T*>(a.v_cache);
  const int slot0 = b % a.kl.slots;
  auto slot_of = [&](int key) {  // of a key of this part
    const int s = slot0 + key - b;
    return s < a.kl.slots ? s : s - a.kl.slots;
  };
  Vec8<T> kv[U], vv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int key = b + (u * 4 + wave) * kpw + sub;
    if (u < uk && key < pos) kv[u] = *reinterpret_cast<const Vec8<T>*>(kc + ring_row(a.kl, g, slot_of(key)) + d0);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int key = b + u * step + first;
    if (u < uv && key < pos) vv[u] = *reinterpret_cast<const Vec8<T>*>(vc + ring_row(a.vl, g, slot_of(key)) + c0);
  }
  const T* const proj = reinterpret_cast<const T*>(a.proj);
  const bool dim8 = (a.dim & 7) == 0, vdim8 = ((a.dim | a.vdim) & 7) == 0;
  float qv[R][8], kn[8] = {}, vn[8] = {};
#pragma unroll
  for (int r = 0; r < R; ++r) row_piece(proj + (int64_t)(h0 + min(r, nr - 1)) * a.dim, d0, a.dim, dim8, qv[r]);
  if (newest) {
    row_piece(proj + (int64_t)(a.heads + g) * a.dim, d0, a.dim, dim8, kn);
    row_piece(proj + (int64_t)(a.heads + a.kv_heads) * a.dim + (int64_t)g * a.vdim, c0, a.vdim, vdim8, vn);
  }
  const float mul = a.scale * temperature(a, pos);  // (while the rows are on their way)
  auto normalise = [&](float (&x)[8]) {
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc = __builtin_fmaf(x[i], x[i], acc);
    const float inv = 1.0f / sqrtf(lanes::sum_of(acc, lpk) / (float)a.dim + a.eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = (float)(T)(x[i] * inv);
  };
#pragma unroll
  for (int r = 0; r < R; ++r) normalise(qv[r]);
  if (newest) {
    normalise(kn);
    Vec8<T> out;
    if (rz == 0 && tid < lpk) {
#pragma unroll
      for (int i = 0; i < 8; ++i) out.v[i] = (T)kn[i];
      *reinterpret_cast<Vec8<T>*>(reinterpret_cast<T*>(a.k_cache) + ring_row(a.kl, g, pos % a.kl.slots) + d0) = out;
    }
    if (rz == 0 && tid < tpv) {
#pragma unroll
      for (int i = 0; i < 8; ++i) out.v[i] = (T)vn[i];
      *reinterpret_cast<Vec8<T>*>(reinterpret_cast<T*>(a.v_cache) + ring_row(a.vl, g, pos % a.vl.slots) + c0) = out;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u >= uk) break;
    const int i = (u * 4 + wave) * kpw + sub, key = b + i;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = key < pos ? (float)kv[u].v[j] : kn[j];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float dot = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) dot = __builtin_fmaf(qv[r][j], x[j], dot);
      dot = lanes::sum_of(dot, lpk);
      if (d0 == 0) sc[r][i] = dot;
    }
  }
  __syncthreads();
  // every wavefront: lane = key
  float p[R], pm[R], pl[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float s = lane < nk && r < nr ? sc[r][lane] * mul - a.slope[h0 + r] * (float)(pos - b - lane) : -INFINITY;
    const float m = lanes::maximum(s), e = r < nr ? expf(s - m) : 0.0f;
    p[r] = e;
    pm[r] = m;
    pl[r] = lanes::sum(e);
  }
  float acc[R][8] = {};
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u >= uv) break;
    const int i = u * step + first;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = b + i < pos ? (float)vv[u].v[j] : vn[j];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float w = __shfl(p[r], i, 64);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[r][j] = __builtin_fmaf(w, i < nk ? x[j] : 0.0f, acc[r][j]);
    }
  }
  // lanes of a wavefront that share columns, then the wavefronts
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      acc[r][j] = lanes::sum_apart(acc[r][j], tpv);
      if (lane < tpv) red[(wave * R + r) * vw + c0 + j] = acc[r][j];
    }
  __syncthreads();
  const bool alone = n_parts == 1 || (SAME && parts == 1);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= nr) break;
    float* const mine = a.parts + ((int64_t)(h0 + r) * n_parts + part) * (2 + a.vdim);
    for (int c = tid; c < a.vdim; c += 256) {
      const float x = (red[r * vw + c] + red[(R + r) * vw + c]) + (red[(2 * R + r) * vw + c] + red[(3 * R + r) * vw + c]);
      if (alone) reinterpret_cast<T*>(a.ctx)[(int64_t)(h0 + r) * a.vdim + c] = (T)(x / pl[r]);
      else put_part<SAME>(mine + 2 + c, x);
    }
    if (!alone && tid == 0) put_part<SAME>(mine, pm[r]), put_part<SAME>(mine + 1, pl[r]);
  }
  if constexpr (SAME) {
    if (alone) return;
    // the parts are out of this die when the workgroup counts itself in; the last one finds all of them
    __shared__ int last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      last = __hip_atomic_fetch_add(a.done + block, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
      if (last) __hip_atomic_store(a.done + block, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    }
    __syncthreads();
    if (!last) return;
    static_assert(R == 1, "heads next to each other would be added up one after the other");
    combine_parts<T, true>(a, h0, n_parts, parts, red);
  }
}

template <typename T, int R, int U, bool SAME>
__global__ __launch_bounds__(256) void window_decode_kernel(WindowAttnArgs a, int chunks) {
  decode_part<T, R, U, SAME>(a, chunks, blockIdx.x, blockIdx.y, gridDim.y);
}

// The same with a product that does not wait for it in the launch (a layer's W_down beside its attention): the first
// groups * n_parts workgroups attend, four of their wavefronts, the others take RW rows of the product each.
template <int R, int U, bool SAME, int RW>
__global__ __launch_bounds__(512) void window_decode_beside_kernel(WindowAttnArgs a, int chunks, int groups, int n_parts, DenseArgs beside) {
  const int block = blockIdx.x;
  if (block >= groups * n_parts) {
    dense_one_rows<8, DENSE_RESIDUAL, IN_READ, RW>(beside, std::false_type(), block - groups * n_parts, 0);
    return;
  }
  if (threadIdx.x >= 256) return;
  decode_part<bf16_t, R, U, SAME>(a, chunks, block % groups, block / groups, n_parts);
}

// a workgroup per head
template <typename T>
__global__ __launch_bounds__(256) void window_combine_kernel(WindowAttnArgs a, int n_parts) {
  __shared__ float red[256];
  const int pos = a.pos.position();
  const int parts = ((a.window > 0 ? min(a.window, pos + 1) : pos + 1) + kPartKeys - 1) / kPartKeys;
  combine_parts<T, false>(a, blockIdx.x, n_parts, parts, red);
}

template <int R, int U, bool SAME>
int launch_decode_beside(const WindowAttnArgs& a, int chunks, int parts, size_t lds, const DenseArgs& product, hipStream_t st) {
  DenseArgs p = product;
  int64_t rows = 0;
  int per_group = 0;
  if (int rc = dense_prepare_beside(&p, &rows, &per_group)) return rc;
  const int groups = a.kv_heads * chunks;
  const int64_t blocks = (int64_t)groups * parts + rows / per_group;
  AWQ_REQUIRE(blocks < (1ll << 31), "too large");
  const dim3 g((unsigned)blocks);
  if (per_group == 8) hipLaunchKernelGGL((window_decode_beside_kernel<R, U, SAME, 8>), g, dim3(512), lds, st, a, chunks, groups, parts, p);
  else hipLaunchKernelGGL((window_decode_beside_kernel<R, U, SAME, 16>), g, dim3(512), lds, st, a, chunks, groups, parts, p);
  return AWQ_OK;
}

// query heads of a workgroup
int decode_heads(int per_group) { return per_group <= 2 ? per_group : per_group <= 4 ? 4 : 8; }

template <typename T, int R, bool SAME>
int launch_decode_parts(const WindowAttnArgs& a, int parts, const DenseArgs* beside, hipStream_t st) {
  const int chunks = (a.heads / a.kv_heads + R - 1) / R;
  const dim3 g((unsigned)(a.kv_heads * chunks), (unsigned)parts);
  const size_t lds = sizeof(float) * 4 * R * a.vl.row;  // (256 floats at least)
  const int row = std::max(a.kl.row, a.vl.row);
  if constexpr (sizeof(T) == 2) {
    if (beside) {
      if (row == 64) return launch_decode_beside<R, 2, SAME>(a, chunks, parts, lds, *beside, st);
      if (row == 128) return launch_decode_beside<R, 4, SAME>(a, chunks, parts, lds, *beside, st);
      return launch_decode_beside<R, 8, SAME>(a, chunks, parts, lds, *beside, st);
    }
  }
  if (row == 64) hipLaunchKernelGGL((window_decode_kernel<T, R, 2, SAME>), g, dim3(256), lds, st, a, chunks);
  else if (row == 128) hipLaunchKernelGGL((window_decode_kernel<T, R, 4, SAME>), g, dim3(256), lds, st, a, chunks);
  else hipLaunchKernelGGL((window_decode_kernel<T, R, 8, SAME>), g, dim3(256), lds, st, a, chunks);
  return AWQ_OK;
}

template <typename T>
int launch_decode(const WindowAttnArgs& a, hipStream_t st, const DenseArgs* beside) {
  const int parts = window_parts(a.window, a.len_bound);
  AWQ_REQUIRE(parts >= 1 && parts <= 65535, "too many keys");
  const int at_once = decode_heads(a.heads / a.kv_heads);
  const bool same = a.done && window_counted_parts(a.heads, a.kv_heads, a.window, a.len_bound);
  const auto launch = same ? launch_decode_parts<T, 1, true>
                           : at_once == 1 ? launch_decode_parts<T, 1, false>
                                          : at_once == 2 ? launch_decode_parts<T, 2, false> : at_once == 4 ? launch_decode_parts<T, 4, false> : launch_decode_parts<T, 8, false>;
  if (int rc = launch(a, parts, beside, st)) return rc;
  AWQ_HIP_TRY(hipGetLastError());
  if (parts > 1 && !same) {
    hipLaunchKernelGGL(window_combine_kernel<T>, dim3((unsigned)a.heads), dim3(256), 0, st, a, parts);
    AWQ_HIP_TRY(hipGetLastError());
  }
  return AWQ_OK;
}

// Many tokens, bfloat16.  128 queries of one head per workgroup, 32 per wavefront; keys and values of 32 positions at
// a time go through LDS.  Operands of v_mfma_f32_32x32x16_bf16, lane (n, kh) = (lane % 32, lane / 32), queries as
// columns throughout:
//     S^T[key][query] = K Q^T,   O^T[c][query] += V^T P^T
// so that a query's maximum, sum and rescaling stay in a lane and its partner, and the weights a lane forms are the
// elements it supplies to the second product (slice j: keys 16 j + 8 (e / 4) + 4 kh + e % 4; V^T by the transposing
// LDS read).  Scores and weights are binary32; a weight enters the product as the sum of two bfloat16 terms.
typedef short short4_t __attribute__((ext_vector_type(4)));
constexpr int kTileQueries = 128, kTileKeys = 32;

template <int DK, int DV, int HALVES>
__global__ __launch_bounds__(256 * HALVES, (DK + DV > 256) ? 1 : 2) void window_tile_kernel(WindowAttnArgs a) {
  constexpr int KS = DK + 8, VS = DV + 16;
  constexpr int KP = DK / 64, VP = DV / 64;  // 16-byte pieces of a tile per thread
  constexpr int kTiles = 2 * kTileKeys * (KS + VS);
  __shared__ __attribute__((aligned(16))) bf16_t tiles[HALVES * kTiles];
  __shared__ float ml[HALVES == 2 ? 1024 : 1];
  const int half = HALVES == 2 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) : 0;
  bf16_t *const ks2 = tiles + half * kTiles, *const vs2 = ks2 + 2 * kTileKeys * KS;
  const int h = blockIdx.x, g = h / (a.heads / a.kv_heads);
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, kh = lane >> 5;
  const int M = (int)a.M, pos0 = a.pos.pos0;
  const int q_first = blockIdx.y * kTileQueries;
  const int qi = q_first + wave * 32 + n, qc = min(qi, M - 1);
  const int pq = pos0 + qc;  // this lane's position
  auto oldest = [&](int p) { return a.window > 0 ? max(0, p - a.window + 1) : 0; };
  const int w_first = pos0 + min(q_first + wave * 32, M - 1), w_last = pos0 + min(q_first + wave * 32 + 31, M - 1);
  const int lo_q = oldest(pq), lo_wave = oldest(w_first), lo_full = oldest(w_last);
  const int k_begin = oldest(pos0 + q_first) & ~(kTileKeys - 1);
  const int k_end = pos0 + min(q_first + kTileQueries - 1, M - 1) + 1;

  const bf16_t* q = reinterpret_cast<const bf16_t*>(a.proj) + (int64_t)qc * a.ldp + (int64_t)h * a.dim;
  bf16x8_t qop[DK / 16];
#pragma unroll
  for (int s = 0; s < DK / 16; ++s) {
    const int at = 16 * s + 8 * kh;
    if (a.dim == DK) {
      qop[s] = *reinterpret_cast<const bf16x8_t*>(q + at);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) qop[s][e] = at + e < a.dim ? q[at + e] : (bf16_t)0.0f;
    }
  }
  f32x16_t o[DV / 32];
#pragma unroll
  for (int d = 0; d < DV / 32; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
  float m_run = -1e30f, l_run = 0.0f;
  constexpr float kLog2e = 1.44269504088896340736f;
  const float mul = a.scale * temperature(a, pq) * kLog2e, slope = a.slope[h] * kLog2e;

  const bf16_t* const kc = reinterpret_cast<const bf16_t*>(a.k_cache);
  const bf16_t* const vc = reinterpret_cast<const bf16_t*>(a.v_cache);
  struct TileRegs {
    bf16x8_t k[KP > 0 ? KP : 1], v[VP > 0 ? VP : 1];
  };
  TileRegs ra, rb;
  auto load_tile = [&](int k0, TileRegs& r) __attribute__((always_inline)) {
    if (k0 >= k_end) return;
    const int slot = k0 % a.kl.slots;  // 32 positions from a multiple of 32 on never wrap
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int pc = tid + i * 256, key = pc / (DK / 8), at = (pc % (DK / 8)) * 8;
      r.k[i] = *reinterpret_cast<const bf16x8_t*>(kc + ring_row(a.kl, g, slot + key) + at);
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int pc = tid + i * 256, key = pc / (DV / 8), at = (pc % (DV / 8)) * 8;
      r.v[i] = *reinterpret_cast<const bf16x8_t*>(vc + ring_row(a.vl, g, slot + key) + at);
    }
  };
  auto store_tile = [&](int half, const TileRegs& r) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int pc = tid + i * 256, key = pc / (DK / 8), at = (pc % (DK / 8)) * 8;
      *reinterpret_cast<bf16x8_t*>(ks2 + (half * kTileKeys + key) * KS + at) = r.k[i];
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int pc = tid + i * 256, key = pc / (DV / 8), at = (pc % (DV / 8)) * 8;
      *reinterpret_cast<bf16x8_t*>(vs2 + (half * kTileKeys + key) * VS + at) = r.v[i];
    }
  };
  // Bound by the chain of a wavefront that has a SIMD nearly to itself, so operands are read four products ahead and the first values
  // ahead of the softmax.  (Two tiles to a softmax: no registers for it with halves, without them no faster.)
  auto step = [&](int k0, int at) __attribute__((always_inline)) {
    if (k0 > w_last || k0 + kTileKeys <= lo_wave) return;  // no query of this wavefront sees a key of the tile
    const bf16_t* const klane = ks2 + (at * kTileKeys + n) * KS + 8 * kh;
    const int L16 = lane & 15;
    const bf16_t* const vlane = vs2 + (at * kTileKeys + 4 * kh + (L16 >> 2)) * VS + 16 * ((lane >> 4) & 1) + 4 * (L16 & 3);
    auto values = [&](int j, int d) __attribute__((always_inline)) {
      const bf16_t* vp = vlane + 16 * j * VS + d * 32;
      const short4_t l = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4_t __attribute__((address_space(3)))*)vp);
      const short4_t u = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4_t __attribute__((address_space(3)))*)(vp + 8 * VS));
      const bf16x4_t l4 = __builtin_bit_cast(bf16x4_t, l), u4 = __builtin_bit_cast(bf16x4_t, u);
      return bf16x8_t{l4[0], l4[1], l4[2], l4[3], u4[0], u4[1], u4[2], u4[3]};
    };
    f32x16_t s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < DK / 16; ++d)
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t*>(klane + 16 * d), qop[d], s, 0, 0, 0);
    bf16x8_t vv[DV / 32];  // (of the first slice)
#pragma unroll
    for (int d = 0; d < DV / 32; ++d) vv[d] = values(0, d);
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int d = 0; d < DK / 16; ++d) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // s[i]: key k0 + 8 (i / 4) + 4 kh + i % 4 for this lane's query
    const float base = (float)(k0 + 4 * kh - pq);  // (sums of whole numbers below 2^24)
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = __builtin_fmaf(s[i], mul, slope * (base + (float)(8 * (i >> 2) + (i & 3))));
    if (k0 + kTileKeys - 1 > w_first || k0 < lo_full) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = k0 + 8 * (i >> 2) + 4 * kh + (i & 3);
        s[i] = key <= pq && key >= lo_q ? s[i] : -INFINITY;
      }
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    const HalfPair best = half_pair(mx);
    mx = fmaxf(best.low, best.high);
    move_maximum<HALVES == 2>(mx, m_run, l_run, o);
    float rs = 0.0f;
    bf16x8_t hi[2], lo[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = __builtin_amdgcn_exp2f(s[i] - m_run);
      rs += p;
      hi[i >> 3][i & 7] = (bf16_t)p;
      lo[i >> 3][i & 7] = (bf16_t)(p - (float)hi[i >> 3][i & 7]);
    }
    const HalfPair sums = half_pair(rs);
    l_run += sums.low + sums.high;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int d = 0; d < DV / 32; ++d) o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv[d], hi[j], o[d], 0, 0, 0);
#pragma unroll
      for (int d = 0; d < DV / 32; ++d) {
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv[d], lo[j], o[d], 0, 0, 0);
        if (j + 1 < 2) vv[d] = values(j + 1, d);
      }
    }
  };
  const int first = k_begin + 2 * kTileKeys * half;
  load_tile(first, ra);
  load_tile(first + kTileKeys, rb);
  // The first products wait for the queries here: inside the loop, where the number of requests on their way is not known, that wait would be one for
  // everything, the next tiles with it.
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  for (int k0 = first; k0 - 2 * kTileKeys * half < k_end; k0 += 2 * HALVES * kTileKeys) {
    __syncthreads();  // the previous tiles' readers are done
    if (k0 < k_end) store_tile(0, ra);
    if (k0 + kTileKeys < k_end) store_tile(1, rb);
    __syncthreads();
    load_tile(k0 + 2 * HALVES * kTileKeys, ra);
    load_tile(k0 + (2 * HALVES + 1) * kTileKeys, rb);
    if (k0 < k_end) step(k0, 0);
    if (k0 + kTileKeys < k_end) step(k0 + kTileKeys, 1);
  }
  constexpr int kOut = DV / 32 / HALVES;  // blocks that this wavefront ends
  f32x16_t ended[kOut];
  if constexpr (HALVES == 2) {
    merge_halves<DV>(o, m_run, l_run, reinterpret_cast<float*>(ks2), reinterpret_cast<const float*>(tiles + (half ^ 1) * kTiles), ml, tid, half, ended);
  } else {
#pragma unroll
    for (int d = 0; d < kOut; ++d) ended[d] = o[d];
  }
  if (qi >= M) return;
  // ended[d][i]: column 32 (kOut half + d) + 8 (i / 4) + 4 kh + i % 4
  const float inv = 1.0f / l_run;
  bf16_t* out = reinterpret_cast<bf16_t*>(a.ctx) + (int64_t)qi * a.ldc + (int64_t)h * a.vdim;
#pragma unroll
  for (int d = 0; d < kOut; ++d)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = 32 * (kOut * half + d) + 8 * u + 4 * kh;
      if (c + 3 < a.vdim && (a.vdim & 3) == 0) {
        bf16x4_t v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (bf16_t)(ended[d][4 * u + j] * inv);
        *reinterpret_cast<bf16x4_t*>(out + c) = v;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (c + j < a.vdim) out[c + j] = (bf16_t)(ended[d][4 * u + j] * inv);
      }
    }
}

// Halves of the keys where a compute unit has a workgroup at most and the longest run of keys is more than two turns of both: 8 heads of
// 128 in a window of 1,024, 2,000 tokens 52 -> 39 us, 16 heads 58 -> 47, 400 tokens of 8 heads 21 -> 17; 90 tokens of 16 heads 7.9 -> 9.7, a
// prompt of 150 tokens of 8 heads 445 -> 460, 32 heads and 2,000 tokens (two workgroups a unit) 84 -> 93.  Wider rows leave no registers
// for two wavefronts.
template <int DK, int DV>
void launch_tile(const WindowAttnArgs& a, hipStream_t st) {
  const dim3 g((unsigned)a.heads, (unsigned)((a.M + kTileQueries - 1) / kTileQueries));
  const int64_t keys = a.window > 0 ? std::min<int64_t>(a.pos.pos0 + a.M, (int64_t)a.window + kTileQueries - 1) : a.pos.pos0 + a.M;
  if constexpr (DK + DV <= 256) {
    if ((int64_t)g.x * g.y <= 256 && keys > 8 * kTileKeys) {
      hipLaunchKernelGGL((window_tile_kernel<DK, DV, 2>), g, dim3(512), 0, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((window_tile_kernel<DK, DV, 1>), g, dim3(256), 0, st, a);
}

template <int DK>
void launch_tiles(const WindowAttnArgs& a, hipStream_t st) {
  if (a.vl.row == 64) launch_tile<DK, 64>(a, st);
  else if (a.vl.row == 128) launch_tile<DK, 128>(a, st);
  else launch_tile<DK, 256>(a, st);
}

// Many tokens, binary32, on v_mfma_f32_16x16x4_f32: sixteen queries of one head per workgroup, whose wavefronts take every eighth tile of
// sixteen keys with a maximum and a sum of their own and meet in LDS at the end.  Operands come straight from the cache, queries as
// columns throughout, lane (r, c) = (lane % 16, lane / 16):
//     S^T[key][query] = K Q^T         instruction (i, e) takes element 16 i + 4 c + e of key r and of query r
//     O^T[col][query] += V^T P^T      instruction (b, j) takes column DV / 16 r + b of key 4 c + j, whose weight the lane has just formed
// A value is not in the sums of a query that does not see it, and a query's bits are its own: they do not depend on the queries beside
// it, nor, without a window, on where the pass begins.
// Bound by the matrix cores' binary32 rate and, for few queries, by the trips to the cache.  All eight wavefronts add the parts up at
// the end, four columns of a query a thread: by one of them, with 32 divisions a lane, 8 heads of 128 took 0.4 to 1.2 us more.
// us, the appending launch included, beside a few queries at a time by vector instructions (window_query_kernel):
//   8 heads of 128, from position 0    333 queries 22 (42)      512 queries 27 (59)
//   12 heads of 128, from position 0   512 queries 43 (84)
//   32 heads of 64, from position 0    333 queries 31 (80)
//   8 heads of 128 behind 3,000 keys, window 1,024   333 queries 39 (106)   2 queries 34.5 (38.5)
//   8 heads of 128, from position 0    4 queries 8.5 (8.0)      64 queries 10.6 (10.0)
//   8 heads of 128 behind 150 keys     4 queries 13.5 (12.3)    32 queries 14.6 (12.7)      (window_few_queries)
template <int DK, int DV>
__global__ __launch_bounds__(512) void window_tile_f32_kernel(WindowAttnArgs a) {
  constexpr int KQ = DK / 16, VB = DV / 16, NW = 8;
  constexpr int PARTS = 16;  // of a score: chains of four or eight products, which round no more than a lane's share and a tree
  __shared__ float most[NW][16], sums[NW][16];
  constexpr int STRIDE = DV + 4;
  __shared__ __attribute__((aligned(16))) float held[NW][16 * STRIDE];
  const int h = blockIdx.x, g = h / (a.heads / a.kv_heads), tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, c = lane >> 4;
  const int M = (int)a.M, pos0 = a.pos.pos0, q0 = blockIdx.y * 16, qi = q0 + r, qc = min(qi, M - 1), pq = pos0 + qc;
  auto oldest = [&](int p) { return a.window > 0 ? max(0, p - a.window + 1) : 0; };
  const int first = pos0 + q0, last = pos0 + min(q0 + 15, M - 1), lo_q = oldest(pq);
  const int k_begin = oldest(first) & ~15, k_end = last + 1;
  const int busy = min(NW, (k_end - k_begin + 15) >> 4);  // wavefronts that have a tile
  const float* const q = reinterpret_cast<const float*>(a.proj) + (int64_t)qc * a.ldp + (int64_t)h * a.dim;
  f32x4_t qv[KQ];
#pragma unroll
  for (int i = 0; i < KQ; ++i) {
    const int at = 16 * i + 4 * c;
    if (a.dim == DK) {
      qv[i] = *reinterpret_cast<const f32x4u_t*>(q + at);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) qv[i][e] = at + e < a.dim ? q[at + e] : 0.0f;
    }
  }
  const float mul = a.scale * temperature(a, pq), slope = a.slope[h];
  const float* const kc = reinterpret_cast<const float*>(a.k_cache);
  const float* const vc = reinterpret_cast<const float*>(a.v_cache);
  f32x4_t k[KQ], v[4][VB / 4], acc[VB];
  float m = -INFINITY, l = 0.0f;
#pragma unroll
  for (int b = 0; b < VB; ++b) acc[b] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  // (16 positions from a multiple of 16 on never wrap)
  auto load_keys = [&](int k0) __attribute__((always_inline)) {
    if (k0 >= k_end) return;
    const int slot = k0 % a.kl.slots, over = k_end - 1 - k0;
    const float* const row = kc + ring_row(a.kl, g, slot + min(r, over)) + 4 * c;
#pragma unroll
    for (int i = 0; i < KQ; ++i) k[i] = *reinterpret_cast<const f32x4_t*>(row + 16 * i);
  };
  auto load_values = [&](int k0) __attribute__((always_inline)) {
    if (k0 >= k_end) return;
    const int slot = k0 % a.vl.slots, over = k_end - 1 - k0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float* const val = vc + ring_row(a.vl, g, slot + min(4 * c + j, over)) + VB * r;
#pragma unroll
      for (int b = 0; b < VB / 4; ++b) v[j][b] = *reinterpret_cast<const f32x4_t*>(val + 4 * b);
    }
  };
  load_keys(k_begin + 16 * wave);
  load_values(k_begin + 16 * wave);
  for (int k0 = k_begin + 16 * wave; k0 < k_end; k0 += 16 * NW) {
    f32x4_t part[PARTS];
#pragma unroll
    for (int i = 0; i < PARTS; ++i) part[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < KQ; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f32x4_t& to = part[(4 * i + e) % PARTS];
        to = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][e], qv[i][e], to, 0, 0, 0);
      }
    load_keys(k0 + 16 * NW);
#pragma unroll
    for (int half = PARTS / 2; half > 0; half /= 2)
#pragma unroll
      for (int i = 0; i < half; ++i) part[i] = part[i] + part[i + half];
    const f32x4_t s = part[0];
    float p[4], top = -INFINITY;
    bool seen[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int key = k0 + 4 * c + j;
      seen[j] = key <= pq && key >= lo_q;
      p[j] = s[j] * mul - slope * (float)(pq - key);
      top = fmaxf(top, seen[j] ? p[j] : -INFINITY);
    }
    top = fmaxf(top, __shfl_xor(top, 16, 64));
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float now = fmaxf(m, top), alpha = m > -INFINITY ? expf(m - now) : 0.0f;
    l *= alpha;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p[j] = seen[j] && p[j] != -INFINITY ? expf(p[j] - now) : 0.0f;
      l += p[j];
    }
    m = now;
#pragma unroll
    for (int b = 0; b < VB; ++b) acc[b] = acc[b] * alpha;
    // where some query does not see some key: values that are not finite go alone, to the queries that see them
    bool odd = false;
    if (k0 + 15 > first || k0 < oldest(last)) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < VB; ++b) odd = odd || !(__builtin_fabsf(v[j][b >> 2][b & 3]) < INFINITY);
      odd = __builtin_amdgcn_ballot_w64(odd) != 0;
      if (odd) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int b = 0; b < VB; ++b)
            if (!(__builtin_fabsf(v[j][b >> 2][b & 3]) < INFINITY)) v[j][b >> 2][b & 3] = 0.0f;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int b = 0; b < VB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j][b >> 2][b & 3], p[j], acc[b], 0, 0, 0);
    if (odd) {
      for (int at = 0; at < min(16, k_end - k0); ++at) {
        const int key = k0 + at;
        const float* const val = vc + ring_row(a.vl, g, key % a.vl.slots);
        float w = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float o = __shfl(p[j], (at >> 2) * 16 + r, 64);
          if ((at & 3) == j) w = o;
        }
        if (key > pq || key < lo_q) continue;
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float x = val[VB * (4 * c + j) + b];
            if (!(__builtin_fabsf(x) < INFINITY)) acc[b][j] = __builtin_fmaf(w, x, acc[b][j]);
          }
      }
    }
    load_values(k0 + 16 * NW);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (c == 0) most[wave][r] = m, sums[wave][r] = l;
  __syncthreads();
  float all = most[0][r];
  for (int w = 1; w < busy; ++w) all = fmaxf(all, most[w][r]);
  const auto factor = [&](float x) { return x > -INFINITY ? expf(x - all) : 0.0f; };
  if (wave < busy) {
    const float mine = factor(m);
    float* const to = held[wave] + r * STRIDE + 4 * VB * c;
#pragma unroll
    for (int b = 0; b < VB; ++b) acc[b] = acc[b] * mine;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int b = 0; b < VB; b += 4) *reinterpret_cast<f32x4_t*>(to + VB * j + b) = f32x4_t{acc[b][j], acc[b + 1][j], acc[b + 2][j], acc[b + 3][j]};
  }
  __syncthreads();
  // all wavefronts add the parts up, four columns of a query a thread
  const int of = tid / (DV / 4), col = 4 * (tid % (DV / 4));
  if (of >= 16 || q0 + of >= M) return;
  float top = most[0][of], total = 0.0f;
  for (int w = 1; w < busy; ++w) top = fmaxf(top, most[w][of]);
  f32x4_t sum = *reinterpret_cast<const f32x4_t*>(held[0] + of * STRIDE + col);
  for (int w = 0; w < busy; ++w) {
    total = __builtin_fmaf(most[w][of] > -INFINITY ? expf(most[w][of] - top) : 0.0f, sums[w][of], total);
    if (w > 0) sum = sum + *reinterpret_cast<const f32x4_t*>(held[w] + of * STRIDE + col);
  }
  sum = sum / total;
  float* const out = reinterpret_cast<float*>(a.ctx) + (int64_t)(q0 + of) * a.ldc + (int64_t)h * a.vdim;
  if (col + 3 < a.vdim) {
    *reinterpret_cast<f32x4u_t*>(out + col) = sum;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < a.vdim) out[col + e] = sum[e];
  }
}

template <int DK>
void launch_tiles_f32(const WindowAttnArgs& a, hipStream_t st) {
  const dim3 g((unsigned)a.heads, (unsigned)((a.M + 15) / 16));
  if (a.vl.row == 64) hipLaunchKernelGGL((window_tile_f32_kernel<DK, 64>), g, dim3(512), 0, st, a);
  else hipLaunchKernelGGL((window_tile_f32_kernel<DK, 128>), g, dim3(512), 0, st, a);
}

template <typename T>
int launch_append(const WindowAttnArgs& a, hipStream_t st) {
  const int row = std::max(a.kl.row, a.vl.row);
  if (sizeof(T) == 2 && ((a.dim | a.vdim) & 7) == 0 && row <= 256) {
    const int lanes = row / 8, per = 256 / lanes;
    const int64_t n = (int64_t)(a.heads + 2 * a.kv_heads) * a.M;
    hipLaunchKernelGGL(window_append8_kernel, dim3((unsigned)((n + per - 1) / per)), dim3(256), 0, st, a, lanes);
    AWQ_HIP_TRY(hipGetLastError());
    return AWQ_OK;
  }
  const dim3 g((unsigned)((a.heads + 2 * a.kv_heads + 3) / 4), (unsigned)a.M);
  hipLaunchKernelGGL(window_append_kernel<T>, g, dim3(256), 0, st, a);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

template <typename T, int QN>
void launch_query_kernel(const WindowAttnArgs& a, hipStream_t st) {
  hipLaunchKernelGGL((window_query_kernel<T, QN>), dim3((unsigned)a.heads, (unsigned)((a.M + QN - 1) / QN)), dim3(256), query_lds(a.kl.row, QN),
                     st, a);
}

template <typename T>
int launch_queries(const WindowAttnArgs& a, hipStream_t st) {
  switch (queries_together(a.heads, a.M)) {
    case 1: launch_query_kernel<T, 1>(a, st); break;
    case 2: launch_query_kernel<T, 2>(a, st); break;
    default: launch_query_kernel<T, 4>(a, st); break;
  }
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

}  // namespace

// the tiled and the one-token kernel have rows of 64, 128 or 256 elements; longer ones go a query at a time
int32_t window_row_padded(int32_t dim) { return dim <= 64 ? 64 : dim <= 128 ? 128 : (int32_t)round_up(dim, 256); }

// The last workgroup reads the parts past the caches and, of heads that share a kv head, one head after the other; a second launch costs
// 2 to 4 us, reads through the caches and has a workgroup per head.  Kugilix of width 1,024, eight layers of attention without window, a
// token at 20, 300, 1,000, 2,500 and 30,000 positions: 16 heads of 64 125, 150, 176, 228 and 1,151 us against 146, 153, 157, 173 and 506 with
// the second launch; 8 heads of 128 132, 157, 176 and 223 against 151, 155, 168 and 180; on 4 kv heads 147, 186, 211 and 272 against 168,
// 177, 184 and 200; on one 239, 361, 463 and 644 against 259, 274, 273 and 283.  So it is for heads with a kv head each and up to 16 parts, where
// what the first positions gain is as much as what the last ones lose.
bool window_counted_parts(int32_t heads, int32_t kv_heads, int64_t window, int64_t max_pos) {
  const int parts = window_parts(window, max_pos);
  return heads == kv_heads && parts > 1 && parts <= 16;
}

int64_t window_parts_floats(int32_t heads, int32_t vdim, int64_t window, int64_t max_pos) {
  return (int64_t)heads * window_parts(window, max_pos) * (2 + vdim);
}

static bool one_token_form(const WindowAttnArgs& a) { return a.kl.row <= 256 && a.vl.row <= 256 && a.M == 1 && a.parts && a.len_bound > 0; }

// Few queries on few keys in binary32: a tile of sixteen queries keeps a compute unit's matrix cores busy for all of them, vector
// instructions form what there is.  Up to 384 rows (query, head) and 320 keys of heads of 65 to 128 values they take 0 to 15 % less
// (5 % more at worst: 12 heads, 32 queries from position 0); above, 8 heads, 64 queries and 64 keys 10.0 us against 10.6, 100 and 148
// 15.4 against 14.6.  Heads of up to 64 are half the tile's work: 32 of them, 4 queries, 7.7 us against 6.8.  Not without a window:
// there a query's bits do not depend on the pass that it comes in.
bool window_few_queries(const WindowAttnArgs& a) {
  return a.window > 0 && a.kl.row == 128 && a.vl.row == 128 && a.heads * a.M <= 384 && std::min<int64_t>(a.pos.pos0, a.window - 1) + a.M <= 320;
}

// Where few workgroups attend: there is one for each part of what the sequence may hold, so most of a long one's without a window
// find nothing to do, and the product's stand behind all of them.  Kugilix, 32 tokens behind 9, us, with [W_o | W_down] behind the
// mixer and with W_down in its launch: width 4,096 (50 M weights), window 1,024 (512 attend) 19,851 and 19,154; no window, 2,048 positions
// (1,024) 19,862 and 20,414, 32,768 (16,384) 19,937 and 21,519.  Width 2,048 (13 M): 2,048 positions (512) 9,156 and 8,816, 4,096 (1,024)
// 9,099 and 8,834 (behind 3,500 10,115 and 10,164), 32,768 (8,192) 9,100 and 9,458.  With the product's workgroups ahead: 19,386 with the window.
bool window_takes_product(const WindowAttnArgs& a, bool f32, int64_t weights) {
  if (f32 || !one_token_form(a)) return false;
  const int per = a.heads / a.kv_heads, at_once = decode_heads(per);
  const int64_t attend = (int64_t)a.kv_heads * ((per + at_once - 1) / at_once) * window_parts(a.window, a.len_bound);
  return attend <= 512 || (attend <= 1024 && weights <= 16 << 20);
}

int launch_window_attention(const WindowAttnArgs& a, bool f32, hipStream_t st, const DenseArgs* beside) {
  AWQ_REQUIRE(a.proj && a.k_cache && a.v_cache && a.ctx && a.slope && a.M >= 1 && a.M <= 65535, "bad arguments");
  AWQ_REQUIRE(a.heads >= 1 && a.kv_heads >= 1 && a.heads % a.kv_heads == 0, "heads must be a multiple of kv_heads");
  AWQ_REQUIRE(a.dim >= 1 && a.dim <= 1024 && a.vdim >= 1 && a.vdim <= kMaxCols, "head sizes must be at most 1024");
  AWQ_REQUIRE(a.kl.slots > 0 && a.kl.slots % 64 == 0 && a.vl.slots == a.kl.slots && a.kl.row == window_row_padded(a.dim) &&
                  a.vl.row == window_row_padded(a.vdim) && a.ldp % 8 == 0 && a.ldc % 8 == 0,
              "bad cache layout");
  AWQ_REQUIRE(!beside || window_takes_product(a, f32, beside->k * beside->seg[0].rows), "no product beside this attention");
  if (one_token_form(a)) return f32 ? launch_decode<float>(a, st, nullptr) : launch_decode<bf16_t>(a, st, beside);
  if (int rc = f32 ? launch_append<float>(a, st) : launch_append<bf16_t>(a, st)) return rc;
  if (f32) {
    if (a.kl.row > 128 || a.vl.row > 128 || a.pos.dyn || window_few_queries(a)) return launch_queries<float>(a, st);
    if (a.kl.row == 64) launch_tiles_f32<64>(a, st);
    else launch_tiles_f32<128>(a, st);
    AWQ_HIP_TRY(hipGetLastError());
    return AWQ_OK;
  }
  if (a.kl.row > 256 || a.vl.row > 256 || a.pos.dyn) return launch_queries<bf16_t>(a, st);
  if (a.kl.row == 64) launch_tiles<64>(a, st);
  else if (a.kl.row == 128) launch_tiles<128>(a, st);
  else launch_tiles<256>(a, st);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}
