// What the kernels of dense products share (dense.hip: bfloat16, dense_f32.hip: binary32): activations, the end of a sum,
// blocks of results on their way to memory, sums of a k that was cut.
#pragma once
#include "layers.hpp"

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
// four floats that need not be aligned
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

__device__ __forceinline__ float sigmoid_f32(float z) { return 1.0f / (1.0f + __expf(-z)); }
__device__ __forceinline__ float sigmoid_exact(float z) { return 1.0f / (1.0f + expf(-z)); }

// exp(z) - 1 - z for z <= 0.  Near zero the difference cancels: there the series z^2/2 + z^3/6 + ...
__device__ __forceinline__ float exp_minus_1_minus(float z) {
  if (z > -0.25f) {
    const float t = z * (1.0f / 7.0f) + 1.0f;
    float s = __builtin_fmaf(z * (1.0f / 6.0f), t, 1.0f);
    s = __builtin_fmaf(z * (1.0f / 5.0f), s, 1.0f);
    s = __builtin_fmaf(z * (1.0f / 4.0f), s, 1.0f);
    s = __builtin_fmaf(z * (1.0f / 3.0f), s, 1.0f);
    return 0.5f * z * z * s;
  }
  return (expf(z) - 1.0f) - z;
}

// `bias` and `lower`: the row's entries, where the activation has them
template <bool F32>
__device__ __forceinline__ float activate_with(const DenseSegment& s, int row, float z, float bias, float lower) {
  if (s.act == DENSE_SILU) return row < s.act_rows ? z * (F32 ? sigmoid_exact(z) : sigmoid_f32(z)) : z;
  if (s.act == DENSE_XIELU) {
    const float h = 0.5f * z;
    return z > 0.0f ? __builtin_fmaf(s.act_pos * z, z, h) : __builtin_fmaf(s.act_neg, exp_minus_1_minus(z), h);
  }
  if (s.act == DENSE_SIGMOID) return F32 ? sigmoid_exact(z + bias) : sigmoid_f32(z + bias);
  if (s.act == DENSE_GELU) {  // (1 + tanh u) / 2 = sigmoid(2 u)
    const float u2 = 1.5957691216057307117f * __builtin_fmaf(0.044715f * z * z, z, z);
    return z * (F32 ? sigmoid_exact(u2) : sigmoid_f32(u2));
  }
  if (s.act == DENSE_LOG_DECAY) {
    z += bias;
    if (F32) return -s.act_pos * (log1pf(expf(-fabsf(z))) + fmaxf(-z, 0.0f));
    // (off by what one rounding of the decay itself is off)
    const float e = __builtin_amdgcn_exp2f(-1.44269504088896340736f * fabsf(z));
    return -s.act_pos * __builtin_fmaf(0.693147180559945309417f, __builtin_amdgcn_logf(1.0f + e), fmaxf(-z, 0.0f));
  }
  if (s.act == DENSE_FORGET) return (1.0f - lower) * sigmoid_exact(-(z + bias));
  return z;
}

// the same for four rows, with one look at which it is
template <bool F32>
__device__ __forceinline__ void activate_four(const DenseSegment& s, int row, f32x4_t& v, const float (&bias)[4], const float (&lower)[4]) {
  switch (s.act) {
#define AWQ_ACTIVATE(ACT)                                                                      \
  case ACT:                                                                                    \
    _Pragma("unroll") for (int j = 0; j < 4; ++j) {                                            \
      __builtin_assume(s.act == ACT);                                                          \
      v[j] = activate_with<F32>(s, row + j, v[j], bias[j], lower[j]);                          \
    }                                                                                          \
    break;
    AWQ_ACTIVATE(DENSE_SILU)
    AWQ_ACTIVATE(DENSE_XIELU)
    AWQ_ACTIVATE(DENSE_SIGMOID)
    AWQ_ACTIVATE(DENSE_GELU)
    AWQ_ACTIVATE(DENSE_LOG_DECAY)
    AWQ_ACTIVATE(DENSE_FORGET)
#undef AWQ_ACTIVATE
  }
}

template <bool F32>
__device__ __forceinline__ float activate(const DenseSegment& s, int row, float z) {
  return activate_with<F32>(s, row, z, s.bias ? s.bias[row] : 0.0f, s.lower ? s.lower[row] : 0.0f);
}

__device__ __forceinline__ float softcap(const DenseSegment& s, float z) { return s.act_pos * tanhf(z / s.act_pos); }

template <bool F32>
__device__ __forceinline__ float glu(float gate, float up) {
  return gate * (F32 ? sigmoid_exact(gate) : sigmoid_f32(gate)) * up;
}

__device__ __forceinline__ int32_t f32_key(float v) {
  if (v != v) return INT32_MIN;  // NaN never wins
  const uint32_t b = __float_as_uint(v);
  if ((b & 0x7fffffffu) == 0) return 0;
  return (b & 0x80000000u) ? -(int32_t)(b & 0x7fffffffu) : (int32_t)b;
}

// the lanes' LDS writes ahead of this are seen by all lanes' reads behind it
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ const DenseSegment& segment_of(const DenseArgs& a, int row) {
  int i = 0;
#pragma unroll
  for (int j = 1; j < kDenseSegments; ++j) i += j < a.n_seg && row >= a.start[j] ? 1 : 0;
  return a.seg[i];
}

// the weight block of this workgroup's product (one token), or -1: it is left out
__device__ __forceinline__ int block_of_product(const DenseArgs& a, int b) {
  const int by_number = a.batch - a.fixed;
  if (!a.ids) return b;
  if (b >= by_number) return a.n_groups + b - by_number;
  const int group = a.ids[b];
  return group < a.n_groups ? group : -1;
}

// one output of one token (DENSE_STORE), `y0` elements into the segment's output
template <typename T>
__device__ __forceinline__ void store_one(const DenseSegment& s, int64_t y0, int64_t t, int row, float v) {
  if (s.act == DENSE_GELU && s.mul) v *= (float)reinterpret_cast<const T*>(s.mul)[t * s.ldmul + row];
  const int64_t at = y0 + t * s.ldy + row;
  if (s.y_f32) reinterpret_cast<float*>(s.y)[at] = v;
  else reinterpret_cast<T*>(s.y)[at] = (T)v;
}

// one finished sum of one token
template <typename T, int OUT>
__device__ __forceinline__ void finish_one(const DenseArgs& a, const DenseSegment& s, int64_t t, int row, float sum, int64_t y0 = 0) {
  if constexpr (OUT == DENSE_STORE) {
    store_one<T>(s, y0, t, row, activate<sizeof(T) == 4>(s, row, sum));
  } else if constexpr (OUT == DENSE_RESIDUAL) {
    const int64_t at = t * s.ldy + row;
    float* y = reinterpret_cast<float*>(s.y);
    float v = y[at] + sum;
    if (a.addend) v += a.addend[at];
    y[at] = v;
  } else {
    reinterpret_cast<float*>(s.y)[t * s.ldy + row] = s.act == DENSE_SOFTCAP ? softcap(s, sum) : sum;
  }
}

constexpr int DENSE_PART = 100;  // the sums of a share of k, to the workspace

// Stores blocks of 32 rows and 32 tokens that a wavefront holds as results of 32 x 32 matrix instructions: acc[t][i] is row
// row_w + 8 (i / 4) + 4 (lane / 32) + i % 4 of token tt0 + 32 t + lane % 32.  A block is turned in LDS, 4 KB of the wavefront's
// own (`turn`), so that eight lanes hold and store the rows of a token side by side; four rows (a piece) of token n are at
// place piece ^ (n % 8).  `rows` and `cut`: the workspace's row length and the share of k (DENSE_PART).
template <typename T, int OUT, bool LISTED, int N>
__device__ __forceinline__ void store_block_rows(const DenseArgs& a, float* turn, const f32x16_t (&acc)[N], int row_w, int tt0, int n_tok,
                                                 const int32_t* list, int rows, int cut) {
  constexpr bool F32 = sizeof(T) == 4;
  typedef T tx4_t __attribute__((ext_vector_type(4), aligned(sizeof(T) == 4 ? 4 : 8)));
  const int lane = threadIdx.x & 63, n = lane & 31, kh = lane >> 5;
  const int64_t y0 = blockIdx.y * a.y_batch;
  const DenseSegment out = segment_of(a, row_w);
  const int local_b = row_w - out.row0;
  const bool gated = OUT == DENSE_STORE && out.act == DENSE_GLU;
  const int n_rows = gated ? out.glu_rows : out.rows;
  if (OUT != DENSE_PART && local_b >= out.rows) return;  // padding
  const bool by_four = ((out.ldy | a.y_batch) & 3) == 0 && !(OUT == DENSE_STORE && out.mul);
  // pieces of a token: 8, or 4 of a gated segment
  const int shift = gated ? 2 : 3, piece = lane & ((1 << shift) - 1);
  const int row = (gated ? local_b / 2 : local_b) + 4 * piece;
  float bias[4] = {}, lower[4] = {};  // of this lane's rows
  if (OUT == DENSE_STORE && out.bias) {
#pragma unroll
    for (int j = 0; j < 4; ++j) bias[j] = out.bias[min(row + j, n_rows - 1)];
  }
  if (OUT == DENSE_STORE && out.lower) {
#pragma unroll
    for (int j = 0; j < 4; ++j) lower[j] = out.lower[min(row + j, n_rows - 1)];
  }
#pragma unroll
  for (int t = 0; t < N; ++t) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (gated && (g & 1)) continue;
      f32x4_t v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = gated ? glu<F32>(acc[t][4 * g + j], acc[t][(4 * g + 4 + j) & 15]) : acc[t][4 * g + j];
      const int p = gated ? g + kh : 2 * g + kh;
      *reinterpret_cast<f32x4_t*>(turn + n * 32 + ((p ^ (n & 7)) << 2)) = v;
    }
    wave_sync();
#pragma unroll 1
    for (int token = lane >> shift; token < 32; token += 64 >> shift) {
      f32x4_t v = *reinterpret_cast<const f32x4_t*>(turn + token * 32 + ((piece ^ (token & 7)) << 2));
      int64_t tok = tt0 + 32 * t + token;
      if (tok >= n_tok) continue;
      if constexpr (LISTED) tok = list[tok];
      if constexpr (OUT == DENSE_PART) {
        *reinterpret_cast<f32x4_t*>(a.workspace + ((int64_t)cut * a.M + tok) * rows + row_w + 4 * piece) = v;
      } else {
        if (OUT == DENSE_STORE && !gated) activate_four<F32>(out, row, v, bias, lower);
        const int64_t at = y0 + tok * out.ldy + row;
        if (row + 3 < n_rows && by_four) {
          if (OUT == DENSE_STORE && !out.y_f32) {
            *reinterpret_cast<tx4_t*>(reinterpret_cast<T*>(out.y) + at) = tx4_t{(T)v[0], (T)v[1], (T)v[2], (T)v[3]};
            continue;
          }
          if (OUT == DENSE_F32 && out.act == DENSE_SOFTCAP) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = softcap(out, v[j]);
          }
          f32x4u_t* y = reinterpret_cast<f32x4u_t*>(reinterpret_cast<float*>(out.y) + at);
          if constexpr (OUT == DENSE_RESIDUAL) {
            v = *y + v;
            if (a.addend) v = v + *reinterpret_cast<const f32x4u_t*>(a.addend + at);
          }
          *y = v;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (row + j >= n_rows) continue;
            if constexpr (OUT == DENSE_STORE) store_one<T>(out, y0, tok, row + j, v[j]);
            else finish_one<T, OUT>(a, out, tok, row + j, v[j]);
          }
        }
      }
    }
    wave_sync();
  }
}

// adds the sums of the workgroups that shared k: a thread takes four rows of a token
template <typename T, int OUT>
__global__ __launch_bounds__(256) void dense_parts_kernel(DenseArgs a, int rows, int cuts) {
  const int row = (blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t tok = blockIdx.y;
  if (row >= rows) return;
  const DenseSegment& s = segment_of(a, row);
  const int local = row - s.row0;
  if (local >= s.rows) return;
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(a.workspace + tok * rows + row);
  const int64_t stride = a.M * rows / 4;
  f32x4_t sum = p[0];
  for (int c = 1; c < cuts; ++c) sum = sum + p[c * stride];
  if constexpr (OUT == DENSE_STORE) {
    if (s.act == DENSE_GLU) {
      if (local & 8) return;
      f32x4_t up = p[2];
      for (int c = 1; c < cuts; ++c) up = up + p[c * stride + 2];
      const int r0 = (local >> 4) * 8 + (local & 7);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (r0 + j < s.glu_rows) store_one<T>(s, 0, tok, r0 + j, glu<sizeof(T) == 4>(sum[j], up[j]));
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (local + j < s.rows) finish_one<T, OUT>(a, s, tok, local + j, sum[j]);
}

}  // namespace

// binary32 (dense_f32.hip)
int launch_dense_one_f32(const DenseArgs& a, int64_t rows, hipStream_t st);
int launch_dense_one_joined_f32(const DenseArgs& a, const JoinArgs& j, int64_t rows, hipStream_t st);
int launch_dense_many_f32(const DenseArgs& a, int64_t rows, hipStream_t st);  // a.tiles: token lists
