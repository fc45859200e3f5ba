// What stands around the products of a sublayer (layers.hpp): token rows, the gated and normalised sum into the residual
// stream with the next norm behind it, PolyNorm.
#include "join_device.hpp"

namespace {

template <typename T, int V>
__global__ __launch_bounds__(256) void embed_tokens_kernel(const T* __restrict__ table, const T* __restrict__ side_table,
                                                           const int32_t* __restrict__ tokens, const int32_t* __restrict__ last,
                                                           PassPos pos, int64_t width, int64_t side_width, float* __restrict__ x,
                                                           T* __restrict__ side) {
  const int t = blockIdx.y;
  int64_t tok;
  if (pos.dyn) {
    tok = pos.dyn->token;
    if (tok < 0) tok = *last;
  } else {
    tok = tokens[t];
  }
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V; i < width + side_width; i += (int64_t)gridDim.x * 256 * V) {
    float v[V];
    if (i < width) {
      read<T, V>(table + tok * width + i, v);
      write<float, V>(x + t * width + i, v);
    } else {
      read<T, V>(side_table + tok * side_width + i - width, v);
      write<T, V>(side + t * side_width + i - width, v);
    }
  }
}

// The same with the first norm behind it: the first workgroup of a token takes its row, four values a thread (launch_embed_tokens says
// which rows), the others what goes with it.  A launch of its own for the norm took 3.5 us for a token, 7.5 and 14.3 for 129
// and 1,024 of width 2,048 and 4,096; in this one it costs less than one.
template <typename T>
__global__ __launch_bounds__(1024) void embed_norm_kernel(const T* __restrict__ table, const T* __restrict__ side_table,
                                                          const int32_t* __restrict__ tokens, const int32_t* __restrict__ last, PassPos pos,
                                                          int64_t width, int64_t side_width, float* __restrict__ x, T* __restrict__ side,
                                                          EmbedNorm norm) {
  __shared__ float sums[16];
  const int t = blockIdx.y, c = 4 * (int)threadIdx.x;
  const bool mine = c < width;
  float w[4] = {};
  if (blockIdx.x == 0 && mine) read<float, 4>(norm.w + c, w);
  int64_t tok;
  if (pos.dyn) {
    tok = pos.dyn->token;
    if (tok < 0) tok = *last;
  } else {
    tok = tokens[t];
  }
  if (blockIdx.x > 0) {
    const int64_t step = (int64_t)(gridDim.x - 1) * blockDim.x * 4;
    for (int64_t i = (int64_t)(blockIdx.x - 1) * blockDim.x * 4 + c; i < side_width; i += step) {
      float v[4];
      read<T, 4>(side_table + tok * side_width + i, v);
      write<T, 4>(side + t * side_width + i, v);
    }
    return;
  }
  float v[4] = {}, sq = 0.0f;
  if (mine) read<T, 4>(table + tok * width + c, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) sq = __builtin_fmaf(v[i], v[i], sq);
  const float inv = 1.0f / sqrtf(group_sum(sq, sums) / (float)width + norm.eps);
  if (!mine) return;
  write<float, 4>(x + t * width + c, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = v[i] * inv * w[i];
  write<T, 4>(reinterpret_cast<T*>(norm.h) + t * norm.ldh + c, v);
}

// A workgroup per token; the sum, then the new residual, wait in LDS.
template <typename T, int V>
__global__ __launch_bounds__(1024) void join_kernel(JoinArgs a) {
  extern __shared__ __attribute__((aligned(16))) float row[];  // [width]
  __shared__ float sums[2][16];
  const int tid = threadIdx.x, step = blockDim.x * V, W = (int)a.width;
  const int64_t t = blockIdx.x;
  const float* const x = a.x + t * W;
  float* const x_out = (a.x_out ? a.x_out : a.x) + t * W;
  const float y_mul = a.y_gate ? 1.0f / (1.0f + expf(-a.y_gate[t])) : 1.0f;
  float sq = 0.0f;
  for (int c = tid * V; c < W; c += step) {
    float v[V] = {};
    if (a.y) {
      read<float, V>(a.y + t * W + c, v);
#pragma unroll
      for (int i = 0; i < V; ++i) v[i] *= y_mul;
    }
    for (int j = 0; j < a.top; ++j) {
      const int64_t p = t * a.top + j;
      const float w = a.weights[p];
      float u[V];
      if (a.ids[p] < a.experts) read<float, V>(a.pairs + p * W + c, u);
      else read<T, V>(reinterpret_cast<const T*>(a.h) + t * a.ldh + c, u);
#pragma unroll
      for (int i = 0; i < V; ++i) v[i] = __builtin_fmaf(w, u[i], v[i]);
    }
    if (a.gate) {
      float g[V];
      read<T, V>(reinterpret_cast<const T*>(a.gate) + t * a.ldg + c, g);
#pragma unroll
      for (int i = 0; i < V; ++i) v[i] *= g[i];
    }
#pragma unroll
    for (int i = 0; i < V; ++i) sq = __builtin_fmaf(v[i], v[i], sq);
    write<float, V>(row + c, v);
  }
  const float inv = 1.0f / sqrtf(group_sum(sq, sums[0]) / (float)W + a.eps);
  sq = 0.0f;
  for (int c = tid * V; c < W; c += step) {
    float v[V], w[V], r[V];
    read<float, V>(row + c, v);
    read<float, V>(a.w_post + c, w);
    read<float, V>(x + c, r);
#pragma unroll
    for (int i = 0; i < V; ++i) {
      r[i] = r[i] + v[i] * inv * w[i];
      sq = __builtin_fmaf(r[i], r[i], sq);
    }
    write<float, V>(x_out + c, r);
    if (a.out) write<float, V>(row + c, r);
  }
  if (!a.out) return;
  const float next = a.w_next ? 1.0f / sqrtf(group_sum(sq, sums[1]) / (float)W + a.eps) : 1.0f;
  T* const out = reinterpret_cast<T*>(a.out) + t * a.ldo;
  for (int c = tid * V; c < W; c += step) {
    float v[V], w[V];
    read<float, V>(row + c, v);
    if (a.w_next) {
      read<float, V>(a.w_next + c, w);
#pragma unroll
      for (int i = 0; i < V; ++i) v[i] = v[i] * next * w[i];
    }
    write<T, V>(out + c, v);
  }
}

// The same where a row is a workgroup's threads times V at most and a token has at most kJoinTop choices, which then wait in
// registers (join_device.hpp): the form above makes three trips to memory, one behind the other, and one more for each choice.
// Tudasun of width 4,096, 64 tokens one by one with 12 launches each: 38.6 -> 37.8 ms; width 1,024 in binary32, 24 tokens:
// 7.73 -> 7.50.
template <typename T, int V>
__global__ __launch_bounds__(1024) void join_row_kernel(JoinArgs a) {
  __shared__ float sums[2][16];
  JoinRow<T, V, 1> row(a, blockIdx.x, blockDim.x);
  row.request_rows();
  row.request_weights();
  float* const x = (a.x_out ? a.x_out : a.x) + row.t * row.W;
  row.finish(sums, [&](int c, const float (&r)[V]) { write<float, V>(x + c, r); });
  if (a.out && row.column(0) < row.W) write<T, V>(reinterpret_cast<T*>(a.out) + row.t * a.ldo + row.column(0), row.r[0]);
}

template <typename T, int V>
__global__ __launch_bounds__(1024) void polynorm_kernel(T* z, int64_t ld, int n, const float* __restrict__ abce, float eps) {
  __shared__ float sums[3][16];
  const int tid = threadIdx.x, step = blockDim.x * V;
  z += blockIdx.x * ld;
  float s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
  for (int c = tid * V; c < n; c += step) {
    float v[V];
    read<T, V>(z + c, v);
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float q = v[i] * v[i], q2 = q * q;
      s1 += q;
      s2 += q2;
      s3 = __builtin_fmaf(q2, q, s3);
    }
  }
  s1 = wave_sum(s1);
  s2 = wave_sum(s2);
  s3 = wave_sum(s3);
  if ((tid & 63) == 0) sums[0][tid >> 6] = s1, sums[1][tid >> 6] = s2, sums[2][tid >> 6] = s3;
  __syncthreads();
  s1 = s2 = s3 = 0.0f;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s1 += sums[0][i], s2 += sums[1][i], s3 += sums[2][i];
  const float m = 1.0f / (float)n;
  const float a = abce[0] / sqrtf(s1 * m + eps), b = abce[1] / sqrtf(s2 * m + eps), c3 = abce[2] / sqrtf(s3 * m + eps), e = abce[3];
  for (int c = tid * V; c < n; c += step) {
    float v[V];
    read<T, V>(z + c, v);
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(c3, v[i], b), v[i], a), v[i], e);
    write<T, V>(z + c, v);
  }
}

// a wavefront per token and head
template <typename T>
__global__ __launch_bounds__(256) void head_norm_kernel(const float* __restrict__ o, const T* __restrict__ gate, int64_t ldg,
                                                        const float* __restrict__ w, T* __restrict__ ctx, int64_t ldc, int heads,
                                                        int vdim, int64_t rows, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t at = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (at >= rows) return;
  const int64_t t = at / heads;
  const int c0 = (int)(at - t * heads) * vdim;
  o += t * heads * vdim + c0;
  float sq = 0.0f;
  for (int c = lane; c < vdim; c += 64) sq = __builtin_fmaf(o[c], o[c], sq);
  const float inv = 1.0f / sqrtf(wave_sum(sq) / (float)vdim + eps);
  for (int c = lane; c < vdim; c += 64) {
    float y = o[c] * inv * w[c];
    if (gate) {
      const float g = (float)gate[t * ldg + c0 + c];
      y *= g / (1.0f + expf(-g));
    }
    ctx[t * ldc + c0 + c] = (T)y;
  }
}

template <typename T>
void embed_tokens(const void* table, const void* side_table, const int32_t* tokens, const int32_t* last, PassPos pos, int64_t M,
                  int64_t width, int64_t side_width, float* x, void* side, hipStream_t st) {
  const bool quads = ((width | side_width) & 3) == 0;
  const dim3 g((unsigned)std::min<int64_t>((width + side_width + 1023) / (quads ? 1024 : 256), 64), (unsigned)M);
  if (quads)
    hipLaunchKernelGGL((embed_tokens_kernel<T, 4>), g, dim3(256), 0, st, (const T*)table, (const T*)side_table, tokens, last, pos, width,
                       side_width, x, (T*)side);
  else
    hipLaunchKernelGGL((embed_tokens_kernel<T, 1>), g, dim3(256), 0, st, (const T*)table, (const T*)side_table, tokens, last, pos, width,
                       side_width, x, (T*)side);
}

// a row of a token is one turn of its workgroup's threads
bool row_form(const JoinArgs& a) {
  const int64_t threads = a.M < 512 ? 1024 : 256;
  return ((a.width | a.ldo | a.ldg | a.ldh) & 3) == 0 && a.width / 4 <= threads && a.top <= kJoinTop;
}

template <typename T>
int join(const JoinArgs& a, hipStream_t st) {
  const size_t lds = (size_t)a.width * 4;
  const bool quads = ((a.width | a.ldo | a.ldg | a.ldh) & 3) == 0;
  const dim3 g((unsigned)a.M);
  const int64_t items = a.width / (quads ? 4 : 1);
  const dim3 b((unsigned)std::min<int64_t>(a.M < 512 ? 1024 : 256, round_up(items, 64)));
  // by measurement above wherever the registers hold a row; wider rows, more choices and odd widths keep the general form
  if (row_form(a)) hipLaunchKernelGGL((join_row_kernel<T, 4>), g, b, 0, st, a);
  else if (quads) hipLaunchKernelGGL((join_kernel<T, 4>), g, b, lds, st, a);
  else hipLaunchKernelGGL((join_kernel<T, 1>), g, b, lds, st, a);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

template <typename T>
int polynorm(void* z, int64_t ld, int64_t n, int64_t M, const float* abce, float eps, hipStream_t st) {
  const bool quads = ((n | ld) & 3) == 0;
  const dim3 b((unsigned)std::min<int64_t>(M < 512 ? 1024 : 256, round_up(n / (quads ? 4 : 1), 64)));
  if (quads) hipLaunchKernelGGL((polynorm_kernel<T, 4>), dim3((unsigned)M), b, 0, st, (T*)z, ld, (int)n, abce, eps);
  else hipLaunchKernelGGL((polynorm_kernel<T, 1>), dim3((unsigned)M), b, 0, st, (T*)z, ld, (int)n, abce, eps);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

}  // namespace

bool embed_takes_norm(int64_t width, int64_t side_width, const EmbedNorm& n) {
  return n.w && n.h && width <= 4096 && ((width | side_width | n.ldh) & 3) == 0 && n.ldh >= width && (((uintptr_t)n.w | (uintptr_t)n.h) & 15) == 0;
}

int launch_embed_tokens(const void* table, const void* side_table, bool f32, const int32_t* tokens, const int32_t* last,
                        PassPos pos, int64_t M, int64_t width, int64_t side_width, float* x, void* side, hipStream_t st, const EmbedNorm* norm) {
  AWQ_REQUIRE(table && x && (pos.dyn ? last != nullptr && M == 1 : tokens != nullptr), "bad arguments");
  AWQ_REQUIRE(M >= 1 && M <= 65535 && width >= 1 && side_width >= 0 && (side_width == 0 || (side_table && side)), "bad shape");
  AWQ_REQUIRE(!norm || embed_takes_norm(width, side_width, *norm), "the norm cannot be part of this launch");
  if (norm) {
    const int64_t threads = std::max<int64_t>(256, round_up((width + 3) / 4, 64)), per = threads * 4;
    const dim3 g((unsigned)(1 + std::min<int64_t>(4, (side_width + per - 1) / per)), (unsigned)M);
    if (f32)
      hipLaunchKernelGGL(embed_norm_kernel<float>, g, dim3((unsigned)threads), 0, st, (const float*)table, (const float*)side_table, tokens, last, pos,
                         width, side_width, x, (float*)side, *norm);
    else
      hipLaunchKernelGGL(embed_norm_kernel<bf16_t>, g, dim3((unsigned)threads), 0, st, (const bf16_t*)table, (const bf16_t*)side_table, tokens, last, pos,
                         width, side_width, x, (bf16_t*)side, *norm);
  } else if (f32) {
    embed_tokens<float>(table, side_table, tokens, last, pos, M, width, side_width, x, side, st);
  } else {
    embed_tokens<bf16_t>(table, side_table, tokens, last, pos, M, width, side_width, x, side, st);
  }
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

// Where the row waits in registers.  Tudasun of width 2,048, 129 tokens: eight launches of 4.3 us less, 884 -> 843 us.  From 512 tokens
// on that is up to a width of 1,024 (row_form): 512 tokens of width 768 751 -> 733 us, of 1,024 801 -> 795, in binary32 1,294 -> 1,267;
// 2,048 tokens the same within 1 %.  Wider rows make three trips to memory in their join as it is: at 1,024 tokens of width 4,096 one
// product is cut, and its shares in the join cost what the launch had.
bool join_adds_shares(const JoinArgs& a) { return row_form(a); }

int launch_join(const JoinArgs& a, bool f32, hipStream_t st) {
  AWQ_REQUIRE(a.x && a.w_post && (a.y || a.top > 0) && a.M >= 1 && a.M < (1ll << 31), "bad arguments");
  AWQ_REQUIRE(a.y_shares == 1 || (a.y_shares > 1 && a.y && join_adds_shares(a) && a.ldy >= a.width && ((a.ldy | a.y_share) & 3) == 0), "bad shares");
  AWQ_REQUIRE(a.width >= 1 && a.width <= 16000, "width must be at most 16000");  // a row in 64 KB of LDS, sums beside it
  AWQ_REQUIRE(a.top == 0 || (a.pairs && a.ids && a.weights && a.h && a.ldh >= a.width), "bad experts");
  AWQ_REQUIRE((!a.out || a.ldo >= a.width) && (!a.gate || a.ldg >= a.width), "bad shape");
  return f32 ? join<float>(a, st) : join<bf16_t>(a, st);
}

int launch_polynorm(void* z, int64_t ld, int64_t n, int64_t M, const float* abce, float eps, bool f32, hipStream_t st) {
  AWQ_REQUIRE(z && abce && n >= 1 && n < (1 << 30) && ld >= n && M >= 1 && M < (1ll << 31), "bad arguments");
  return f32 ? polynorm<float>(z, ld, n, M, abce, eps, st) : polynorm<bf16_t>(z, ld, n, M, abce, eps, st);
}

int launch_head_norm(const float* o, const void* gate, int64_t ldg, const float* w, void* ctx, int64_t ldc, int32_t heads,
                     int32_t vdim, int64_t M, float eps, bool f32, hipStream_t st) {
  AWQ_REQUIRE(o && w && ctx && heads >= 1 && vdim >= 1 && M >= 1 && ldc >= (int64_t)heads * vdim, "bad arguments");
  const int64_t rows = M * heads;
  AWQ_REQUIRE(rows < (1ll << 32), "too large");
  const dim3 g((unsigned)((rows + 3) / 4));
  if (f32)
    hipLaunchKernelGGL(head_norm_kernel<float>, g, dim3(256), 0, st, o, (const float*)gate, ldg, w, (float*)ctx, ldc, heads, vdim,
                       rows, eps);
  else
    hipLaunchKernelGGL(head_norm_kernel<bf16_t>, g, dim3(256), 0, st, o, (const bf16_t*)gate, ldg, w, (bf16_t*)ctx, ldc, heads, vdim,
                       rows, eps);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}
