// Dense products of binary32 weights with one token or many (layers.hpp).
#include "dense_device.hpp"
#include "join_device.hpp"

#include <math.h>

#include <type_traits>

namespace {

// --- one token -----------------------------------------------------------------------------------------------
// Bound by the weights' bytes.  A wavefront takes R rows (R = 2, 4: among them both rows of a gated pair) against one
// reading of the input, a workgroup of four wavefronts 4 R rows; a lane's sum of a row takes every 64th piece of four
// inputs whatever R is.  Rows of 1,024 inputs: 32,768 of them (a vocabulary's logits, R = 4) 29 us, 4.6 TB/s; four blocks of
// 1,536 gated rows (R = 2) 6.8 us, where a wavefront that took the two rows of a pair one after the other, beside one
// that had none, took 9.8; below 8,192 rows one each, so that 1,024 rows still make 256 workgroups.
// JQ: the input is formed here, the end of the sublayer ahead (JoinArgs, JQ turns of the workgroup's threads)
template <int OUT, int R, int JQ = 0>
__global__ __launch_bounds__(256) void dense_one_f32_kernel(DenseArgs a, std::conditional_t<JQ != 0, JoinArgs, std::false_type> join) {
  extern __shared__ __attribute__((aligned(16))) float formed[];  // [k]
  __shared__ unsigned long long candidates[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // rows of the wavefront: row(0), and with R = 2 row(0) + 8, with R = 4 row(0) + 1, + 8, + 9
  const int base = R == 1 ? blockIdx.x * 4 : R == 2 ? (blockIdx.x >> 1) * 16 + (blockIdx.x & 1) * 4 : blockIdx.x * 16;
  const int row0 = base + wave * (R == 4 ? 2 : 1);
  auto row_of = [&](int i) { return row0 + (R == 4 ? (i & 1) + 8 * (i >> 1) : 8 * i); };
  const DenseSegment& s = segment_of(a, base);
  const int local0 = base - s.row0;
  if (local0 >= s.rows) return;
  const int group = block_of_product(a, blockIdx.y);
  if (group < 0) return;
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
  if constexpr (JQ != 0) {
    __shared__ float sums[2][16];
    f32x4_t wv[4][R];  // the first weights, behind the request for the row
    const bool first = at + 64 * 3 < (int)k4;
    joined_input<float, JQ>(join, blockIdx.x == 0 && blockIdx.y == 0, (int)a.k, formed, sums, [&]() {
      if (!first) return;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < R; ++i) wv[u][i] = __builtin_nontemporal_load(w + row_of(i) * k4 + at + 64 * u);
    });
    if (first) {
#pragma unroll
      for (int u = 0; u < 4; ++u) add(wv[u], reinterpret_cast<const f32x4_t*>(formed)[at + 64 * u]);
      at += 64 * 4;
    }
  }
  auto pieces = [&](auto count) __attribute__((always_inline)) {
    constexpr int N = decltype(count)::value;
    f32x4_t wv[N][R], xv[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
#pragma unroll
      for (int i = 0; i < R; ++i) wv[u][i] = __builtin_nontemporal_load(w + row_of(i) * k4 + at + 64 * u);
      if constexpr (JQ != 0) xv[u] = reinterpret_cast<const f32x4_t*>(formed)[at + 64 * u];
      else xv[u] = x[at + 64 * u];
    }
#pragma unroll
    for (int u = 0; u < N; ++u) add(wv[u], xv[u]);
    at += 64 * N;
  };
  while (at + 64 * (U - 1) < (int)k4) pieces(std::integral_constant<int, U>());
  // the rest together as well: one by one 1,536 rows of 1,536 inputs took 6.0 us, now 4.7, 1,024 of 1,024 4.8 and 3.7
  if constexpr (U > 4)
    if (at + 64 * 3 < (int)k4) pieces(std::integral_constant<int, 4>());
  if (at + 64 < (int)k4) pieces(std::integral_constant<int, 2>());
  if (at < (int)k4) pieces(std::integral_constant<int, 1>());
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
// On v_mfma_f32_32x32x2_f32: a workgroup of four wavefronts takes 64 rows and 32 TW C tokens, steps of 32 inputs.  Two
// wavefronts share the rows, TW the tokens (C accumulators each) and KW the inputs of a step, whose sums meet in LDS.
// Weights and tokens go through LDS, 128 bytes per row and step, the eight 16-byte pieces of row r at positions c ^ (r & 7),
// requested a step ahead into registers.  Lane (n, kh) reads piece 2 j + kh of row n of both operands, and instruction e
// multiplies element e of the two: the inputs of a step are met in another order on both sides alike.
// Up to about 50 tokens bound by the weights' bytes (2 operations per token and 4 bytes against 134 TFLOP/s and 5.1 TB/s),
// beyond by the matrix cores.  Where the tiles do not fill the device, k is cut over `cuts` workgroups and a second launch
// adds their sums, as in bfloat16.  333 tokens, sums added: 1,024 rows of 4,096 inputs 39 us, 7,168 of 1,024 57, 32,768 of 1,024
// 212 (106 TFLOP/s); 4 x 4 sums per thread without matrix cores took 270, 135 and 482.  20 tokens on 1,024 x 4,096: 18, was 273.
template <int TW, int KW, int C, int OUT, bool LISTED = false>
__global__ __launch_bounds__(256) void dense_many_f32_kernel(DenseArgs a, int row_tiles, int tok_tiles, int cuts) {
  static_assert(TW * KW == 2, "four wavefronts, two of them share the rows");
  constexpr int TOK = 32 * TW * C, NL = (64 + TOK) / 32;  // pieces per thread and step
  __shared__ __attribute__((aligned(16))) float tiles[2][(64 + TOK) * 32];
  const int total = row_tiles * tok_tiles * cuts;
  // workgroups whose indices agree modulo 8 share a die: each die walks its own run of row tiles
  const int per = (total + 7) >> 3;
  const int work = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (work >= total) return;
  const int rc = work / tok_tiles, tile = work - rc * tok_tiles, tt0 = LISTED ? 0 : tile * TOK;
  const int rt = rc / cuts, cut = rc - rt * cuts;
  int64_t group = blockIdx.y;
  int n_tok = (int)min((int64_t)1 << 30, a.M);
  const int32_t* list = nullptr;
  if constexpr (LISTED) {
    const DenseTile run = a.tiles[tile];
    if (run.count == 0) return;
    group = run.group;
    n_tok = run.count;
    list = a.list + run.first;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, kh = lane >> 5;
  const int rw = wave & 1, tw = TW == 2 ? wave >> 1 : 0, kw = KW == 2 ? wave >> 1 : 0;
  const DenseSegment& s = segment_of(a, rt * 64);
  if (rt * 64 >= a.seg[a.n_seg - 1].row0 + a.seg[a.n_seg - 1].rows) return;  // padding
  const int all_steps = (int)(a.k >> 5);
  const int first_step = (int)((int64_t)all_steps * cut / cuts);
  const int steps = (int)((int64_t)all_steps * (cut + 1) / cuts) - first_step;

  // this thread's pieces of a step: place tid % 8 of rows tid / 8 + 32 i, the first two of them weights
  const float* src[NL];
  const int lr = tid >> 3, at = (tid & 7) << 2;
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    if (i < 2) {
      src[i] = reinterpret_cast<const float*>(a.w) + group * a.w_batch + (int64_t)(rt * 64 + lr + 32 * i) * a.k;
    } else {
      int64_t tok = min(tt0 + lr + 32 * (i - 2), n_tok - 1);
      if constexpr (LISTED) tok = list[tok] / a.list_div;
      src[i] = reinterpret_cast<const float*>(s.x) + blockIdx.y * a.x_batch + tok * s.ldx;
    }
    src[i] += first_step * 32 + at;
  }
  const int place = lr * 32 + (((tid & 7) ^ (lr & 7)) << 2);
  f32x4_t next[NL];
  auto request = [&](int step) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i) next[i] = *reinterpret_cast<const f32x4u_t*>(src[i] + step * 32);
  };
  auto keep = [&](float* to) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<f32x4_t*>(to + i * 1024 + place) = next[i];
  };
  f32x16_t acc[C];
#pragma unroll
  for (int t = 0; t < C; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
  request(0);
  keep(tiles[0]);
  __syncthreads();
  for (int st = 0; st < steps; ++st) {
    if (st + 1 < steps) request(st + 1);
    const float* const now = tiles[st & 1];
#pragma unroll
    for (int jj = 0; jj < 4 / KW; ++jj) {
      const int piece = ((2 * (jj + kw * 2) + kh) ^ (n & 7)) << 2;
      const f32x4_t wv = *reinterpret_cast<const f32x4_t*>(now + (rw * 32 + n) * 32 + piece);
      f32x4_t xv[C];
#pragma unroll
      for (int t = 0; t < C; ++t) xv[t] = *reinterpret_cast<const f32x4_t*>(now + (64 + (tw * C + t) * 32 + n) * 32 + piece);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < C; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[e], xv[t][e], acc[t], 0, 0, 0);
    }
    if (st + 1 < steps) keep(tiles[(st + 1) & 1]);  // its readers passed the barrier behind the step before
    __syncthreads();
  }
  if constexpr (KW == 2) {
    float* const other = tiles[0] + rw * 1024;
    if (kw == 1) {
#pragma unroll
      for (int i = 0; i < 16; ++i) other[i * 64 + lane] = acc[0][i];
    }
    __syncthreads();
    if (kw == 1) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[0][i] += other[i * 64 + lane];
    wave_sync();
  }
  store_block_rows<float, OUT, LISTED>(a, tiles[0] + wave * 1024, acc, rt * 64 + rw * 32, tt0 + tw * C * 32, n_tok, list, row_tiles * 64,
                                       cut);
}

template <int OUT>
int launch_one(const DenseArgs& a, int64_t rows, hipStream_t st) {
  bool pairs = false;
  for (int i = 0; i < a.n_seg; ++i) pairs |= a.seg[i].act == DENSE_GLU;
  const int64_t all = rows * a.batch;
  const std::false_type no;
  if (OUT == DENSE_ARGMAX || all >= 16384)
    hipLaunchKernelGGL((dense_one_f32_kernel<OUT, 4>), dim3((unsigned)(rows / 16), (unsigned)a.batch), dim3(256), 0, st, a, no);
  else if (pairs || all >= 8192)
    hipLaunchKernelGGL((dense_one_f32_kernel<OUT, 2>), dim3((unsigned)(rows / 8), (unsigned)a.batch), dim3(256), 0, st, a, no);
  else
    hipLaunchKernelGGL((dense_one_f32_kernel<OUT, 1>), dim3((unsigned)(rows / 4), (unsigned)a.batch), dim3(256), 0, st, a, no);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

// The time of a product of many tokens in us, but for what all forms of it share, for the choice between tiles of 32, 64 and 128
// tokens and shares of k: a step of a workgroup that has its compute unit to itself, the steps of several on one, weights
// at 4.6 TB/s, the shares' sums written and read at 6.8 TB/s.  Fitted to 1,190 timings (eight shapes from 256 x 1,536 to 32,768
// x 1,024, 3 to 512 tokens, 1 to 16 shares; 5 % off in the mean square with 7.3 us added).  The form it picks takes 2.9 % longer
// on average than the fastest timed; two workgroups per compute unit whatever the size, as it was, 7.4 %, up to 30 %.
float many_time(const DenseArgs& a, int64_t rows, int tile, int64_t cuts) {
  const float alone = tile == 32 ? 0.52f : tile == 64 ? 0.65f : 1.18f, beside = tile == 32 ? 0.32f : tile == 64 ? 0.56f : 1.05f;
  const float steps = (float)(((a.k >> 5) + cuts - 1) / cuts);
  const float per_unit = ceilf((float)(rows / 64 * ((a.M + tile - 1) / tile) * cuts * a.batch) / 256.0f);
  float t = std::max(steps * alone, (float)rows * (float)a.k * (float)a.batch * 4.0f / 4.6e6f);
  if (per_unit > 1.0f) t = std::max(t, steps * beside * per_unit);
  if (cuts > 1) t += 2.3f + (float)cuts * (float)a.M * (float)rows * 8.0f / 6.8e6f;
  return t;
}

template <int OUT, bool LISTED>
int launch_tiles(const DenseArgs& a, int64_t rows, int tile, int tok_tiles, int cuts, hipStream_t st) {
  const int row_tiles = (int)(rows / 64);
  const dim3 grid((unsigned)(((int64_t)row_tiles * tok_tiles * cuts + 7) / 8 * 8), (unsigned)a.batch);
  if (tile == 32)
    hipLaunchKernelGGL((dense_many_f32_kernel<1, 2, 1, OUT, LISTED>), grid, dim3(256), 0, st, a, row_tiles, tok_tiles, cuts);
  else if (tile == 64)
    hipLaunchKernelGGL((dense_many_f32_kernel<2, 1, 1, OUT, LISTED>), grid, dim3(256), 0, st, a, row_tiles, tok_tiles, cuts);
  else
    hipLaunchKernelGGL((dense_many_f32_kernel<2, 1, 2, OUT, LISTED>), grid, dim3(256), 0, st, a, row_tiles, tok_tiles, cuts);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

template <int OUT>
int launch_many(const DenseArgs& a, int64_t rows, hipStream_t st) {
  int64_t most = 1;  // shares of k: at least four steps each
  if (a.workspace && a.batch == 1 && a.M <= 65535)
    most = std::max<int64_t>(1, std::min(std::min<int64_t>(16, a.k >> 7), a.workspace_floats / (a.M * rows)));
  int tile = 32;
  int64_t cuts = 1;
  float best = HUGE_VALF;
  for (int t = 32; t <= 128; t *= 2)
    for (int64_t c = 1; c <= most; ++c) {
      const float time = many_time(a, rows, t, c);
      if (time < best) best = time, tile = t, cuts = c;
    }
  const int64_t tok_tiles = (a.M + tile - 1) / tile, tiles = rows / 64 * tok_tiles;
  AWQ_REQUIRE(tiles < (1ll << 26), "too large");
  if (cuts == 1) return launch_tiles<OUT, false>(a, rows, tile, (int)tok_tiles, 1, st);
  if (int rc = launch_tiles<DENSE_PART, false>(a, rows, tile, (int)tok_tiles, (int)cuts, st)) return rc;
  hipLaunchKernelGGL((dense_parts_kernel<float, OUT>), dim3((unsigned)((rows / 4 + 255) / 256), (unsigned)a.M), dim3(256), 0, st, a,
                     (int)rows, (int)cuts);
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

int launch_dense_one_joined_f32(const DenseArgs& a, const JoinArgs& j, int64_t rows, hipStream_t st) {
  const size_t lds = (size_t)a.k * 4;
  bool pairs = false;
  for (int i = 0; i < a.n_seg; ++i) pairs |= a.seg[i].act == DENSE_GLU;
  const auto launch = [&](auto q) {
    constexpr int Q = decltype(q)::value;
    if (rows >= 2048) hipLaunchKernelGGL((dense_one_f32_kernel<DENSE_STORE, 4, Q>), dim3((unsigned)(rows / 16)), dim3(256), lds, st, a, j);
    else if (pairs) hipLaunchKernelGGL((dense_one_f32_kernel<DENSE_STORE, 2, Q>), dim3((unsigned)(rows / 8)), dim3(256), lds, st, a, j);
    else hipLaunchKernelGGL((dense_one_f32_kernel<DENSE_STORE, 1, Q>), dim3((unsigned)(rows / 4)), dim3(256), lds, st, a, j);
  };
  if (j.width <= 1024) launch(std::integral_constant<int, 1>{});
  else launch(std::integral_constant<int, 2>{});
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

int launch_dense_many_f32(const DenseArgs& a, int64_t rows, hipStream_t st) {
  if (a.tiles) return launch_tiles<DENSE_STORE, true>(a, rows, a.tile_tokens <= 32 ? 32 : 64, a.max_tiles, 1, st);
  switch (a.out) {
    case DENSE_STORE: return launch_many<DENSE_STORE>(a, rows, st);
    case DENSE_RESIDUAL: return launch_many<DENSE_RESIDUAL>(a, rows, st);
    default: return launch_many<DENSE_F32>(a, rows, st);
  }
}
