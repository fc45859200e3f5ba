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
// Four numbers as sums of three bfloat16 terms: the upper halves of the numbers, of what that leaves, and of what is left then.  Eight
// bits of significand each, so the sum is the number itself, down to 2^-110: there the last terms leave the range of bfloat16.
struct Split4 {
  uint2 part[3];
};
__device__ __forceinline__ uint2 upper_halves(const f32x4_t v) {
  return make_uint2(__builtin_amdgcn_perm(__float_as_uint(v[1]), __float_as_uint(v[0]), 0x07060302u),
                    __builtin_amdgcn_perm(__float_as_uint(v[3]), __float_as_uint(v[2]), 0x07060302u));
}
__device__ __forceinline__ Split4 split4(f32x4_t v) {
  Split4 s;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    s.part[p] = upper_halves(v);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] -= __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u);
  }
  return s;
}

// On v_mfma_f32_32x32x16_bf16, whose products are exact and which does 16 times the operations of v_mfma_f32_32x32x2_f32: both
// operands as three terms each and all products of two terms but the one of the last two, which is 2^-30 of the whole at most.  (A
// second and a third term's product is up to 2^-22 of the whole, and cut terms have the sign of their number: without these two a
// product came out smaller by 0.7 x 2^-24 on average and 7.8 x 2^-24 at most.)  Where a step's weights are bfloat16 numbers, as a
// checkpoint in bfloat16 has them, three products are left and nothing is left out.  The first terms' products have a sum of their
// own, which is rounded once per 16 inputs.
// A workgroup of four wavefronts takes 32 RW rows and 32 TW C tokens, steps of 32 inputs; KW wavefronts share the inputs of a step,
// whose sums meet in LDS.  Weights and tokens are requested two steps ahead into registers, split once and go through LDS, a term's
// 64 bytes per row and step, the four 16-byte pieces of row r at positions c ^ (r / 4 & 3).  Where the tiles do not fill the device, k
// is cut over `cuts` workgroups and a second launch adds their sums, as in bfloat16.
// Bound by the splitting (vector instructions) beside the matrix cores, at few tokens by the weights' bytes.  333 tokens, us, on
// v_mfma_f32_32x32x2_f32 before, weights that are bfloat16 numbers, and weights that are not: 1,024 rows of 4,096 inputs 40, 27, 39;
// 7,168 of 1,024 58, 34, 57; 32,768 of 1,024 220, 111, 207.  Up to 64 tokens weights that are not take more than before,
// up to 15 % with 256 inputs and 11 % with more, weights that are mostly less (1,024 x 4,096, 33 tokens: 18.0, 17.3 and 18.2 us).
// Off from 64 bits (norm) by 0.8e-7 to 1.8e-7 with 300 to 1,024 rows of 64 to 4,096 inputs, either way; before 1.1e-7 to 2.2e-7.
// An infinity has no such terms (what it leaves is NaN), and numbers below 2^-110 not all of theirs: a wavefront that finds sums that
// are not finite, or other than zero and below 2^-100, forms them again, in binary32.  (Inputs of 2^-115 were off by 37 x 2^-24 of the
// result, of 2^-120 by 1,180, and still are beside operands so large that the sum is 2^-100 and more.)
template <int RW, int TW, int KW, int C, int OUT, bool LISTED = false>
__global__ __launch_bounds__(256, 2) void dense_many_f32_kernel(DenseArgs a, int row_tiles, int tok_tiles, int cuts) {
  static_assert(RW * TW * KW == 4 && (KW == 1 || (KW == 2 && C == 1)), "four wavefronts");
  constexpr int ROWS = 32 * RW, TOK = 32 * TW * C, NW = ROWS / 32, NL = (ROWS + TOK) / 32;  // pieces per thread and step, NW of weights
  constexpr int PLANE = (ROWS + TOK) * 32;
  __shared__ __attribute__((aligned(16))) bf16_t planes[2][3][PLANE];
  __shared__ __attribute__((aligned(16))) int wide[4];  // by wavefront that split them: some of the weights so far were no bfloat16 numbers
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
  const int rw = wave % RW, tw = TW > 1 ? wave / RW : 0, kw = KW > 1 ? wave / RW : 0;
  const DenseSegment& s = segment_of(a, rt * ROWS);
  if (rt * ROWS >= a.seg[a.n_seg - 1].row0 + a.seg[a.n_seg - 1].rows) return;  // padding
  const int all_steps = (int)(a.k >> 5);
  const int first_step = (int)((int64_t)all_steps * cut / cuts);
  const int steps = (int)((int64_t)all_steps * (cut + 1) / cuts) - first_step;
  const float* const w_rows = reinterpret_cast<const float*>(a.w) + group * a.w_batch + (int64_t)rt * ROWS * a.k + first_step * 32;
  const float* const x_rows = reinterpret_cast<const float*>(s.x) + blockIdx.y * a.x_batch + first_step * 32;
  auto token = [&](int i) __attribute__((always_inline)) {
    int64_t tok = min(tt0 + i, n_tok - 1);
    if constexpr (LISTED) tok = list[tok] / a.list_div;
    return tok;
  };

  // this thread's pieces of a step: place tid % 8 of rows tid / 8 + 32 i, the first NW of them weights
  const float* src[NL];
  const int lr = tid >> 3, at = (tid & 7) << 2;
#pragma unroll
  for (int i = 0; i < NL; ++i) src[i] = (i < NW ? w_rows + (int64_t)(lr + 32 * i) * a.k : x_rows + token(lr + 32 * (i - NW)) * s.ldx) + at;
  const int place = lr * 32 + ((((tid & 7) >> 1) ^ ((lr >> 2) & 3)) << 3) + (tid & 1) * 4;
  typedef f32x4_t Step[NL];
  auto request = [&](Step& to, int step) __attribute__((always_inline)) {
    step = min(step, steps - 1);
#pragma unroll
    for (int i = 0; i < NL; ++i) to[i] = *reinterpret_cast<const f32x4u_t*>(src[i] + step * 32);
  };
  int dirty = 3;  // buffers whose second and third terms of this wavefront's weights may be other than zero
  auto keep = [&](const Step& from, int buf) __attribute__((always_inline)) {
    bf16_t* const to = planes[buf][0] + place;
    uint32_t below = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) below |= __float_as_uint(from[i][e]);
    const bool any = __builtin_amdgcn_ballot_w64((below & 0xffffu) != 0) != 0;
    if (any || (dirty >> buf & 1)) {
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        const Split4 w = split4(from[i]);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(to + p * PLANE + i * 1024) = w.part[p];
      }
      if (lane == 0 && (any || dirty == 3)) wide[wave] = any ? 1 : 0;
      dirty = any ? dirty | 1 << buf | 4 : dirty & ~(1 << buf);
    } else {
#pragma unroll
      for (int i = 0; i < NW; ++i) *reinterpret_cast<uint2*>(to + i * 1024) = upper_halves(from[i]);
    }
#pragma unroll
    for (int i = NW; i < NL; ++i) {
      const Split4 x = split4(from[i]);
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(to + p * PLANE + i * 1024) = x.part[p];
    }
  };
  f32x16_t acc[C], low[C];
#pragma unroll
  for (int t = 0; t < C; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = low[t][i] = 0.0f;
  auto multiply = [&](int buf, bool all) __attribute__((always_inline)) {
#pragma unroll
    for (int jj = 0; jj < 2 / KW; ++jj) {
      const int piece = ((2 * (jj + kw) + kh) ^ ((n >> 2) & 3)) << 3;
      auto term = [&](int p, int row) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8_t*>(planes[buf][p] + (row + n) * 32 + piece);
      };
      bf16x8_t xv[3][C];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int t = 0; t < C; ++t) xv[p][t] = term(p, ROWS + (tw * C + t) * 32);
      auto add = [&](f32x16_t (&to)[C], bf16x8_t wv, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < C; ++t) to[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, xv[p][t], to[t], 0, 0, 0);
      };
      const bf16x8_t w0 = term(0, rw * 32);
      if (all) {
        const bf16x8_t w1 = term(1, rw * 32), w2 = term(2, rw * 32);
        add(low, w2, 1);
        add(low, w1, 2);
        add(low, w2, 0);
        add(low, w1, 1);
        add(low, w1, 0);
      }
      add(low, w0, 2);
      add(acc, w0, 0);
      add(low, w0, 1);
    }
  };
  auto step = [&](Step& now, Step& after, int st) __attribute__((always_inline)) {
    // `now` is in LDS already; `after` arrives for the step behind this one
    __syncthreads();
    typedef int int4_t __attribute__((ext_vector_type(4)));
    const int4_t some = *reinterpret_cast<const volatile int4_t*>(wide);
    const bool all = __builtin_amdgcn_readfirstlane(some[0] | some[1] | some[2] | some[3]) != 0;
    request(now, st + 2);
    multiply(st & 1, all);
    if (st + 1 < steps) keep(after, (st + 1) & 1);  // its readers passed the barrier
  };
  Step even, odd;
  request(even, 0);
  request(odd, 1);
  keep(even, 0);
  for (int st = 0;;) {
    step(even, odd, st);
    if (++st == steps) break;
    step(odd, even, st);
    if (++st == steps) break;
  }
#pragma unroll
  for (int t = 0; t < C; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] += low[t][i];
  __syncthreads();
  float* const turns = reinterpret_cast<float*>(&planes[0][0][0]);
  if constexpr (KW == 2) {
    float* const other = turns + rw * 1024;
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
  const auto holds = [](float v) __attribute__((always_inline)) {
    const uint32_t size = __float_as_uint(v) & 0x7fffffffu, least = __float_as_uint(0x1p-100f);
    return (int)(size - least < 0x7f800000u - least) | (int)(size == 0);
  };
#pragma unroll
  for (int t = 0; t < C; ++t) {
    int all = 1;
#pragma unroll
    for (int i = 0; i < 16; ++i) all &= holds(acc[t][i]);
    if (__builtin_amdgcn_ballot_w64(all == 0) == 0) continue;
    f32x16_t again;
#pragma unroll
    for (int i = 0; i < 16; ++i) again[i] = 0.0f;
    const float *w = w_rows + (int64_t)(rw * 32 + n) * a.k + kh, *x = x_rows + token((tw * C + t) * 32 + n) * s.ldx + kh;
    for (int i = 0; i < 32 * steps; i += 2) again = __builtin_amdgcn_mfma_f32_32x32x2f32(w[i], x[i], again, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (!holds(acc[t][i])) acc[t][i] = again[i];
  }
  store_block_rows<float, OUT, LISTED>(a, turns + wave * 1024, acc, rt * ROWS + rw * 32, tt0 + tw * C * 32, n_tok, list, row_tiles * ROWS,
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

// The tiles of a product of many tokens: few rows and tokens make many workgroups, four, three and two of which a compute unit holds.
struct Form {
  int rows, tokens;
  float alone, beside, end;  // a step of a workgroup that has its unit to itself, and of one of several; the end of a tile
};
constexpr int kForms = 3;
constexpr Form kForm[kForms] = {{64, 32, 0.4714f, 0.2758f, 0.0706f}, {64, 64, 0.7176f, 0.3196f, 0.018f}, {128, 64, 0.7455f, 0.5484f, 0.0376f}};

// The time of a product in us, but for what all forms of it share: what the choice of a form and of a number of shares of k needs.  Fitted
// for the choice, not for the time, to 5,997 timings (20 shapes from 256 x 256 to 32,768 x 1,024, 2 to 512 tokens, 1 to 16 shares; weights that
// are bfloat16 numbers).  The 0.25 us of a share is fitted apart, to 700 products (50 shapes, 8 to 333 tokens, weights of either kind, all
// forms timed): with 0.37, as the fit of all gave it, 1,024 x 4,096 at 33 to 64 tokens went in 8 shares instead of 16 and took 6 to 9 %
// longer.  The form it picks takes 0.8 % longer on average than the fastest timed, 11 % at the 99th of 100.
float many_time(const DenseArgs& a, int64_t rows, const Form& f, int64_t cuts) {
  const float steps = (float)(((a.k >> 5) + cuts - 1) / cuts);
  const float per_unit = ceilf((float)(rows / f.rows * ((a.M + f.tokens - 1) / f.tokens) * cuts * a.batch) / 256.0f);
  float t = std::max(steps * f.alone, (float)rows * (float)a.k * (float)a.batch * 4.0f / 7.169e6f);
  if (per_unit > 1.0f) t = std::max(t, steps * f.beside * per_unit);
  if (cuts > 1) return t + 2.743f + (float)cuts * (0.25f + (float)a.M * (float)rows * 8.0f / 4.476e6f);
  return t + per_unit * f.end;
}

template <int OUT, bool LISTED>
int launch_tiles(const DenseArgs& a, int64_t rows, int form, int tok_tiles, int cuts, hipStream_t st) {
  const int row_tiles = (int)(rows / kForm[form].rows);
  const dim3 grid((unsigned)(((int64_t)row_tiles * tok_tiles * cuts + 7) / 8 * 8), (unsigned)a.batch);
  if (form == 0)
    hipLaunchKernelGGL((dense_many_f32_kernel<2, 1, 2, 1, OUT, LISTED>), grid, dim3(256), 0, st, a, row_tiles, tok_tiles, cuts);
  else if (form == 1)
    hipLaunchKernelGGL((dense_many_f32_kernel<2, 2, 1, 1, OUT, LISTED>), grid, dim3(256), 0, st, a, row_tiles, tok_tiles, cuts);
  else
    hipLaunchKernelGGL((dense_many_f32_kernel<4, 1, 1, 2, OUT, LISTED>), grid, dim3(256), 0, st, a, row_tiles, tok_tiles, cuts);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

struct Choice {
  int form = 0;
  int64_t cuts = 1;
};
Choice choose(const DenseArgs& a, int64_t rows) {
  int64_t most = 1;  // shares of k: at least four steps each
  if (a.workspace && a.batch == 1 && a.M <= 65535)
    most = std::max<int64_t>(1, std::min(std::min<int64_t>(16, a.k >> 7), a.workspace_floats / (a.M * rows)));
  Choice best_of;
  float best = HUGE_VALF;
  for (int f = 0; f < kForms; ++f)
    for (int64_t c = 1; c <= most; ++c) {
      const float time = many_time(a, rows, kForm[f], c);
      if (time < best) best = time, best_of = Choice{f, c};
    }
  return best_of;
}

template <int OUT>
int launch_many(const DenseArgs& a, int64_t rows, hipStream_t st) {
  const auto [form, cuts] = choose(a, rows);
  const int64_t tok_tiles = (a.M + kForm[form].tokens - 1) / kForm[form].tokens, tiles = rows / 64 * tok_tiles;
  AWQ_REQUIRE(tiles < (1ll << 26), "too large");
  if (cuts == 1) return launch_tiles<OUT, false>(a, rows, form, (int)tok_tiles, 1, st);
  if (int rc = launch_tiles<DENSE_PART, false>(a, rows, form, (int)tok_tiles, (int)cuts, st)) return rc;
  if (OUT == DENSE_F32 && a.shares) {
    *a.shares = (int32_t)cuts;
    return AWQ_OK;
  }
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

DenseForm dense_form_f32(const DenseArgs& a, int64_t rows) {
  const Choice c = choose(a, rows);
  return DenseForm{kForm[c.form].tokens / 32, kForm[c.form].rows / 64, (int32_t)c.cuts};
}

int launch_dense_many_f32(const DenseArgs& a, int64_t rows, hipStream_t st) {
  if (a.tiles) return launch_tiles<DENSE_STORE, true>(a, rows, a.tile_tokens <= 32 ? 0 : 1, a.max_tiles, 1, st);
  switch (a.out) {
    case DENSE_STORE: return launch_many<DENSE_STORE>(a, rows, st);
    case DENSE_RESIDUAL: return launch_many<DENSE_RESIDUAL>(a, rows, st);
    default: return launch_many<DENSE_F32>(a, rows, st);
  }
}
