// Dense products of bfloat16 weights with one token or many, packing of weights, the launch of any product (layers.hpp).
#include "dense_one_device.hpp"

#include <math.h>

#include <type_traits>

namespace {
template <int NW, int OUT, int IN, int RW, int TAPS = 0>
__global__ __launch_bounds__(NW * 64) void dense_one_kernel(DenseArgs a, typename OneExtra<IN>::type ahead) {
  dense_one_rows<NW, OUT, IN, RW, TAPS>(a, ahead, blockIdx.x, blockIdx.y);
}

// --- few tokens, bfloat16 ----------------------------------------------------------------------------------
// The one-token kernel with NT tiles of 16 tokens in the columns of v_mfma_f32_16x16x32_bf16: bound by the weights' bytes and by
// the tokens, which every workgroup reads out of its die's L2 (NT tiles beside R of weights).  A workgroup owns 16 R rows
// and all of k, so that nothing is left for a second launch to add.  9 tokens: 7,168 x 1,024 4.9 us, 4,096 x 4,096 8.0, 28,672 x
// 4,096 42.7 (5.5 TB/s); as tiles of 64 tokens with k cut over workgroups and a second launch 12.3, 18.8 and 58.5.
template <int NW, int NT, int R, int OUT, bool LISTED>
__global__ __launch_bounds__(NW * 64) void dense_few_kernel(DenseArgs a) {
  constexpr int PS = 20;  // floats per token of a wavefront's sums
  __shared__ __attribute__((aligned(16))) float part[NW * R * NT * 16 * PS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = blockIdx.x * 16 * R;
  const DenseSegment& s = segment_of(a, row0);
  const int local = row0 - s.row0;
  if (local >= s.rows) return;  // padding
  int64_t group = blockIdx.y;
  int n_tok = (int)a.M;
  const int32_t* list = nullptr;
  if constexpr (LISTED) {
    const DenseTile run = a.tiles[blockIdx.y];
    if (run.count == 0) return;
    group = run.group;
    n_tok = run.count;
    list = a.list + run.first;
  }
  const int steps = (int)(a.k >> 5);
  const int per = (steps + NW - 1) / NW;
  const int s0 = min(wave * per, steps), s1 = min(s0 + per, steps);
  const int r = lane & 15, c = lane >> 4;
  const bf16x8_t* w = reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const bf16_t*>(a.w) + group * a.w_batch) +
                      ((int64_t)(row0 >> 5) * (a.k >> 4) + (c >> 1)) * 64 + 32 * (c & 1) + (row0 & 16) + r;
  const bf16x8_t* x[NT];  // (rows 16 .. 31 of a block of weights are 16 pieces behind rows 0 .. 15)
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    int64_t tok = min(16 * t + r, n_tok - 1);
    if constexpr (LISTED) tok = list[tok] / a.list_div;
    x[t] = reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const bf16_t*>(s.x) + (LISTED ? 0 : blockIdx.y * a.x_batch) + tok * s.ldx) + c;
  }
  f32x4_t acc[R][NT];
#pragma unroll
  for (int b = 0; b < R; ++b)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[b][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int U = R * NT == 1 ? 8 : 4;
  int i = s0;
  for (; i + U <= s1; i += U) {
    bf16x8_t wv[U][R], xv[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int b = 0; b < R; ++b) wv[u][b] = __builtin_nontemporal_load(w + (int64_t)(i + u) * 128 + 16 * b);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t) xv[u][t] = x[t][(i + u) * 4];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int b = 0; b < R; ++b) acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[u][b], xv[u][t], acc[b][t], 0, 0, 0);
  }
  for (; i < s1; ++i) {
#pragma unroll
    for (int b = 0; b < R; ++b) {
      const bf16x8_t wv = __builtin_nontemporal_load(w + (int64_t)i * 128 + 16 * b);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, x[t][i * 4], acc[b][t], 0, 0, 0);
    }
  }
  // acc[b][t][j]: row 16 b + 4 c + j of token 16 t + r
#pragma unroll
  for (int b = 0; b < R; ++b)
#pragma unroll
    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4_t*>(part + (((wave * R + b) * NT + t) * 16 + r) * PS + 4 * c) = acc[b][t];
  __syncthreads();
  const int64_t y0 = blockIdx.y * a.y_batch;
  for (int at = tid; at < R * NT * 256; at += NW * 64) {
    const int b = at / (NT * 256), token = (at >> 4) % (NT * 16), row = at & 15;
    const int here = local + 16 * b;
    float sum = 0.0f;
#pragma unroll
    for (int v = 0; v < NW; ++v) sum += part[((v * R + b) * NT * 16 + token) * PS + row];
    int64_t tok = token;
    if constexpr (LISTED) tok = list[min(token, n_tok - 1)];
    if constexpr (OUT == DENSE_STORE) {
      if (s.act == DENSE_GLU) {
        const float up = __shfl_down(sum, 8, 16);
        if (token < n_tok && row < 8 && here / 2 + row < s.glu_rows)
          store_one<bf16_t>(s, LISTED ? 0 : y0, tok, here / 2 + row, glu<false>(sum, up));
        continue;
      }
    }
    if (token < n_tok && here + row < s.rows) finish_one<bf16_t, OUT>(a, s, tok, here + row, sum, LISTED ? 0 : y0);
  }
}

// --- many tokens, bfloat16 ---------------------------------------------------------------------------------
// A workgroup of four wavefronts takes 128 RB rows and 32 TT tokens: 32 RB rows per wavefront as RB x TT accumulators of
// v_mfma_f32_32x32x16_bf16.  The weights go from memory into registers in operand order, every byte once per
// workgroup; the tokens go through LDS (global_load_lds_dwordx4, 128 bytes per token and step of 64 inputs, the
// eight 16-byte pieces of row r at positions c ^ (r & 7)).  Both are requested two steps ahead.  Where the tiles do not
// fill the device, k is cut over `cuts` workgroups whose sums go to the workspace, [cut][token][row]; a second launch
// adds them in order.  At 2,048 tokens bound by the matrix cores: 28,672 x 4,096 434 us, 1.11 PFLOP/s (requested a step ahead, with
// a wait for everything on its way at each barrier, 474); at few by the trips to memory (33 tokens, 4,096 x 4,096: 17.8,
// was 19.9).
// LISTED: the tokens come from runs of a list, each with a weight block of its own.
// HALVES 2: four more wavefronts, which take the second half of k with tiles of their own (halves_pay).
template <int TT, int RB, int OUT, bool LISTED = false, int HALVES = 1>
__global__ __launch_bounds__(HALVES * 256, 2) void dense_many_kernel(DenseArgs a, int row_tiles, int tok_tiles, int cuts) {
  // three arrays, so that the compiler can tell which reads a request on its way may touch
  constexpr int kTile = 32 * TT * 64;
  __shared__ __attribute__((aligned(16))) bf16_t tiles0[HALVES * kTile];
  __shared__ __attribute__((aligned(16))) bf16_t tiles1[HALVES * kTile];
  __shared__ __attribute__((aligned(16))) bf16_t tiles2[HALVES * kTile];
  const int total = row_tiles * tok_tiles * cuts;
  // workgroups whose indices agree modulo 8 share a die: each die walks its own run of row tiles
  const int per = (total + 7) >> 3;
  const int work = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (work >= total) return;
  const int rc = work / tok_tiles, tile = work - rc * tok_tiles, tt0 = LISTED ? 0 : tile * 32 * TT;
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
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = HALVES == 2 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) : 0;
  bf16_t *const tile0 = tiles0 + half * kTile, *const tile1 = tiles1 + half * kTile, *const tile2 = tiles2 + half * kTile;
  const int n = lane & 31, kh = lane >> 5;
  const DenseSegment& s = segment_of(a, rt * 128 * RB);
  const int all_steps = (int)(a.k >> 6);
  const int first_of_cut = (int)((int64_t)all_steps * cut / cuts);
  const int steps = ((int)((int64_t)all_steps * (cut + 1) / cuts) - first_of_cut) / HALVES;
  const int first_step = first_of_cut + half * steps;
  const int64_t k16 = a.k >> 4;

  // this lane's pieces of the token tile
  const bf16_t* src[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) {
    const int row = (wave * TT + i) * 8 + (lane >> 3);
    int64_t tok = min(tt0 + row, n_tok - 1);
    if constexpr (LISTED) tok = list[tok] / a.list_div;
    src[i] = reinterpret_cast<const bf16_t*>(s.x) + blockIdx.y * a.x_batch + tok * s.ldx + first_step * 64 +
             (((lane & 7) ^ (row & 7)) << 3);
  }
  const bf16_t* const x_first = reinterpret_cast<const bf16_t*>(s.x);
  auto request = [&](bf16_t* tile, int step) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      const bf16_t* from = step < steps ? src[i] + step * 64 : x_first;
      __builtin_amdgcn_global_load_lds((gptr_t)from, (lptr_t)(tile + (wave * TT + i) * 8 * 64), 16, 0, 0);
    }
  };
  const bf16x8_t* wp = reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const bf16_t*>(a.w) + group * a.w_batch) +
                       ((int64_t)(rt * 4 + wave) * RB * k16 + first_step * 4) * 64;
  auto weights = [&](bf16x8_t (&wv)[RB][4], int step, int j) __attribute__((always_inline)) {
    const int at = step < steps ? lane : 0;
    step = min(step, steps - 1);
#pragma unroll
    for (int b = 0; b < RB; ++b) wv[b][j] = wp[(b * k16 + step * 4 + j) * 64 + at];
  };
  f32x16_t acc[RB][TT];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[b][t][i] = 0.0f;
  auto read_x = [&](const bf16_t* tile, int j, bf16x8_t (&xv)[TT]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TT; ++t) xv[t] = *reinterpret_cast<const bf16x8_t*>(tile + (32 * t + n) * 64 + (((2 * j + kh) ^ (n & 7)) << 3));
  };
  auto multiply = [&](const bf16x8_t (&wv)[RB][4], int j, const bf16x8_t (&xv)[TT]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int b = 0; b < RB; ++b) acc[b][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[b][j], xv[t], acc[b][t], 0, 0, 0);
  };
  // The order in which a slice of a step (16 of its inputs) is issued: the next slice's reads between the first products, the
  // weights of two steps on behind them.
  auto spread = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if (RB == 2) __builtin_amdgcn_sched_group_barrier(0x008, TT, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, RB, 0);
  };
  // Step st multiplies tile st % 3 and set st % 2 of the weights.  Both were requested two steps ago, so that a trip to memory
  // has two steps of products to hide behind: at the wait the 4 RB + TT requests of the step between may still be on their
  // way.  A slice's weights are requested into the registers that the slice has just used.  Past the end every lane
  // requests the same piece, which is not used.  The compiler need not keep the weights' requests of those steps: at the
  // wait ahead of a last step the youngest 4 RB + TT are then TT past the end and the 4 RB for that step's own weights, whose
  // use waits for them.  That leaves no request to spare, and needs a step's tokens to be requested ahead of its weights.
  bf16x8_t w0[RB][4], w1[RB][4];
  auto step = [&](const bf16_t* now, bf16x8_t (&w)[RB][4], bf16_t* later, int st) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0x0f70 | (4 * RB + TT));  // vmcnt(4 RB + TT)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();  // this step's tile is whole, the readers of the tile ahead of it are done
    asm volatile("" ::: "memory");
    request(later, st + 2);
    bf16x8_t xa[TT], xb[TT];
    read_x(now, 0, xa);
    __builtin_amdgcn_sched_barrier(0);
    read_x(now, 1, xb);
    multiply(w, 0, xa);
    weights(w, st + 2, 0);
    spread();
    read_x(now, 2, xa);
    multiply(w, 1, xb);
    weights(w, st + 2, 1);
    spread();
    read_x(now, 3, xb);
    multiply(w, 2, xa);
    weights(w, st + 2, 2);
    spread();
    multiply(w, 3, xb);
    weights(w, st + 2, 3);
    __builtin_amdgcn_sched_barrier(0);
  };
  request(tile0, 0);
#pragma unroll
  for (int j = 0; j < 4; ++j) weights(w0, 0, j);
  __builtin_amdgcn_sched_barrier(0);
  request(tile1, 1);
#pragma unroll
  for (int j = 0; j < 4; ++j) weights(w1, 1, j);
  int st = 0;
  for (; st + 6 <= steps; st += 6) {
    step(tile0, w0, tile2, st);
    step(tile1, w1, tile0, st + 1);
    step(tile2, w0, tile1, st + 2);
    step(tile0, w1, tile2, st + 3);
    step(tile1, w0, tile0, st + 4);
    step(tile2, w1, tile1, st + 5);
  }
  if (st < steps) {
    step(tile0, w0, tile2, st);
    if (st + 1 < steps) {
      step(tile1, w1, tile0, st + 1);
      if (st + 2 < steps) {
        step(tile2, w0, tile1, st + 2);
        if (st + 3 < steps) {
          step(tile0, w1, tile2, st + 3);
          if (st + 4 < steps) step(tile1, w0, tile0, st + 4);
        }
      }
    }
  }
  const int row_w = (rt * 4 + wave) * 32 * RB;
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no request is on its way into the tiles any more
  __syncthreads();                     // the last step's readers are done
  if constexpr (HALVES == 2) {
    // the halves of a sum meet: the first half of the wavefronts finishes the first half of the tokens
    constexpr int TH = TT / 2;
    float* const to = reinterpret_cast<float*>(half ? tiles0 : tiles1);
    const float* const from = reinterpret_cast<const float*>(half ? tiles1 : tiles0);
    f32x16_t mine[RB][TH];
#pragma unroll
    for (int b = 0; b < RB; ++b) {
#pragma unroll
      for (int t = 0; t < TH; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) to[(t * 16 + i) * 256 + tid] = half ? acc[b][t][i] : acc[b][TH + t][i];
      __syncthreads();
#pragma unroll
      for (int t = 0; t < TH; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float other = from[(t * 16 + i) * 256 + tid];
          mine[b][t][i] = half ? other + acc[b][TH + t][i] : acc[b][t][i] + other;
        }
      __syncthreads();
    }
    float* const turn = reinterpret_cast<float*>(half ? tiles1 : tiles0) + wave * 1024;
#pragma unroll
    for (int b = 0; b < RB; ++b)
      store_block_rows<bf16_t, OUT, LISTED>(a, turn, mine[b], row_w + 32 * b, tt0 + half * 32 * TH, n_tok, list, row_tiles * 128 * RB, cut);
  } else {
    float* const turn = reinterpret_cast<float*>(TT == 4 ? tile0 : (wave < 2 ? tile0 : tile1)) + (TT == 4 ? wave : wave & 1) * 1024;
#pragma unroll
    for (int b = 0; b < RB; ++b)
      store_block_rows<bf16_t, OUT, LISTED>(a, turn, acc[b], row_w + 32 * b, tt0, n_tok, list, row_tiles * 128 * RB, cut);
  }
}

template <typename S>
__global__ __launch_bounds__(256) void dense_pack_kernel(const S* __restrict__ src, int64_t rows, int64_t cols, void* w,
                                                         int64_t k, int64_t row0, int64_t col0, int f32, int form) {
  const int64_t n = rows * cols;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    int64_t r = i / cols, c = i % cols;
    if (form == PACK_TRANSPOSED) {
      const int64_t was = r;
      r = c;
      c = was;
    } else if (form != PACK_PLAIN) {
      r = (r >> 3) * 16 + (r & 7) + (form == PACK_UP ? 8 : 0);
    }
    r += row0;
    c += col0;
    if (f32)
      reinterpret_cast<float*>(w)[r * k + c] = (float)src[i];
    else
      reinterpret_cast<bf16_t*>(w)[(((r >> 5) * (k >> 4) + (c >> 4)) * 64 + ((c >> 3) & 1) * 32 + (r & 31)) * 8 + (c & 7)] =
          (bf16_t)(float)src[i];
  }
}

constexpr int kFewTokens = 32;

// Up to 2,048 rows 16 of them a workgroup leave half of the compute units or more without one, and a unit takes in no more than
// about 30 KB a us.  8 rows against 16: 1,024 x 4,096 4.8 and 6.1 us, 1,536 x 6,144 6.7 and 8.9, 2,048 x 8,192 9.6 and 11.8, 1,024 x
// 16,384 12.2 and 17.8; from 2,304 rows on 16 are faster (2,304 x 9,216 13.9 against 15.3, 3,072 x 3,072 6.4 against 7.7), and with
// up to 1,024 inputs neither is (3.5).  Both rows of a gated pair, and the rows of a candidate, are in one workgroup of 16.
bool eight_rows(const DenseArgs& a, int64_t rows) {
  bool eight = a.k > 1024 && rows * a.batch <= 2048;
  for (int i = 0; i < a.n_seg; ++i) eight = eight && a.seg[i].act != DENSE_GLU;
  return eight;
}

template <int OUT, int IN, int RW>
void launch_one_rows(const DenseArgs& a, int64_t rows, size_t lds, hipStream_t st) {
  const dim3 g((unsigned)(rows / RW), (unsigned)a.batch);
  const std::false_type no;
  if (a.k > 8192) hipLaunchKernelGGL((dense_one_kernel<16, OUT, IN, RW>), g, dim3(1024), lds, st, a, no);
  else if (a.k > 1024) hipLaunchKernelGGL((dense_one_kernel<8, OUT, IN, RW>), g, dim3(512), lds, st, a, no);
  else hipLaunchKernelGGL((dense_one_kernel<4, OUT, IN, RW>), g, dim3(256), lds, st, a, no);
}

template <int OUT, int IN>
int launch_one_as(const DenseArgs& a, int64_t rows, hipStream_t st) {
  const size_t lds = IN == IN_GATED ? (size_t)a.gate_k * 2 : 0;
  const bool eight = OUT != DENSE_ARGMAX && eight_rows(a, rows);
  if constexpr (OUT != DENSE_ARGMAX) {
    if (eight) launch_one_rows<OUT, IN, 8>(a, rows, lds, st);
  }
  if (!eight) launch_one_rows<OUT, IN, 16>(a, rows, lds, st);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

template <int OUT>
int launch_one(const DenseArgs& a, int64_t rows, hipStream_t st) {
  if constexpr (OUT == DENSE_RESIDUAL)
    if (a.gate_o) return launch_one_as<OUT, IN_GATED>(a, rows, st);
  return launch_one_as<OUT, IN_READ>(a, rows, st);
}

template <int OUT>
int launch_one_normed(const DenseArgs& a, const NormConvArgs& n, int64_t rows, hipStream_t st) {
  const dim3 g((unsigned)(rows / 16));
  const size_t lds = (size_t)a.k * 2;
  if (n.conv) hipLaunchKernelGGL((dense_one_kernel<8, OUT, IN_NORMED, 16, kFusedTaps>), g, dim3(512), lds, st, a, n);
  else hipLaunchKernelGGL((dense_one_kernel<8, OUT, IN_NORMED, 16>), g, dim3(512), lds, st, a, n);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

int launch_one_joined(const DenseArgs& a, const JoinArgs& j, int64_t rows, hipStream_t st) {
  const size_t lds = (size_t)a.k * 2;
  const auto launch = [&](auto in) {
    constexpr int IN = decltype(in)::value;
    if (eight_rows(a, rows)) hipLaunchKernelGGL((dense_one_kernel<8, DENSE_STORE, IN, 8>), dim3((unsigned)(rows / 8)), dim3(512), lds, st, a, j);
    else hipLaunchKernelGGL((dense_one_kernel<8, DENSE_STORE, IN, 16>), dim3((unsigned)(rows / 16)), dim3(512), lds, st, a, j);
  };
  if (j.width <= 2048) launch(std::integral_constant<int, IN_JOINED>{});
  else launch(std::integral_constant<int, IN_JOINED_2>{});
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

// 32 rows per workgroup read the tokens half as often, 16 make twice the workgroups: 8,192 x 1,024 at 9 tokens 6.9 against 5.2 us,
// 16,384 x 4,096 at 16 tokens 25.4 against 32.0, at 32 tokens 32.3 against 46.7
bool few_pairs(int64_t rows, int64_t tokens, int64_t blocks) { return rows * blocks >= (tokens <= 16 ? 16384 : 8192); }

// The time of such a launch in us, without its first 1.5: what the workgroups of a compute unit take in, at the rates at which
// one does for one and for two tiles of tokens, or the weights out of memory.
float few_time(const DenseArgs& a, int64_t rows) {
  const int64_t R = few_pairs(rows, a.M, a.batch) ? 32 : 16, per_unit = (rows / R * a.batch + 255) / 256;
  return std::max((float)per_unit * (float)((R + a.M) * a.k) * 2.0f / (a.M <= 16 ? 36e3f : 28e3f),
                  (float)rows * (float)a.k * (float)a.batch * 2.0f / 5.4e6f);
}

// up to 32 tokens, or tiles of as many
template <int OUT, bool LISTED>
int launch_few(const DenseArgs& a, int64_t rows, int tokens, int blocks, hipStream_t st) {
  const bool pairs = few_pairs(rows, tokens, blocks);
  const dim3 g((unsigned)(rows / (pairs ? 32 : 16)), (unsigned)blocks);
  const auto launch = [&](auto waves) {
    constexpr int NW = decltype(waves)::value;
    const dim3 t(NW * 64);
    if (tokens <= 16) {
      if (pairs) hipLaunchKernelGGL((dense_few_kernel<NW, 1, 2, OUT, LISTED>), g, t, 0, st, a);
      else hipLaunchKernelGGL((dense_few_kernel<NW, 1, 1, OUT, LISTED>), g, t, 0, st, a);
    } else {
      if (pairs) hipLaunchKernelGGL((dense_few_kernel<NW, 2, 2, OUT, LISTED>), g, t, 0, st, a);
      else hipLaunchKernelGGL((dense_few_kernel<NW, 2, 1, OUT, LISTED>), g, t, 0, st, a);
    }
  };
  if (a.k > 8192) launch(std::integral_constant<int, 16>{});
  else if (a.k > 1024) launch(std::integral_constant<int, 8>{});
  else launch(std::integral_constant<int, 4>{});
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

// The forms of a product of many tokens: tiles of 256 or 128 rows and 64 or 128 tokens.  Small tiles put more workgroups on the
// device, and three or four of them on a compute unit instead of two, so that fewer shares of k (and often no second launch) are
// needed; large ones read less.  2,048 x 2,048 at 129 tokens 14.2 -> 11.9 us with 128 rows, 8,192 x 2,048 18.2 -> 13.2, 4,096 x 4,096
// at 512 30.8 -> 23.4, 1,024 x 1,024 at 64 to 1,024 tokens 12 -> 8.4.
struct ManyForm {
  int tt, rb;         // 32 tt tokens, 128 rb rows
  int resident;       // workgroups that the device holds
  float wait, root;   // a step of a workgroup that has its unit to itself waits for memory, the longer the more weights are on their way
  float step;         // a step of one of several workgroups
  float end;          // the end of a tile, of binary32 outputs that are not added to others
};
constexpr ManyForm kManyForms[4] = {{2, 2, 512, 0.5296f, 0.0068f, 0.4825f, 2.9902f},
                                    {2, 1, 1024, 0.4289f, 0.0f, 0.3366f, 0.0f},
                                    {4, 2, 512, 0.7263f, 0.0f, 0.6619f, 4.8844f},
                                    {4, 1, 768, 0.5590f, 0.0f, 0.4261f, 1.6886f}};

// the shares' sums, written, read and added one after the other
float shares_time(const DenseArgs& a, int64_t rows, int64_t cuts) {
  return 2.71f + (float)cuts * (0.3703f + (float)a.M * (float)rows * 8.0f / 2.708e6f);
}
// Two wavefronts per SIMD, each with a half of k, where a tile of a product has a compute unit to itself (at most 256 of them): one
// waits for its trips to memory and its tokens, two have products for each other.  us, with four wavefronts and with eight:
//   1,024 x 512    129 tokens    8.1   7.7       4,096 x 4,096     512 tokens   32.6   29.3
//   2,048 x 1,024  333 tokens   10.3   9.6       4,096 x 4,096   1,000 tokens   41.6   38.9
//   2,048 x 2,048  512 tokens   14.2  12.5       8,192 x 8,192     512 tokens   86.3   76.9
//   6,144 x 2,048  200 tokens   18.9  16.7       2,048 x 8,192   2,048 tokens   84.4   75.6
//   12,288 x 2,048 129 tokens   23.9  21.8       4,096 x 16,384  2,048 tokens    250    241
// Not for shares of k, which are short already (1,024 x 4,096 at 512 tokens in four 16.2, 17.1), nor for tokens of a list, whose tiles
// are mostly without any (no gain).
bool halves_pay(int64_t groups, int64_t steps, int64_t cuts) { return cuts == 1 && groups <= 256 && steps >= 8 && steps % 2 == 0; }

// The time of a product in us, but for what all forms of it share: what the choice of a form and of a number of shares of k needs.
// The numbers are fitted for the choice, not for the time, to 49,600 timings (2,153 products: 111 shapes from 256 x 64 to 32,768 x 1,024,
// 28,672 x 8,192 and 4,096 x 16,384, 33 to 2,048 tokens, all forms, 1 to 16 shares, every kind of output, weights from memory).  The form
// it picks takes 0.7 % longer on average than the fastest timed, 11 % at the 99th of 100; against tiles of 256 rows alone, by an
// estimate of their own, it is 13 % faster on average (21 % with up to 512 inputs, 6 % beyond 4,096) and for one product in 170 slower by 5 %
// or more, 17 % at most.  Fitted to binary32 outputs and mostly to 1,024 to 4,096 inputs, it was for one in ten of the longer ones
// and wherever 2,816 to 4,096 rows of 512 met 1,500 tokens or more: 10,752 x 15,232 at 98 tokens 77 -> 89 us, now 74; 3,328 x 512 at 1,500, added to
// the stream, 19.3 -> 24.7, now 15.5.  The choice costs the host 0.1 to 1 us.
float many_time(const DenseArgs& a, int64_t rows, const ManyForm& f, int64_t cuts) {
  const int64_t row_tiles = rows / (128 * f.rb), tok_tiles = (a.M + 32 * f.tt - 1) / (32 * f.tt);
  const float groups = (float)(row_tiles * tok_tiles * cuts * a.batch), steps = (float)(((a.k >> 6) + cuts - 1) / cuts);
  const float wait = f.wait + f.root * sqrtf((float)std::min<int64_t>(256, row_tiles * cuts * a.batch));
  const float per_unit = ceilf(groups / 256.0f);
  float t = steps * wait * ceilf(groups / (float)f.resident);
  // What eight wavefronts give, where that was timed for the choice.  (Beyond 4,096 inputs the choice is the one without, and they only
  // make it faster; sums that another launch adds anyway are cheaper in shares.)
  if (halves_pay((int64_t)groups, a.k >> 6, cuts) && a.k <= 4096 && !a.shares) t -= steps * (f.rb == 1 ? 0.05f : 0.02f);
  if (per_unit > 1.0f) t = std::max(t, steps * per_unit * f.step);
  t = std::max(t, (float)rows * (float)a.k * (float)a.batch * 2.0f / 9.12e6f);
  return cuts > 1 ? t + shares_time(a, rows, cuts) : t + per_unit * f.end * (a.out == DENSE_F32 ? 1.0f : 1.7f);
}

template <int OUT, bool LISTED>
void launch_form(const DenseArgs& a, const ManyForm& f, int64_t rows, int64_t tok_tiles, int64_t cuts, hipStream_t st) {
  const int row_tiles = (int)(rows / (128 * f.rb));
  const dim3 grid((unsigned)((row_tiles * tok_tiles * cuts + 7) / 8 * 8), (unsigned)a.batch);
  const auto launch = [&](auto halves) {
    constexpr int H = decltype(halves)::value;
    const dim3 b(H * 256);
    if (f.tt == 2 && f.rb == 2) hipLaunchKernelGGL((dense_many_kernel<2, 2, OUT, LISTED, H>), grid, b, 0, st, a, row_tiles, (int)tok_tiles, (int)cuts);
    else if (f.tt == 2) hipLaunchKernelGGL((dense_many_kernel<2, 1, OUT, LISTED, H>), grid, b, 0, st, a, row_tiles, (int)tok_tiles, (int)cuts);
    else if (f.rb == 2) hipLaunchKernelGGL((dense_many_kernel<4, 2, OUT, LISTED, H>), grid, b, 0, st, a, row_tiles, (int)tok_tiles, (int)cuts);
    else hipLaunchKernelGGL((dense_many_kernel<4, 1, OUT, LISTED, H>), grid, b, 0, st, a, row_tiles, (int)tok_tiles, (int)cuts);
  };
  if constexpr (!LISTED && OUT != DENSE_PART) {
    if (halves_pay(row_tiles * tok_tiles * a.batch, a.k >> 6, cuts)) return launch(std::integral_constant<int, 2>{});
  }
  launch(std::integral_constant<int, 1>{});
}

template <int OUT>
int launch_many(const DenseArgs& a, int64_t rows, hipStream_t st) {
  const DenseForm c = dense_form(a, rows);
  if (c.tt == 0) return launch_few<OUT, false>(a, rows, (int)a.M, a.batch, st);
  const ManyForm* form = kManyForms;
  while (form->tt != c.tt || form->rb != c.rb) ++form;
  const int64_t tok_tiles = (a.M + 32 * form->tt - 1) / (32 * form->tt);
  if (c.cuts > 1) {
    launch_form<DENSE_PART, false>(a, *form, rows, tok_tiles, c.cuts, st);
    AWQ_HIP_TRY(hipGetLastError());
    if (OUT == DENSE_F32 && a.shares) {
      *a.shares = c.cuts;
      return AWQ_OK;
    }
    hipLaunchKernelGGL((dense_parts_kernel<bf16_t, OUT>), dim3((unsigned)((rows / 4 + 255) / 256), (unsigned)a.M), dim3(256), 0, st, a,
                       (int)rows, (int)c.cuts);
  } else {
    launch_form<OUT, false>(a, *form, rows, tok_tiles, 1, st);
  }
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

// tokens with weight blocks of their own
int launch_listed(const DenseArgs& a, int64_t rows, hipStream_t st) {
  if (a.tile_tokens <= kFewTokens) return launch_few<DENSE_STORE, true>(a, rows, a.tile_tokens, a.max_tiles, st);
  // 128 rows where 64 tokens meet a weight block, and where 128 do and 256 rows would be at most two workgroups per compute unit, of
  // which not all have tokens: Tudasun 2,048 at 129 tokens 1,010 -> 957 us, 1,536 at 300 (128 tokens) 888 -> 856; 4,096 at 1,024, 1,104
  // workgroups of 256 rows, 3,436 and with 128 rows 3,608
  const bool few_groups = rows / 256 * a.max_tiles <= 512;
  launch_form<DENSE_STORE, true>(a, kManyForms[a.tile_tokens <= 64 ? 1 : few_groups ? 3 : 2], rows, a.max_tiles, 1, st);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

}  // namespace

// A product of few tokens goes the way whose time is estimated to be the shorter; what the other way's estimate leaves out is 7 us
// more, and it takes the weights' time at least.  Workgroups that leave compute units idle and long rows, which read the tokens more than the
// weights, are against the few-token kernel: 6,144 x 12,288 at 20 tokens 54 us, below 36.  Of 520 products (52 shapes from 256 x 64 to
// 28,672 x 8,192, 2 to 32 tokens, both ways timed) the choice is 0.6 % off on average and 16 % at most.
DenseForm dense_form(const DenseArgs& a, int64_t rows) {
  constexpr float kManyMore = 7.0f;
  const float few = a.M <= kFewTokens ? few_time(a, rows) : HUGE_VALF;
  DenseForm form;
  // (mostly known without an estimate of the other way's forms)
  if (few < (float)rows * (float)a.k * (float)a.batch * 2.0f / 5.8e6f + kManyMore) return form;
  int64_t most = 1;  // shares of k: at least four steps each
  if (a.workspace && a.batch == 1 && a.M <= 65535)
    most = std::max<int64_t>(1, std::min(std::min<int64_t>(16, a.k >> 8), a.workspace_floats / (a.M * rows)));
  float best = HUGE_VALF;
  for (const ManyForm& f : kManyForms)
    for (int64_t c = 1; c <= most && (c == 1 || shares_time(a, rows, c) < best); ++c) {
      const float t = many_time(a, rows, f, c);
      if (t < best) best = t, form = DenseForm{f.tt, f.rb, (int32_t)c};
    }
  if (few < best + kManyMore) return DenseForm();
  return form.tt ? form : DenseForm{4, 2, 1};  // (a product too long for the estimate)
}

bool dense_gate_fused(int64_t n, int64_t k_padded, int64_t M, bool f32) {
  return !f32 && M == 1 && n % 4 == 0 && n > 0 && n <= k_padded && k_padded % kDenseKAlign == 0 && k_padded <= 16384;
}

int64_t dense_weight_bytes(int64_t rows_padded, int64_t k_padded, bool f32) { return rows_padded * k_padded * (f32 ? 4 : 2); }

int launch_dense_pack(const void* src, bool src_f32, int64_t rows, int64_t cols, void* w, int64_t k_padded, int64_t row0,
                      int64_t col0, bool f32, hipStream_t st, int form) {
  AWQ_REQUIRE(rows > 0 && cols > 0 && k_padded % kDenseKAlign == 0 && col0 % 8 == 0 &&
                  col0 + (form == PACK_TRANSPOSED ? rows : cols) <= k_padded,
              "bad block");
  const unsigned grid = (unsigned)std::min<int64_t>((rows * cols + 255) / 256, 65536);
  if (src_f32)
    hipLaunchKernelGGL(dense_pack_kernel<float>, dim3(grid), dim3(256), 0, st, (const float*)src, rows, cols, w, k_padded,
                       row0, col0, f32 ? 1 : 0, form);
  else
    hipLaunchKernelGGL(dense_pack_kernel<bf16_t>, dim3(grid), dim3(256), 0, st, (const bf16_t*)src, rows, cols, w, k_padded,
                       row0, col0, f32 ? 1 : 0, form);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

// Up to 2,048 values, where every workgroup's reading of row, weights, taps and state (36 bytes a value) costs as much as the launch:
// Kugilix, 64 tokens after 100, with it and without: width 1,280 13.5 and 14.6 ms, 1,664 15.6 and 16.1, 2,048 18.4 and 18.5.  And up to 24
// groups: a wavefront takes every eighth, each a trip to memory behind the one ahead.  A token of four layers with it
// and without: 24 groups of 1,536 values 114 and 116 us, 16 of 1,024 98 and 102, 20 of 640 82 and 86; 32 of 2,048 134 and 134, 32 of 1,024
// 108 and 102, 40 of 640 94 and 86, 256 of 1,024 276 and 102.
bool dense_norm_fused(const NormConvArgs& n, bool f32) {
  const int64_t part = n.groups > 0 && n.width % n.groups == 0 ? n.width / n.groups : 0;
  return !f32 && n.M == 1 && n.width <= 2048 && n.groups >= 4 && n.groups <= 24 && part % 4 == 0 && part > 0 && part <= 256 && !n.rows && n.ld % kDenseKAlign == 0 &&
         (!n.conv || n.taps == kFusedTaps) && (((uintptr_t)n.x | (uintptr_t)n.w1 | (uintptr_t)n.w2 | (uintptr_t)n.conv) & 15) == 0;
}

// Every workgroup of the product reads the rows and the norms' weights, 24 bytes a value and more, and adds them up for itself: up to
// 4,096 rows at width 4,096 (or as many values in all) that costs less than the launch.  Tudasun, 24 tokens after 48, without it, up to
// 1 M values (the token input's products only), up to 16 M and always: width 1,024 5.97, 5.96, 5.60 and 5.73 ms, 1,536 6.95, 7.01, 6.60
// and 6.76, 2,048 8.00, 7.98, 7.56 and 7.67, 2,816 10.4, 10.4, 10.3 and 10.9; 4,096, 64 after 128, 37.2, 37.2, 37.0 and 39.7; width
// 1,024 in binary32 6.97, 7.08, 6.84 and 6.98.
bool dense_join_fused(const JoinArgs& j, int64_t rows, bool f32) {
  return j.M == 1 && j.y_shares == 1 && j.out && j.x_out && j.x_out != j.x && (j.top == 0 || j.out != j.h) && j.top <= kJoinTop && j.width <= (f32 ? 2048 : 4096) &&
         ((j.width | j.ldo | j.ldg | j.ldh) & 3) == 0 && j.ldo % kDenseKAlign == 0 && rows * j.width <= 16 << 20;
}

// every workgroup reads the operands of the end, the last of them behind the first one's outputs
static bool writes_operand_of(const DenseArgs& a, const JoinArgs& j) {
  const void* const operands[] = {j.x, j.y, j.y_gate, j.pairs, j.ids, j.weights, j.top > 0 ? j.h : nullptr, j.gate};
  for (int i = 0; i < a.n_seg; ++i)
    for (const void* p : operands)
      if (p && p == a.seg[i].y) return true;
  return false;
}

int dense_prepare_beside(DenseArgs* a, int64_t* rows, int* per_group) {
  const DenseSegment& s = a->seg[0];
  if (a->ldk == 0) a->ldk = a->k;
  AWQ_REQUIRE(a->w && a->M == 1 && a->n_seg == 1 && a->out == DENSE_RESIDUAL && a->batch == 1 && !a->gate_o && !a->ids && !a->tiles,
              "the product cannot be part of another launch");
  AWQ_REQUIRE(a->k > 0 && a->k % kDenseKAlign == 0 && a->ldk >= a->k && a->ldk % kDenseKAlign == 0 && s.x && s.y && s.rows > 0 && s.row0 == 0 &&
                  s.rows < (1 << 30),
              "bad product");
  a->start[0] = 0;
  *rows = round_up(s.rows, kDenseRowAlign);
  *per_group = eight_rows(*a, *rows) ? 8 : 16;
  return AWQ_OK;
}

int launch_dense(const DenseArgs& args, bool f32, hipStream_t st, const NormConvArgs* norm, const JoinArgs* join) {
  DenseArgs a = args;
  if (a.ldk == 0) a.ldk = a.k;
  AWQ_REQUIRE(a.w && a.M >= 1 && a.k > 0 && a.k % kDenseKAlign == 0, "bad product");
  AWQ_REQUIRE(a.ldk == a.k || (a.ldk > a.k && a.ldk % kDenseKAlign == 0 && a.M == 1 && !f32 && !a.tiles), "bad length of the block's rows");
  AWQ_REQUIRE(a.n_seg >= 1 && a.n_seg <= kDenseSegments, "too few or too many segments");
  for (int i = 0; i < a.n_seg; ++i) {
    const DenseSegment& s = a.seg[i];
    const bool shares = i > 0 && s.x == a.seg[i - 1].x;
    AWQ_REQUIRE(s.x && s.y && s.rows > 0 && s.row0 % (shares ? kDenseSharedAlign : kDenseRowAlign) == 0 && s.ldx % 8 == 0,
                "bad segment");
    AWQ_REQUIRE(i == 0 || s.row0 >= a.seg[i - 1].row0 + a.seg[i - 1].rows, "segments overlap");
    AWQ_REQUIRE(s.act != DENSE_GLU || (a.out == DENSE_STORE && s.glu_rows > 0 && s.rows == dense_glu_rows(s.glu_rows)), "bad gated segment");
    AWQ_REQUIRE((s.act != DENSE_SIGMOID && s.act != DENSE_LOG_DECAY && s.act != DENSE_FORGET) || s.bias, "a segment lacks its bias");
    AWQ_REQUIRE(s.act != DENSE_FORGET || s.lower, "a segment lacks its lower bound");
    a.start[i] = s.row0;
  }
  AWQ_REQUIRE(!a.gate_o || (a.out == DENSE_RESIDUAL && a.n_seg == 1 && dense_gate_fused(a.gate_n, a.gate_k, a.M, f32) && a.gate_g &&
                            a.gate_w && a.gate_k <= a.k),
              "the gated norm cannot be part of this product");
  const DenseSegment& last = a.seg[a.n_seg - 1];
  const int64_t rows = round_up(last.row0 + last.rows, kDenseRowAlign);
  AWQ_REQUIRE(rows < (1ll << 30) && a.M < (1ll << 30), "too large");
  AWQ_REQUIRE(a.batch >= 1 && a.batch <= 65535 && (a.batch == 1 || (a.out == DENSE_STORE && a.w_batch % 8 == 0 && a.x_batch % 8 == 0)),
              "bad batch");
  AWQ_REQUIRE(!a.ids || (a.M == 1 && a.n_groups >= 0), "weight blocks by number take one token");
  AWQ_REQUIRE(a.fixed == 0 || (a.ids && a.fixed > 0 && a.fixed <= a.batch), "bad number of fixed weight blocks");
  if (a.tiles) {
    AWQ_REQUIRE(a.out == DENSE_STORE && a.list && a.list_div >= 1 && a.batch == 1 && a.max_tiles >= 1 && a.max_tiles <= 65535 &&
                    a.tile_tokens >= 1 && a.tile_tokens <= (f32 ? 64 : 128),
                "bad list of tokens");
    return f32 ? launch_dense_many_f32(a, rows, st) : launch_listed(a, rows, st);
  }
  AWQ_REQUIRE(a.out >= DENSE_STORE && a.out <= DENSE_ARGMAX, "unknown output");
  AWQ_REQUIRE(!a.shares || (a.out == DENSE_F32 && a.n_seg == 1 && last.act == DENSE_NONE), "the shares of this product cannot be left");
  if (a.shares) *a.shares = 1;
  AWQ_REQUIRE(a.out != DENSE_ARGMAX || (a.M == 1 && a.best), "sampling takes one token");
  if (norm) {
    AWQ_REQUIRE(dense_norm_fused(*norm, f32) && a.M == 1 && a.k == norm->ld && a.batch == 1 && !a.gate_o && a.n_seg <= (norm->w2 ? 2 : 1) &&
                    (a.out == DENSE_STORE || a.out == DENSE_ARGMAX) && norm->x && norm->w1 && (!norm->conv || (norm->state[0] && norm->state[1])),
                "the norm cannot be part of this product");
    return a.out == DENSE_STORE ? launch_one_normed<DENSE_STORE>(a, *norm, rows, st) : launch_one_normed<DENSE_ARGMAX>(a, *norm, rows, st);
  }
  if (join) {
    AWQ_REQUIRE(dense_join_fused(*join, rows, f32) && a.M == 1 && a.k == join->ldo && a.batch == 1 && !a.ids && !a.gate_o && a.out == DENSE_STORE &&
                    join->x && join->w_post && (join->y || join->top > 0),
                "the end of the sublayer cannot be part of this product");
    AWQ_REQUIRE(!writes_operand_of(a, *join), "the product writes what the end of the sublayer in it reads");
    return f32 ? launch_dense_one_joined_f32(a, *join, rows, st) : launch_one_joined(a, *join, rows, st);
  }
  if (f32) return a.M == 1 ? launch_dense_one_f32(a, rows, st) : launch_dense_many_f32(a, rows, st);
  switch (a.out) {
    case DENSE_STORE: return a.M == 1 ? launch_one<DENSE_STORE>(a, rows, st) : launch_many<DENSE_STORE>(a, rows, st);
    case DENSE_RESIDUAL: return a.M == 1 ? launch_one<DENSE_RESIDUAL>(a, rows, st) : launch_many<DENSE_RESIDUAL>(a, rows, st);
    case DENSE_F32: return a.M == 1 ? launch_one<DENSE_F32>(a, rows, st) : launch_many<DENSE_F32>(a, rows, st);
    default: return launch_one<DENSE_ARGMAX>(a, rows, st);
  }
}
