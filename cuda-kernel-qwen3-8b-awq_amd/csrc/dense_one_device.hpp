// A product of bfloat16 weights with one token: the rows of a workgroup, for the launches that it is all of (dense.hip) and those that
// it shares (window_attention.hip, linear_attention.hip).
#pragma once
#include "dense_device.hpp"
#include "join_device.hpp"
#include "lane_sums.hpp"

#include <type_traits>

namespace {
// --- one token, bfloat16 -----------------------------------------------------------------------------------
// A workgroup owns RW rows and all of k, its wavefronts a run of k each; a load of a wavefront is pieces of 16 RW contiguous
// bytes of the block.  v_mfma_f32_16x16x32_bf16 with the token in the columns: the matrix unit does the additions, and nothing
// but loads stands between the wavefront and memory.  With RW = 8 the 16 rows of the instruction are 8 rows at two steps of 32
// inputs next to each other, and a column holds the inputs of the step whose rows it meets.
// Eight steps of a wavefront are requested at once, and what is left of its run as well: one by one 1,536 rows of 1,536 inputs took
// 5.7 us, now 4.0, 1,152 of 1,152 4.9 and 3.6.  Requesting the next eight ahead of these products cost more in wavefronts per unit
// (81 registers instead of 62) than it gained: 28,672 x 4,096 40 -> 44 us.
// IN_GATED: the first gate_k inputs are formed here, RMS norm of o times w times sigmoid(g) (token_ops.hip has it as a
// launch of its own for many tokens): every workgroup normalises for itself while its first weights are on their way.
// IN_NORMED: all inputs are formed here, the grouped norms and the convolution of NormConvArgs (norm_conv4_kernel in token_ops.hip),
// the first norm's for segment 0, the second's for segment 1.  A launch between two products costs 3.5 to 4 us whatever it does, the
// norms in every workgroup about two: Kugilix's q, k, v and W_up at width 1,024 8.8 us with the launch ahead, now 6.6; with the row
// requested behind the weights, and the statistic through LDS, 7.4 (a compute unit's requests are served in order).
constexpr int kFusedTaps = 4;
// IN_JOINED, _2: all inputs are formed here, the end of the sublayer ahead (JoinArgs, one and two turns of the workgroup's threads).
enum OneInput { IN_READ, IN_GATED, IN_NORMED, IN_JOINED, IN_JOINED_2 };
template <int IN>
struct OneExtra {
  typedef std::false_type type;
};
template <>
struct OneExtra<IN_NORMED> {
  typedef NormConvArgs type;
};
template <>
struct OneExtra<IN_JOINED> {
  typedef JoinArgs type;
};
template <>
struct OneExtra<IN_JOINED_2> {
  typedef JoinArgs type;
};

// A group of the norm is a wavefront's, at most four channels a lane.  Everything is requested ahead of the statistic and in two
// parts, so that the first of the weights can go between them; the inputs ahead of the pass for both parities, since which one it
// is comes out of memory too.
template <int NW, int TAPS>
struct NormedInput {
  static constexpr int BACK = TAPS > 0 ? TAPS - 1 : 0, KN = TAPS > 0 ? TAPS : 1, HN = BACK > 0 ? BACK : 1;
  const NormConvArgs& a;
  const bool conv;
  const float* const w;
  const int part, lane, wave;
  int pos = 0, par = 0;
  f32x4_t x, wv, taps[KN], past[2][HN];
  __device__ __forceinline__ NormedInput(const NormConvArgs& n, bool second)
      : a(n), conv(TAPS > 0 && !second), w(second ? n.w2 : n.w1), part((int)n.width / n.groups), lane(threadIdx.x & 63),
        wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {}
  __device__ __forceinline__ bool mine(int g) const { return g < a.groups && 4 * lane < part; }
  __device__ __forceinline__ void request_row(int g) {
    x = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    if (mine(g)) x = *reinterpret_cast<const f32x4_t*>(a.x + g * part + 4 * lane);
    if (conv) pos = a.pos.position(), par = a.pos.parity();
  }
  __device__ __forceinline__ void request_constants(int g) {
    if (!mine(g)) return;
    const int c = g * part + 4 * lane;
    wv = *reinterpret_cast<const f32x4_t*>(w + c);
    if (conv) {
#pragma unroll
      for (int i = 0; i < TAPS; ++i) taps[i] = *reinterpret_cast<const f32x4_t*>(a.conv + (int64_t)c * TAPS + 4 * i);
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int j = 0; j < BACK; ++j) past[p][j] = *reinterpret_cast<const f32x4_t*>(a.state[p] + (int64_t)j * a.width + c);
    }
  }
  __device__ __forceinline__ void finish(int g, bool keeps, bf16_t* in) {
    float sq = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) sq = __builtin_fmaf(x[e], x[e], sq);
    const float inv = 1.0f / sqrtf(lanes::sum(sq) / (float)part + a.eps);
    if (!mine(g)) return;
    const int c = g * part + 4 * lane;
    const f32x4_t h = x * inv * wv;
    f32x4_t y = h;
    if (conv) {
      f32x4_t before[HN];
#pragma unroll
      for (int j = 0; j < BACK; ++j) {
        before[j] = par ? past[1][j] : past[0][j];
        if (pos - BACK + j < 0) before[j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // four channels of TAPS taps each, contiguous
        auto tap = [&](int j) { return taps[(e * TAPS + j) >> 2][(e * TAPS + j) & 3]; };
#pragma unroll
        for (int j = 0; j < BACK; ++j) y[e] = __builtin_fmaf(tap(j), before[j][e], y[e]);
        y[e] = __builtin_fmaf(tap(BACK), h[e], y[e]);
      }
      if (keeps) {
        float* const after = a.state[par ^ 1] + c;
#pragma unroll
        for (int j = 0; j + 1 < BACK; ++j) *reinterpret_cast<f32x4_t*>(after + (int64_t)j * a.width) = before[j + 1];
        *reinterpret_cast<f32x4_t*>(after + (int64_t)(BACK - 1) * a.width) = h;
      }
    }
    bf16x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (bf16_t)y[e];
    *reinterpret_cast<bf16x4_t*>(in + c) = o;
  }
  __device__ __forceinline__ void rest(bool keeps, int k, bf16_t* in) {
    for (int g = wave + NW; g < a.groups; g += NW) {
      request_row(g);
      request_constants(g);
      finish(g, keeps, in);
    }
    for (int c = (int)a.width + (int)threadIdx.x; c < k; c += NW * 64) in[c] = (bf16_t)0.0f;
    __syncthreads();
  }
};

template <int NW, int OUT, int IN, int RW, int TAPS = 0>
__device__ __forceinline__ void dense_one_rows(const DenseArgs& a, const typename OneExtra<IN>::type& ahead, const int block, const int product) {
  constexpr bool JOINED = IN == IN_JOINED || IN == IN_JOINED_2;
  constexpr int SP = 16 / RW;  // steps of an instruction
  extern __shared__ __attribute__((aligned(16))) bf16_t formed[];  // the inputs that are formed here
  __shared__ float part[NW][16];
  __shared__ float squares[NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = block * RW;
  const DenseSegment& s = segment_of(a, row0);
  const int local = row0 - s.row0;
  if (local >= s.rows) return;  // padding
  const int group = block_of_product(a, product);
  if (group < 0) return;
  const int steps = (int)(a.k >> 5);  // even: k is a multiple of 64
  const int per = ((steps + SP - 1) / SP + NW - 1) / NW;
  const int s0 = min(wave * per * SP, steps), s1 = min(s0 + per * SP, steps);
  const int r = lane & 15, c = lane >> 4, sub = r / RW;
  // piece of (row, 8-wide chunk c of step i): block (row / 32, 2 i + c / 2), lane 32 (c % 2) + row % 32
  const bf16x8_t* w = reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const bf16_t*>(a.w) + group * a.w_batch) +
                      ((int64_t)(row0 >> 5) * (a.ldk >> 4) + (c >> 1) + 2 * sub) * 64 + 32 * (c & 1) + (row0 & (32 - RW)) + r % RW;
  const bf16x8_t* x = reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const bf16_t*>(s.x) + product * a.x_batch) + c + 4 * sub;
  f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int U = IN == IN_NORMED || JOINED ? 4 : 8;
  constexpr int US = U * SP;
  // The inputs of the rest (8 rows: of a turn too) are requested before the first product, which takes registers for all of them: 512 x
  // 5,888 5.8 -> 5.4 us, 512 x 768 3.3 -> 2.9.  Not with 16 wavefronts of 16 rows, of which a unit then holds one workgroup instead of two:
  // 9,728 x 8,704 29.7 -> 32.6.
  constexpr bool kHold = RW == 8 || NW < 16;
  bf16x8_t wv[U];
  auto weights = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) wv[u] = __builtin_nontemporal_load(w + (int64_t)(i + u * SP) * 128);
  };
  auto input = [&](int i) __attribute__((always_inline)) {
    if (IN == IN_NORMED || JOINED || (IN == IN_GATED && (i + sub) * 32 < a.gate_k)) return reinterpret_cast<const bf16x8_t*>(formed)[(i + sub) * 4 + c];
    return x[i * 4];
  };
  int i = s0;
  if constexpr (IN == IN_NORMED) {
    NormedInput<NW, TAPS> in(ahead, a.n_seg > 1 && row0 >= a.start[1]);
    in.request_row(in.wave);
    __builtin_amdgcn_sched_barrier(0);
    in.request_constants(in.wave);
    __builtin_amdgcn_sched_barrier(0);
    if (i + US <= s1) weights(i);
    __builtin_amdgcn_sched_barrier(0);
    in.finish(in.wave, block == 0, formed);
    in.rest(block == 0, (int)a.k, formed);
  } else if constexpr (JOINED) {
    __shared__ float sums[2][16];
    joined_input<bf16_t, IN == IN_JOINED ? 1 : 2>(ahead, block == 0 && product == 0, (int)a.k, formed, sums, [&]() {
      if (i + US <= s1) weights(i);
    });
  } else {
    if (i + US <= s1) weights(i);
  }
  if constexpr (IN == IN_GATED) {
    constexpr int NT = NW * 64;
    const bf16_t* gate = reinterpret_cast<const bf16_t*>(a.gate_g);
    float sq = 0.0f;
    for (int j = tid * 4; j < a.gate_n; j += NT * 4) {
      const f32x4_t o = *reinterpret_cast<const f32x4_t*>(a.gate_o + j);
#pragma unroll
      for (int e = 0; e < 4; ++e) sq = __builtin_fmaf(o[e], o[e], sq);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
    if (lane == 0) squares[wave] = sq;
    __syncthreads();
    float all = 0.0f;
#pragma unroll
    for (int v = 0; v < NW; ++v) all += squares[v];
    const float inv = 1.0f / sqrtf(all / (float)a.gate_n + a.gate_eps);
    for (int j = tid * 4; j < a.gate_k; j += NT * 4) {
      bf16x4_t y = {(bf16_t)0.0f, (bf16_t)0.0f, (bf16_t)0.0f, (bf16_t)0.0f};
      if (j < a.gate_n) {
        const f32x4_t o = *reinterpret_cast<const f32x4_t*>(a.gate_o + j), gw = *reinterpret_cast<const f32x4_t*>(a.gate_w + j);
        const bf16x4_t g = *reinterpret_cast<const bf16x4_t*>(gate + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = (bf16_t)(o[e] * inv * gw[e] * sigmoid_exact((float)g[e]));
      }
      *reinterpret_cast<bf16x4_t*>(formed + j) = y;
    }
    __syncthreads();
  }
  for (; i + US <= s1; i += US) {
    if (i != s0) weights(i);
    bf16x8_t xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = input(i + u * SP);
    if (RW == 8) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[u], xv[u], acc, 0, 0, 0);
  }
  // The rest together as well, as many requests as there are steps: with the last one's repeated up to four or eight, 9,728 x 1,280 took
  // 7.4 us and 9,728 x 8,704 34.8, one step behind the other 6.4 and 29.6, now 6.4 and 29.7.  Behind the function's end, where the
  // compiler puts what it is told is rare: 2 % of a token of Kugilix of width 1,024, none of whose runs has a rest.  (A run is whole
  // instructions: the number of steps is even.)
  auto some = [&](auto count) __attribute__((always_inline)) {
    constexpr int N = decltype(count)::value;
    bf16x8_t xv[N];
#pragma unroll
    for (int u = 0; u < N; ++u) wv[u] = __builtin_nontemporal_load(w + (int64_t)(i + u * SP) * 128);
#pragma unroll
    for (int u = 0; u < N; ++u) xv[u] = input(i + u * SP);
    if (kHold) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < N; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[u], xv[u], acc, 0, 0, 0);
    i += N * SP;
  };
  if (__builtin_expect(i < s1, 0)) {
    if (IN == IN_GATED && s1 - i >= 4 * SP) some(std::integral_constant<int, 4>{});
    const int left = (s1 - i) / SP;  // less than U
    if (left == 1) some(std::integral_constant<int, 1>{});
    else if (left == 2) some(std::integral_constant<int, 2>{});
    else if (left == 3) some(std::integral_constant<int, 3>{});
    if constexpr (IN == IN_READ) {
      if (left == 4) some(std::integral_constant<int, 4>{});
      else if (left == 5) some(std::integral_constant<int, 5>{});
      else if (left == 6) some(std::integral_constant<int, 6>{});
      else if (left == 7) some(std::integral_constant<int, 7>{});
    }
  }
  // lane (c, r): rows 4 c .. + 3 of the instruction against column r, which is theirs where r / RW is 4 c / RW
  if (r == 4 * c / RW * RW) {
#pragma unroll
    for (int j = 0; j < 4; ++j) part[wave][4 * c + j] = acc[j];
  }
  __syncthreads();
  if (tid >= RW) return;
  float sum = 0.0f;
#pragma unroll
  for (int v = 0; v < NW; ++v) {
    float one = part[v][tid];
#pragma unroll
    for (int j = 1; j < SP; ++j) one += part[v][j * RW + tid];
    sum += one;
  }
  const int row = local + tid;
  const int64_t y0 = product * a.y_batch;
  if constexpr (OUT == DENSE_STORE && RW == 16) {
    if (s.act == DENSE_GLU) {
      const float up = __shfl_down(sum, 8, 16);
      if (tid < 8 && local / 2 + tid < s.glu_rows) store_one<bf16_t>(s, y0, 0, local / 2 + tid, glu<false>(sum, up));
      return;
    }
  }
  if (row < s.rows) finish_one<bf16_t, OUT>(a, s, 0, row, sum, y0);
  if constexpr (OUT == DENSE_ARGMAX) {
    if (s.act == DENSE_SOFTCAP) sum = softcap(s, sum);
    unsigned long long b = row < s.rows ? awq_pack_candidate(f32_key(sum), (uint32_t)row) : 0ull;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
      const unsigned long long o = __shfl_xor(b, off, 16);
      b = o > b ? o : b;
    }
    if (tid == 0) a.best[block] = b;
  }
}

}  // namespace
