// Linear attention whose state decays per channel (layers.hpp): per head S <- diag(decay_t) S + k_t v_t^T, o_t = S^T q_t.
#include "lane_sums.hpp"
#include "layers.hpp"
#include "segment_join.hpp"

#include <type_traits>

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// decay and key of one channel and token; without keys of its own the layer writes 1 - decay
__device__ __forceinline__ void decay_and_key(float g, bool keys, float k, float& decay, float& key) {
  decay = keys ? exp2f(g) : 1.0f - g;
  key = keys ? k : g;
}

// The recurrence token by token: a wavefront holds kCols columns of the state, lane l the rows l, l + 64, ... of each.
// Used for one token.  A workgroup takes 4 kCols columns.
template <typename T, int DPL, int kCols>
__global__ __launch_bounds__(256) void gated_step_kernel(GatedStateArgs a) {
  const int head = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int dimp = DPL * 64;
  const T* q = reinterpret_cast<const T*>(a.q) + (int64_t)head * a.dim;
  const T* k = reinterpret_cast<const T*>(a.k) + (int64_t)head * a.dim;
  const T* v = reinterpret_cast<const T*>(a.v) + (int64_t)head * a.vdim;
  const float* g = a.g + (int64_t)head * a.dim;
  float* o = a.o + (int64_t)head * a.vdim;
  const int64_t ldo = (int64_t)a.heads * a.vdim;
  const bool keys = a.k != nullptr, fresh = a.pos.position() == 0;
  const int col0 = (blockIdx.y * 4 + wave) * kCols;
  if (col0 >= a.vdim) return;
  float* state = a.state + ((int64_t)head * a.vdim + col0) * dimp;
  const int nc = min(kCols, a.vdim - col0);
  float s[kCols][DPL];
#pragma unroll
  for (int c = 0; c < kCols; ++c)
#pragma unroll
    for (int i = 0; i < DPL; ++i) s[c][i] = fresh || c >= nc ? 0.0f : state[c * dimp + i * 64 + lane];
  for (int64_t t = 0; t < a.M; ++t) {
    float qv[DPL], kv[DPL], dv[DPL], out[kCols];
#pragma unroll
    for (int i = 0; i < DPL; ++i) {
      const int d = i * 64 + lane;
      qv[i] = kv[i] = dv[i] = 0.0f;
      if (d < a.dim) {
        qv[i] = (float)q[t * a.ldp + d] * a.q_scale;
        decay_and_key(g[t * a.ldg + d], keys, keys ? (float)k[t * a.ldp + d] : 0.0f, dv[i], kv[i]);
      }
    }
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const float vv = c < nc ? (float)v[t * a.ldp + col0 + c] : 0.0f;
      out[c] = 0.0f;
#pragma unroll
      for (int i = 0; i < DPL; ++i) {
        s[c][i] = __builtin_fmaf(kv[i], vv, dv[i] * s[c][i]);
        out[c] = __builtin_fmaf(s[c][i], qv[i], out[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) out[c] += __shfl_xor(out[c], off, 64);
      if (lane == c && c < nc) o[t * ldo + col0 + c] = out[c];
    }
  }
#pragma unroll
  for (int c = 0; c < kCols; ++c)
    if (c < nc)
#pragma unroll
      for (int i = 0; i < DPL; ++i) state[c * dimp + i * 64 + lane] = s[c][i];
}

// The same for several tokens: fewer than the chunked form takes, wider heads, linear attention with few tokens or a decay of
// zero (HEAD: one decay per head).  A token's sums are those of a pass of its own, bit for bit.  Bound, token by token, by the
// trip of a token's inputs through memory and by the exchanges that end its sums, so the inputs of G tokens are requested
// together and left in LDS for the four wavefronts (a decay is formed once instead of four times), and sixteen sums are ended
// at a time.  8 heads of 128, 9 tokens: decays per head 4.1 us, per channel 4.5 (a token after the other 11.7 to 17.4; the chunked
// form 4.9 to 5.2, at 2 to 40 times the error); 15 tokens 4.2 and 4.6.  Two columns per wavefront: four took 4.9 and 5.3.
template <int DPL>
constexpr int few_tokens() { return DPL <= 4 ? 16 : 8; }  // 48 KB of LDS at most
template <int DPL>
constexpr int few_cols() { return DPL <= 4 ? 2 : 4; }

// x of lane ^ 1, 2, 4 or 8
template <int OFF>
__device__ __forceinline__ float other_lane(float x) {
  const int v = __float_as_int(x);
  if constexpr (OFF == 4) return __int_as_float(__builtin_amdgcn_ds_swizzle(v, (4 << 10) | 31));
  constexpr int kControl = OFF == 1 ? 0xb1 : OFF == 2 ? 0x4e : 0x128;  // quad_perm 1 0 3 2, quad_perm 2 3 0 1, row_ror:8
  return __int_as_float(__builtin_amdgcn_update_dpp(0, v, kControl, 0xf, 0xf, true));
}

// Sixteen sums over all lanes, number lane / 4 in x[0]: at each of the first four exchanges a lane hands over the half of its
// sums that it does not end with.  Each is added up as by an exchange of it at every distance from 32 to 1, bit for bit.
__device__ __forceinline__ void sixteen_sums(float (&x)[16], int lane) {
  typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const u32x2_t p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[i]), __float_as_uint(x[i + 8]), false, false);
    x[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u32x2_t p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[i]), __float_as_uint(x[i + 4]), false, false);
    x[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float low = x[i], high = x[i + 2];
    x[i] = (lane & 8 ? high : low) + other_lane<8>(lane & 8 ? low : high);
  }
  const float low = x[0], high = x[1];
  x[0] = (lane & 4 ? high : low) + other_lane<4>(lane & 4 ? low : high);
  x[0] += other_lane<2>(x[0]);
  x[0] += other_lane<1>(x[0]);
}

// One token with the head's norm and gate behind the recurrence: a workgroup per head, the recurrence as above.  Bound by the trips to
// memory and by what a compute unit takes in and gives out (the head's state both ways), so everything is requested at once:
// the state before the position is known (what it holds ahead of position 0 is not used), norm and gate ahead of the sums,
// which are ended together.  32 heads of 128 5.4 us; with the state requested behind the position, and each sum
// by itself, 8.2.
template <int N>
__device__ __forceinline__ void ended_sums(float (&x)[N], int lane) {  // N = 8, 4: number lane / (64 / N) in x[0], in the order of sixteen_sums
  typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const u32x2_t p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[i]), __float_as_uint(x[i + N / 2]), false, false);
    x[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const u32x2_t p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[i]), __float_as_uint(x[i + N / 4]), false, false);
    x[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  if constexpr (N == 8) x[0] = (lane & 8 ? x[1] : x[0]) + other_lane<8>(lane & 8 ? x[0] : x[1]);
  else x[0] += other_lane<8>(x[0]);
  x[0] += other_lane<4>(x[0]);
  x[0] += other_lane<2>(x[0]);
  x[0] += other_lane<1>(x[0]);
}

template <typename T, int DPL, int kCols>
__global__ __launch_bounds__(1024) void gated_head_kernel(GatedStateArgs a) {
  extern __shared__ float row[];  // [vdim]
  __shared__ float sums[16];
  const int head = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
  const int dimp = DPL * 64;
  const T* q = reinterpret_cast<const T*>(a.q) + (int64_t)head * a.dim;
  const T* k = reinterpret_cast<const T*>(a.k) + (int64_t)head * a.dim;
  const T* v = reinterpret_cast<const T*>(a.v) + (int64_t)head * a.vdim;
  const T* gate = reinterpret_cast<const T*>(a.gate) + (int64_t)head * a.vdim;
  const float* g = a.g + (int64_t)head * a.dim;
  const bool keys = a.k != nullptr;
  float qv[DPL], kv[DPL], gv[DPL], s[kCols][DPL], vv = 0.0f;
  auto request = [&](int col0) __attribute__((always_inline)) {
    const float* state = a.state + (int64_t)head * a.vdim * dimp;
#pragma unroll
    for (int c = 0; c < kCols; ++c)
#pragma unroll
      for (int i = 0; i < DPL; ++i) s[c][i] = state[(int64_t)min(col0 + c, a.vdim - 1) * dimp + i * 64 + lane];
    vv = (float)v[min(col0 + lane % kCols, a.vdim - 1)];
  };
#pragma unroll
  for (int i = 0; i < DPL; ++i) {
    const int d = min(i * 64 + lane, a.dim - 1);
    qv[i] = (float)q[d];
    gv[i] = g[d];
    kv[i] = keys ? (float)k[d] : 0.0f;
  }
  const int first = wave * kCols;
  if (first < a.vdim) request(first);
  const int c0 = min(tid, a.vdim - 1);
  float norm = a.norm[c0], z = a.gate ? (float)gate[c0] : 0.0f;
  const bool fresh = a.pos.position() == 0;
  float dv[DPL];
#pragma unroll
  for (int i = 0; i < DPL; ++i) {
    decay_and_key(gv[i], keys, kv[i], dv[i], kv[i]);
    qv[i] *= a.q_scale;
    if (i * 64 + lane >= a.dim) qv[i] = kv[i] = dv[i] = 0.0f;
  }
  for (int col0 = first; col0 < a.vdim; col0 += waves * kCols) {
    if (col0 != first) request(col0);
    float out[kCols];
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const float one = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(vv), c));
      out[c] = 0.0f;
#pragma unroll
      for (int i = 0; i < DPL; ++i) {
        s[c][i] = __builtin_fmaf(kv[i], one, dv[i] * (fresh ? 0.0f : s[c][i]));
        out[c] = __builtin_fmaf(s[c][i], qv[i], out[c]);
      }
      if (col0 + c < a.vdim)
#pragma unroll
        for (int i = 0; i < DPL; ++i) a.state[((int64_t)head * a.vdim + col0 + c) * dimp + i * 64 + lane] = s[c][i];
    }
    ended_sums(out, lane);
    const int c = lane / (64 / kCols);
    if (lane % (64 / kCols) == 0 && col0 + c < a.vdim) row[col0 + c] = out[0];
  }
  __syncthreads();
  float sq = 0.0f;
  for (int c = tid; c < a.vdim; c += blockDim.x) sq = __builtin_fmaf(row[c], row[c], sq);
  sq = lanes::sum(sq);
  if (lane == 0) sums[wave] = sq;
  __syncthreads();
  const float all = lanes::sum<16>((lane & 15) < waves ? sums[lane & 15] : 0.0f);
  const float inv = 1.0f / sqrtf(all / (float)a.vdim + a.eps);
  T* ctx = reinterpret_cast<T*>(a.ctx) + (int64_t)head * a.vdim;
  for (int c = tid; c < a.vdim; c += blockDim.x) {
    if (c != tid) norm = a.norm[c], z = a.gate ? (float)gate[c] : 0.0f;
    float y = row[c] * inv * norm;
    if (a.gate) y *= z / (1.0f + expf(-z));
    ctx[c] = (T)y;
  }
}

template <typename T, int DPL, bool HEAD>
__global__ __launch_bounds__(256) void gated_few_kernel(GatedStateArgs a) {
  constexpr int kCols = few_cols<DPL>(), J = 16 / kCols;  // J tokens a step
  constexpr int G = few_tokens<DPL>(), D = DPL * 64, N = G * DPL / 4;  // N pieces of 64 channels of a token per wavefront
  __shared__ float qs[G * D], ks[G * D], ds[HEAD ? 1 : G * D];
  const int head = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col0 = (blockIdx.y * 4 + wave) * kCols, nc = min(kCols, a.vdim - col0);
  const T* const q = reinterpret_cast<const T*>(a.q) + (int64_t)head * a.dim;
  const bool keys = HEAD || a.k != nullptr, fresh = a.pos.position() == 0;
  const T* const k = keys ? reinterpret_cast<const T*>(a.k) + (int64_t)head * a.dim : q;
  const T* const v = reinterpret_cast<const T*>(a.v) + (int64_t)head * a.vdim;
  const float* const g = HEAD ? a.head_decay : a.g + (int64_t)head * a.dim;
  const float of_head = HEAD ? a.head_decay[head] : 0.0f;
  float* const o = a.o + (int64_t)head * a.vdim + col0;
  const int64_t ldo = (int64_t)a.heads * a.vdim;
  float* const state = a.state + ((int64_t)head * a.vdim + col0) * D;
  float s[kCols][DPL];
#pragma unroll
  for (int c = 0; c < kCols; ++c)
#pragma unroll
    for (int i = 0; i < DPL; ++i) s[c][i] = fresh || c >= nc ? 0.0f : state[c * D + i * 64 + lane];
  for (int64_t t0 = 0; t0 < a.M; t0 += G) {
    const int n = (int)min((int64_t)G, a.M - t0);
    T qr[N], kr[N], vr;
    float gr[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {  // (behind the last token and channel: read again, not kept)
      const int piece = i * 4 + wave, d = min(piece % DPL * 64 + lane, a.dim - 1);
      const int64_t t = t0 + min(piece / DPL, n - 1);
      qr[i] = q[t * a.ldp + d];
      kr[i] = k[t * a.ldp + d];
      if constexpr (!HEAD) gr[i] = g[t * a.ldg + d];
    }
    // lane kCols t + c: column c of token t
    vr = v[(t0 + min(lane / kCols, n - 1)) * a.ldp + min(col0 + lane % kCols, a.vdim - 1)];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int piece = i * 4 + wave, at = piece * 64 + lane;
      const bool there = piece % DPL * 64 + lane < a.dim;
      float decay = 0.0f, key;
      if constexpr (HEAD) key = (float)kr[i];
      else decay_and_key(gr[i], keys, (float)kr[i], decay, key);
      qs[at] = there ? (float)qr[i] * a.q_scale : 0.0f;
      ks[at] = there ? key : 0.0f;
      if constexpr (!HEAD) ds[at] = there ? decay : 0.0f;
    }
    __syncthreads();
    const float value = lane % kCols < nc ? (float)vr : 0.0f;
    for (int tj = 0; tj < n; tj += J) {
      float qv[J][DPL], kv[J][DPL], dv[J][DPL], out[16];
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int i = 0; i < DPL; ++i) {
          const int at = (tj + j) * D + i * 64 + lane;
          qv[j][i] = qs[at];
          kv[j][i] = ks[at];
          dv[j][i] = HEAD ? of_head : ds[at];
        }
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int c = 0; c < kCols; ++c) {
          float& sum = out[j * kCols + c];
          sum = 0.0f;
          if (tj + j >= n) continue;
          const float vv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(value), (tj + j) * kCols + c));
#pragma unroll
          for (int i = 0; i < DPL; ++i) {
            s[c][i] = __builtin_fmaf(kv[j][i], vv, dv[j][i] * s[c][i]);
            sum = __builtin_fmaf(s[c][i], qv[j][i], sum);
          }
        }
      sixteen_sums(out, lane);
      const int t = tj + (lane >> 2) / kCols, c = (lane >> 2) % kCols;
      if ((lane & 3) == 0 && t < n && c < nc) o[(t0 + t) * ldo + c] = out[0];
    }
    if (t0 + G < a.M) __syncthreads();  // the group is read
  }
#pragma unroll
  for (int c = 0; c < kCols; ++c)
    if (c < nc)
#pragma unroll
      for (int i = 0; i < DPL; ++i) state[c * D + i * 64 + lane] = s[c][i];
}

// Many tokens on the binary32 matrix instruction (v_mfma_f32_16x16x4_f32), C tokens (a chunk) after the other in blocks
// of 16.  Inside a block, with L_t the sum of the logarithms of the decays up to and with token t (a number per
// channel), T that of all 16, S the state ahead of the block and
//     Q_t = q_t 2^(L_t - T/2),   K_s = k_s 2^(T/2 - L_s),   R = 2^(T/2) S,
// the outputs and the state behind the block are
//     o_t = R^T Q_t + sum over s <= t of (Q_t . K_s) v_s,   S <- 2^(T/2) (R + sum over s of K_s v_s^T).
// A workgroup takes 16 columns of one head's state.  Wavefronts 4 .. 7 form a chunk's Q, K and 2^(T/2) in LDS (two channels
// and eight tokens a thread) and add up and store the outputs of the chunk before the running one, while wavefronts 0 .. 3
// go through the running one: wavefront w holds the D / 4 rows from w D / 4 on of the state in its accumulators and takes
// them for both sums over channels as well, so that nothing passes between wavefronts inside a chunk.
// Operands, lane (n, j) = (lane % 16, lane / 16), step i: an accumulator holds rows 4 j + i of column n, and used as an
// operand it is just that for an order of the summed index of 4 j + i.
//     A^T[s][t] = K Q^T,  O^T[c][t] = R^T Q^T + V^T (A^T, s <= t),  R[d][c] += K^T V
// HEAD: one decay per head (linear attention in binary32).  Its powers are factors of whole sums then,
//     o_t = decay^(t+1) S^T q_t + sum over s <= t of decay^(t-s) (q_t . k_s) v_s,
//     S <- decay^n S + sum over s < n of k_s decay^(n-1-s) v_s    (n tokens in the block),
// rounded once from 64 bits; the state's, which every block meets again, is a sum of two numbers.  333 tokens, 8 heads of 128:
// 23 us, a token after the other 395; outputs 7.8e-8 off, by the recurrence 8.4e-8 (exponentials of the logarithm as factors
// of q and k: 29 us, 1.8e-7).
// Where a channel of a block decays by more than 2^-kSafe the factors could leave the range of binary32: such a block goes
// token by token, in the same accumulators.  So does a block with a value that is infinite or NaN, which the weights of zero
// that stand for s > t would bring to the tokens ahead of it.
constexpr int kBlock = 16;
constexpr float kSafe = 200.0f;
constexpr int kValueStride = 20;

template <typename T>
struct Pair {
  typedef T type __attribute__((ext_vector_type(2)));
};
typedef float f32x2_t __attribute__((ext_vector_type(2)));

template <int D>
constexpr int chunk_blocks() { return 256 / D; }
template <int D>
constexpr int chunk_lds() {
  constexpr int B = chunk_blocks<D>(), C = B * kBlock;
  return 2 * (2 * C * (D + 4) + C * kValueStride + B * D + 4 * B * 256) * 4;
}

// EVEN: dim is even, two channels make one load; keys: there are keys beside the decays.
// Where heads and columns leave compute units without a workgroup, a pass is cut into segments (a.seg_tokens, blockIdx.z) that go side by
// side, in two launches.  AHEAD: for every segment but the last the state that it adds to an empty one and what it leaves of
// a row of the state ahead of it; the first starts from the state itself and keeps a copy.  Then the outputs, every segment starting from
// those sums, and the last one's state.  The workspace holds
//     [segments][heads][vdim][dimp]: the state ahead of the pass, then what the segments but the last add,
//     [segments - 1][heads][dimp]: the root of what is left of a row (not HEAD).
// (MODE 0: a pass in one piece, 1: AHEAD, 2: outputs of segments.  One piece without the segments' arguments in the way: 16 tokens, 8 heads of 128
// 4.88 us, with them 5.10, 4 heads of 256 4.94 and 5.19.)
template <typename T, int D, bool EVEN, bool keys, bool HEAD, int MODE>
__global__ __launch_bounds__(512) void gated_chunk_kernel(GatedStateArgs a) {
  constexpr bool AHEAD = MODE == 1, SEGMENTS = MODE != 0;
  static_assert(keys || !HEAD, "a head's decay leaves no keys");
  constexpr int B = chunk_blocks<D>(), C = B * kBlock, S4 = D + 4, VS = kValueStride;
  constexpr int NT = D / 64;                  // tiles of 16 state rows per wavefront
  constexpr int kHalf = kBlock / 2;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* const qs2 = lds;                     // [2][C][S4]
  float* const ks2 = qs2 + 2 * C * S4;        // [2][C][S4]
  float* const vs2 = ks2 + 2 * C * S4;        // [2][C][VS]
  float* const ts2 = vs2 + 2 * C * VS;        // [2][B][D]: 2^(T/2)
  float* const red2 = ts2 + 2 * B * D;        // [2][4][B][256]
  __shared__ int unsafe[3][B];                // of the running chunk, the one being formed, and one to be cleared
  const int head = blockIdx.x, c0 = blockIdx.y * 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int segment = SEGMENTS ? blockIdx.z : 0;
  const int64_t tok0 = SEGMENTS ? (int64_t)segment * a.seg_tokens : 0;
  const int M = (int)(SEGMENTS ? min((int64_t)a.seg_tokens, a.M - tok0) : a.M);  // tokens of this segment, counted from tok0
  const int nv = min(16, a.vdim - c0), chunks = (M + C - 1) / C;
  const T* const q = reinterpret_cast<const T*>(a.q) + tok0 * a.ldp + (int64_t)head * a.dim;
  const T* const k = keys ? reinterpret_cast<const T*>(a.k) + tok0 * a.ldp + (int64_t)head * a.dim : q;
  const T* const v = reinterpret_cast<const T*>(a.v) + tok0 * a.ldp + (int64_t)head * a.vdim + c0;
  const float* const g = HEAD ? a.head_decay : a.g + tok0 * a.ldg + (int64_t)head * a.dim;
  const float of_head = HEAD ? a.head_decay[head] : 0.0f;
  __shared__ float power[HEAD ? kBlock + 1 : 1], power_rest[HEAD ? kBlock + 1 : 1];  // of the decay: their sum is the n-th
  if constexpr (HEAD) {
    if (tid <= kBlock) {
      double x = 1.0;
      for (int i = 0; i < tid; ++i) x *= (double)of_head;
      power[tid] = (float)x;
      power_rest[tid] = (float)(x - (double)(float)x);
    }
  }
  if (tid < 3 * B) unsafe[tid / B][tid % B] = 0;
  __syncthreads();

  if (wave >= 4) {
    const int p = tid - 256;
    const int pair = (p >> 6) * 32 + (lane & 31), half = lane >> 5;
    const int d = (pair % (D / 2)) * 2, blk = pair / (D / 2);
    const bool has[2] = {d < a.dim, d + 1 < a.dim};
    const int dc = has[0] ? d : 0, t0 = blk * kBlock + half * kHalf;  // this thread's tokens of a chunk
    T vr[B];
    f32x2_t gr[kHalf];
    typename Pair<T>::type qr[kHalf], kr[kHalf];
    auto two = [&](const auto* x) __attribute__((always_inline)) {
      typedef typename Pair<std::remove_cv_t<std::remove_reference_t<decltype(*x)>>>::type P;
      if constexpr (EVEN) return *reinterpret_cast<const P*>(x);
      else return P{x[0], x[has[1] ? 1 : 0]};
    };
    auto load = [&](int chunk) __attribute__((always_inline)) {
      const int at = chunk * C;
#pragma unroll
      for (int t = 0; t < kHalf; ++t) {
        const int64_t tok = min(at + t0 + t, M - 1);
        if constexpr (!HEAD) gr[t] = two(g + tok * a.ldg + dc);
        if constexpr (!AHEAD) qr[t] = two(q + tok * a.ldp + dc);
        if constexpr (keys) kr[t] = two(k + tok * a.ldp + dc);
      }
#pragma unroll
      for (int i = 0; i < B; ++i) vr[i] = v[(int64_t)min(at + i * 16 + (p >> 4), M - 1) * a.ldp + min(p & 15, nv - 1)];
    };
    auto form = [&](int chunk) __attribute__((always_inline)) {
      const int at = chunk * C + t0, par = chunk & 1;
      float* const qs = qs2 + (par * C + t0) * S4 + d;
      float* const ks = ks2 + (par * C + t0) * S4 + d;
      auto values = [&]() __attribute__((always_inline)) {  // (behind the last token and column: they meet keys of zero, or are not stored)
#pragma unroll
        for (int i = 0; i < B; ++i) {
          const float x = (float)vr[i];
          vs2[(par * C + i * 16 + (p >> 4)) * VS + (p & 15)] = x;
          if (!(fabsf(x) < INFINITY)) unsafe[chunk % 3][i] = 1;
        }
      };
      if constexpr (HEAD) {
#pragma unroll
        for (int t = 0; t < kHalf; ++t) {
          f32x2_t qv, kv;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const bool there = has[e] && at + t < M;
            if constexpr (!AHEAD) qv[e] = there ? (float)qr[t][e] * a.q_scale : 0.0f;
            kv[e] = there ? (float)kr[t][e] : 0.0f;
          }
          if constexpr (!AHEAD) *reinterpret_cast<f32x2_t*>(qs + t * S4) = qv;
          *reinterpret_cast<f32x2_t*>(ks + t * S4) = kv;
        }
        values();
        return;
      }
      f32x2_t L[kHalf];
      float sum[2] = {0.0f, 0.0f};
#pragma unroll
      for (int t = 0; t < kHalf; ++t)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float x = has[e] && at + t < M ? gr[t][e] : 0.0f;
          gr[t][e] = x;
          // (a decay of zero: nothing of binary32 is left behind 2^-150)
          sum[e] += fmaxf(keys ? x : __builtin_amdgcn_logf(1.0f - x), -150.0f);
          L[t][e] = sum[e];
        }
      f32x2_t mid, ahead;  // T / 2, and what the block's first half adds to the second
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float other = __shfl_xor(sum[e], 32, 64);
        mid[e] = 0.5f * (sum[e] + other);
        ahead[e] = half ? other : 0.0f;
      }
      if (half == 0 && fminf(mid[0], mid[1]) < -0.5f * kSafe) unsafe[chunk % 3][blk] = 1;
#pragma unroll
      for (int t = 0; t < kHalf; ++t) {
        f32x2_t qv, kv;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const bool there = has[e] && at + t < M;
          const float x = L[t][e] + ahead[e] - mid[e];
          if constexpr (!AHEAD) qv[e] = (there ? (float)qr[t][e] * a.q_scale : 0.0f) * __builtin_amdgcn_exp2f(x);
          kv[e] = (keys ? (there ? (float)kr[t][e] : 0.0f) : gr[t][e]) * __builtin_amdgcn_exp2f(-x);
        }
        if constexpr (!AHEAD) *reinterpret_cast<f32x2_t*>(qs + t * S4) = qv;
        *reinterpret_cast<f32x2_t*>(ks + t * S4) = kv;
      }
      if (half == 0)
        *reinterpret_cast<f32x2_t*>(ts2 + (par * B + blk) * D + d) =
            f32x2_t{__builtin_amdgcn_exp2f(mid[0]), __builtin_amdgcn_exp2f(mid[1])};
      values();
    };
    auto store = [&](int chunk) __attribute__((always_inline)) {
      if (p >= C * 4) return;
      const int t = p >> 2, c = (p & 3) * 4;  // four columns of a token
      const float* const red = red2 + (chunk & 1) * 4 * B * 256 + t * 16 + c;
      f32x4_t sum = *reinterpret_cast<const f32x4_t*>(red);
#pragma unroll
      for (int w = 1; w < 4; ++w) sum = sum + *reinterpret_cast<const f32x4_t*>(red + w * B * 256);
      if (chunk * C + t >= M) return;
      float* const out = a.o + ((tok0 + chunk * C + t) * a.heads + head) * a.vdim + c0 + c;
      if (c + 3 < nv && (a.vdim & 3) == 0) {
        *reinterpret_cast<f32x4_t*>(out) = sum;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < nv) out[e] = sum[e];
      }
    };
    load(0);
    form(0);
    if (chunks > 1) load(1);
    __syncthreads();
    for (int i = 0; i < chunks; ++i) {
      if (p < B) unsafe[(i + 2) % 3][p] = 0;
      if (i + 1 < chunks) form(i + 1);
      if (i + 2 < chunks) load(i + 2);
      if (!AHEAD && i > 0) store(i - 1);
      __syncthreads();
    }
    if constexpr (!AHEAD) store(chunks - 1);
    return;
  }

  const int n = lane & 15, j4 = (lane >> 4) * 4;
  const int dimp = (a.dim + 63) & ~63;
  const int row0 = wave * (D / 4);        // this wavefront's rows of the state
  const int64_t column = ((int64_t)head * a.vdim + c0 + n) * dimp, states = (int64_t)a.heads * a.vdim * dimp;
  float* const state = a.state + column;
  f32x4_t s[NT];                          // s[i]: rows row0 + 16 i + j4 .. + 3 of column n
  f32x4_t left[NT];                       // AHEAD, not HEAD: the root of the product of the decays
  const double over = HEAD && MODE == 2 && segment > 1 ? segment_power(of_head, a.seg_tokens) : 0.0;
  const bool fresh = a.pos.position() == 0;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int d = row0 + 16 * i + j4;
    const bool there = d < dimp && n < nv;
    s[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    left[i] = f32x4_t{1.0f, 1.0f, 1.0f, 1.0f};
    if constexpr (MODE != 2) {
      if (!fresh && there && segment == 0) s[i] = *reinterpret_cast<const f32x4_t*>(state + d);
      if (AHEAD && segment == 0 && there) *reinterpret_cast<f32x4_t*>(a.workspace + column + d) = s[i];
    } else if (there) {
      const float* const from = a.workspace + column + d;
      s[i] = *reinterpret_cast<const f32x4_t*>(from + (segment == 0 ? 0 : states));
      for (int j = 2; j <= segment; ++j) {
        const f32x4_t add = *reinterpret_cast<const f32x4_t*>(from + j * states);
        if constexpr (HEAD) {
#pragma unroll
          for (int e = 0; e < 4; ++e) s[i][e] = behind_segment(s[i][e], over, add[e]);
          continue;
        }
        const f32x4_t f =
            *reinterpret_cast<const f32x4_t*>(a.workspace + (int64_t)gridDim.z * states + ((int64_t)(j - 1) * a.heads + head) * dimp + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[i][e] = behind_segment(s[i][e], of_root(f[e]), add[e]);
      }
    }
  }
  // HEAD: a power that is no number, or leaves the range where a product with it is as exact as others, is not used; nor is any
  // for a state that is not finite (the power's second number may be 0)
  bool whole = !HEAD || (power[kBlock] > 0x1p-100f && power[kBlock] < 0x1p100f);
  if constexpr (HEAD) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) whole = whole && fabsf(s[i][e]) < INFINITY;
    whole = __all(whole);
  }
  float state_power = 0.0f, state_power_rest = 0.0f, out_power = 0.0f, out_power_rest = 0.0f, back[4] = {}, to_end[4] = {};
  if constexpr (HEAD) {
    state_power = power[kBlock], state_power_rest = power_rest[kBlock];
    out_power = power[n + 1], out_power_rest = power_rest[n + 1];
#pragma unroll
    for (int i = 0; i < 4; ++i) back[i] = power[max(n - j4 - i, 0)], to_end[i] = power[kBlock - 1 - j4 - i];
  }
  __syncthreads();
  for (int chunk = 0; chunk < chunks; ++chunk) {
    const int par = chunk & 1;
    const float* const qs = qs2 + par * C * S4;
    const float* const ks = ks2 + par * C * S4;
    const float* const vs = vs2 + par * C * VS;
    const float* const ts = ts2 + par * B * D;
    float* const red = red2 + par * 4 * B * 256;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      f32x4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
      float vv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) vv[i] = vs[(b * kBlock + j4 + i) * VS + n];
      if (unsafe[chunk % 3][b] == 0 && whole) {
        if constexpr (HEAD) {
          const int here = min(kBlock, M - chunk * C - b * kBlock);  // tokens of the block
          if (here > 0) {
            f32x4_t w[2 * NT], ot[2 * NT];  // an accumulator per 8 rows: the sums over rows are short chains, added in pairs
#pragma unroll
            for (int i = 0; i < 2 * NT; ++i) w[i] = ot[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < NT; ++i) {
              const f32x4_t qv = *reinterpret_cast<const f32x4_t*>(qs + (b * kBlock + n) * S4 + row0 + 16 * i + j4);
              const f32x4_t kv = *reinterpret_cast<const f32x4_t*>(ks + (b * kBlock + n) * S4 + row0 + 16 * i + j4);
#pragma unroll
              for (int e = 0; e < 4 && !AHEAD; ++e) {
                const int j = 2 * i + (e & 1);
                w[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[e], qv[e], w[j], 0, 0, 0);
                ot[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[i][e], qv[e], ot[j], 0, 0, 0);
              }
            }
            float f = state_power, f_rest = state_power_rest, later[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) later[e] = to_end[e] * vv[e];
            if (here < kBlock) {  // the last block
              f = power[here];
              f_rest = power_rest[here];
#pragma unroll
              for (int e = 0; e < 4; ++e) later[e] = j4 + e < here ? power[max(here - 1 - j4 - e, 0)] * vv[e] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < NT; ++i) {
#pragma unroll
              for (int e = 0; e < 4; ++e) s[i][e] = __builtin_fmaf(s[i][e], f, s[i][e] * f_rest);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ks[(b * kBlock + j4 + e) * S4 + row0 + 16 * i + n], later[e], s[i], 0, 0, 0);
            }
            if constexpr (!AHEAD) {
#pragma unroll
              for (int half = NT; half > 0; half >>= 1)
#pragma unroll
                for (int i = 0; i < half; ++i) w[i] = w[i] + w[i + half], ot[i] = ot[i] + ot[i + half];
              // w[0][i]: key token j4 + i, query token n
#pragma unroll
              for (int i = 0; i < 4; ++i) o[i] = __builtin_fmaf(ot[0][i], out_power, ot[0][i] * out_power_rest);
#pragma unroll
              for (int i = 0; i < 4; ++i) o = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[i], j4 + i <= n ? w[0][i] * back[i] : 0.0f, o, 0, 0, 0);
            }
          }
        } else {
          f32x4_t w = {0.0f, 0.0f, 0.0f, 0.0f}, f[NT];
#pragma unroll
          for (int i = 0; i < NT; ++i) {
            f[i] = *reinterpret_cast<const f32x4_t*>(ts + b * D + row0 + 16 * i + j4);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[i][e] *= f[i][e];
            if constexpr (AHEAD) {
#pragma unroll
              for (int e = 0; e < 4; ++e) left[i][e] = times_decay(left[i][e], f[i][e], 0x1p-126f);
              continue;
            }
            const f32x4_t qv = *reinterpret_cast<const f32x4_t*>(qs + (b * kBlock + n) * S4 + row0 + 16 * i + j4);
            const f32x4_t kv = *reinterpret_cast<const f32x4_t*>(ks + (b * kBlock + n) * S4 + row0 + 16 * i + j4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              w = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[e], qv[e], w, 0, 0, 0);
              o = __builtin_amdgcn_mfma_f32_16x16x4f32(s[i][e], qv[e], o, 0, 0, 0);
            }
          }
#pragma unroll
          for (int i = 0; i < NT; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ks[(b * kBlock + j4 + e) * S4 + row0 + 16 * i + n], vv[e], s[i], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[i][e] *= f[i][e];
          }
          // w[i]: key token j4 + i, query token n
#pragma unroll
          for (int i = 0; i < 4 && !AHEAD; ++i) o = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[i], j4 + i <= n ? w[i] : 0.0f, o, 0, 0, 0);
        }
      } else {
        if constexpr (HEAD) whole = false;
        constexpr bool kLeft = AHEAD && !HEAD;
        double product[kLeft ? 4 * NT : 1];  // of the block's decays
        if constexpr (kLeft)
#pragma unroll
          for (int i = 0; i < 4 * NT; ++i) product[i] = 1.0;
        for (int t = 0; t < kBlock && chunk * C + b * kBlock + t < M; ++t) {
          const int64_t tok = chunk * C + b * kBlock + t;
          const float value = vs[(b * kBlock + t) * VS + n];
          float out = 0.0f;
#pragma unroll
          for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int r = row0 + 16 * i + j4 + e;
              if (r >= a.dim) continue;
              float decay = of_head, key;
              if constexpr (HEAD) key = (float)k[tok * a.ldp + r];
              else decay_and_key(g[tok * a.ldg + r], keys, keys ? (float)k[tok * a.ldp + r] : 0.0f, decay, key);
              s[i][e] = __builtin_fmaf(key, value, decay * s[i][e]);
              if constexpr (kLeft) product[4 * i + e] = times_decay(product[4 * i + e], (double)decay, 0x1p-252);
              out = __builtin_fmaf(s[i][e], (float)q[tok * a.ldp + r] * a.q_scale, out);
            }
          out += __shfl_xor(out, 16, 64);
          out += __shfl_xor(out, 32, 64);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = __shfl(out, j4 + i, 64);
            if (n == t) o[i] = x;
          }
        }
        if constexpr (kLeft)
#pragma unroll
          for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const double x = product[4 * i + e];
              left[i][e] = times_decay(left[i][e], (float)__builtin_copysign(sqrt(__builtin_fabs(x)), x), 0x1p-126f);
            }
      }
      if constexpr (!AHEAD) *reinterpret_cast<f32x4_t*>(red + (wave * B + b) * 256 + n * 16 + j4) = o;
    }
    __syncthreads();
  }
  if (MODE == 2 && segment != (int)gridDim.z - 1) return;
  if (n < nv)
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int d = row0 + 16 * i + j4;
      if (d < dimp) *reinterpret_cast<f32x4_t*>(AHEAD ? a.workspace + (segment + 1) * states + column + d : state + d) = s[i];
    }
  if (AHEAD && !HEAD && n == 0 && c0 == 0)
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int d = row0 + 16 * i + j4;
      if (d < dimp)
        *reinterpret_cast<f32x4_t*>(a.workspace + (int64_t)(gridDim.z + 1) * states + ((int64_t)segment * a.heads + head) * dimp + d) = left[i];
    }
}

// Segments of a pass: as many as have a compute unit for each workgroup (a workgroup's LDS leaves no place for a second), where they pay: a
// chunk of the launch ahead takes about 0.8 of one of outputs, and a launch more with the states between as long as three.
// Heads of 128: 10 heads, 1,800 tokens (57 chunks, 3 segments) 144 -> 32 + 54 us; 16 heads, 700 tokens (22 chunks, 2 segments)
// as long as in one.
constexpr int kMaxSegments = 16;
int segment_tokens(const GatedStateArgs& a, int chunk) {
  const int64_t blocks = (int64_t)a.heads * ((a.vdim + 15) / 16), chunks = (a.M + chunk - 1) / chunk;
  int64_t n = std::min<int64_t>(std::min<int64_t>(256 / blocks, kMaxSegments), chunks);
  const int64_t floats = (int64_t)a.heads * (a.vdim + 1) * round_up(a.dim, 64);  // of a segment
  if (a.workspace) n = std::min(n, a.workspace_floats / floats);
  if (!a.workspace || n < 2) return 0;
  const int64_t of_one = (chunks + n - 1) / n;
  return 10 * chunks > 18 * of_one + 30 ? (int)of_one * chunk : 0;
}

template <typename T, int D, bool EVEN, bool KEYS, bool HEAD, int MODE>
int launch_chunk_kernel(const GatedStateArgs& a, unsigned segments, hipStream_t st) {
  static bool raised = false;  // more LDS than the default limit of a launch
  if (!raised) {
    AWQ_HIP_TRY(hipFuncSetAttribute((const void*)gated_chunk_kernel<T, D, EVEN, KEYS, HEAD, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    chunk_lds<D>()));
    raised = true;
  }
  const dim3 g((unsigned)a.heads, (unsigned)((a.vdim + 15) / 16), segments);
  hipLaunchKernelGGL((gated_chunk_kernel<T, D, EVEN, KEYS, HEAD, MODE>), g, dim3(512), chunk_lds<D>(), st, a);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

template <typename T, int D, bool EVEN, bool KEYS, bool HEAD = false>
int launch_chunk_form(const GatedStateArgs& u, hipStream_t st) {
  if constexpr (EVEN) {
    GatedStateArgs a = u;
    a.seg_tokens = segment_tokens(a, chunk_blocks<D>() * kBlock);
    if (a.seg_tokens) {
      const unsigned ahead = (unsigned)((a.M - 1) / a.seg_tokens);
      if (int rc = launch_chunk_kernel<T, D, EVEN, KEYS, HEAD, 1>(a, ahead, st)) return rc;
      return launch_chunk_kernel<T, D, EVEN, KEYS, HEAD, 2>(a, ahead + 1, st);
    }
  }
  return launch_chunk_kernel<T, D, EVEN, KEYS, HEAD, 0>(u, 1, st);
}
template <typename T, int D>
int launch_chunks(const GatedStateArgs& a, hipStream_t st) {
  const uintptr_t parts = (uintptr_t)a.q | (uintptr_t)a.k;  // two values of T, two floats
  const bool even = a.dim % 2 == 0 && a.ldp % 2 == 0 && a.ldg % 2 == 0 && parts % (2 * sizeof(T)) == 0 && (uintptr_t)a.g % 8 == 0;
  if constexpr (sizeof(T) == 4)
    if (a.head_decay) return even ? launch_chunk_form<T, D, true, true, true>(a, st) : launch_chunk_form<T, D, false, true, true>(a, st);
  if (a.k) return even ? launch_chunk_form<T, D, true, true>(a, st) : launch_chunk_form<T, D, false, true>(a, st);
  return even ? launch_chunk_form<T, D, true, false>(a, st) : launch_chunk_form<T, D, false, false>(a, st);
}

template <typename T, int DPL>
void launch_steps(const GatedStateArgs& a, hipStream_t st) {
  constexpr int kHeadCols = DPL <= 4 ? 8 : 4, kCols = 4;
  const auto groups = [&](int cols) { return dim3((unsigned)a.heads, (unsigned)((a.vdim + 4 * cols - 1) / (4 * cols))); };
  if (a.ctx)
    hipLaunchKernelGGL((gated_head_kernel<T, DPL, kHeadCols>), dim3((unsigned)a.heads),
                       dim3((unsigned)std::min<int64_t>(1024, (a.vdim + kHeadCols - 1) / kHeadCols * 64)), (size_t)a.vdim * 4, st, a);
  else if (a.head_decay)
    hipLaunchKernelGGL((gated_few_kernel<T, DPL, true>), groups(few_cols<DPL>()), dim3(256), 0, st, a);
  else if (a.M == 1)
    hipLaunchKernelGGL((gated_step_kernel<T, DPL, kCols>), groups(kCols), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((gated_few_kernel<T, DPL, false>), groups(few_cols<DPL>()), dim3(256), 0, st, a);
}

template <typename T>
int launch_any_steps(const GatedStateArgs& a, hipStream_t st) {
  switch ((a.dim + 63) / 64) {
    case 1: launch_steps<T, 1>(a, st); break;
    case 2: launch_steps<T, 2>(a, st); break;
    case 3: launch_steps<T, 3>(a, st); break;
    case 4: launch_steps<T, 4>(a, st); break;
    case 5: launch_steps<T, 5>(a, st); break;
    case 6: launch_steps<T, 6>(a, st); break;
    case 7: launch_steps<T, 7>(a, st); break;
    default: launch_steps<T, 8>(a, st); break;
  }
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

// Tokens from which on a chunk is used, 5.0 us for one.  Its factors are exponentials of sums of logarithms, further off than the
// decays themselves: without keys the state behind 9 tokens 1.2e-7, token by token 4.7e-8.
constexpr int kChunkFrom = 16;

template <typename T>
int launch(const GatedStateArgs& a, hipStream_t st) {
  if (a.M < kChunkFrom || a.dim > 256) return launch_any_steps<T>(a, st);
  if (a.dim <= 64) return launch_chunks<T, 64>(a, st);
  return a.dim <= 128 ? launch_chunks<T, 128>(a, st) : launch_chunks<T, 256>(a, st);
}

// linear attention's arguments, but for the decay
template <typename T>
GatedStateArgs of_linear(const LinearAttnArgs& u) {
  const T* p = reinterpret_cast<const T*>(u.proj);
  const int64_t keys = (int64_t)u.heads * u.dim;
  GatedStateArgs a;
  a.q = p;
  a.k = p + keys;
  a.v = p + 2 * keys;
  a.ldp = u.ldp;
  a.heads = u.heads;
  a.dim = u.dim;
  a.vdim = u.vdim;
  a.state = u.state;
  a.o = u.o;
  a.M = u.M;
  a.pos = u.pos;
  a.workspace = u.workspace;
  a.workspace_floats = u.workspace_floats;
  return a;
}

}  // namespace

int launch_linear_few(const LinearAttnArgs& u, bool f32, hipStream_t st) {
  GatedStateArgs a = f32 ? of_linear<float>(u) : of_linear<bf16_t>(u);
  a.head_decay = u.decay;
  return f32 ? launch_any_steps<float>(a, st) : launch_any_steps<bf16_t>(a, st);
}

int launch_linear_chunks_f32(const LinearAttnArgs& u, hipStream_t st) {
  GatedStateArgs a = of_linear<float>(u);
  a.head_decay = u.decay;
  if (a.dim <= 64) return launch_chunks<float, 64>(a, st);
  return a.dim <= 128 ? launch_chunks<float, 128>(a, st) : launch_chunks<float, 256>(a, st);
}

int launch_gated_state(const GatedStateArgs& a, bool f32, hipStream_t st) {
  AWQ_REQUIRE(a.q && a.v && a.g && a.state && (a.o || a.ctx) && a.M >= 1 && a.M < (1 << 30), "bad arguments");
  AWQ_REQUIRE(a.heads >= 1 && a.heads <= 65535 && a.dim >= 1 && a.dim <= 512 && a.vdim >= 1 && a.vdim <= 8192, "bad shape");
  AWQ_REQUIRE(!a.ctx || (a.M == 1 && a.norm), "the heads' norm in the launch is for one token");
  return f32 ? launch<float>(a, st) : launch<bf16_t>(a, st);
}
