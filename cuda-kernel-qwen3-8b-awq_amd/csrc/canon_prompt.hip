// Prompt positions together with the arithmetic of the one-token step, bit for bit (awq_prefill; Inference.cu:1304-1343
// runs them one after the other).  A token's products, norms and attention are those of gemv.hip, ops.hip and
// attention.hip; only the weights are read once for many tokens.
//
// Products.  A block's value is fma(-z, S, D) * (s * c) with D = sum q I an integer below 2^24 (awq_canon_math.h), so
// whatever forms D exactly keeps every bit.  The 16-bit integers I have at most 11 significant bits (they are rounded
// binary16 values over a power of two), so I is a binary16 number and so is a nibble, and one v_mfma_f32_16x16x32_f16
// forms D of 16 rows, 16 tokens and one block: its 32 products and all their partial sums are integers below 2^24.
// Where the zero-points are integers up to 16, q - z takes q's place: |sum (q - z) I| <= 16 * 32 * 32752 < 2^24, so the
// sum is what the fma returns and the fma is left out.  What remains per block value is a multiply by s * c and an
// addition in the order of awq_tree_sum: the vector pipes are what is busiest (two instructions per 32 weights and
// token, half of them the tree; 128 tokens of 12,288 x 4,096: 54 % of the time, the matrix pipes 18 %, on 192 workgroups for
// 256 compute units), not the matrix cores and not the weights' bytes.
//
// 36 layers of 4096 x 12288: 128 positions one after the other take 112 ms, together 6.4; 16 take 14 and 2.5.
#include <type_traits>

#include "gemv_device.hpp"

namespace {

typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// One block's fixed point for a value of it (awq_block_fixed): the exponent field of the block's largest magnitude
// gives c, 1 / c and the integer as a binary16 number.  A block that holds an infinity or a NaN: c a NaN, integers 0.
struct BlockScale {
  float c, inv;
  bool finite;
};
__device__ __forceinline__ BlockScale block_scale(uint32_t max_bits) {  // max of the magnitudes' bit patterns
  const uint32_t e = max_bits >> 10;
  const uint32_t cbits = (max(e, 1u) + 98u) << 23;
  return BlockScale{__builtin_bit_cast(float, e == 31u ? 0x7fc00000u : cbits), __builtin_bit_cast(float, 0x7f000000u - cbits), e != 31u};
}
__device__ __forceinline__ float block_int(half_t x, const BlockScale& b) {  // rounds to nearest even; zero is +0
  const float magic = 12582912.0f;
  const float i = __builtin_fmaf((float)x, b.inv, magic) - magic;
  return b.finite ? i : 0.0f;
}
// (x & mask) | bits in one instruction: the three-operand encoding takes no literals, so the mask travels in a scalar and the
// bits in a vector register
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t bits) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
  return r;
}
__device__ __forceinline__ float4_t add4(float4_t a, float4_t b) { return float4_t{a[0] + b[0], a[1] + b[1], a[2] + b[2], a[3] + b[3]}; }
__device__ __forceinline__ uint32_t magnitude(half_t v) { return __builtin_bit_cast(unsigned short, v) & 0x7fffu; }

}  // namespace

// Where the integers of token t, block b, element e lie: pieces of 1 KB per (16 tokens, block), the matrix instruction's
// operand -- lane (e / 8) * 16 + t % 16, element e % 8.
__device__ __forceinline__ int64_t canon_op_at(int64_t nblk, int tok, int64_t blk, int e) {
  return (((int64_t)(tok >> 4) * nblk + blk) * 64 + (e >> 3) * 16 + (tok & 15)) * 8 + (e & 7);
}
// ... and c and S of (t, b): [t / 16][b / 4][t % 16][b % 4]
__device__ __forceinline__ int64_t canon_scale_at(int64_t nblk, int tok, int64_t blk) {
  return (((int64_t)(tok >> 4) * (nblk >> 2) + (blk >> 2)) * 16 + (tok & 15)) * 4 + (blk & 3);
}

namespace {

// ---------------------------------------------------------------------------
// Product of up to 16 N tokens (blockIdx.y: which of them), 32 RS rows (blockIdx.x) and a run of KB = KS BW blocks
// (blockIdx.z), KS = 8 / RS.  Wavefront (rw, kw) multiplies rows 32 rw .. + 31 by blocks BW kw .. + BW - 1 of the run,
// a power of two of them that is a subtree of awq_tree_sum.  The tokens' operands pass through LDS, SB blocks of every
// kw at a time (two slabs, filled through registers a slab ahead), and serve RS wavefronts; a wavefront's weights are
// requested PD slabs ahead, four bytes per lane and block, and become operands once for all tokens.  The sum over
// blocks is a binary counter: pend[l] holds the finished left sibling of level l.
// ---------------------------------------------------------------------------
struct ProductParams {
  const uint32_t* wq;
  const half_t *scale, *zp;
  int32_t m, nblk, mg, kg;
  CanonTokens x;
  int32_t M, tiles;
  float* part;         // CANON_PARTS: [blockIdx.z][M][m]
  CanonTokens y;       // CANON_GELU: nblk = m / 32
  CanonQkv qkv;        // CANON_QKV
};

template <int N, int RS, int BW, bool ZI, int OUT>
__global__ __launch_bounds__(512, 2) void canon_product_kernel(ProductParams p) {
  constexpr int R = 2, KS = 8 / RS, KB = KS * BW, SB = RS == 4 || N <= 2 ? 4 : 2, NS = BW / SB, PD = NS < 4 ? NS : 4;
  constexpr int PIECES = KS * SB * N, NP = PIECES / 8;  // of 1 KB per slab, and per wavefront
  constexpr int LP = PD == 1 ? 0 : PD == 2 ? 1 : 2, LU = NS / PD == 1 ? 0 : NS / PD == 2 ? 1 : 2;  // levels within PD slabs, above
  static_assert(PD == 1 << LP && NS / PD == 1 << LU && PIECES % 8 == 0 && BW % SB == 0, "power-of-two runs");
  constexpr bool TOP_LDS = LU == 2 && N == 4;
  constexpr int kSlab = PIECES * 512;  // halves
  __shared__ __attribute__((aligned(16))) half_t xs[2][kSlab];
  __shared__ __attribute__((aligned(16))) float table[N * KB * 16];  // s * c, [n][block / 4][token][block % 4]
  __shared__ __attribute__((aligned(16))) float4_t top[TOP_LDS ? 8 * N * R * 64 : 1];
  static_assert(2 * kSlab * 2 >= 8 * N * R * 1024, "the sums' exchange takes the slabs' place");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave % KS, rw = wave / KS;
  const int g = lane >> 4, col = lane & 15;
  const int row0 = blockIdx.x * (32 * RS) + 32 * rw;  // this wavefront's first row
  const int tile0 = blockIdx.y * N;
  const int64_t blk0 = (int64_t)blockIdx.z * KB;

  // slab s of this wavefront's pieces: piece (kw', b, n) is block BW kw' + SB s + b of token tile n
  const u32x4* src[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int pc = wave * NP + i, n = pc % N, b = pc / N % SB, kk = pc / (N * SB);
    const int tile = min(tile0 + n, p.tiles - 1);  // (a tile past the last repeats it and is not stored)
    src[i] = reinterpret_cast<const u32x4*>(p.x.op) + ((int64_t)tile * p.nblk + blk0 + kk * BW + b) * 64 + lane;
  }
  u32x4 in[NP];
  auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) in[i] = src[i][s * (SB * 64)];
  };
  auto put = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NP; ++i) *reinterpret_cast<u32x4*>(&xs[s & 1][(wave * NP + i) * 512 + lane * 8]) = in[i];
  };
  const uint32_t* wp[R];
#pragma unroll
  for (int r = 0; r < R; ++r)
    wp[r] = p.wq + ((int64_t)(row0 / 16 + r) * p.nblk + blk0 + kw * BW) * 64 + col * 4 + g;
  uint32_t w[PD][SB][R];
  auto request = [&](int s, uint32_t (&dst)[SB][R]) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < SB; ++b)
#pragma unroll
      for (int r = 0; r < R; ++r) dst[b][r] = __builtin_nontemporal_load(wp[r] + (s * SB + b) * 64);
  };
  const int gi = ((row0 >> 7) % p.kg) % p.mg;
  const half_t sh = p.scale[gi], zh = p.zp[gi];
  fetch(0);
  // the table: 4 KB units of 64 blocks and 16 tokens
  constexpr int kTableUnits = N * KB * 4;  // of 16 bytes
  float4_t cs[(kTableUnits + 511) / 512];
#pragma unroll
  for (int i = 0; i < (kTableUnits + 511) / 512; ++i) {
    const int u = min(tid + i * 512, kTableUnits - 1), n = u / (KB * 4), at = u % (KB * 4);
    cs[i] = *reinterpret_cast<const float4_t*>(p.x.c + ((int64_t)min(tile0 + n, p.tiles - 1) * p.nblk + blk0) * 16 + at * 4);
  }
#pragma unroll
  for (int u = 0; u < PD; ++u) request(u, w[u]);
  put(0);
  const float s = (float)sh, zn = -(float)zh;
#pragma unroll
  for (int i = 0; i < (kTableUnits + 511) / 512; ++i)
    if (tid + i * 512 < kTableUnits) {
      const float4_t v = cs[i];
      *reinterpret_cast<float4_t*>(table + (tid + i * 512) * 4) = float4_t{s * v[0], s * v[1], s * v[2], s * v[3]};
    }
  if (NS > 1) fetch(1);
  __syncthreads();

  // q - z (ZI) or q of a dword's eight weights in element order: 1024 + q and 64 + q are one masked word each
  const half_t off_lo = ZI ? -((half_t)1024.0f + zh) : (half_t)-1024.0f, off_hi = ZI ? -((half_t)64.0f + zh) : (half_t)-64.0f;
  const half2_t lo2 = half2_t{off_lo, off_lo}, hi2 = half2_t{off_hi, off_hi};
  auto operand = [&](uint32_t v) __attribute__((always_inline)) {
    const uint32_t v8 = v >> 8;
    const half2_t a = as_half2(and_or(v, 0x000f000fu, 0x64006400u)) + lo2, b = as_half2(and_or(v, 0x00f000f0u, 0x54005400u)) + hi2;
    const half2_t c = as_half2(and_or(v8, 0x000f000fu, 0x64006400u)) + lo2, d = as_half2(and_or(v8, 0x00f000f0u, 0x54005400u)) + hi2;
    return half8_t{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
  };

  // pend[l]: the finished left sibling of level l; the levels within PD slabs are known when the loop is unrolled, of the
  // (at most two) above them the upper one lies in LDS where registers are short
  float4_t pend[LP + 1][N][R];
  float4_t(&cur)[N][R] = pend[LP];
  float4_t up[N][R], upper[TOP_LDS ? 1 : N][R];
  auto slabs = [&](int it, auto LAST) __attribute__((always_inline)) {
    constexpr bool last = decltype(LAST)::value;  // nothing of a further round is requested
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      const int sl = it * PD + u;
      if (!last || u + 1 < PD) put(sl + 1);
      if (!last || u + 2 < PD) fetch(sl + 2);
      half8_t wop[SB][R];
#pragma unroll
      for (int b = 0; b < SB; ++b)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          asm volatile("" : "+v"(w[u][b][r]));  // (the operands of later slabs would be formed, and held, early)
          wop[b][r] = operand(w[u][b][r]);
        }
      if (!last) request(sl + PD, w[u]);
      const half_t* const slab = &xs[sl & 1][kw * (SB * N * 512) + lane * 8];
      half8_t xo[2][SB];
#pragma unroll
      for (int b = 0; b < SB; ++b) xo[0][b] = *reinterpret_cast<const half8_t*>(slab + b * N * 512);
#pragma unroll
      for (int n = 0; n < N; ++n) {
        if (n + 1 < N)
#pragma unroll
          for (int b = 0; b < SB; ++b) xo[(n + 1) & 1][b] = *reinterpret_cast<const half8_t*>(slab + (b * N + n + 1) * 512);
        float sc[SB];
        const float* const t = table + ((n * KB + kw * BW + sl * SB) >> 2) * 64 + col * 4 + (SB == 2 ? (sl & 1) * 2 : 0);
        if constexpr (SB == 4) {
          const float4_t v = *reinterpret_cast<const float4_t*>(t);
#pragma unroll
          for (int b = 0; b < SB; ++b) sc[b] = v[b];
        } else {
          const float2_t v = *reinterpret_cast<const float2_t*>(t);
          sc[0] = v[0], sc[1] = v[1];
        }
        float S[SB];
        if constexpr (!ZI) {
          const float* const sp = p.x.s + canon_scale_at(p.nblk, min(tile0 + n, p.tiles - 1) * 16 + col, blk0 + kw * BW + sl * SB);
#pragma unroll
          for (int b = 0; b < SB; ++b) S[b] = sp[b];
        }
        float4_t v[SB][R];
#pragma unroll
        for (int b = 0; b < SB; ++b)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const float4_t D = __builtin_amdgcn_mfma_f32_16x16x32_f16(wop[b][r], xo[n & 1][b], float4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[b][r][i] = (ZI ? D[i] : __builtin_fmaf(zn, S[b], D[i])) * sc[b];
          }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float4_t t4;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if constexpr (SB == 4) t4[i] = (v[0][r][i] + v[1][r][i]) + (v[2][r][i] + v[3][r][i]);
            else t4[i] = v[0][r][i] + v[1][r][i];
            asm volatile("" : "+v"(t4[i]));  // (summed here, not where the pair is: products take four times the registers)
          }
          // a finished pair moves a level up
          bool open = true;
#pragma unroll
          for (int l = 0; l < LP; ++l)
            if (open) {
              if ((u >> l) & 1) t4 = add4(pend[l][n][r], t4);
              else pend[l][n][r] = t4, open = false;
            }
          if (open) cur[n][r] = t4;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
    }
    auto all = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < N; ++n)
#pragma unroll
        for (int r = 0; r < R; ++r) f(n, r);
    };
    if constexpr (LU > 0) {
      if ((it & 1) == 0) {
        all([&](int n, int r) { up[n][r] = cur[n][r]; });
      } else {
        all([&](int n, int r) { cur[n][r] = add4(up[n][r], cur[n][r]); });
        if constexpr (LU > 1) {
          auto at = [&](int n, int r) -> float4_t& {
            if constexpr (TOP_LDS) return top[((wave * N + n) * R + r) * 64 + lane];
            else return upper[n][r];
          };
          if (it == 1) all([&](int n, int r) { at(n, r) = cur[n][r]; });
          else all([&](int n, int r) { cur[n][r] = add4(at(n, r), cur[n][r]); });
        }
      }
    }
  };
#pragma unroll 1
  for (int it = 0; it < NS / PD - 1; ++it) slabs(it, std::false_type{});
  slabs(NS / PD - 1, std::true_type{});

  // the wavefronts of a row range exchange their subtrees' sums; wavefront kw finishes token tiles kw, kw + KS, ..
  float4_t* const red = reinterpret_cast<float4_t*>(&xs[0][0]);
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int r = 0; r < R; ++r) red[((wave * N + n) * R + r) * 64 + lane] = cur[n][r];
  __syncthreads();
  for (int n = kw; n < N; n += KS) {
    const int tok = (tile0 + n) * 16 + col;
    if (tile0 + n >= p.tiles) break;
    float4_t sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float4_t v[KS];
#pragma unroll
      for (int k = 0; k < KS; ++k) v[k] = red[(((rw * KS + k) * N + n) * R + r) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (KS == 2) sum[r][i] = v[0][i] + v[1][i];
        else sum[r][i] = (v[0][i] + v[1][i]) + (v[2][i] + v[3][i]);
      }
    }
    if constexpr (OUT == CANON_PARTS) {
      if (tok < p.M)
#pragma unroll
        for (int r = 0; r < R; ++r)
          *reinterpret_cast<float4_t*>(p.part + ((int64_t)blockIdx.z * p.M + tok) * p.m + row0 + 16 * r + 4 * g) = sum[r];
    } else if constexpr (OUT == CANON_GELU) {  // Inference.cu:271-279; the 32 rows are one block of the product that follows
      half_t h[R][4];
      uint32_t mm = 0;
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          h[r][i] = to_half_rn(awq_gelu_f32((float)(half_t)sum[r][i]));
          mm = max(mm, magnitude(h[r][i]));
        }
      mm = max(mm, (uint32_t)__shfl_xor((int)mm, 16, 64));
      mm = max(mm, (uint32_t)__shfl_xor((int)mm, 32, 64));
      const BlockScale bs = block_scale(mm);
      const int64_t blk = row0 >> 5;
      float S = 0.0f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        half4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = block_int(h[r][i], bs);
          S += f;
          v[i] = (half_t)f;
        }
        *reinterpret_cast<half4_t*>(p.y.op + canon_op_at(p.m >> 5, tok, blk, 16 * r + 4 * g)) = v;
      }
      S += __shfl_xor(S, 16, 64);
      S += __shfl_xor(S, 32, 64);
      if (g == 0) {
        const int64_t at = canon_scale_at(p.m >> 5, tok, blk);
        p.y.c[at] = bs.c;
        p.y.s[at] = S;
      }
    } else {  // split, rotary on Q and K, K/V appended (Inference.cu:1070-1103)
      if (tok < p.M) {
        const int H = p.m / 3;
        const int part = row0 / H, head = row0 % H >> 7, pos = p.qkv.pos0 + tok;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int d = (row0 & 127) + 16 * r + 4 * g;
          half4_t v = half4_t{(half_t)sum[r][0], (half_t)sum[r][1], (half_t)sum[r][2], (half_t)sum[r][3]};
          if (part < 2) {
            const half2_t c2 = *reinterpret_cast<const half2_t*>(p.qkv.cos_t + (int64_t)pos * 64 + (d >> 1));
            const half2_t s2 = *reinterpret_cast<const half2_t*>(p.qkv.sin_t + (int64_t)pos * 64 + (d >> 1));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const half_t a = v[2 * j], b = v[2 * j + 1];
              const half_t ac = a * c2[j], bsn = b * s2[j], as = a * s2[j], bc = b * c2[j];
              v[2 * j] = ac - bsn;
              v[2 * j + 1] = as + bc;
            }
          }
          if (part == 0) {
            *reinterpret_cast<half4_t*>(p.qkv.q_out + (int64_t)tok * H + head * AWQ_HEAD_DIM + d) = v;
          } else {
            *reinterpret_cast<half4_t*>((part == 1 ? p.qkv.k_cache : p.qkv.v_cache) + kv_row(p.qkv.kv, head, pos) + d) = v;
            half_t* const again = part == 1 ? p.qkv.k_parts : p.qkv.v_parts;
            if (again && pos < p.qkv.parts_pos)
              *reinterpret_cast<half4_t*>(again + (((int64_t)head * 8 + (d >> 4)) * p.qkv.parts_pos + pos) * 16 + (d & 15)) = v;
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// What stands between two products, a workgroup per token of 4,096 values: the product's parts are added in
// awq_tree_sum's order, the residual added (Inference.cu:1149-1155), the row normed (:111-145 in rmsnorm_kernel's order)
// and put into block fixed point.  gamma null: the residual stream only.
// ---------------------------------------------------------------------------
constexpr int kCanonHidden = 4096;

template <int P>
__global__ __launch_bounds__(256) void canon_norm_kernel(const float* __restrict__ part, half_t* __restrict__ hidden,
                                                         const half_t* __restrict__ gamma, float eps, CanonTokens out, int M) {
  constexpr int E = kCanonHidden / 256;
  __shared__ float buf[256];
  __shared__ __attribute__((aligned(16))) half_t xn[kCanonHidden];
  const int tid = threadIdx.x, tok = blockIdx.x;
  const bool real = tok < M;  // the tokens that fill the last tile: zeros
  if (real) {
    half_t* const row = hidden + (int64_t)tok * kCanonHidden;
    half_t x[E];
#pragma unroll
    for (int j = 0; j < E; ++j) x[j] = row[tid + 256 * j];
    if constexpr (P > 0) {
      float v[P][E];
#pragma unroll
      for (int q = 0; q < P; ++q)
#pragma unroll
        for (int j = 0; j < E; ++j) v[q][j] = part[((int64_t)q * M + tok) * kCanonHidden + tid + 256 * j];
#pragma unroll
      for (int j = 0; j < E; ++j) {
        float t;
        if constexpr (P == 2) t = v[0][j] + v[1][j];
        else if constexpr (P == 3) t = (v[0][j] + v[1][j]) + v[2][j];
        else t = (v[0][j] + v[1][j]) + (v[2][j] + v[3][j]);
        x[j] = x[j] + (half_t)t;
        row[tid + 256 * j] = x[j];
      }
    }
    if (!gamma) return;
    half_t gm[E];
#pragma unroll
    for (int j = 0; j < E; ++j) gm[j] = gamma[tid + 256 * j];
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) acc = __builtin_fmaf((float)x[j], (float)x[j], acc);
    buf[tid] = acc;
    __syncthreads();
    const int l = tid & 63;
    float t = (buf[l] + buf[l + 128]) + (buf[l + 64] + buf[l + 192]);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) t += __shfl_xor(t, d, 64);
    const half_t sc = rsqrt_half(t / (float)kCanonHidden + eps);
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const half_t n = x[j] * sc;
      xn[tid + 256 * j] = n * gm[j];
    }
    __syncthreads();
  } else if (!gamma) {
    return;
  }
  // units of eight values, four threads a block
#pragma unroll
  for (int u = tid; u < kCanonHidden / 8; u += 256) {
    half8_t v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (half_t)0.0f;
    if (real) v = *reinterpret_cast<const half8_t*>(xn + 8 * u);
    uint32_t mm = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) mm = max(mm, magnitude(v[i]));
    mm = max(mm, dpp_u<kDppXor1>(mm));
    mm = max(mm, dpp_u<kDppXor2>(mm));
    const BlockScale bs = block_scale(mm);
    float S = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float f = block_int(v[i], bs);
      S += f;
      v[i] = (half_t)f;
    }
    S += dpp_f<kDppXor1>(S);
    S += dpp_f<kDppXor2>(S);
    *reinterpret_cast<half8_t*>(out.op + canon_op_at(kCanonHidden / 32, tok, u >> 2, (u & 3) * 8)) = v;
    if ((u & 3) == 0) {
      const int64_t at = canon_scale_at(kCanonHidden / 32, tok, u >> 2);
      out.c[at] = bs.c;
      out.s[at] = S;
    }
  }
}

// ---------------------------------------------------------------------------
// Attention of four consecutive prompt positions of a head, a wavefront's lanes and sums as in attention_kernel
// (attention.hip): sixteen lanes of eight dimensions per key, exponentials summed by chunks of 64 positions, a chunk's
// context by four chains.  A key or value row is read once for the four queries.  The context goes out in block fixed
// point: a head's 128 dimensions are four blocks of the product that follows.
// ---------------------------------------------------------------------------
constexpr int kCanonQueries = 4;

template <int CTRL>
__device__ __forceinline__ float add_dpp(float v) { return v + dpp_f<CTRL>(v); }
constexpr int kDppMirror = 0x140;  // lane i <-> 15 - i within 16
__device__ __forceinline__ float sum16(float v) {
  return add_dpp<kDppMirror>(add_dpp<kDppHalfMirror>(add_dpp<kDppXor2>(add_dpp<kDppXor1>(v))));
}
// v + lane ^ 16, then + lane ^ 32
__device__ __forceinline__ float sum_rows(float v) { return sum_rows_of_16(v); }

__global__ __launch_bounds__(256) void canon_attention_kernel(const half_t* __restrict__ q, const half_t* __restrict__ kc,
                                                              const half_t* __restrict__ vc, KvLayout kv, int pos0, int M,
                                                              int use_len_hi, int L_cap, CanonTokens out) {
  constexpr int QG = kCanonQueries, NW = 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* const s = lds;                              // [QG][L_cap]
  float* const cs = s + QG * L_cap;                  // [QG][L_cap / 64]
  float* const cv = cs + QG * (L_cap >> 6);          // [NW][QG][128]
  float* const wmax = cv + NW * QG * AWQ_HEAD_DIM;   // [NW][QG]
  const int head = blockIdx.x, H = gridDim.x * AWQ_HEAD_DIM, tok0 = blockIdx.y * QG;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tq = lane >> 4, dl = lane & 15;
  const float scale = 1.0f / sqrtf((float)AWQ_HEAD_DIM);  // Inference.cu:218
  int L[QG], Lmax = 1;
  float qf[QG][8];
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    const int tok = min(tok0 + g, M - 1), pos = pos0 + tok;
    L[g] = use_len_hi ? pos + 1 : max(pos, 1);  // Inference.cu:1118 before :1331 in layer 0
    Lmax = max(Lmax, L[g]);
    const half8_t v = *reinterpret_cast<const half8_t*>(q + (int64_t)tok * H + head * AWQ_HEAD_DIM + 8 * dl);
#pragma unroll
    for (int i = 0; i < 8; ++i) qf[g][i] = (float)v[i];
  }
  const int nch = (Lmax + 63) >> 6;

  float lmax[QG];
#pragma unroll
  for (int g = 0; g < QG; ++g) lmax[g] = -1e9f;
  constexpr int U = 4;
  for (int t0 = 4 * wave; t0 < Lmax; t0 += 4 * NW * U) {
    half8_t k[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = min(t0 + 4 * NW * u + tq, Lmax - 1);
      k[u] = *reinterpret_cast<const half8_t*>(kc + kv_row(kv, head, t) + 8 * dl);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + 4 * NW * u + tq;
#pragma unroll
      for (int g = 0; g < QG; ++g) {
        float part = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) part = __builtin_fmaf(qf[g][i], (float)k[u][i], part);
        const float sc = sum16(part) * scale;
        if (t < L[g]) {
          if (dl == 0) s[g * L_cap + t] = sc;
          lmax[g] = fmaxf(lmax[g], sc);
        }
      }
    }
  }
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    float v = lmax[g];
#pragma unroll
    for (int d = 16; d <= 32; d <<= 1) v = fmaxf(v, __shfl_xor(v, d, 64));  // (the sixteen lanes of a key hold the same)
    if (lane == 0) wmax[wave * QG + g] = v;
  }
  __syncthreads();
  // exponentials and their sums by chunk (Inference.cu:239-249)
  for (int chunk = wave; chunk < nch; chunk += NW) {
    const int t = (chunk << 6) + lane;
#pragma unroll
    for (int g = 0; g < QG; ++g) {
      const float mx = fmaxf(fmaxf(wmax[g], wmax[QG + g]), fmaxf(wmax[2 * QG + g], wmax[3 * QG + g]));
      float e = 0.0f;
      if (t < L[g]) {
        e = awq_expf(s[g * L_cap + t] - mx);
        s[g * L_cap + t] = e;
      }
      e = sum_rows(sum16(e));
      if (lane == 0) cs[g * (L_cap >> 6) + chunk] = e;
    }
  }
  __syncthreads();
  float Z[QG];
#pragma unroll
  for (int g = 0; g < QG; ++g) {
    Z[g] = cs[g * (L_cap >> 6)];
    const int n = (L[g] + 63) >> 6;
    for (int c = 1; c < n; ++c) Z[g] += cs[g * (L_cap >> 6) + c];
  }
  // weighted sum of V (Inference.cu:251-265), NW chunks at a time; wavefront g then adds query g's chunk vectors in order
  float o0 = 0.0f, o1 = 0.0f;
  const int my_n = (L[wave] + 63) >> 6;
  for (int c0 = 0; c0 < nch; c0 += NW) {
    const int chunk = c0 + wave, base = chunk << 6;
    if (chunk < nch) {
      half8_t v[16];
#pragma unroll
      for (int nl = 0; nl < 16; ++nl)
        v[nl] = *reinterpret_cast<const half8_t*>(vc + kv_row(kv, head, min(base + 4 * nl + tq, Lmax - 1)) + 8 * dl);
#pragma unroll
      for (int g = 0; g < QG; ++g) {
        const float p_lane = base + lane < L[g] ? s[g * L_cap + base + lane] / Z[g] : 0.0f;
        float acc[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int nl = 0; nl < 16; ++nl) {
          const bool in = base + 4 * nl + tq < L[g];
          const float pp = __shfl(p_lane, 4 * nl + tq, 64);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float r = __builtin_fmaf(pp, (float)v[nl][i], acc[i]);
            acc[i] = in ? r : acc[i];
          }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = sum_rows(acc[i]);
        if (tq == 0)
#pragma unroll
          for (int i = 0; i < 8; ++i) cv[(wave * QG + g) * AWQ_HEAD_DIM + 8 * dl + i] = acc[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w)
      if (c0 + w < my_n) {
        const float2_t v = *reinterpret_cast<const float2_t*>(&cv[(w * QG + wave) * AWQ_HEAD_DIM + 2 * lane]);
        o0 = c0 + w == 0 ? v[0] : o0 + v[0];
        o1 = c0 + w == 0 ? v[1] : o1 + v[1];
      }
    __syncthreads();
  }
  static_assert(NW == QG, "a wavefront per query");
  const int tok = tok0 + wave;
  const half_t h0 = tok < M ? (half_t)o0 : (half_t)0.0f, h1 = tok < M ? (half_t)o1 : (half_t)0.0f;
  uint32_t mm = max(magnitude(h0), magnitude(h1));
  mm = max(mm, dpp_u<kDppXor1>(mm));
  mm = max(mm, dpp_u<kDppXor2>(mm));
  mm = max(mm, dpp_u<kDppHalfMirror>(mm));
  mm = max(mm, dpp_u<kDppMirror>(mm));
  const BlockScale bs = block_scale(mm);
  const float f0 = block_int(h0, bs), f1 = block_int(h1, bs);
  const float S = sum16(f0 + f1);
  const int64_t nblk = H >> 5, blk = head * 4 + tq;
  *reinterpret_cast<half2_t*>(out.op + canon_op_at(nblk, tok, blk, 2 * dl)) = half2_t{(half_t)f0, (half_t)f1};
  if (dl == 0) {
    const int64_t at = canon_scale_at(nblk, tok, blk);
    out.c[at] = bs.c;
    out.s[at] = S;
  }
}

template <int N, int RS, bool ZI>
int launch_product(const ProductParams& p, int out, int kb, hipStream_t st) {
  const dim3 grid((unsigned)(p.m / (32 * RS)), (unsigned)((p.tiles + N - 1) / N), (unsigned)(p.nblk / kb)), block(512);
  constexpr int full = 128 * RS / 8, quarter = 32 * RS / 8;
  if (out == CANON_QKV) hipLaunchKernelGGL((canon_product_kernel<N, RS, full, ZI, CANON_QKV>), grid, block, 0, st, p);
  else if (out == CANON_GELU) hipLaunchKernelGGL((canon_product_kernel<N, RS, full, ZI, CANON_GELU>), grid, block, 0, st, p);
  else if (kb == 128) hipLaunchKernelGGL((canon_product_kernel<N, RS, full, ZI, CANON_PARTS>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((canon_product_kernel<N, RS, quarter, ZI, CANON_PARTS>), grid, block, 0, st, p);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

template <int N, int RS>
int launch_product_zi(const ProductParams& p, bool zi, int out, int kb, hipStream_t st) {
  return zi ? launch_product<N, RS, true>(p, out, kb, st) : launch_product<N, RS, false>(p, out, kb, st);
}

}  // namespace

int canon_prompt_parts(int64_t m, int64_t k) { return (int)(m == kCanonHidden && k == kCanonHidden ? 4 : k / 4096); }

bool canon_prompt_supported(int64_t hidden, int64_t inter) {
  return hidden == kCanonHidden && inter % 4096 == 0 && inter / 4096 <= 4 && awq_group_period(3 * hidden, hidden) == 1 &&
         awq_group_period(hidden, hidden) == 1 && awq_group_period(inter, hidden) == 1 && awq_group_period(hidden, inter) == 1;
}

// A layer of a pass of up to 16 positions against the steps it takes the place of.  A step's attention cuts the sequence over workgroups,
// the pass's gives a workgroup four queries of a head and all their keys.  Us per layer, pass and step: at position 0 63 and 20.8 with
// inter 4,096, 71 and 26.1 with 12,288, 73 and 32.4 with 16,384; at 1,500 of 12,288 141 and 33.0, at 2,000 170 and 36.6.  12 layers, 3
// positions from 0, 1,000 and 2,000 on: single 940, 1,098 and 1,319 us, together 857, 1,455 and 2,039; 4: 1,236, 1,449 and 1,735
// against 850, 1,462 and 2,051; 8 are faster together everywhere (2,000: 2,033 against 3,413).
int64_t canon_prompt_from(int64_t inter, int64_t pos0) {
  const float at = (float)pos0, wide = (float)inter;
  return (int64_t)ceilf((61.0f + 0.001f * wide + 0.0495f * at) / (18.1f + 0.00065f * wide + 0.0052f * at));
}

int launch_canon_norm(const float* part, int parts, half_t* hidden, const half_t* gamma, float eps, CanonTokens out, int64_t M,
                      hipStream_t st) {
  AWQ_REQUIRE(M >= 1 && M <= kCanonTokens && (parts == 0 || (parts >= 2 && parts <= 4 && part)), "bad arguments");
  const dim3 grid((unsigned)(gamma ? round16(M) : M)), block(256);
  if (parts == 0) hipLaunchKernelGGL((canon_norm_kernel<0>), grid, block, 0, st, part, hidden, gamma, eps, out, (int)M);
  else if (parts == 2) hipLaunchKernelGGL((canon_norm_kernel<2>), grid, block, 0, st, part, hidden, gamma, eps, out, (int)M);
  else if (parts == 3) hipLaunchKernelGGL((canon_norm_kernel<3>), grid, block, 0, st, part, hidden, gamma, eps, out, (int)M);
  else hipLaunchKernelGGL((canon_norm_kernel<4>), grid, block, 0, st, part, hidden, gamma, eps, out, (int)M);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}

int launch_canon_product(const void* wq, const half_t* scale, const half_t* zp, bool zp_small, int64_t m, int64_t k, CanonTokens x,
                         int64_t M, int out, float* part, CanonTokens y, const CanonQkv& qkv, hipStream_t st) {
  AWQ_REQUIRE(m % 128 == 0 && k % 4096 == 0 && awq_group_period(m, k) == 1, "shape");
  AWQ_REQUIRE(M >= 1 && M <= kCanonTokens, "token count out of range");
  AWQ_REQUIRE(out == CANON_PARTS ? part != nullptr : k == 4096, "a finished sum needs all of k in a workgroup");
  ProductParams p;
  p.wq = (const uint32_t*)wq;
  p.scale = scale;
  p.zp = zp;
  p.m = (int)m;
  p.nblk = (int)(k / 32);
  p.mg = (int)(m / 128);
  p.kg = (int)(k / 128);
  p.x = x;
  p.M = (int)M;
  p.tiles = (int)(round16(M) / 16);
  p.part = part;
  p.y = y;
  p.qkv = qkv;
  const int kb = out == CANON_PARTS ? p.nblk / canon_prompt_parts(m, k) : 128;
  // Up to four tiles of 16 tokens in a workgroup; 64 rows a workgroup where all tokens are in one, else 128.
  const int groups = (p.tiles + 3) / 4, n = (p.tiles + groups - 1) / groups;
  if (groups == 1) {
    if (n == 1) return launch_product_zi<1, 2>(p, zp_small, out, kb, st);
    if (n == 2) return launch_product_zi<2, 2>(p, zp_small, out, kb, st);
    if (n == 3) return launch_product_zi<3, 2>(p, zp_small, out, kb, st);
    return launch_product_zi<4, 2>(p, zp_small, out, kb, st);
  }
  if (n == 3) return launch_product_zi<3, 4>(p, zp_small, out, kb, st);
  return launch_product_zi<4, 4>(p, zp_small, out, kb, st);
}

int launch_canon_attention(const half_t* q, const half_t* kc, const half_t* vc, KvLayout kv, int n_heads, int64_t pos0, int64_t M,
                           int use_len_hi, CanonTokens out, hipStream_t st) {
  AWQ_REQUIRE(M >= 1 && M <= kCanonTokens && pos0 >= 0 && pos0 + M <= kCanonPositions, "positions out of range");
  const int L_cap = (int)((pos0 + M + 63) / 64 * 64);
  const size_t lds = ((size_t)kCanonQueries * (L_cap + L_cap / 64) + 4 * kCanonQueries * AWQ_HEAD_DIM + 4 * kCanonQueries) * 4;
  hipLaunchKernelGGL(canon_attention_kernel, dim3((unsigned)n_heads, (unsigned)(round16(M) / kCanonQueries)), dim3(256), lds, st, q, kc,
                     vc, kv, (int)pos0, (int)M, use_len_hi, L_cap, out);
  AWQ_HIP_TRY(hipGetLastError());
  return AWQ_OK;
}
