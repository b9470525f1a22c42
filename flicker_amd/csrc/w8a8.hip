// w8a8: SmoothQuant int8 QKV projection for gfx950 (int8 MFMA, int32 accumulate).
//
// The reference projects x @ w in bf16 (src/flicker/nn.py:13-14, called for the QKV
// projection at src/flicker/modules.py:128,132,186) and has no quantisation.  This file
// implements the replacement defined by the formula below; every integer and every
// float32 rounding is reproduced exactly (each float op is one IEEE f32 operation with
// round-to-nearest-even; division and sqrt correctly rounded; rint ties-to-even):
//
//   calibration   s_j = sqrt(max_t |X[t,j]|) / sqrt(max_o |W[j,o]|)  (1 if either is 0)
//                 inv_s_j = 1 / s_j
//   weight        Wh[j,o] = f32(W[j,o]) * s_j;  w_o = max_j |Wh[j,o]| / 127 (1 if 0)
//                 Wq[j,o] = clamp(rint(Wh[j,o] / w_o), -127, 127)           int8
//   activation    Xh[t,j] = f32(X[t,j]) * inv_s_j;  a_t = max_j |Xh[t,j]| / 127 (1 if 0)
//                 Xq[t,j] = clamp(rint(Xh[t,j] / a_t), -127, 127)           int8
//   GEMM          acc[t,o] = sum_j Xq[t,j] * Wq[j,o]                          int32, exact
//   rescale       Y[t,o] = bf16((f32(acc[t,o]) * a_t) * w_o)
//
// Layouts: X (M, K) and W (K, N) bf16 row-major with row strides (W as the reference
// stores it: in x out); Xq (M, K) int8; the quantised weight is stored transposed,
// WqT (N, K) int8, so both GEMM operands are K-contiguous rows; Y (M, N) bf16 with a
// row stride; optional acc (M, N) int32.
//
// GEMM.  A block of 8 waves (two per SIMD) owns a 256 (n) x 256 (m) output tile and
// computes it transposed, Y^T = WqT . Xq^T, with v_mfma_i32_16x16x64_i8: A operand = 16 WqT
// rows x 64 k bytes, B operand = 16 Xq rows x 64 k bytes, both one ds_read_b128 per lane.
// Under random int8 data the chip runs at its power limit, where the 16x16x64 form does the
// same ops on less energy than 32x32x32 (a quarter of the accumulator traffic per
// instruction; an MFMA stream with random operands issues 12-17% more ops per second).  In
// the 16x16 accumulator a lane owns one token and 4 consecutive output channels.  Each wave
// holds a 128 (n) x 64 (m) sub-tile: 32 accumulators of 4 int32 (128 registers), 12 operand
// reads per 32 MFMAs.  k advances in 128-byte stages (one full 128-byte line per operand
// row) through two 64 KiB LDS buffers filled by global_load_lds_dwordx4 (no registers); a
// row's 16-byte chunk c is stored at c ^ gswz(row), which keeps every operand read on
// distinct banks.  Integer sums are exact in any order, so the products are those of any
// other tiling, bit for bit.  The epilogue rescales into LDS and
// stores whole 256-byte output rows.  Blocks are renumbered so consecutive output tiles
// share an XCD (and its L2), and grouped so that 4 token tiles sweep the channel tiles
// together.
//
// A launch of more than one round (the Klein projection: 648 tiles, 2.53 rounds of 256 CUs)
// takes the rounds order: each XCD runs whole rounds of 32 of its tiles, then cuts the tiles
// left over into tiles of 192 tokens (waves of 128 x 48: three token fragments), so the
// partial last round has up to 4/3 as many blocks with 3/4 of the work each (measured 1-5%
// faster for the plain GEMM, 3-6% with the qk_prep epilogue).
//
// A launch of few tiles (a short text stream, a small image) takes tiles of 128 channels x 64 or
// 128 tokens instead, two waves per 128 x 32 position (gemm_tile_split; launch_group's rule).
//
// A launch takes up to two problems (GemmGroup; the activation quantiser likewise takes a
// QuantGroup): a double block's text and image projections share one grid, so the small
// text projection runs on the CUs the image projection leaves idle in its last round.

#include <algorithm>

#include "qk_math.h"

namespace {

using flk::f32x4;
using flk::i32x4;
using flk::i32x16;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kQMax = 127.0f;

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
  return v;
}

__device__ __forceinline__ float absmax_scale(float amax) { return amax > 0.0f ? amax / kQMax : 1.0f; }

// The codes clamp(rint(v / a), -127, 127) of 4 elements, packed, without a division each: a their
// absmax scale (|v / a| <= 127.0001), r = 1 / a rounded once, so that v * r is within 2^-23 |q|
// < 1.6e-5 of the correctly rounded quotient q.  Adding 1.5 * 2^23 rounds the exact product to its
// integer t, whose two's complement is then the sum's low byte; when the product is within
// 0.5 - 2^-15 of t, q rounds to t too.  Otherwise -- near a tie, or not finite -- the lane divides.
__device__ __forceinline__ uint32_t quantize4(const float (&v)[4], float a, float r) {
  constexpr float kRound = 12582912.0f;
  uint32_t u[4];
  bool near = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float sum = __builtin_fmaf(v[i], r, kRound);
    const float off = __builtin_fmaf(v[i], r, -(sum - kRound));
    near |= !(fabsf(off) < 0.5f - 0x1p-15f);
    u[i] = __float_as_uint(sum);
  }
  if (near) {
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = (uint32_t)(int)fminf(fmaxf(__builtin_rintf(v[i] / a), -kQMax), kQMax);
  }
  // bytes 0 of two words each: perm selects from the second argument (0-3) and the first (4-7), 0x0c = 0
  return __builtin_amdgcn_perm(u[1], u[0], 0x0c0c0400u) | __builtin_amdgcn_perm(u[3], u[2], 0x04000c0cu);
}

template <int kCtrl>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF, false));
}

template <int kCtrl>
__device__ __forceinline__ double dpp_move(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, kCtrl, 0xF, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), kCtrl, 0xF, 0xF, false);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

__device__ __forceinline__ void unpack_bf16x8(const uint4& r, float (&f)[8]) {
  f[0] = flk::bf16_lo(r.x); f[1] = flk::bf16_hi(r.x);
  f[2] = flk::bf16_lo(r.y); f[3] = flk::bf16_hi(r.y);
  f[4] = flk::bf16_lo(r.z); f[5] = flk::bf16_hi(r.z);
  f[6] = flk::bf16_lo(r.w); f[7] = flk::bf16_hi(r.w);
}

// ---------------------------------------------------------------- calibration ----------

// s = sqrt(xa) / sqrt(wa) (1 where either maximum is 0).
__device__ __forceinline__ float smooth_factor(float xa, float wa) {
  return xa > 0.0f && wa > 0.0f ? __builtin_sqrtf(xa) / __builtin_sqrtf(wa) : 1.0f;
}

// out[r] = max_c |x[r, c]|; one wave per row, 8 columns per lane step (cols % 8 == 0).
// HBM-bound: 3072 rows are only three waves a SIMD, so kRowUnroll loads per lane are in flight
// (3072 x 9216, with the factors: one load 15.1 us, 6 11.4, 9 11.5; as two launches 16.6).
// kSmooth: out holds the smoothing factors of the row maxima and xa instead, and inv their inverses
// (a weight's rows are its input channels): one launch less before a weight's quantisation.
template <int kRowUnroll, bool kSmooth>
__global__ __launch_bounds__(256) void absmax_rows_kernel(const uint16_t* __restrict__ x, int64_t rows,
                                                          int64_t cols, int64_t stride,
                                                          float* __restrict__ out, const float* __restrict__ xa,
                                                          float* __restrict__ inv) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= rows) return;
  const uint16_t* p = x + row * stride;
  float xrow = 0.0f;
  if constexpr (kSmooth) xrow = xa[row];   // before the row: its latency hides behind the row's
  float m = 0.0f;
  for (int64_t c = (int64_t)lane * 8; c < cols; c += 512 * kRowUnroll) {
    uint4 v[kRowUnroll];
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u)   // a chunk past the row's end repeats this pass's first
      v[u] = *reinterpret_cast<const uint4*>(p + (c + 512 * u < cols ? c + 512 * u : c));
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) {
      float f[8];
      unpack_bf16x8(v[u], f);
#pragma unroll
      for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(f[i]));
    }
  }
  m = wave_max(m);
  if (lane == 0) {
    if constexpr (kSmooth) {
      m = smooth_factor(xrow, m);
      inv[row] = 1.0f / m;
    }
    out[row] = m;
  }
}

// The start of a merged column maximum: 0, or the running maximum that is accumulated into (a NaN
// or a negative value there counts as 0, as fmaxf against the first |x| does).
__global__ __launch_bounds__(256) void absmax_init_kernel(int64_t cols, int accumulate, float* __restrict__ out) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c < cols) out[c] = accumulate ? fmaxf(out[c], 0.0f) : 0.0f;
}

// Column maxima of one block's 128 columns over rows r, r + 16, ... of [r, r1): 16 lane groups
// of 8 columns x 16 row groups, kColUnroll rows' loads in flight per thread (a load past r1
// repeats the thread's first row), reduced through LDS into threads 0-127 (one column each).
// kScaled: the maximum of |x * s[row]|.
constexpr int kColUnroll = 8;
constexpr int kColRows = 16 * kColUnroll;   // rows one pass of a block's loads covers

template <bool kScaled>
__device__ __forceinline__ float column_absmax(float (&red)[16][129], const uint16_t* __restrict__ x, int64_t stride,
                                               int64_t r0, int64_t r1, int64_t cols, int64_t c0,
                                               const float* __restrict__ s) {
  const int cg = threadIdx.x & 15, rg = threadIdx.x >> 4;
  float m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (c0 + cg * 8 < cols) {
    const uint16_t* col = x + c0 + cg * 8;
    for (int64_t r = r0 + rg; r < r1; r += kColRows) {
      uint4 v[kColUnroll];
      float sj[kColUnroll];
#pragma unroll
      for (int i = 0; i < kColUnroll; ++i) {
        const int64_t ri = r + 16 * i < r1 ? r + 16 * i : r;
        v[i] = *reinterpret_cast<const uint4*>(col + ri * stride);
        if constexpr (kScaled) sj[i] = s[ri];
      }
#pragma unroll
      for (int i = 0; i < kColUnroll; ++i) {
        float f[8];
        unpack_bf16x8(v[i], f);
#pragma unroll
        for (int j = 0; j < 8; ++j) m[j] = fmaxf(m[j], fabsf(kScaled ? f[j] * sj[i] : f[j]));
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) red[rg][cg * 8 + j] = m[j];
  __syncthreads();
  float v = 0.0f;
  if (threadIdx.x < 128) {
#pragma unroll
    for (int g = 0; g < 16; ++g) v = fmaxf(v, red[g][threadIdx.x]);
  }
  return v;
}

// out[c] = max(out[c], max_r |x[r, c]|).  HBM-bound: the rows are cut over blockIdx.y so that the
// pass fills the chip (one block per 128 columns alone was 24 blocks at 3072 channels, each a
// serial walk of the rows).  kMerge: out set by absmax_init_kernel; block maxima are finite or +inf
// and never negative, so their int bits order as the floats do and an integer atomic merges them.
// 4608 x 3072 (28 MB): 6.5 us + 1.6 us to set out, 103 us before.  Otherwise one cut holds all the
// rows (flk_absmax_cols' rule) and its block writes out itself.
template <bool kMerge>
__global__ __launch_bounds__(256) void absmax_cols_kernel(const uint16_t* __restrict__ x, int64_t rows,
                                                          int64_t cols, int64_t stride, int64_t rows_per_block,
                                                          int accumulate, float* __restrict__ out) {
  __shared__ float red[16][129];
  const int64_t c0 = (int64_t)blockIdx.x * 128, r0 = blockIdx.y * rows_per_block;
  const float v = column_absmax<false>(red, x, stride, r0, min(rows, r0 + rows_per_block), cols, c0, nullptr);
  const int64_t c = c0 + threadIdx.x;
  if (threadIdx.x >= 128 || c >= cols) return;
  if constexpr (kMerge) {
    if (v > 0.0f) atomicMax(reinterpret_cast<int*>(out) + c, __float_as_int(v));
  } else {
    out[c] = accumulate ? fmaxf(v, out[c]) : v;
  }
}

__global__ void smooth_factors_kernel(const float* __restrict__ xa, const float* __restrict__ wa, int64_t k,
                                      float* __restrict__ s, float* __restrict__ inv_s) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k) return;
  const float v = smooth_factor(xa[i], wa[i]);
  s[i] = v;
  inv_s[i] = 1.0f / v;
}

// ---------------------------------------------------------------- quantisation ---------

// Weight (offline), three launches.  The first cuts the rows of W over blockIdx.y and writes each
// cut's column maxima of |Wh| to part (cut, channel); the second takes their maximum -> w_scale;
// the third quantises.  part is the front of the WqT buffer itself, which the third launch then
// overwrites: cuts are of 128 rows or more, the last of 64 or more, so their 4 bytes per channel
// fit the K bytes per channel many times over.  HBM-bound; one block per 64 channels walking all
// the rows twice filled 144 CUs and waited on each row: 3072 x 9216 took 91 us, 30 us now (10.4 +
// 2.0 + 17.3).  One launch with 32 channels of all the rows in registers, W read once, took 37.
__global__ __launch_bounds__(256) void weight_absmax_kernel(const uint16_t* __restrict__ w, int64_t w_stride,
                                                            const float* __restrict__ s, int K, int N,
                                                            int64_t rows_per_block, float* __restrict__ part) {
  __shared__ float red[16][129];
  const int64_t c0 = (int64_t)blockIdx.x * 128, r0 = blockIdx.y * rows_per_block;
  const float v = column_absmax<true>(red, w, w_stride, r0, min((int64_t)K, r0 + rows_per_block), N, c0, s);
  const int64_t c = c0 + threadIdx.x;
  if (threadIdx.x < 128 && c < N) part[(int64_t)blockIdx.y * N + c] = v;
}

__global__ __launch_bounds__(256) void weight_scale_kernel(const float* __restrict__ part, int cuts, int N,
                                                           float* __restrict__ w_scale) {
  const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  float v = 0.0f;
#pragma unroll 8
  for (int i = 0; i < cuts; ++i) v = fmaxf(v, part[(int64_t)i * N + n]);
  w_scale[n] = absmax_scale(v);
}

// Codes and transposes a tile of 128 rows (k) x 64 channels.  A thread takes 4 consecutive k (raw, of
// smoothing factors sj) of 8 channels, so that four codes leave as one 32-bit LDS write and a WqT
// row piece as 128 contiguous bytes; the 33-word pitch spreads the 64 words of a wave's write over
// the banks.
typedef uint32_t WeightTile[64][33];

__device__ __forceinline__ void code_weights(WeightTile& tile, const uint4 (&raw)[4], const float (&sj)[4],
                                             const float (&sc)[8], const float (&rc)[8]) {
  const int cg = threadIdx.x & 7, rq = threadIdx.x >> 3;
  float f[4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i) unpack_bf16x8(raw[i], f[i]);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v[4] = {f[0][j] * sj[0], f[1][j] * sj[1], f[2][j] * sj[2], f[3][j] * sj[3]};
    tile[cg * 8 + j][rq] = quantize4(v, sc[j], rc[j]);
  }
}

__device__ __forceinline__ void store_weights(const WeightTile& tile, int8_t* __restrict__ wqt, int n0, int64_t k0,
                                              int K, int N) {
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int n = (threadIdx.x >> 3) + it * 32, ch = threadIdx.x & 7;
    if (n0 + n < N && k0 + ch * 16 < K)
      *reinterpret_cast<uint4*>(wqt + (int64_t)(n0 + n) * K + k0 + ch * 16) =
          uint4{tile[n][ch * 4], tile[n][ch * 4 + 1], tile[n][ch * 4 + 2], tile[n][ch * 4 + 3]};
  }
}

__global__ __launch_bounds__(256) void quantize_weight_kernel(const uint16_t* __restrict__ w, int64_t w_stride,
                                                              const float* __restrict__ s, int K, int N,
                                                              int8_t* __restrict__ wqt,
                                                              const float* __restrict__ w_scale) {
  __shared__ WeightTile tile;
  const int n0 = blockIdx.x * 64, nc = n0 + (threadIdx.x & 7) * 8;
  const bool active = nc < N;
  float sc[8], rc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) sc[j] = active ? w_scale[nc + j] : 1.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) rc[j] = 1.0f / sc[j];
  // One tile, but for a K past the grid's 65535 tiles.
  for (int64_t k0 = (int64_t)blockIdx.y * 128; k0 < K; k0 += (int64_t)gridDim.y * 128) {
    const int64_t kr = k0 + (threadIdx.x >> 3) * 4;
    if (active && kr < K) {
      uint4 raw[4];
      float sj[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        raw[i] = *reinterpret_cast<const uint4*>(w + (kr + i) * w_stride + nc);
        sj[i] = s[kr + i];
      }
      code_weights(tile, raw, sj, sc, rc);
    }
    __syncthreads();
    store_weights(tile, wqt, n0, k0, K, N);
    __syncthreads();
  }
}

// All of a short weight's rows (K <= 128 kTiles) in one launch: a block holds its 64 channels in
// registers between the maxima and the codes.  Bound by latency: the three launches above take 7 us
// however small the weight (us, three launches and one, at 3072 channels: k = 64 8.1 / 3.9, 128
// 8.2 / 4.0, 256 8.4 / 5.5, 384 8.6 / 6.9, 512 8.9 / 8.4; 512 x 27648 19.4 / 12.7).
template <int kTiles>
__global__ __launch_bounds__(256) void quantize_weight_short_kernel(const uint16_t* __restrict__ w, int64_t w_stride,
                                                                    const float* __restrict__ s, int K, int N,
                                                                    int8_t* __restrict__ wqt,
                                                                    float* __restrict__ w_scale) {
  __shared__ WeightTile tile;
  __shared__ float red[32][65], scale[64];
  const int cg = threadIdx.x & 7, rq = threadIdx.x >> 3;
  const int n0 = blockIdx.x * 64, nc = n0 + cg * 8;
  const bool active = nc < N;
  uint4 raw[kTiles][4];
  float sj[kTiles][4];
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = t * 128 + rq * 4 + i;
      const bool in = active && k < K;
      raw[t][i] = in ? *reinterpret_cast<const uint4*>(w + k * w_stride + nc) : uint4{0, 0, 0, 0};
      sj[t][i] = in ? s[k] : 0.0f;
    }
  float m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float f[8];
      unpack_bf16x8(raw[t][i], f);
#pragma unroll
      for (int j = 0; j < 8; ++j) m[j] = fmaxf(m[j], fabsf(f[j] * sj[t][i]));
    }
#pragma unroll
  for (int j = 0; j < 8; ++j) red[rq][cg * 8 + j] = m[j];
  __syncthreads();
  if (threadIdx.x < 64) {
    float v = 0.0f;
#pragma unroll
    for (int g = 0; g < 32; ++g) v = fmaxf(v, red[g][threadIdx.x]);
    v = absmax_scale(v);
    scale[threadIdx.x] = v;
    if (n0 + (int)threadIdx.x < N) w_scale[n0 + threadIdx.x] = v;
  }
  __syncthreads();
  float sc[8], rc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    sc[j] = scale[cg * 8 + j];
    rc[j] = 1.0f / sc[j];
  }
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    if (t > 0) __syncthreads();
    code_weights(tile, raw[t], sj[t], sc, rc);
    __syncthreads();
    store_weights(tile, wqt, n0, t * 128, K, N);
  }
}

// op over the 64 lanes of a wave: the 16-lane rows by DPP, then the rows by lane shuffles.
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  v = op(v, dpp_move<0xB1>(v));    // quad_perm 1,0,3,2
  v = op(v, dpp_move<0x4E>(v));    // quad_perm 2,3,0,1
  v = op(v, dpp_move<0x141>(v));   // row_half_mirror
  v = op(v, dpp_move<0x140>(v));   // row_mirror
  v = op(v, __shfl_xor(v, 16));
  return op(v, __shfl_xor(v, 32));
}

// ... and over the kRowWaves waves of a row, through LDS; every thread of the block calls it.
template <int kRowWaves, typename T, typename Op>
__device__ __forceinline__ T row_reduce(T v, T (&slot)[4], Op op) {
  v = wave_reduce(v, op);
  if constexpr (kRowWaves > 1) {
    const int wave = threadIdx.x >> 6, first = wave / kRowWaves * kRowWaves;
    if ((threadIdx.x & 63) == 0) slot[wave] = v;
    __syncthreads();
    v = slot[first];
#pragma unroll
    for (int i = 1; i < kRowWaves; ++i) v = op(v, slot[first + i]);
  }
  return v;
}

// One activation of a quantisation launch (rows of M tokens, all of width K).
struct QuantProblem {
  const uint16_t* x;
  int64_t x_stride;
  const float* inv_s;
  int M;
  int8_t* xq;
  float* a_scale;
  const uint16_t* shift;    // kModulate: modulation rows of each batch entry
  const uint16_t* scale;
  int64_t mod_stride;
  int tokens_per_batch;
  uint16_t* x_mod;          // kModulate: optional store of the modulated input
  int64_t x_mod_stride;
};

// Up to two activations in one launch (a double block's text and image streams): blocks
// [0, first_blocks) take p[0], the rest p[1]; 4 / kRowWaves rows per block.
struct QuantGroup {
  QuantProblem p[2];
  int first_blocks;
  int K;
};

// Activation (per forward): kRowWaves waves per token row, the row held in registers
// (kChunks x 8 elements per lane), its sums and its absmax reduced across the waves.
//
// kModulate: the row is first the block input x and becomes the projection input
//   X = bf16(bf16((bf16(1 + scale) * bf16(layer_norm(x)))) + shift)      (modules.py:38-40)
// with layer_norm(x) = bf16((x - mean) * (1 / sqrt(var + 1e-6))) (nn.py:17-21), the mean and
// the variance each summed in float64 and rounded to float32 once (bf16 inputs make the f64
// sum of the row exact, so the mean does not depend on the summation order), every other
// step one f32 operation.  scale / shift are the modulation rows of the token's batch entry;
// X is optionally stored (bf16) for other consumers of the modulated input.
//
// What bounds it is the latency of the chain load -> sum -> sum -> absmax -> codes and the L2
// reads of the modulation and the factors (8 bytes a channel for 2 of x), then VALU work: every
// load is issued before the first reduction, reductions cross lanes by DPP, and a code takes
// five instructions (quantize4).  Two rows per wave, which share those reads, gain only past
// ~9000 rows (4%) and lose up to 15% below.
//
// kFull: the lanes' chunks end with the row (K = 512 kRowWaves kChunks).
template <int kRowWaves, int kChunks, bool kFull, bool kModulate>
__global__ __launch_bounds__(256) void quantize_act_kernel(const QuantGroup grp) {
  __shared__ double sums[4], squares[4];
  __shared__ float maxima[4];
  const bool second = (int)blockIdx.x >= grp.first_blocks;
  const QuantProblem& P = second ? grp.p[1] : grp.p[0];   // wave-uniform, read from the kernel arguments
  const int M = P.M, K = grp.K;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int block = (int)blockIdx.x - (second ? grp.first_blocks : 0);
  const int64_t row_id = (int64_t)block * (4 / kRowWaves) + wave / kRowWaves;
  const bool live = row_id < M;               // waves past the end repeat the last row and store nothing
  const int row = live ? (int)row_id : M - 1;
  const int nch = K >> 3;
  const int first = wave % kRowWaves * 64 + lane;   // the lane's chunks: first, first + 64 kRowWaves, ...
  auto chunk = [&](int c) { return first + c * 64 * kRowWaves; };
  auto valid = [&](int c) { return kFull || chunk(c) < nch; };

  // Every load unconditional (a chunk past the row's end re-reads chunk 0 and counts as zeros).
  // x is read once: nontemporal loads cost a cached x 1.6 us at 4608 x 3072, but leave the caches
  // to the codes and the weight (3473 tokens, modulated, then projected: 118.0 -> 114.7 us).
  uint4 raw[kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const u32x4* src = reinterpret_cast<const u32x4*>(P.x + (int64_t)row * P.x_stride);
    const u32x4 v = __builtin_nontemporal_load(src + (valid(c) ? chunk(c) : 0));
    raw[c] = uint4{v.x, v.y, v.z, v.w};
  }
  uint32_t shift[kChunks][4], plus[kChunks][4];   // bf16 pairs: shift and bf16(1 + scale)
  if constexpr (kModulate) {
    const int64_t b = row / P.tokens_per_batch;
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const int at = valid(c) ? chunk(c) : 0;
      const uint4 sh = reinterpret_cast<const uint4*>(P.shift + b * P.mod_stride)[at];
      const uint4 sc = reinterpret_cast<const uint4*>(P.scale + b * P.mod_stride)[at];
      const uint32_t sw[4] = {sh.x, sh.y, sh.z, sh.w}, tw[4] = {sc.x, sc.y, sc.z, sc.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        shift[c][i] = sw[i];
        plus[c][i] = flk::pack_bf16x2(1.0f + flk::bf16_lo(tw[i]), 1.0f + flk::bf16_hi(tw[i]));
      }
    }
  }
  f32x4 si[kChunks][2];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int at = valid(c) ? chunk(c) : 0;
    si[c][0] = reinterpret_cast<const f32x4*>(P.inv_s)[2 * at];
    si[c][1] = reinterpret_cast<const f32x4*>(P.inv_s)[2 * at + 1];
  }
  float xr[kChunks][8];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    if (!valid(c)) raw[c] = uint4{0, 0, 0, 0};
    unpack_bf16x8(raw[c], xr[c]);
  }

  if constexpr (kModulate) {
    auto add = [](double p, double q) { return p + q; };
    double sum = 0.0, ssq = 0.0;
#pragma unroll
    for (int c = 0; c < kChunks; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += (double)xr[c][i];
    const float mean = (float)(row_reduce<kRowWaves>(sum, sums, add) / (double)K);
#pragma unroll
    for (int c = 0; c < kChunks; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        xr[c][i] = xr[c][i] - mean;
        const float sq = xr[c][i] * xr[c][i];
        ssq += (double)(valid(c) ? sq : 0.0f);
      }
    const float var = (float)(row_reduce<kRowWaves>(ssq, squares, add) / (double)K);
    const float inv = 1.0f / sqrtf(var + 1e-6f);
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      uint32_t out[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t base = flk::pack_bf16x2(xr[c][2 * i] * inv, xr[c][2 * i + 1] * inv);
        const uint32_t prod = flk::pack_bf16x2(flk::bf16_lo(plus[c][i]) * flk::bf16_lo(base),
                                               flk::bf16_hi(plus[c][i]) * flk::bf16_hi(base));
        out[i] = flk::pack_bf16x2(flk::bf16_lo(prod) + flk::bf16_lo(shift[c][i]),
                                  flk::bf16_hi(prod) + flk::bf16_hi(shift[c][i]));
        xr[c][2 * i] = valid(c) ? flk::bf16_lo(out[i]) : 0.0f;
        xr[c][2 * i + 1] = valid(c) ? flk::bf16_hi(out[i]) : 0.0f;
      }
      if (P.x_mod && live && valid(c))
        reinterpret_cast<uint4*>(P.x_mod + (int64_t)row * P.x_mod_stride)[chunk(c)] =
            uint4{out[0], out[1], out[2], out[3]};
    }
  }

  float amax = 0.0f;
#pragma unroll
  for (int c = 0; c < kChunks; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      xr[c][i] *= si[c][i >> 2][i & 3];
      amax = fmaxf(amax, fabsf(xr[c][i]));
    }
  const float a = absmax_scale(row_reduce<kRowWaves>(amax, maxima, [](float p, float q) { return fmaxf(p, q); }));
  const float ra = 1.0f / a;
  if (!live) return;
  uint2* dst = reinterpret_cast<uint2*>(P.xq + (int64_t)row * K);
#pragma unroll
  for (int c = 0; c < kChunks; ++c)
    if (valid(c)) {
      const float lo[4] = {xr[c][0], xr[c][1], xr[c][2], xr[c][3]}, hi[4] = {xr[c][4], xr[c][5], xr[c][6], xr[c][7]};
      dst[chunk(c)] = uint2{quantize4(lo, a, ra), quantize4(hi, a, ra)};
    }
  if (first == 0) P.a_scale[row] = a;
}

// ---------------------------------------------------------------- GEMM -----------------

constexpr int kGT = 256;                 // tile edge: tokens and output channels
constexpr int kGK = 128;                 // k bytes per stage: one full 128-byte line per row
constexpr int kGHalf = kGT * kGK;        // one operand's stage: 32 KiB
constexpr int kGStage = 2 * kGHalf;      // WqT rows, then Xq rows; two stages fill 128 KiB
constexpr int kGWaves = 8;               // two waves per SIMD
constexpr int kGThreads = kGWaves * 64;
constexpr int kGWaveN = 128;             // a wave's output channels (8 fragments of 16)
constexpr int kGNF = kGWaveN / 16;       // channel fragments per wave
constexpr int kGCopies = kGT / kGWaves / 8;   // WqT copy instructions per wave and stage (4)
constexpr int kGT192 = 192;              // token edge of the tiles that re-tile a partial last round
constexpr int kGRing = 4;                // channel-fragment registers in flight
constexpr int kMaxDim = INT32_MAX - kGT;  // largest token / channel count: a tile past it stays within int
constexpr int kGLead = 3;                // groups between a channel fragment's read and its MFMAs
static_assert(kGNF % kGRing == 0 && kGRing > kGLead, "the fragment ring must divide the groups of a step");
#ifndef FLK_GEMM_GROUP
#define FLK_GEMM_GROUP 4
#endif
constexpr int kGroup = FLK_GEMM_GROUP;   // token tiles that sweep the channel tiles together
constexpr int kXcds = 8;
constexpr int kCUs = 256;                // MI355X compute units

// LDS slot of 16-byte chunk c in row r is c ^ gswz(r).  gfx950's LDS serves 256 B per clock
// from 64 banks, i.e. two 128-byte operand rows; a b128 read is served as lanes 0-7 with
// 32-39, 8-15 with 40-47, and so on.  An operand read takes rows r0 .. r0+15 (lane % 16) and
// chunks 4 ks + perm(lane / 16), perm = 0, 2, 1, 3: lanes l and l + 32 then read chunks c and
// c ^ 1 of the same 8 rows, which the swizzle spreads over the 16 slots of a bank line (as it
// does the 16 rows of lanes l .. l + 15).
__device__ __forceinline__ int gswz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

__device__ __forceinline__ const uint8_t* a_frag(const uint8_t* stage, int nf, int wn) {
  return stage + (wn * kGWaveN + nf * 16) * kGK;
}
template <int kWaveM>
__device__ __forceinline__ const uint8_t* b_frag(const uint8_t* stage, int mf, int wm) {
  return stage + kGHalf + (wm * kWaveM + mf * 16) * kGK;
}

// The fused epilogue's qk_prep parameters (see flk_w8a8_qk_prep): output row m of the
// projection is token t = m % length of batch b = m / length, and its 128-channel head
// groups are q heads 0..H-1, then k heads, then v heads.
struct QkEpilogue {
  const float* cos;
  const float* sin;
  int64_t table_stride;
  const void* q_scale;
  const void* k_scale;
  float q_gain;
  int length, heads;
  uint16_t* out[3];
  int64_t out_length, out_offset;
};

// One projection Y = X W^T of a launch (xq M x K, wqt N x K), with its outputs.
struct GemmProblem {
  const int8_t* xq;
  const int8_t* wqt;
  const float* a_scale;
  const float* w_scale;
  uint16_t* y;            // plain epilogue: Y rows of y_stride elements
  int64_t y_stride;
  int32_t* acc_out;       // kAcc: the exact int32 products
  int M, K, N, tiles_m, tiles_n;
  QkEpilogue qe;          // kQk: qk_prep epilogue
};

// Up to two projections in one launch, so that a small one (a double block's 512 text
// tokens: 72 tiles) fills the CUs the large one (the image tokens) leaves idle in its last
// round.  Logical blocks [0, first_blocks) take p[0], the rest p[1].
struct GemmGroup {
  GemmProblem p[2];
  int first_blocks;
  int units;    // tiles of both problems (first_blocks + p[1]'s, or first_blocks alone)
  int rounds;   // rounds order (w8a8_gemm_kernel)
};

// The epilogue of a wave's 128 channels from nw x 16 kMF tokens from mw, of which tokens below
// m_limit are stored; out_lds holds 16 kMF rows of 256 bytes.  kAcc, kQk, kScaleF32 as for
// w8a8_gemm_kernel.
template <bool kAcc, bool kQk, bool kScaleF32, int kMF>
__device__ __forceinline__ void gemm_epilogue(uint8_t* out_lds, const GemmProblem& P, const i32x4 (&acc)[kGNF][kMF],
                                              int mw, int nw, int m_limit) {
  constexpr int kWaveM = 16 * kMF;
  const int lane = threadIdx.x & 63;
  const int l16 = lane & 15, h4 = lane >> 4;
  const float* __restrict__ a_scale = P.a_scale;
  const float* __restrict__ w_scale = P.w_scale;
  uint16_t* __restrict__ y = P.y;
  const int64_t y_stride = P.y_stride;
  int32_t* __restrict__ acc_out = P.acc_out;
  const int M = P.M, N = P.N;
  const QkEpilogue& qe = P.qe;
  if constexpr (kAcc) {
    // Exact int32 products, straight from the accumulators: the lane owns token l16 and
    // channels 4 * (lane / 16) .. +3 of each 16 x 16 fragment.
#pragma unroll
    for (int nf = 0; nf < kGNF; ++nf) {
      const int n = nw + nf * 16 + h4 * 4;
#pragma unroll
      for (int mf = 0; mf < kMF; ++mf) {
        const int m = mw + mf * 16 + l16;
        if (n < N && m < m_limit) *reinterpret_cast<i32x4*>(acc_out + (int64_t)m * N + n) = acc[nf][mf];
      }
    }
  }

  // Epilogue.  The lane owns token m = mf*16 + l16 and channels n = nf*16 + 4 h4 .. +3 of the
  // wave's 128 x 64 sub-tile.  Rescaled bf16 values go to this wave's 16 KiB of the (now
  // idle) LDS as [m][n] rows of 256 B whose 16-byte chunks are XOR-swizzled by m & 15; then
  // the wave reads back 4 rows per instruction (16 lanes x 16 B per row) and writes each
  // row's 256 contiguous bytes with 16-byte nontemporal stores (Y is streamed out: 1-2%
  // faster, and a qk_prep pass reading Y next measured no slower).
  float am[kMF];
#pragma unroll
  for (int mf = 0; mf < kMF; ++mf) am[mf] = a_scale[min(mw + mf * 16 + l16, M - 1)];
  __syncthreads();   // every wave is done reading the operand stages
#pragma unroll
  for (int nf = 0; nf < kGNF; ++nf) {
    // w_o of the lane's 4 channels (clamped at the edge; clamped values are never stored)
    const f32x4 w4 = *reinterpret_cast<const f32x4*>(w_scale + min(nw + nf * 16 + h4 * 4, N - 4));
#pragma unroll
    for (int mf = 0; mf < kMF; ++mf) {
      const int ml = mf * 16 + l16;
      const float y0 = ((float)acc[nf][mf][0] * am[mf]) * w4.x;
      const float y1 = ((float)acc[nf][mf][1] * am[mf]) * w4.y;
      const float y2 = ((float)acc[nf][mf][2] * am[mf]) * w4.z;
      const float y3 = ((float)acc[nf][mf][3] * am[mf]) * w4.w;
      uint2 packed;
      packed.x = flk::pack_bf16x2(y0, y1);
      packed.y = flk::pack_bf16x2(y2, y3);
      const int chunk = (nf * 2 + (h4 >> 1)) ^ (ml & 15);
      *reinterpret_cast<uint2*>(out_lds + ml * 256 + chunk * 16 + (h4 & 1) * 8) = packed;
    }
  }
  // Each wave reads back only what it wrote itself: its LDS writes complete in order before
  // its reads (the compiler waits on lgkmcnt), so no barrier is needed here.
  constexpr int kReads = kWaveM / 4;
  const int n_lane = nw + (lane & 15) * 8;
  if constexpr (kQk) {
    // The wave's 128 channels are one head of the q|k|v thirds (N = 3 H 128, tiles 128-aligned);
    // each 16-lane row of a read-back is one token's finished bf16 head row -- the input of
    // qk_prep, rounded exactly as the unfused path stores it in Y.
    const int head_g = nw / flk::kQkHeadDim;
    if (nw >= N) return;
    const int sec = head_g / qe.heads, h = head_g - sec * qe.heads;
    float sc[8];
    if (sec < 2) flk::load_scale8<kScaleF32>(sec == 0 ? qe.q_scale : qe.k_scale, l16, sc);
    uint16_t* const out = qe.out[sec];
    // Row m = b * length + t.  One division for the lane's first row; each read-back moves 4
    // rows on, which wraps into the next batch entry at most once when length >= 4 (shorter
    // sequences divide per row).  A division per row measured 2.4% of the fused kernel.
    const int len = qe.length;
    const bool short_seq = len < 4;
    const int m_first = mw + (lane >> 4);
    int b = m_first / len, t = m_first - b * len;
#pragma unroll 4
    for (int it = 0; it < kReads; ++it) {
      const int ml = it * 4 + (lane >> 4);
      const int m = mw + ml;
      if (it > 0) {
        if (short_seq) {
          b = m / len;
          t = m - b * len;
        } else {
          t += 4;
          if (t >= len) {
            t -= len;
            ++b;
          }
        }
      }
      const uint4 v = *reinterpret_cast<const uint4*>(out_lds + ml * 256 + ((l16 ^ (ml & 15)) * 16));
      if (m >= m_limit) continue;   // uniform over the 16-lane row, so the DPP rows stay whole
      uint4 r = v;
      if (sec < 2) {
        float c[8], s[8];
        flk::load_table8(qe.cos + (int64_t)t * qe.table_stride, l16, c);
        flk::load_table8(qe.sin + (int64_t)t * qe.table_stride, l16, s);
        r = sec == 0 ? flk::norm_rotate<kScaleF32, true>(v, sc, c, s, qe.q_gain)
                     : flk::norm_rotate<kScaleF32, false>(v, sc, c, s, 1.0f);
      }
      const int64_t o = (((int64_t)b * qe.heads + h) * qe.out_length + qe.out_offset + t) * flk::kQkHeadDim + l16 * 8;
      *reinterpret_cast<uint4*>(out + o) = r;
    }
    return;
  }
  const bool wide = (y_stride & 7) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;   // 16-byte rows
#pragma unroll 8
  for (int it = 0; it < kReads; ++it) {
    const int ml = it * 4 + (lane >> 4);
    const uint4 v = *reinterpret_cast<const uint4*>(out_lds + ml * 256 + (((lane & 15) ^ (ml & 15)) * 16));
    const int m = mw + ml;
    if (m < m_limit && n_lane < N) {
      uint16_t* dst = y + (int64_t)m * y_stride + n_lane;
      if (wide && n_lane + 8 <= N) {
        __builtin_nontemporal_store(u32x4{v.x, v.y, v.z, v.w}, reinterpret_cast<u32x4*>(dst));
      } else {
        *reinterpret_cast<uint2*>(dst) = uint2{v.x, v.y};
        if (n_lane + 8 <= N) *reinterpret_cast<uint2*>(dst + 4) = uint2{v.z, v.w};
      }
    }
  }
}

// One output tile: channels n0 .. n0 + 255 and tokens m0 .. m0 + 64 kMF - 1 (kMF = 4: 256
// tokens; 3: 192), of which tokens below m_limit are stored.  Each of the 2 (channels) x 4
// (tokens) waves holds 128 channels x 16 kMF tokens.  kAcc, kQk, kScaleF32 as for
// w8a8_gemm_kernel.
template <bool kAcc, bool kQk, bool kScaleF32, int kMF>
__device__ __forceinline__ void gemm_tile(uint8_t* smem, const GemmProblem& P, int m0, int n0, int m_limit) {
  constexpr int kWaveM = 16 * kMF;   // a wave's tokens
  constexpr int kBCopies = kMF;      // Xq copy instructions per wave and stage (8 kMF rows)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int8_t* __restrict__ xq = P.xq;
  const int8_t* __restrict__ wqt = P.wqt;
  const int M = P.M, K = P.K, N = P.N;

  // Copy sources: this wave fills rows wave*32 .. +31 of WqT and wave*8kMF .. +8kMF-1 of Xq,
  // 8 rows (64 lanes x 16 B) per instruction; lane i lands at row i/8, slot i%8, and fetches
  // chunk slot^gswz.
  // Rows past the matrix edge repeat the last row (their results are never stored).  The
  // tile's first row (plus the stage's k offset) is a scalar base; lanes add 32-bit offsets.
  const int8_t* abase = wqt + (int64_t)n0 * K;
  const int8_t* bbase = xq + (int64_t)m0 * K;
  uint32_t aoff[kGCopies], boff[kBCopies];
#pragma unroll
  for (int i = 0; i < kGCopies; ++i) {
    const int row = wave * (kGT / kGWaves) + i * 8 + (lane >> 3);
    aoff[i] = (uint32_t)min(row, N - 1 - n0) * (uint32_t)K + (uint32_t)(((lane & 7) ^ gswz(row)) * 16);
  }
#pragma unroll
  for (int i = 0; i < kBCopies; ++i) {
    const int row = wave * 8 * kMF + i * 8 + (lane >> 3);
    boff[i] = (uint32_t)min(row, M - 1 - m0) * (uint32_t)K + (uint32_t)(((lane & 7) ^ gswz(row)) * 16);
  }
  uint8_t* const a_lds = smem + wave * (kGT / kGWaves) * kGK;   // this wave's WqT rows in stage 0
  uint8_t* const b_lds = smem + kGHalf + wave * 8 * kMF * kGK;  // ... and its Xq rows

  const int KT = K / kGK;
  const int wn = wave >> 2, wm = wave & 3;     // 2 (channels) x 4 (tokens) waves
  const int l16 = lane & 15, h4 = lane >> 4;
  const int hperm = ((h4 & 1) << 1) | (h4 >> 1);
  int off[2];   // fragment read offsets of k steps 0, 1: row l16, chunk 4 ks + perm(lane / 16)
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) off[ks] = l16 * kGK + (((4 * ks + hperm) ^ gswz(l16)) * 16);

  i32x4 acc[kGNF][kMF];
#pragma unroll
  for (int a = 0; a < kGNF; ++a)
#pragma unroll
    for (int b = 0; b < kMF; ++b) acc[a][b] = i32x4{};

  // Two stages of 128 k bytes, two 64-byte k steps each.  Stage kt: step 0 reads step 1's
  // fragments as it goes; step 1 reads its own last channel fragments in groups 0-4, then --
  // every wave done reading stage kt, stage kt+1 landed everywhere (the barrier) -- refills
  // stage kt's buffer with stage kt+2 and reads stage kt+1's first fragments in groups 5-7.
  // Past the last stage the copies repeat it (into the buffer no later step reads), so
  // every stage issues the same copies and vmcnt(0) is exact.
  const int k1 = min(1, KT - 1) * kGK;
  auto copy_stage = [&](int k_off, int buf) {   // WqT and Xq copies alternating
#pragma unroll
    for (int i = 0; i < kGCopies; ++i) {
      flk::dma16_at(abase + k_off, aoff[i], a_lds + buf * kGStage + i * 8 * kGK);
      if (i < kBCopies) flk::dma16_at(bbase + k_off, boff[i], b_lds + buf * kGStage + i * 8 * kGK);
    }
  };
  copy_stage(0, 0);
  copy_stage(k1, 1);
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kGCopies + kBCopies) : "memory");   // stage 0 landed
  __syncthreads();
  i32x4 ring[kGRing], b0[kMF], b1[kMF];
#pragma unroll
  for (int mf = 0; mf < kMF; ++mf) b0[mf] = *reinterpret_cast<const i32x4*>(b_frag<kWaveM>(smem, mf, wm) + off[0]);
#pragma unroll
  for (int nf = 0; nf < kGLead; ++nf) ring[nf] = *reinterpret_cast<const i32x4*>(a_frag(smem, nf, wn) + off[0]);

  auto mfma_group = [&](int nf, const i32x4 (&b)[kMF]) {
#pragma unroll
    for (int mf = 0; mf < kMF; ++mf)
      acc[nf][mf] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[nf % kGRing], b[mf], acc[nf][mf], 0, 0, 0);
  };
  auto afrag = [&](const uint8_t* st, int nf, int o) { return *reinterpret_cast<const i32x4*>(a_frag(st, nf, wn) + o); };
  auto bfrag = [&](const uint8_t* st, int mf, int o) { return *reinterpret_cast<const i32x4*>(b_frag<kWaveM>(st, mf, wm) + o); };

  for (int kt = 0; kt < KT; ++kt) {
    const uint8_t* cs = smem + (kt & 1) * kGStage;          // stage kt
    const uint8_t* ns = smem + ((kt + 1) & 1) * kGStage;    // stage kt+1
    const int k_next = min(kt + 2, KT - 1) * kGK;
    // step 0
#pragma unroll
    for (int nf = 0; nf < kGNF; ++nf) {
      mfma_group(nf, b0);
      const int nl = nf + kGLead;
      ring[nl % kGRing] = nl < kGNF ? afrag(cs, nl, off[0]) : afrag(cs, nl - kGNF, off[1]);
      if (nf < kMF) b1[nf] = bfrag(cs, nf, off[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // step 1, groups reading stage kt
#pragma unroll
    for (int nf = 0; nf < kGNF - kGLead; ++nf) {
      mfma_group(nf, b1);
      ring[(nf + kGLead) % kGRing] = afrag(cs, nf + kGLead, off[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // stage kt read, kt+1 landed
    copy_stage(k_next, kt & 1);
    // step 1, groups reading stage kt+1 (its step 0 fragments)
#pragma unroll
    for (int nf = kGNF - kGLead; nf < kGNF; ++nf) {
      mfma_group(nf, b1);
      ring[(nf + kGLead) % kGRing] = afrag(ns, nf + kGLead - kGNF, off[0]);
      const int j = nf - (kGNF - kGLead);           // 0, 1, 2
      if constexpr (kMF == 4) {                     // token fragments 0-1, 2, 3
        if (j == 0) {
          b0[0] = bfrag(ns, 0, off[0]);
          b0[1] = bfrag(ns, 1, off[0]);
        } else {
          b0[j + 1] = bfrag(ns, j + 1, off[0]);
        }
      } else {                                      // token fragments 0, 1, 2
        b0[j] = bfrag(ns, j, off[0]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  gemm_epilogue<kAcc, kQk, kScaleF32, kMF>(smem + wave * (kWaveM * 256), P, acc, m0 + wm * kWaveM,
                                           n0 + wn * kGWaveN, m_limit);
}

// The same product for launches whose 256 x 256 tiles leave most CUs idle: tiles of 128 channels x
// 32 kWM tokens, taken by 2 kWM waves.  A 128 x 32 position is held by two waves that take the two
// 64-byte halves of every 128-byte k stage; their int32 sums (exact in any order) are exchanged
// through LDS at the end, each wave finishing 16 of the 32 tokens.  Few blocks run a serial chain
// of stages, so what bounds it is a stage's latency: two waves per SIMD on one position halve the
// chain's MFMAs per wave (four waves with whole stages: 27 us against 22.6 at 512 tokens).
template <bool kAcc, bool kQk, bool kScaleF32, int kWM, int kBuffers>
__device__ __forceinline__ void gemm_tile_split(uint8_t* smem, const GemmProblem& P, int m0, int n0, int m_limit) {
  constexpr int kMF = 2, kWaveM = 16 * kMF, kWaves = 2 * kWM, kTM = kWM * kWaveM;
  constexpr int kABytes = kGWaveN * kGK, kStage = kABytes + kTM * kGK;
  constexpr int kAC = kGWaveN / 8 / kWaves, kBC = kTM / 8 / kWaves;   // copies per wave and stage (8 rows each)
  static_assert(kGWaveN % (8 * kWaves) == 0 && kTM % (8 * kWaves) == 0, "whole copies per wave");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int M = P.M, K = P.K, N = P.N;
  const int8_t* abase = P.wqt + (int64_t)n0 * K;
  const int8_t* bbase = P.xq + (int64_t)m0 * K;
  uint32_t aoff[kAC], boff[kBC];
#pragma unroll
  for (int i = 0; i < kAC; ++i) {
    const int row = (wave * kAC + i) * 8 + (lane >> 3);
    aoff[i] = (uint32_t)min(row, N - 1 - n0) * (uint32_t)K + (uint32_t)(((lane & 7) ^ gswz(row)) * 16);
  }
#pragma unroll
  for (int i = 0; i < kBC; ++i) {
    const int row = (wave * kBC + i) * 8 + (lane >> 3);
    boff[i] = (uint32_t)min(row, M - 1 - m0) * (uint32_t)K + (uint32_t)(((lane & 7) ^ gswz(row)) * 16);
  }
  const int kg = wave / kWM, wm = wave % kWM;   // half of the k stages, 32-token position
  const int l16 = lane & 15, h4 = lane >> 4;
  const int hperm = ((h4 & 1) << 1) | (h4 >> 1);
  const int off = l16 * kGK + (((4 * kg + hperm) ^ gswz(l16)) * 16);
  const int b_off = off + kABytes + wm * kWaveM * kGK;

  i32x4 acc[kGNF][kMF];
#pragma unroll
  for (int a = 0; a < kGNF; ++a)
#pragma unroll
    for (int b = 0; b < kMF; ++b) acc[a][b] = i32x4{};

  const int KT = K / kGK;
  auto copy_stage = [&](int kt, uint8_t* dst) {
    const int k_off = min(kt, KT - 1) * kGK;
#pragma unroll
    for (int i = 0; i < kAC; ++i) flk::dma16_at(abase + k_off, aoff[i], dst + (wave * kAC + i) * 8 * kGK);
#pragma unroll
    for (int i = 0; i < kBC; ++i) flk::dma16_at(bbase + k_off, boff[i], dst + kABytes + (wave * kBC + i) * 8 * kGK);
  };
#pragma unroll
  for (int i = 0; i < kBuffers; ++i) copy_stage(i, smem + i * kStage);
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"((kBuffers - 1) * (kAC + kBC)) : "memory");
  __syncthreads();
  auto afrag = [&](const uint8_t* st, int nf) { return *reinterpret_cast<const i32x4*>(st + off + nf * 16 * kGK); };
  auto bfrag = [&](const uint8_t* st, int mf) { return *reinterpret_cast<const i32x4*>(st + b_off + mf * 16 * kGK); };
  i32x4 ring[kGRing], b0[kMF], b1[kMF];
#pragma unroll
  for (int mf = 0; mf < kMF; ++mf) b0[mf] = bfrag(smem, mf);
#pragma unroll
  for (int nf = 0; nf < kGLead; ++nf) ring[nf] = afrag(smem, nf);

  int cb = 0;   // byte offset of stage kt's buffer
  auto step = [&](int kt, i32x4 (&b)[kMF], i32x4 (&bn)[kMF]) {
    uint8_t* cs = smem + cb;
    cb = cb == (kBuffers - 1) * kStage ? 0 : cb + kStage;
    const uint8_t* ns = smem + cb;
#pragma unroll
    for (int nf = 0; nf < kGNF; ++nf) {
#pragma unroll
      for (int mf = 0; mf < kMF; ++mf)
        acc[nf][mf] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[nf % kGRing], b[mf], acc[nf][mf], 0, 0, 0);
      const int nl = nf + kGLead;
      ring[nl % kGRing] = nl < kGNF ? afrag(cs, nl) : afrag(ns, nl - kGNF);
      if (nf >= kGNF - kGLead) {
        const int j = nf - (kGNF - kGLead);
#pragma unroll
        for (int mf = 0; mf < kMF; ++mf)
          if (mf * kGLead / kMF == j) bn[mf] = bfrag(ns, mf);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (nf == kGNF - kGLead - 1) {
        // every wave has read stage kt; stage kt+1 has landed everywhere
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((kBuffers - 2) * (kAC + kBC)) : "memory");
        copy_stage(kt + kBuffers, cs);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  int kt = 0;
  for (; kt + 2 <= KT; kt += 2) {
    step(kt, b0, b1);
    step(kt + 1, b1, b0);
  }
  if (kt < KT) step(kt, b0, b1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // Wave kg of a position keeps token fragment kg and gives the other one away.
  i32x4* const sums = reinterpret_cast<i32x4*>(smem) + lane;
  constexpr int kSum = kGNF * 64;   // one wave's fragments
  static_assert(kWaves * kSum * 16 <= kBuffers * kStage, "the exchanged sums fit the idle stages");
  i32x4 sum[kGNF][1];
#pragma unroll
  for (int nf = 0; nf < kGNF; ++nf) {
    sums[wave * kSum + nf * 64] = kg ? acc[nf][0] : acc[nf][1];
    sum[nf][0] = kg ? acc[nf][1] : acc[nf][0];
  }
  __syncthreads();
#pragma unroll
  for (int nf = 0; nf < kGNF; ++nf) sum[nf][0] += sums[((1 - kg) * kWM + wm) * kSum + nf * 64];
  gemm_epilogue<kAcc, kQk, kScaleF32, 1>(smem + wave * (16 * 256), P, sum, m0 + wm * kWaveM + kg * 16, n0, m_limit);
}

// Logical tile u of a problem -> its token and channel tiles: kGroup token tiles sweep the
// channel tiles together (consecutive logical tiles share a channel tile's WqT rows).
__device__ __forceinline__ void tile_of(int u, int tiles_m, int tiles_n, int& mt, int& nt) {
  const int group_tiles = kGroup * tiles_n;
  const int group = u / group_tiles;
  const int first_m = group * kGroup;
  const int gm = min(kGroup, tiles_m - first_m);
  const int in_group = u - group * group_tiles;
  mt = first_m + in_group % gm;
  nt = in_group / gm;
}

// The rounds order's 192-token tiles: logical tiles [first, end) of a launch's problems (p[0]'s
// tiles, then p[1]'s) taken as runs of one channel tile (consecutive token tiles of one group
// of one problem), each run's tokens cut into 192-token tiles, the last one short.  The j-th
// such tile, or false past the last.  The host's gemm_rounds_grid counts them the same way.
__device__ __forceinline__ bool leftover_tile(const GemmGroup& grp, int first, int end, int j, int& second, int& m0,
                                              int& n0, int& m_end) {
  for (int u = first; u < end;) {
    second = u >= grp.first_blocks;
    const GemmProblem& P = second ? grp.p[1] : grp.p[0];
    const int base = second ? grp.first_blocks : 0;
    const int p_end = second ? end : min(end, grp.first_blocks);
    const int group_tiles = kGroup * P.tiles_n;
    const int group = (u - base) / group_tiles;
    const int first_m = group * kGroup;
    const int gm = min(kGroup, P.tiles_m - first_m);
    const int in_group = u - base - group * group_tiles;
    const int r = in_group % gm;
    const int run = min(gm - r, p_end - u);
    const int s = (first_m + r) * kGT, e = min((first_m + r + run) * kGT, P.M);
    const int count = (e - s + kGT192 - 1) / kGT192;
    if (j < count) {
      m0 = s + j * kGT192;
      m_end = min(m0 + kGT192, e);
      n0 = (in_group / gm) * kGT;
      return true;
    }
    j -= count;
    u += run;
  }
  return false;
}

// kAcc: also write the exact int32 products (a test and debugging path).
// kQk: instead of Y, run qk_prep on each finished bf16 head row (kScaleF32: float32 norm
// scales) and write head-major q, k, v.
template <bool kAcc, bool kQk = false, bool kScaleF32 = false>
__global__ __launch_bounds__(kGThreads, 2) void w8a8_gemm_kernel(const GemmGroup grp) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kGStage];
  const int xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;   // blocks are dealt round-robin over XCDs
  if (grp.rounds) {
    // Rounds order: each XCD takes a contiguous range of the logical tiles (of one problem,
    // then the next), runs whole rounds of 32 of them, and cuts the ones left over into
    // 192-token tiles, so the partial last round has up to 4/3 as many blocks with 3/4 of the
    // work each.
    constexpr int C = kCUs / kXcds;
    const int ux0 = (int)((int64_t)xcd * grp.units / kXcds);
    const int n = (int)((int64_t)(xcd + 1) * grp.units / kXcds) - ux0;
    const int full = n / C * C;
    if (local < full) {
      const int u = ux0 + local;
      const bool second = u >= grp.first_blocks;
      const GemmProblem& P = second ? grp.p[1] : grp.p[0];
      int mt, nt;
      tile_of(u - (second ? grp.first_blocks : 0), P.tiles_m, P.tiles_n, mt, nt);
      gemm_tile<kAcc, kQk, kScaleF32, 4>(smem, P, mt * kGT, nt * kGT, P.M);
      return;
    }
    int second, m0, n0, m_end;
    if (!leftover_tile(grp, ux0 + full, ux0 + n, local - full, second, m0, n0, m_end)) return;
    gemm_tile<kAcc, kQk, kScaleF32, 3>(smem, second ? grp.p[1] : grp.p[0], m0, n0, m_end);
    return;
  }
  // Tile order: renumber so that each XCD runs a contiguous range of logical tiles (of one
  // problem, then the next).
  const int nblocks = gridDim.x;
  const int per = nblocks / kXcds, extra = nblocks % kXcds;
  const int logical_all = xcd * per + min(xcd, extra) + local;
  const bool second = logical_all >= grp.first_blocks;
  const GemmProblem& P = second ? grp.p[1] : grp.p[0];   // wave-uniform, read from the kernel arguments
  int mt, nt;
  tile_of(logical_all - (second ? grp.first_blocks : 0), P.tiles_m, P.tiles_n, mt, nt);
  gemm_tile<kAcc, kQk, kScaleF32, 4>(smem, P, mt * kGT, nt * kGT, P.M);
}

// A launch of few tiles (launch_group): one tile of 128 channels x 32 kWM tokens per block, through
// kBuffers LDS stages, kPerCU blocks to a CU.
template <bool kAcc, bool kQk, bool kScaleF32, int kWM, int kBuffers, int kPerCU>
__global__ __launch_bounds__(kWM * 128, kPerCU * kWM / 2) void w8a8_gemm_split_kernel(const GemmGroup grp) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kBuffers * (kGWaveN + 32 * kWM) * kGK];
  const int xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;   // blocks are dealt round-robin over XCDs
  const int per = gridDim.x / kXcds, extra = gridDim.x % kXcds;
  const int logical = xcd * per + min(xcd, extra) + local;
  const bool second = logical >= grp.first_blocks;
  const GemmProblem& P = second ? grp.p[1] : grp.p[0];   // wave-uniform, read from the kernel arguments
  int mt, nt;
  tile_of(logical - (second ? grp.first_blocks : 0), P.tiles_m, P.tiles_n, mt, nt);
  gemm_tile_split<kAcc, kQk, kScaleF32, kWM, kBuffers>(smem, P, mt * 32 * kWM, nt * kGWaveN, P.M);
}

inline hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }

// Rows per block of a column-maximum launch with `blocks` blocks of 128 columns: one pass of
// kColRows rows while the grid stays under ~8 blocks per CU, more passes beyond that.
int64_t column_rows(int64_t rows, int64_t blocks) {
  const int64_t cuts = std::max<int64_t>(1, 8 * kCUs / blocks);
  const int64_t per = (rows + cuts - 1) / cuts;
  return (per + kColRows - 1) / kColRows * kColRows;
}

// Rows of a column maximum that one block per 128 columns takes in one launch: up to 512 rows are
// four passes of its loads, less than a second launch costs (us at 3072 columns, cuts and one
// block: 128 rows 4.2 / 2.6, 256 4.2 / 2.9, 512 4.2 / 3.7; 8 columns 4.6 / 5.4 at 512).
constexpr int64_t kOneCutRows = 4 * kColRows;

}  // namespace

namespace {

int check_rows(const void* x, int64_t rows, int64_t cols, int64_t row_stride, const float* out) {
  if (rows < 0 || cols < 0 || row_stride < cols) return FLK_E_INVALID;
  if (rows == 0) return FLK_OK;
  if (!x || !out || cols == 0) return FLK_E_INVALID;
  if (cols % 8 || row_stride % 8 || !flk_host_aligned(x, 16) || !flk_host_aligned(out, 4)) return FLK_E_ALIGN;
  return (rows + 3) / 4 > INT32_MAX ? FLK_E_INVALID : FLK_OK;
}

// As many loads in flight per lane as a row has chunks of 512, six for longer rows (six for all, us:
// 8192 x 64 4.3 against 3.1, 3072 x 128 3.0 / 2.5, 8192 x 1544 4.4 / 3.9).
template <bool kSmooth>
void launch_absmax_rows(const uint16_t* x, int64_t rows, int64_t cols, int64_t stride, float* out, const float* xa,
                        float* inv, void* stream) {
#define FLK_ROWS(U)                                                                                              \
  hipLaunchKernelGGL((absmax_rows_kernel<U, kSmooth>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0,           \
                     as_stream(stream), x, rows, cols, stride, out, xa, inv)
  switch ((cols + 511) / 512) {
    case 0: case 1: FLK_ROWS(1); break;
    case 2: FLK_ROWS(2); break;
    case 3: FLK_ROWS(3); break;
    case 4: FLK_ROWS(4); break;
    default: FLK_ROWS(6); break;
  }
#undef FLK_ROWS
}

}  // namespace

extern "C" int flk_absmax_rows(const void* x, int64_t rows, int64_t cols, int64_t row_stride, float* out,
                               void* stream) {
  const int st = check_rows(x, rows, cols, row_stride, out);
  if (st != FLK_OK || rows == 0) return st;
  launch_absmax_rows<false>(static_cast<const uint16_t*>(x), rows, cols, row_stride, out, nullptr, nullptr, stream);
  return flk_launch_status();
}

extern "C" int flk_weight_smooth(const void* w, int64_t k, int64_t n, int64_t w_row_stride, const float* x_absmax,
                                 float* s, float* inv_s, void* stream) {
  const int st = check_rows(w, k, n, w_row_stride, s);
  if (st != FLK_OK || k == 0) return st;
  if (!x_absmax || !inv_s) return FLK_E_INVALID;
  if (!flk_host_aligned(x_absmax, 4) || !flk_host_aligned(inv_s, 4)) return FLK_E_ALIGN;
  launch_absmax_rows<true>(static_cast<const uint16_t*>(w), k, n, w_row_stride, s, x_absmax, inv_s, stream);
  return flk_launch_status();
}

extern "C" int flk_absmax_cols(const void* x, int64_t rows, int64_t cols, int64_t row_stride, int accumulate,
                               float* out, void* stream) {
  if (rows < 0 || cols < 0 || row_stride < cols) return FLK_E_INVALID;
  if (cols == 0 || (rows == 0 && accumulate)) return FLK_OK;
  if (!out || (rows > 0 && !x)) return FLK_E_INVALID;
  if (cols % 8 || row_stride % 8 || (x && !flk_host_aligned(x, 16)) || !flk_host_aligned(out, 4))
    return FLK_E_ALIGN;
  const int64_t blocks = (cols + 127) / 128;
  if (blocks > INT32_MAX) return FLK_E_INVALID;
  const uint16_t* xp = static_cast<const uint16_t*>(x);
  const hipStream_t st = as_stream(stream);
  // Few rows, or blocks that fill the chip without cuts (640 x 131072: two cuts 27.7 us, one 26.3).
  if (rows <= kOneCutRows || blocks >= 4 * kCUs) {
    hipLaunchKernelGGL(absmax_cols_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, st, xp, rows, cols, row_stride,
                       rows, accumulate, out);
    return flk_launch_status();
  }
  const int64_t per = column_rows(rows, blocks);
  hipLaunchKernelGGL(absmax_init_kernel, dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, st, cols, accumulate, out);
  hipLaunchKernelGGL(absmax_cols_kernel<true>, dim3((unsigned)blocks, (unsigned)((rows + per - 1) / per)), dim3(256), 0,
                     st, xp, rows, cols, row_stride, per, accumulate, out);
  return flk_launch_status();
}

extern "C" int flk_smooth_factors(const float* x_absmax, const float* w_absmax, int64_t k, float* s,
                                  float* inv_s, void* stream) {
  if (k < 0) return FLK_E_INVALID;
  if (k == 0) return FLK_OK;
  if (!x_absmax || !w_absmax || !s || !inv_s) return FLK_E_INVALID;
  const int64_t blocks = (k + 255) / 256;
  if (blocks > INT32_MAX) return FLK_E_INVALID;
  hipLaunchKernelGGL(smooth_factors_kernel, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), x_absmax,
                     w_absmax, k, s, inv_s);
  return flk_launch_status();
}

extern "C" int flk_quantize_weight(const void* w, int64_t w_row_stride, const float* s, int k, int n,
                                   int8_t* wq_t, float* w_scale, void* stream) {
  if (k < 0 || n < 0 || w_row_stride < n) return FLK_E_INVALID;
  if (k == 0 || n == 0) return FLK_OK;
  if (k > INT32_MAX - 64 || n > INT32_MAX - 64) return FLK_E_INVALID;   // a block's last row / column index
  if (!w || !s || !wq_t || !w_scale) return FLK_E_INVALID;
  if (k % 64 || n % 8 || w_row_stride % 8) return FLK_E_UNSUPPORTED;
  if (!flk_host_aligned(w, 16) || !flk_host_aligned(wq_t, 16) || !flk_host_aligned(s, 4) ||
      !flk_host_aligned(w_scale, 4))
    return FLK_E_ALIGN;
  const hipStream_t hs = as_stream(stream);
  const uint16_t* wp = static_cast<const uint16_t*>(w);
  const dim3 channels((unsigned)((n + 63) / 64));
#define FLK_SHORT(T) \
  hipLaunchKernelGGL(quantize_weight_short_kernel<T>, channels, dim3(256), 0, hs, wp, w_row_stride, s, k, n, wq_t, w_scale)
  if (k <= 512) {
    if (k <= 128) FLK_SHORT(1);
    else if (k <= 256) FLK_SHORT(2);
    else if (k <= 384) FLK_SHORT(3);
    else FLK_SHORT(4);
    return flk_launch_status();
  }
#undef FLK_SHORT
  const int64_t col_blocks = ((int64_t)n + 127) / 128;
  const int64_t per = column_rows(k, col_blocks);
  const int cuts = (int)(((int64_t)k + per - 1) / per);
  const int64_t k_tiles = std::min<int64_t>(((int64_t)k + 127) / 128, 65535);   // grid y
  float* part = reinterpret_cast<float*>(wq_t);
  hipLaunchKernelGGL(weight_absmax_kernel, dim3((unsigned)col_blocks, (unsigned)cuts), dim3(256), 0, hs, wp,
                     w_row_stride, s, k, n, per, part);
  hipLaunchKernelGGL(weight_scale_kernel, dim3((unsigned)(((int64_t)n + 255) / 256)), dim3(256), 0, hs, part, cuts, n,
                     w_scale);
  hipLaunchKernelGGL(quantize_weight_kernel, dim3((unsigned)((n + 63) / 64), (unsigned)k_tiles), dim3(256), 0, hs, wp,
                     w_row_stride, s, k, n, wq_t, w_scale);
  return flk_launch_status();
}

namespace {

// Waves that share a row of K elements: two for the hidden widths, so that a row's chain of
// reductions is half as long and twice the rows' loads are in flight (one wave per row,
// 4608 x 3072: 13.1 us, modulated 21.2; two: 10.4, 18.4; 512 rows: 5.2 -> 3.5).  A row of at most
// three chunks a lane is one wave: sharing it only adds the exchange (two waves, then one, us:
// 4608 x 1024 6.6 / 4.7, 67584 x 1024 62 / 35, modulated 113 / 71; 4608 x 1536 modulated
// 12.9 / 10.3; 512 x 1032 modulated 5.0 / 5.2 is the most it loses).
int row_waves(int k) { return k <= 1536 ? 1 : k <= 4096 ? 2 : 4; }

template <bool kModulate>
int launch_quantize_act(const QuantGroup& g, int64_t blocks, void* stream) {
  if (blocks > INT32_MAX) return FLK_E_INVALID;
  const int waves = row_waves(g.K);
  const int chunks = (g.K / 8 + 64 * waves - 1) / (64 * waves);
  const bool full = g.K == 512 * waves * chunks;
  const dim3 grid((unsigned)blocks), block(256);
  const hipStream_t st = as_stream(stream);
#define FLK_QA(W, C) \
  if (full) hipLaunchKernelGGL((quantize_act_kernel<W, C, true, kModulate>), grid, block, 0, st, g); \
  else hipLaunchKernelGGL((quantize_act_kernel<W, C, false, kModulate>), grid, block, 0, st, g)
  if (waves == 1 && chunks == 1) { FLK_QA(1, 1); }
  else if (waves == 1 && chunks == 2) { FLK_QA(1, 2); }
  else if (waves == 1) { FLK_QA(1, 3); }
  else if (waves == 2 && chunks == 2) { FLK_QA(2, 2); }
  else if (waves == 2 && chunks == 3) { FLK_QA(2, 3); }
  else if (waves == 2) { FLK_QA(2, 4); }
  else if (chunks <= 3) { FLK_QA(4, 3); }
  else { FLK_QA(4, 4); }
#undef FLK_QA
  return flk_launch_status();
}

// Status of a checked problem with nothing to launch (empty input).
constexpr int kNoWork = 1;

// Checks one modulated activation (flk_quantize_act_modulated's arguments) and fills its
// problem: FLK_OK, kNoWork, or an error status.
int modulated_problem(const void* x, int64_t x_row_stride, const void* shift, const void* scale,
                      int64_t mod_batch_stride, int tokens_per_batch, const float* inv_s, int m, int k, int8_t* xq,
                      float* a_scale, void* x_mod, int64_t x_mod_row_stride, QuantProblem& p) {
  if (m < 0 || k < 0 || x_row_stride < k || mod_batch_stride < 0 || (x_mod && x_mod_row_stride < k))
    return FLK_E_INVALID;
  if (m == 0 || k == 0) return kNoWork;   // an empty input (its sequence length may be 0 too)
  if (tokens_per_batch <= 0 || m > INT32_MAX - 4) return FLK_E_INVALID;
  if (!x || !shift || !scale || !inv_s || !xq || !a_scale) return FLK_E_INVALID;
  if ((m - 1) / tokens_per_batch > 0 && mod_batch_stride < k) return FLK_E_INVALID;
  if (k % 8 || k > 8192) return FLK_E_UNSUPPORTED;
  if (x_row_stride % 8 || mod_batch_stride % 8 || !flk_host_aligned(x, 16) || !flk_host_aligned(shift, 16) ||
      !flk_host_aligned(scale, 16) || !flk_host_aligned(inv_s, 16) || !flk_host_aligned(xq, 8) ||
      !flk_host_aligned(a_scale, 4) || (x_mod && (!flk_host_aligned(x_mod, 16) || x_mod_row_stride % 8)))
    return FLK_E_ALIGN;
  p = QuantProblem{static_cast<const uint16_t*>(x), x_row_stride, inv_s, m, xq, a_scale,
                   static_cast<const uint16_t*>(shift), static_cast<const uint16_t*>(scale), mod_batch_stride,
                   tokens_per_batch, static_cast<uint16_t*>(x_mod), x_mod_row_stride};
  return FLK_OK;
}

int64_t row_blocks(const QuantProblem& p, int k) {
  const int rows = 4 / row_waves(k);
  return ((int64_t)p.M + rows - 1) / rows;
}

}  // namespace

extern "C" int flk_quantize_act(const void* x, int64_t x_row_stride, const float* inv_s, int m, int k,
                                int8_t* xq, float* a_scale, void* stream) {
  if (m < 0 || k < 0 || x_row_stride < k) return FLK_E_INVALID;
  if (m == 0 || k == 0) return FLK_OK;
  if (m > INT32_MAX - 4) return FLK_E_INVALID;   // the last block's row index
  if (!x || !inv_s || !xq || !a_scale) return FLK_E_INVALID;
  if (k % 8 || k > 8192) return FLK_E_UNSUPPORTED;
  if (x_row_stride % 8 || !flk_host_aligned(x, 16) || !flk_host_aligned(inv_s, 16) || !flk_host_aligned(xq, 8) ||
      !flk_host_aligned(a_scale, 4))
    return FLK_E_ALIGN;
  const QuantProblem p{static_cast<const uint16_t*>(x), x_row_stride, inv_s, m, xq, a_scale, nullptr, nullptr, 0, 1,
                       nullptr, 0};
  const int64_t blocks = row_blocks(p, k);
  return launch_quantize_act<false>(QuantGroup{{p, p}, (int)std::min<int64_t>(blocks, INT32_MAX), k}, blocks,
                                    stream);
}

extern "C" int flk_quantize_act_modulated(const void* x, int64_t x_row_stride, const void* shift,
                                          const void* scale, int64_t mod_batch_stride, int tokens_per_batch,
                                          const float* inv_s, int m, int k, int8_t* xq, float* a_scale,
                                          void* x_mod, int64_t x_mod_row_stride, void* stream) {
  QuantProblem p{};
  const int st = modulated_problem(x, x_row_stride, shift, scale, mod_batch_stride, tokens_per_batch, inv_s, m, k,
                                   xq, a_scale, x_mod, x_mod_row_stride, p);
  if (st != FLK_OK) return st == kNoWork ? FLK_OK : st;
  const int64_t blocks = row_blocks(p, k);
  return launch_quantize_act<true>(QuantGroup{{p, p}, (int)std::min<int64_t>(blocks, INT32_MAX), k}, blocks,
                                   stream);
}

extern "C" int flk_quantize_act_modulated_pair(
    const void* x0, int64_t x_row_stride0, const void* shift0, const void* scale0, int64_t mod_batch_stride0,
    int tokens_per_batch0, const float* inv_s0, int m0, int8_t* xq0, float* a_scale0, void* x_mod0,
    int64_t x_mod_row_stride0,
    const void* x1, int64_t x_row_stride1, const void* shift1, const void* scale1, int64_t mod_batch_stride1,
    int tokens_per_batch1, const float* inv_s1, int m1, int8_t* xq1, float* a_scale1, void* x_mod1,
    int64_t x_mod_row_stride1, int k, void* stream) {
  QuantGroup g{};
  g.K = k;
  const int st0 = modulated_problem(x0, x_row_stride0, shift0, scale0, mod_batch_stride0, tokens_per_batch0, inv_s0,
                                    m0, k, xq0, a_scale0, x_mod0, x_mod_row_stride0, g.p[0]);
  if (st0 != FLK_OK && st0 != kNoWork) return st0;
  const int st1 = modulated_problem(x1, x_row_stride1, shift1, scale1, mod_batch_stride1, tokens_per_batch1, inv_s1,
                                    m1, k, xq1, a_scale1, x_mod1, x_mod_row_stride1, g.p[1]);
  if (st1 != FLK_OK && st1 != kNoWork) return st1;
  if (st0 == kNoWork && st1 == kNoWork) return FLK_OK;
  // An empty problem gives its place to the other one, which then takes every block.
  if (st0 == kNoWork) g.p[0] = g.p[1];
  if (st1 == kNoWork) g.p[1] = g.p[0];
  const bool both = st0 == FLK_OK && st1 == FLK_OK;
  const int64_t b0 = row_blocks(g.p[0], k);
  const int64_t blocks = both ? b0 + row_blocks(g.p[1], k) : b0;
  g.first_blocks = (int)std::min<int64_t>(b0, INT32_MAX);
  return launch_quantize_act<true>(g, blocks, stream);
}

namespace {

int64_t tiles(int size, int edge) { return ((int64_t)size + edge - 1) / edge; }

// Grid of the rounds order of a launch (w8a8_gemm_kernel), or 0 when it is not the choice: it
// needs a full round of 32 tiles on every XCD, tiles left over, and at most one round of
// 192-token tiles for them (counted as leftover_tile walks them).
int64_t gemm_rounds_grid(const GemmGroup& g) {
  constexpr int C = kCUs / kXcds;
  const int64_t units = g.units;
  if (units < kCUs) return 0;
  int64_t most = 0, left_max = 0;
  for (int x = 0; x < kXcds; ++x) {
    const int64_t ux0 = x * units / kXcds, n = (x + 1) * units / kXcds - ux0;
    const int64_t full = n / C * C;
    int64_t count = 0;
    for (int64_t u = ux0 + full; u < ux0 + n;) {
      const bool second = u >= g.first_blocks;
      const GemmProblem& p = second ? g.p[1] : g.p[0];
      const int64_t base = second ? g.first_blocks : 0;
      const int64_t p_end = second ? ux0 + n : std::min<int64_t>(ux0 + n, g.first_blocks);
      const int64_t group_tiles = (int64_t)kGroup * p.tiles_n;
      const int64_t group = (u - base) / group_tiles, first_m = group * kGroup;
      const int64_t gm = std::min<int64_t>(kGroup, p.tiles_m - first_m);
      const int64_t r = (u - base - group * group_tiles) % gm;
      const int64_t run = std::min(gm - r, p_end - u);
      const int64_t e = std::min<int64_t>((first_m + r + run) * kGT, p.M);
      count += (e - (first_m + r) * kGT + kGT192 - 1) / kGT192;
      u += run;
    }
    if (count > C) return 0;
    left_max = std::max(left_max, n - full);
    most = std::max(most, full + count);
  }
  return left_max > 0 ? most * kXcds : 0;
}

// Fills a launch's tiles of tm tokens x tn channels (of p[0] alone unless both); returns their count.
int64_t plan_tiles(GemmGroup& g, bool both, int tm, int tn) {
  for (GemmProblem& p : g.p) {
    p.tiles_m = (int)tiles(p.M, tm);
    p.tiles_n = (int)tiles(p.N, tn);
  }
  const int64_t first = (int64_t)g.p[0].tiles_m * g.p[0].tiles_n;
  g.first_blocks = (int)std::min<int64_t>(first, INT32_MAX);
  const int64_t units = first + (both ? (int64_t)g.p[1].tiles_m * g.p[1].tiles_n : 0);
  g.units = (int)std::min<int64_t>(units, INT32_MAX);
  return units;
}

// Launches p[0], and p[1] when both.  A round of 256 x 256 tiles takes ~34 us at K = 3072 however
// few blocks it has, so a launch takes the smallest of these tiles that fit the chip at once, the
// shortest chain per CU (us, plain GEMM with 3072 x 9216 weights, 256 x 256 tiles first):
//   128 x 64, one block per CU             17 tokens: 33.2 -> 10.3    128 tokens: 34.3 -> 11.3
//   128 x 128, one per CU, four stages    256 tokens: 34.6 -> 15.1    384 tokens: 34.6 -> 15.5
//   128 x 128, two per CU, two stages     512 tokens: 34.7 -> 22.6    896 tokens: 39.4 -> 29.3
// Past that 256 x 256 tiles, with half the stage copies per product, are faster: at 1152 tokens
// (648 tiles of 128 x 128) 41.7 against 46.2, at 4608 129 against 149.  The lines are in tiles, not
// sizes: over N = 128 to 27648 and K = 512 to 8192 (165 shapes on the small tiles' side, plain, 44
// with the qk_prep epilogue) none was slower than in 256 x 256 tiles.
template <bool kAcc, bool kQk, bool kScaleF32>
int launch_group(GemmGroup g, bool both, void* stream) {
  if (!both) g.p[1] = g.p[0];
  const hipStream_t st = as_stream(stream);
  int64_t blocks = plan_tiles(g, both, 64, kGWaveN);
  if (blocks <= kCUs) {
    hipLaunchKernelGGL((w8a8_gemm_split_kernel<kAcc, kQk, kScaleF32, 2, 4, 1>), dim3((unsigned)blocks), dim3(256), 0,
                       st, g);
    return flk_launch_status();
  }
  blocks = plan_tiles(g, both, 128, kGWaveN);
  if (blocks <= kCUs) {
    hipLaunchKernelGGL((w8a8_gemm_split_kernel<kAcc, kQk, kScaleF32, 4, 4, 1>), dim3((unsigned)blocks), dim3(512), 0,
                       st, g);
    return flk_launch_status();
  }
  if (blocks <= 2 * kCUs) {
    hipLaunchKernelGGL((w8a8_gemm_split_kernel<kAcc, kQk, kScaleF32, 4, 2, 2>), dim3((unsigned)blocks), dim3(512), 0,
                       st, g);
    return flk_launch_status();
  }
  blocks = plan_tiles(g, both, kGT, kGT);
  const int64_t rounds = blocks <= INT32_MAX ? gemm_rounds_grid(g) : 0;
  g.rounds = rounds > 0;
  if (rounds) blocks = rounds;
  if (blocks > INT32_MAX) return FLK_E_INVALID;
  hipLaunchKernelGGL((w8a8_gemm_kernel<kAcc, kQk, kScaleF32>), dim3((unsigned)blocks), dim3(kGThreads), 0, st, g);
  return flk_launch_status();
}

// Checks one fused projection + qk_prep (flk_w8a8_qk_prep's arguments) and fills its
// problem.  FLK_OK = launch, kNoWork = empty (nothing to launch), else an error status.

int qk_problem(const int8_t* xq, const int8_t* wq_t, const float* a_scale, const float* w_scale, int k,
               const float* cos, const float* sin, int64_t table_row_stride, const void* q_scale,
               const void* k_scale, float q_gain, int batch, int length, int num_heads, int head_dim,
               void* q_out, void* k_out, void* v_out, int64_t out_length, int64_t out_offset, GemmProblem& p) {
  if (head_dim != flk::kQkHeadDim) return FLK_E_UNSUPPORTED;
  if (batch < 0 || length < 0 || num_heads <= 0 || k < 0 || out_offset < 0 || out_offset + length > out_length)
    return FLK_E_INVALID;
  if (batch == 0 || length == 0) return kNoWork;
  if (!xq || !wq_t || !a_scale || !w_scale || !cos || !sin || !q_scale || !k_scale || !q_out || !k_out ||
      !v_out || k == 0 || table_row_stride < head_dim)
    return FLK_E_INVALID;
  if (k % 128) return FLK_E_UNSUPPORTED;
  if ((int64_t)k * 127 * 127 > INT32_MAX) return FLK_E_UNSUPPORTED;
  const int64_t m64 = (int64_t)batch * length, n = 3LL * num_heads * head_dim;
  if (m64 > kMaxDim || n > kMaxDim) return FLK_E_INVALID;
  if (!flk_host_aligned(xq, 16) || !flk_host_aligned(wq_t, 16) || !flk_host_aligned(w_scale, 16) ||
      !flk_host_aligned(a_scale, 4) || !flk_host_aligned(cos, 16) || !flk_host_aligned(sin, 16) ||
      table_row_stride % 4 || !flk_host_aligned(q_scale, 16) || !flk_host_aligned(k_scale, 16) ||
      !flk_host_aligned(q_out, 16) || !flk_host_aligned(k_out, 16) || !flk_host_aligned(v_out, 16))
    return FLK_E_ALIGN;
  p = GemmProblem{};
  p.xq = xq;
  p.wqt = wq_t;
  p.a_scale = a_scale;
  p.w_scale = w_scale;
  p.M = (int)m64;
  p.K = k;
  p.N = (int)n;
  p.qe = QkEpilogue{cos, sin, table_row_stride, q_scale, k_scale, q_gain, length, num_heads,
                    {static_cast<uint16_t*>(q_out), static_cast<uint16_t*>(k_out), static_cast<uint16_t*>(v_out)},
                    out_length, out_offset};
  return FLK_OK;
}

int launch_qk(const GemmGroup& g, bool both, int scale_is_f32, void* stream) {
  return scale_is_f32 ? launch_group<false, true, true>(g, both, stream)
                      : launch_group<false, true, false>(g, both, stream);
}

}  // namespace

extern "C" int flk_w8a8_gemm(const int8_t* xq, const int8_t* wq_t, const float* a_scale, const float* w_scale,
                             int m, int k, int n, void* y, int64_t y_row_stride, int32_t* acc_or_null,
                             void* stream) {
  if (m < 0 || k < 0 || n < 0 || y_row_stride < n) return FLK_E_INVALID;
  if (m == 0 || n == 0) return FLK_OK;
  if (m > kMaxDim || n > kMaxDim) return FLK_E_INVALID;
  if (!xq || !wq_t || !a_scale || !w_scale || !y || k == 0) return FLK_E_INVALID;
  if (k % 128 || n % 4) return FLK_E_UNSUPPORTED;
  if ((int64_t)k * 127 * 127 > INT32_MAX) return FLK_E_UNSUPPORTED;   // int32 accumulation must be exact
  if (!flk_host_aligned(xq, 16) || !flk_host_aligned(wq_t, 16) || !flk_host_aligned(w_scale, 16) ||
      !flk_host_aligned(a_scale, 4) || !flk_host_aligned(y, 8) || y_row_stride % 4 ||
      (acc_or_null && !flk_host_aligned(acc_or_null, 16)))
    return FLK_E_ALIGN;
  GemmGroup g{};
  GemmProblem& p = g.p[0];
  p.xq = xq;
  p.wqt = wq_t;
  p.a_scale = a_scale;
  p.w_scale = w_scale;
  p.y = static_cast<uint16_t*>(y);
  p.y_stride = y_row_stride;
  p.acc_out = acc_or_null;
  p.M = m;
  p.K = k;
  p.N = n;
  return acc_or_null ? launch_group<true, false, false>(g, false, stream)
                     : launch_group<false, false, false>(g, false, stream);
}

extern "C" int flk_w8a8_qk_prep(const int8_t* xq, const int8_t* wq_t, const float* a_scale, const float* w_scale,
                                int k, const float* cos, const float* sin, int64_t table_row_stride,
                                const void* q_scale, const void* k_scale, int scale_is_f32, float q_gain, int batch,
                                int length, int num_heads, int head_dim, void* q_out, void* k_out, void* v_out,
                                int64_t out_length, int64_t out_offset, void* stream) {
  GemmGroup g{};
  const int st = qk_problem(xq, wq_t, a_scale, w_scale, k, cos, sin, table_row_stride, q_scale, k_scale, q_gain,
                            batch, length, num_heads, head_dim, q_out, k_out, v_out, out_length, out_offset, g.p[0]);
  if (st != FLK_OK) return st == kNoWork ? FLK_OK : st;
  return launch_qk(g, false, scale_is_f32, stream);
}

extern "C" int flk_w8a8_qk_prep_pair(
    const int8_t* xq0, const int8_t* wq_t0, const float* a_scale0, const float* w_scale0, const float* cos0,
    const float* sin0, const void* q_scale0, const void* k_scale0, int length0, int64_t out_offset0,
    const int8_t* xq1, const int8_t* wq_t1, const float* a_scale1, const float* w_scale1, const float* cos1,
    const float* sin1, const void* q_scale1, const void* k_scale1, int length1, int64_t out_offset1, int k,
    int64_t table_row_stride, int scale_is_f32, float q_gain, int batch, int num_heads, int head_dim, void* q_out,
    void* k_out, void* v_out, int64_t out_length, void* stream) {
  GemmGroup g{};
  const int st0 = qk_problem(xq0, wq_t0, a_scale0, w_scale0, k, cos0, sin0, table_row_stride, q_scale0, k_scale0,
                             q_gain, batch, length0, num_heads, head_dim, q_out, k_out, v_out, out_length,
                             out_offset0, g.p[0]);
  if (st0 != FLK_OK && st0 != kNoWork) return st0;
  const int st1 = qk_problem(xq1, wq_t1, a_scale1, w_scale1, k, cos1, sin1, table_row_stride, q_scale1, k_scale1,
                             q_gain, batch, length1, num_heads, head_dim, q_out, k_out, v_out, out_length,
                             out_offset1, g.p[1]);
  if (st1 != FLK_OK && st1 != kNoWork) return st1;
  if (st0 == kNoWork && st1 == kNoWork) return FLK_OK;
  // An empty problem gives its place to the other one, which then takes every block.
  if (st0 == kNoWork) g.p[0] = g.p[1];
  return launch_qk(g, st0 == FLK_OK && st1 == FLK_OK, scale_is_f32, stream);
}
