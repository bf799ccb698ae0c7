// BinaryWeightAffine / BinaryConnectAffine forward in one launch, for layers too small (or too oddly shaped) for the
// forms that stream a large W: block = 32 rows of x x 64 output columns, the whole of K.
//
// The general path is a chain of launches -- signs and packed bits of W, alpha, the digit operand of x, the product --
// each of which takes 4 to 20 us on a small layer although its work is a fraction of one: the chain's length is the
// time.  Here a block reads its 32 rows of x and its 64 columns of W itself: x becomes three int8 digits under one
// power-of-two scale per row (gemm_layout.hpp), a weight becomes the byte +1 / -1 (or Sign(0)), both in registers in
// exactly the places v_mfma_i32_32x32x32_i8 wants them -- lane (h, c) of a wavefront holds rows 16 h .. 16 h + 15 of
// column c, read as 128-byte runs of a row of W, and the sixteen values k = 16 h .. of row c of x.  The wavefronts walk
// every kWaves-th k tile; nothing goes through LDS but the rows' maxima, the |W| sums and the final exchange.  Every
// block adds the |W| sums of its columns in the same order, so all use the same alpha.  Wb is written by further blocks of
// the launch, element by element: stores between a wavefront's loads would make the loads behind them wait for
// the stores' completion (one in-order counter), 2 us per tile.  The integer sums are exact, combined in double and rounded once: the outputs are those of the
// digit operand and the packed bits.  No alignment is asked for: rows of W and x start at any multiple of four bytes.
//
// What bounds it is latency: two round trips to memory (x and the first two k tiles of W, then the other two), the
// exchanges and the launch.  Forward in a graph, the chain -> this, blocks of 64 columns (the narrow ones below, where
// they apply, take 60 to 85 % of it): 20 x 250 x 250 (rows x inputs x outputs) 42 -> 9.8 us,
// 800 x 816 x 632 40 -> 16, 64 x 1001 x 1003 48 -> 14.6, 512^3 29 -> 12, 1024^3 43 -> 31 (two rounds of blocks; 4096 x
// 512 x 512, two rounds as well, 34 -> 31; at three the chain is the faster one: 1000 x 300 x 3000 33 against 36).
//
// A row of x with a NaN or an infinity is recomputed by its blocks in fp32 in the reference's order.
#include "common.hpp"
#include "gemm_layout.hpp"
#include "internal.hpp"

#include <hip/hip_ext.h>

namespace nbla_hip {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));

constexpr int kFusedRows = 32;
constexpr int kFusedTiles = 4;                 // k tiles of x a wavefront keeps in registers, at most
constexpr uint32_t kOutside = 0x80000000u;     // a byte offset past the end of any buffer here

struct FusedArgs {
  const float *x, *W;
  float *Wb, *alpha; // alpha null: BinaryConnectAffine
  const float *bias;
  float *y;
  int M, K, N, n_tiles, products; // products: blocks that multiply, the rest write Wb
  float zero_to, inv_k;
  uint32_t x_bytes, w_bytes;
};

// sign.hpp:48-50; +-0 and NaN are exactly the values that are neither less nor greater than zero
__device__ __forceinline__ float fused_sign(float v, float zero_to) {
  const float one = __uint_as_float((__float_as_uint(v) & 0x80000000u) | 0x3f800000u);
  return __builtin_islessgreater(v, 0.0f) ? one : zero_to;
}

// Largest shift s with rint(amax * 2^s) <= kDigitMax (the scale rule of the digit operand).
__device__ __forceinline__ int fused_shift(uint32_t amax_bits) {
  int s = 22 - binade_exponent(binade_of(amax_bits));
  if (rintf(ldexpf(__uint_as_float(amax_bits), s)) > (float)kDigitMax)
    --s;
  return s;
}

// kTiles: k tiles of a wavefront (kWaves * kTiles of them cover K); kFrags: fragments of 32 columns of a block.
template <int kWaves, int kTiles, int kFrags>
__global__ __launch_bounds__(64 * kWaves, 2) void binary_affine_fused(FusedArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kFusedCols = 32 * kFrags;
  extern __shared__ __attribute__((aligned(16))) int s_red[]; // [wave][32][lane]
  __shared__ uint32_t s_max[kWaves][kFusedRows], s_nonfinite[kWaves][kFusedRows];
  __shared__ float s_cs[kWaves][2][kFusedCols];
  __shared__ int s_shift[kFusedRows];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if ((int)blockIdx.x >= a.products) { // Wb = Sign(W), sixteen elements per thread and step
    const int64_t total = (int64_t)a.K * a.N, step = (int64_t)(gridDim.x - a.products) * (64 * kWaves) * 4;
    for (int64_t i = ((int64_t)(blockIdx.x - a.products) * (64 * kWaves) + tid) * 4; i < total; i += 4 * step) {
      f32x4_t v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = *reinterpret_cast<const f32x4_u *>(a.W + min(i + j * step, total - 4));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4_t o;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          o[c] = fused_sign(v[j][c], a.zero_to);
        if (i + j * step < total)
          *reinterpret_cast<f32x4_u *>(a.Wb + min(i + j * step, total - 4)) = o; // (the last four elements once more)
      }
    }
    return;
  }
  const int tile_m = (int)blockIdx.x / a.n_tiles, tile_n = (int)blockIdx.x - tile_m * a.n_tiles;
  const int n0 = tile_n * kFusedCols, m0 = tile_m * kFusedRows;
  const int k_tiles = (a.K + kTileK - 1) / kTileK;
  const uint32_t row_bytes = (uint32_t)a.N * 4;
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x), 0, (int)a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.W), 0, (int)a.w_bytes, 0x00020000);
  const uint32_t col_off = (uint32_t)half * 16 * row_bytes + (uint32_t)(n0 + r) * 4;

  // sixteen rows of the lane's two columns in k tile t (t < k_tiles); rows past K repeat the last one or read as zero
  auto load_w = [&](int t, float (&w)[kFrags][16]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t soff = (uint32_t)min(t * kTileK + j, a.K - 1) * row_bytes;
#pragma unroll
      for (int f = 0; f < kFrags; ++f)
        w[f][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(wr, (int)(col_off + 128 * f), (int)soff, 0));
    }
  };
  const int zero_byte = (int)a.zero_to;
  float cs[kFrags] = {};
  i32x16_t acc[kFrags][kDigits];
#pragma unroll
  for (int f = 0; f < kFrags; ++f)
#pragma unroll
    for (int d = 0; d < kDigits; ++d)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[f][d][q] = 0;
  // the tile's bytes, and its magnitudes to the column sums
  auto take_tile = [&](int t, float (&w)[kFrags][16], uint4_t (&b)[kFrags]) __attribute__((always_inline)) {
    const int k0 = t * kTileK + 16 * half;
    if (t * kTileK + kTileK > a.K) { // uniform: the last tile
#pragma unroll
      for (int j = 0; j < 16; ++j)
#pragma unroll
        for (int f = 0; f < kFrags; ++f)
          w[f][j] = k0 + j < a.K ? w[f][j] : 0.0f;
    }
#pragma unroll
    for (int f = 0; f < kFrags; ++f)
#pragma unroll
      for (int j4 = 0; j4 < 4; ++j4) {
        uint32_t byte[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int j = 4 * j4 + c;
          const float v = w[f][j];
          cs[f] += fabsf(v);
          byte[c] = (uint32_t)(__builtin_islessgreater(v, 0.0f) ? ((int)__float_as_uint(v) >> 31) | 1 : zero_byte);
        }
        const uint32_t lo = __builtin_amdgcn_perm(byte[1], byte[0], 0x0c0c0400u);
        const uint32_t hi = __builtin_amdgcn_perm(byte[3], byte[2], 0x04000c0cu);
        b[f][j4] = lo | hi;
      }
  };
  auto multiply = [&](const uint4_t (&xd)[kDigits], const uint4_t (&b)[kFrags]) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < kFrags; ++f)
#pragma unroll
      for (int d = 0; d < kDigits; ++d)
        acc[f][d] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4_t, xd[d]),
                                                          __builtin_bit_cast(i32x4_t, b[f]), acc[f][d], 0, 0, 0);
  };

  // x: the row's values of the wavefront's k tiles, its largest finite magnitude over all wavefronts, the digits
  f32x4_t xv[kTiles][4];
  const bool row_in = m0 + r < a.M;
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    const int k0 = (wave + kWaves * i) * kTileK + 16 * half;
    const uint32_t off = (uint32_t)((m0 + r) * a.K + k0) * 4;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      xv[i][v] = __builtin_bit_cast(
          f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(row_in && k0 + 4 * v < a.K ? off + 16 * v : kOutside),
                                                         0, 0));
  }
  float w0[kFrags][16], w1[kFrags][16];
  load_w(min(wave, k_tiles - 1), w0);
  if constexpr (kTiles > 1)
    load_w(min(wave + kWaves, k_tiles - 1), w1);
  uint32_t amax = 0u, bad = 0u;
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    const int k0 = (wave + kWaves * i) * kTileK + 16 * half;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float v = k0 + j < a.K ? xv[i][j >> 2][j & 3] : 0.0f;
      xv[i][j >> 2][j & 3] = v;
      const uint32_t m = __float_as_uint(v) & 0x7fffffffu;
      const bool fin = m < 0x7f800000u;
      amax = max(amax, fin ? m : 0u);
      bad |= fin ? 0u : 1u;
    }
  }
  amax = max(amax, (uint32_t)__shfl_xor((int)amax, 32));
  bad |= (uint32_t)__shfl_xor((int)bad, 32);
  if (half == 0)
    s_max[wave][r] = amax, s_nonfinite[wave][r] = bad;
  __syncthreads();
#pragma unroll
  for (int v = 0; v < kWaves; ++v)
    amax = max(amax, s_max[v][r]), bad |= s_nonfinite[v][r];
  const int shift = amax ? fused_shift(amax) : 0;
  if (wave == 0 && half == 0)
    s_shift[r] = bad ? kBadRow : shift;
  uint4_t xd[kTiles][kDigits];
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    int q[16];
    uint32_t words[3][4];
#pragma unroll
    for (int j = 0; j < 16; ++j)
      q[j] = bad ? 0 : (int)rintf(ldexpf(xv[i][j >> 2][j & 3], shift));
    pack_digits(q, words);
#pragma unroll
    for (int d = 0; d < kDigits; ++d)
      xd[i][d] = uint4_t{words[d][0], words[d][1], words[d][2], words[d][3]};
  }
  static_assert(kTiles == 1 || kTiles == 2 || kTiles == 4, "one tile, a pair or two pairs");
  uint4_t b[kFrags];
  if (wave < k_tiles) {
    take_tile(wave, w0, b);
    if constexpr (kTiles > 2)
      load_w(min(wave + 2 * kWaves, k_tiles - 1), w0);
    multiply(xd[0], b);
  }
  if constexpr (kTiles > 1)
    if (wave + kWaves < k_tiles) {
      take_tile(wave + kWaves, w1, b);
      if constexpr (kTiles > 2)
        load_w(min(wave + 3 * kWaves, k_tiles - 1), w1);
      multiply(xd[1], b);
    }
  if constexpr (kTiles > 2) {
    if (wave + 2 * kWaves < k_tiles) {
      take_tile(wave + 2 * kWaves, w0, b);
      multiply(xd[2], b);
    }
    if (wave + 3 * kWaves < k_tiles) {
      take_tile(wave + 3 * kWaves, w1, b);
      multiply(xd[3], b);
    }
  }

  // ---- the wavefronts' sums, one fragment of 32 columns at a time: each finishes 16 / kWaves accumulator registers
#pragma unroll
  for (int f = 0; f < kFrags; ++f)
    s_cs[wave][half][32 * f + r] = cs[f];
  int any_bad = 0;
#pragma unroll
  for (int f = 0; f < kFrags; ++f) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      s_red[(wave * 32 + 2 * q) * 64 + lane] = acc[f][0][q] * 256 + acc[f][1][q]; // below 2^30 for K up to 2^14
      s_red[(wave * 32 + 2 * q + 1) * 64 + lane] = acc[f][2][q];
    }
    __syncthreads();
    const int n = n0 + 32 * f + r;
    float al = 1.0f;
    if (a.alpha) {
      float sum = 0.0f;
#pragma unroll
      for (int v = 0; v < kWaves; ++v)
        sum += s_cs[v][0][32 * f + r] + s_cs[v][1][32 * f + r];
      al = sum * a.inv_k; // binary_weight_affine.cpp:68: the sum times the rounded reciprocal
      if (tile_m == 0 && wave == 0 && half == 0 && n < a.N)
        a.alpha[n] = al;
    }
    const float bias = a.bias ? a.bias[n < a.N ? n : a.N - 1] : -0.0f;
#pragma unroll
    for (int i = 0; i < 16 / kWaves; ++i) {
      const int q = wave * (16 / kWaves) + i;
      int hi = 0, lo = 0;
#pragma unroll
      for (int v = 0; v < kWaves; ++v)
        hi += s_red[(v * 32 + 2 * q) * 64 + lane], lo += s_red[(v * 32 + 2 * q + 1) * 64 + lane];
      const int row = 8 * (q >> 2) + 4 * half + (q & 3), m = m0 + row, shift = s_shift[row];
      any_bad |= shift == kBadRow && m < a.M;
      // the exact sum, rounded once
      float v = ldexpf((float)((double)hi * 256.0 + (double)lo), -shift);
      v = v * al;
      v = v + bias;
      if (m < a.M && n < a.N && shift != kBadRow)
        a.y[(int64_t)m * a.N + n] = v;
    }
    __syncthreads();
  }
  // rows of x with a NaN or an infinity (affine.cpp:87-95 propagates them output by output: Inf * w = +-Inf,
  // Inf - Inf = NaN): fp32 dot products with the scaled signs in ascending k
  if (!__syncthreads_or(any_bad))
    return;
  for (int row = 0; row < kFusedRows; ++row) {
    const int n = n0 + tid;
    if (s_shift[row] != kBadRow || m0 + row >= a.M || tid >= kFusedCols || n >= a.N)
      continue;
    float al = 1.0f;
    if (a.alpha) {
      float sum = 0.0f;
      for (int v = 0; v < kWaves; ++v)
        sum += s_cs[v][0][tid] + s_cs[v][1][tid];
      al = sum * a.inv_k;
    }
    float sum = 0.0f;
    for (int k = 0; k < a.K; ++k) {
      const float v = a.W[(int64_t)k * a.N + n];
      const float s = fused_sign(v, a.zero_to);
      sum = sum + a.x[(int64_t)(m0 + row) * a.K + k] * (a.alpha ? s * al : s);
    }
    a.y[(int64_t)(m0 + row) * a.N + n] = a.bias ? sum + a.bias[n] : sum;
  }
#endif
}

template <int kWaves, int kTiles, int kFrags> int run_fused(FusedArgs &a, hipStream_t stream) {
  static std::atomic<uint64_t> configured{0};
  constexpr int lds = kWaves * 32 * 64 * 4;
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(binary_affine_fused<kWaves, kTiles, kFrags>), lds,
                                   configured, "hipFuncSetAttribute(binary_affine_fused LDS size)");
  if (rc)
    return rc;
  a.n_tiles = (int)ceil_div(a.N, 32 * kFrags), a.products = (int)(a.n_tiles * ceil_div(a.M, kFusedRows));
  int64_t writers = ceil_div((int64_t)a.K * a.N, (int64_t)64 * kWaves * 16);
  if (writers > 512)
    writers = 512;
  const dim3 grid((unsigned)(a.products + writers));
  hipEvent_t start, stop;
  if (product_timer_next(&start, &stop))
    hipExtLaunchKernelGGL((binary_affine_fused<kWaves, kTiles, kFrags>), grid, dim3(64 * kWaves), lds, stream, start,
                          stop, 0, a);
  else
    hipLaunchKernelGGL((binary_affine_fused<kWaves, kTiles, kFrags>), grid, dim3(64 * kWaves), lds, stream, a);
  NBLA_HIP_LAUNCH_CHECK("binary_affine_fused");
  return NBLA_HIP_OK;
}

constexpr int kWideCols = 64; // columns of a block of two fragments

} // namespace

bool fused_affine_applies(const float *W, const float *Wb, int64_t M, int64_t K, int64_t N, float zero_to) {
  // the sign is a byte: of what Sign(0) may be -1, 0 and 1 are in use; a wavefront's registers hold the whole of a row in
  // four k tiles; 32-bit offsets, the tiles' rows past the end of x and W included
  // (Wb in the place of W: other blocks would still read what a block has overwritten)
  if (!Wb || (Wb < W + K * N && W < Wb + K * N))
    return false;
  if (!(zero_to == 1.0f || zero_to == -1.0f || zero_to == 0.0f) || K > 8 * kFusedTiles * kTileK || K * N < 4 ||
      (K + 64) * N * 4 >= (1ll << 31) || (M + kFusedRows) * (K + 512) * 4 >= (1ll << 31))
    return false;
  // Two rounds of blocks at most: of 512 (four wavefronts, two blocks to a CU) or of 256.
  const int64_t blocks = ceil_div(M, kFusedRows) * ceil_div(N, kWideCols);
  return blocks <= (K <= 4 * kFusedTiles * kTileK ? 1024 : 512);
}

int launch_fused_affine(const float *x, const float *W, float *Wb, float *alpha, const float *bias,
                        float *y, int64_t M, int64_t K, int64_t N, float zero_to, hipStream_t stream) {
  FusedArgs a;
  a.x = x, a.W = W, a.Wb = Wb, a.alpha = alpha, a.bias = bias, a.y = y;
  a.M = (int)M, a.K = (int)K, a.N = (int)N;
  a.zero_to = zero_to, a.inv_k = (float)1 / K;
  a.x_bytes = (uint32_t)(M * K * 4), a.w_bytes = (uint32_t)(K * N * 4);
  // Few blocks: the chain of one block is the time, so blocks of one fragment of columns, K over eight wavefronts and no
  // more k tiles in a wavefront than there are (20 x 250 x 250: 9.1 -> 4.9 us).
  // (Twice as many blocks with one k tile, where a block has little to do: 1000 x 120 x 500 8.5 -> 6.9; with more it is
  // slower, 800 x 816 x 632 17 -> 22.)
  if (ceil_div(M, kFusedRows) * ceil_div(N, kWideCols) <= (K <= 8 * kTileK ? 256 : 128)) {
    if (K <= 8 * kTileK)
      return run_fused<8, 1, 1>(a, stream);
    if (K <= 16 * kTileK)
      return run_fused<8, 2, 1>(a, stream);
    return run_fused<8, 4, 1>(a, stream);
  }
  return K <= 4 * kFusedTiles * kTileK ? run_fused<4, 4, 2>(a, stream) : run_fused<8, 4, 2>(a, stream);
}

} // namespace nbla_hip
