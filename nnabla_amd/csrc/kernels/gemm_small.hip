// A product of two real-valued matrices in one launch, for sizes whose time on the digit path is that of its chain of
// launches: y[m, n] = sum_k A(m, k) B(k, n) (+ bias[n]), block = 32 rows x 64 columns, the whole contraction.
//
// The digit path (gemm_digits.hip) prepares both operands -- clear, column maxima, shifts, digits, row digits -- and
// follows the product with the sum of its split and a look for non-finite values: seven to nine launches of 2 to 11 us
// each.  Here a wavefront reads its k tiles of A and B straight into the lanes that v_mfma_f32_32x32x16_bf16 wants them
// in and splits each value into three bf16 numbers that add up to it exactly (8 bits each, 24 in all; bf16 has fp32's
// exponents, so no scale and no pass over the data is needed before).  Six of the nine products are taken -- the three
// left out are below 2^-25 of a term -- the leading one into an accumulator of its own, so that the corrections' sums
// cost it no roundings.  The wavefronts walk every kWaves-th tile, two tiles in registers and two in flight, and their
// sums are added in double and rounded once.
//
// bf16 products lose bits below 2^-126 and sums overflow at 2^128 (up to 2^13 products, of either sign one after the
// other): rows of A and columns of B whose largest magnitude is outside 2^-50 .. 2^56, or that hold a NaN or an infinity, are marked, and the block recomputes the marked ones'
// outputs one by one in double (affine.cpp:87-95 propagates NaN and Inf output by output).
//
// What bounds it: the splitting, ten vector operations per value (a value of A is split by every column block), and for
// the smallest sizes two round trips to memory.  Digit path -> this, rows x inputs x outputs, forward: 20 x 250 x 250
// 35.2 -> 7.5 us, 512^3 40.6 -> 9.5, 200 x 1000 x 1000 43.7 -> 14.8, 1024^3 53 -> 29, 128 x 4096 x 4096 88 -> 45; weight
// gradient at 200 x 1000 x 1000 36.4 -> 13.3, input gradient 31.9 -> 15.3.  Off float64 (relative, 2-norm): 3e-8 to 1.0e-7
// where the digits are 1.6e-7 to 8.6e-7 off.
//
// With signs, Sign(B) stands for B, exact in one bf16 part: three products, no splitting of B.  The input gradient of a
// small binary layer is dy alpha . Sign(W)^T this way, 29 us as packed signs, digits and product in four launches: 20 x
// 250 x 250 5.0, 512^3 8.7, 200 x 368 x 257 6.4, 64 x 1000 x 1000 11.6, 600 x 700 x 800 (32) 16.2; off float64 3.6e-8, the
// digits 1.5e-7.
#include "bf16_parts.hpp"
#include "common.hpp"
#include "gemm_layout.hpp"
#include "internal.hpp"

namespace nbla_hip {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kWavesPerBlock = 8; // one block to a CU, two wavefronts to a SIMD
constexpr int kRows = 32, kWideCols = 64, kTile = 32; // rows and columns of a block (or 32 columns); a tile of the contraction: two MFMA steps
constexpr uint32_t kOutside = 0x80000000u;        // a byte offset past the end of any buffer here
constexpr uint32_t kLeast = (127u - 50u) << 23, kMost = (127u + 56u) << 23; // magnitudes, as bits

struct SmallArgs {
  const float *a, *b;
  const float *bias; // may be null
  float *y;          // [M, N], rows N apart
  int M, K, N, n_tiles, accumulate;
  uint32_t a_bytes, b_bytes;
  const float *kscale; // may be null; with signs only: A(m, k) is multiplied by kscale[k] first, rounded once
  float zero_to;       // with signs: what stands for a value of B that is neither negative nor positive (-1, 0 or 1)
};

// The sixteen values k = 32 t + 16 half .. of one row (column) of an operand with `count` of them, `f` the lane's own.
// kAcross: [K][count], lanes side by side in memory; otherwise [count][K], a lane's values side by side.  Values past
// the ends read as zero or as some other element of the operand.
template <bool kAcross>
__device__ __forceinline__ void load_tile(const __amdgpu_buffer_rsrc_t rsrc, int t, int half, int f, int count, int K,
                                          float (&v)[16]) {
  if (kAcross) {
    const uint32_t row = (uint32_t)count * 4;
    const uint32_t off = (uint32_t)half * 16 * row + (uint32_t)f * 4;
#pragma unroll
    for (int j = 0; j < 16; ++j)
      v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          rsrc, (int)off, (int)((uint32_t)min(t * kTile + j, K - 1) * row), 0));
  } else {
    const int k0 = t * kTile + 16 * half;
    const uint32_t off = ((uint32_t)f * K + k0) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4_t w = __builtin_bit_cast(
          f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                       rsrc, (int)(f < count && k0 + 4 * q < K ? off + 16 * q : kOutside), 0, 0));
#pragma unroll
      for (int c = 0; c < 4; ++c)
        v[4 * q + c] = w[c];
    }
  }
}

// eight of the sixteen values (s: which) as bf16 operands
__device__ __forceinline__ void split3(const float (&v)[16], int s, uint4_t &hi, uint4_t &mid, uint4_t &lo) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    uint32_t h, m, l;
    split3_pair(v[8 * s + 2 * p], v[8 * s + 2 * p + 1], h, m, l);
    hi[p] = h, mid[p] = m, lo[p] = l;
  }
}

__device__ __forceinline__ f32x16_t mma(const uint4_t &a, const uint4_t &b, f32x16_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
#else
  return c;
#endif
}

// Sign(v), which bf16 holds in one part.
__device__ __forceinline__ float small_sign(float v, float zero_to) {
  const float one = __uint_as_float((__float_as_uint(v) & 0x80000000u) | 0x3f800000u);
  return __builtin_islessgreater(v, 0.0f) ? one : zero_to;
}

// kFrags: fragments of 32 columns of a block.  kSigns: Sign(B) in the place of B, three products instead of six.
template <int kWaves, int kFrags, bool kAAcross, bool kBAcross, bool kSigns>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_small(SmallArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kCols = 32 * kFrags;
  extern __shared__ __attribute__((aligned(16))) float s_red[]; // [wave][32][lane]
  __shared__ uint32_t s_max_a[kWaves][kRows], s_max_b[kWaves][kCols];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile_m = (int)blockIdx.x / a.n_tiles, tile_n = (int)blockIdx.x - tile_m * a.n_tiles;
  const int m0 = tile_m * kRows, n0 = tile_n * kCols;
  const int k_tiles = (a.K + kTile - 1) / kTile;
  const __amdgpu_buffer_rsrc_t ar =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.a), 0, (int)a.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t br =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.b), 0, (int)a.b_bytes, 0x00020000);

  f32x16_t acc[kFrags][2];
#pragma unroll
  for (int f = 0; f < kFrags; ++f)
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[f][d][q] = 0.0f;
  uint32_t max_a = 0u, max_b[kFrags] = {};

  struct Tile {
    float av[16], bv[kFrags][16], sc[kSigns ? 16 : 1];
  };
  auto load = [&](int t, Tile &w) __attribute__((always_inline)) {
    load_tile<kAAcross>(ar, t, half, m0 + r, a.M, a.K, w.av);
#pragma unroll
    for (int f = 0; f < kFrags; ++f)
      load_tile<kBAcross>(br, t, half, n0 + 32 * f + r, a.N, a.K, w.bv[f]);
    if (kSigns) {
#pragma unroll
      for (int j = 0; j < 16; ++j)
        w.sc[j] = a.kscale ? a.kscale[min(t * kTile + 16 * half + j, a.K - 1)] : 1.0f;
    }
  };
  auto take = [&](int t, Tile &w) __attribute__((always_inline)) {
    if (kSigns) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        if (a.kscale)
          w.av[j] = w.av[j] * w.sc[j];
#pragma unroll
        for (int f = 0; f < kFrags; ++f)
          w.bv[f][j] = small_sign(w.bv[f][j], a.zero_to);
      }
    }
    if (t * kTile + kTile > a.K) { // uniform: the last tile
      const int k0 = t * kTile + 16 * half;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const bool in = k0 + j < a.K;
        w.av[j] = in ? w.av[j] : 0.0f;
#pragma unroll
        for (int f = 0; f < kFrags; ++f)
          w.bv[f][j] = in ? w.bv[f][j] : 0.0f;
      }
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      max_a = max(max_a, __float_as_uint(w.av[j]) & 0x7fffffffu);
#pragma unroll
      for (int f = 0; f < kFrags; ++f)
        if (!kSigns)
          max_b[f] = max(max_b[f], __float_as_uint(w.bv[f][j]) & 0x7fffffffu);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      uint4_t ah, am, al;
      split3(w.av, s, ah, am, al);
#pragma unroll
      for (int f = 0; f < kFrags; ++f) {
        uint4_t bh, bm, bl;
        if (kSigns) {
#pragma unroll
          for (int p = 0; p < 4; ++p)
            bh[p] = __builtin_amdgcn_perm(__float_as_uint(w.bv[f][8 * s + 2 * p + 1]), __float_as_uint(w.bv[f][8 * s + 2 * p]),
                                          0x07060302u);
          acc[f][0] = mma(ah, bh, acc[f][0]);
          acc[f][1] = mma(al, bh, acc[f][1]);
          acc[f][1] = mma(am, bh, acc[f][1]);
          continue;
        }
        split3(w.bv[f], s, bh, bm, bl);
        acc[f][0] = mma(ah, bh, acc[f][0]);
        acc[f][1] = mma(ah, bl, acc[f][1]);
        acc[f][1] = mma(al, bh, acc[f][1]);
        acc[f][1] = mma(am, bm, acc[f][1]);
        acc[f][1] = mma(ah, bm, acc[f][1]);
        acc[f][1] = mma(am, bh, acc[f][1]);
      }
    }
  };
  Tile w0, w1;
  if (wave < k_tiles)
    load(wave, w0);
  if (wave + kWaves < k_tiles)
    load(wave + kWaves, w1);
  for (int t = wave; t < k_tiles; t += 2 * kWaves) {
    take(t, w0);
    if (t + 2 * kWaves < k_tiles)
      load(t + 2 * kWaves, w0);
    if (t + kWaves < k_tiles)
      take(t + kWaves, w1);
    if (t + 3 * kWaves < k_tiles)
      load(t + 3 * kWaves, w1);
  }

  max_a = max(max_a, (uint32_t)__shfl_xor((int)max_a, 32));
#pragma unroll
  for (int f = 0; f < kFrags; ++f)
    max_b[f] = max(max_b[f], (uint32_t)__shfl_xor((int)max_b[f], 32));
  if (half == 0) {
    s_max_a[wave][r] = m0 + r < a.M ? max_a : 0u;
#pragma unroll
    for (int f = 0; f < kFrags; ++f)
      s_max_b[wave][32 * f + r] = n0 + 32 * f + r < a.N ? max_b[f] : 0u;
  }
  // ---- the wavefronts' sums, one fragment of 32 columns at a time: each finishes 16 / kWaves accumulator registers
#pragma unroll
  for (int f = 0; f < kFrags; ++f) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      s_red[(wave * 32 + 2 * q) * 64 + lane] = acc[f][0][q];
      s_red[(wave * 32 + 2 * q + 1) * 64 + lane] = acc[f][1][q];
    }
    __syncthreads();
    const int n = n0 + 32 * f + r;
    const float bias = a.bias ? a.bias[n < a.N ? n : a.N - 1] : -0.0f;
#pragma unroll
    for (int i = 0; i < 16 / kWaves; ++i) {
      const int q = wave * (16 / kWaves) + i;
      double sum = 0.0;
#pragma unroll
      for (int v = 0; v < kWaves; ++v)
        sum += (double)s_red[(v * 32 + 2 * q) * 64 + lane] + (double)s_red[(v * 32 + 2 * q + 1) * 64 + lane];
      const int m = m0 + 8 * (q >> 2) + 4 * half + (q & 3);
      if (m < a.M && n < a.N) {
        const int64_t o = (int64_t)m * a.N + n;
        // (a marked output that is added to y is left for the pass below)
        uint32_t big_a = 0u, big_b = 0u;
#pragma unroll
        for (int v = 0; v < kWaves; ++v)
          big_a = max(big_a, s_max_a[v][m - m0]), big_b = max(big_b, s_max_b[v][n - n0]);
        if (big_a <= kMost && big_b <= kMost && (big_a >= kLeast || big_a == 0u) && (big_b >= kLeast || big_b == 0u)) {
          const float v = (float)sum + bias;
          a.y[o] = a.accumulate ? a.y[o] + v : v;
        }
      }
    }
    __syncthreads();
  }
  // ---- marked rows and columns
  auto mark = [&](const uint32_t *col, int stride) __attribute__((always_inline)) {
    uint32_t big = 0u;
    for (int v = 0; v < kWaves; ++v)
      big = max(big, col[v * stride]);
    return big > kMost || (big != 0u && big < kLeast);
  };
  bool marked = false;
  if (tid < kCols)
    marked = mark(&s_max_b[0][tid], kCols) || (tid < kRows && mark(&s_max_a[0][tid], kRows));
  static_assert(kCols >= kRows, "a thread per row among those of the columns");
  if (!__syncthreads_or(marked))
    return;
  for (int i = tid; i < kRows * kCols; i += 64 * kWaves) {
    const int row = i / kCols, col = i - row * kCols, m = m0 + row, n = n0 + col;
    if (m >= a.M || n >= a.N || !(mark(&s_max_a[0][row], kRows) || mark(&s_max_b[0][col], kCols)))
      continue;
    double sum = 0.0;
    for (int k = 0; k < a.K; ++k) {
      float av = kAAcross ? a.a[(int64_t)k * a.M + m] : a.a[(int64_t)m * a.K + k];
      float bv = kBAcross ? a.b[(int64_t)k * a.N + n] : a.b[(int64_t)n * a.K + k];
      if (kSigns) {
        av = a.kscale ? av * a.kscale[k] : av;
        bv = small_sign(bv, a.zero_to);
      }
      sum = sum + (double)av * (double)bv;
    }
    const int64_t o = (int64_t)m * a.N + n;
    const float v = (float)sum + (a.bias ? a.bias[n] : -0.0f);
    a.y[o] = a.accumulate ? a.y[o] + v : v;
  }
#endif
}

template <int kFrags, bool kAAcross, bool kBAcross, bool kSigns = false> int run_small(SmallArgs &a, hipStream_t stream) {
  constexpr int kWaves = kWavesPerBlock;
  static std::atomic<uint64_t> configured{0};
  constexpr int lds = kWaves * 32 * 64 * 4;
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(gemm_small<kWaves, kFrags, kAAcross, kBAcross, kSigns>), lds,
                                   configured, "hipFuncSetAttribute(gemm_small LDS size)");
  if (rc)
    return rc;
  a.n_tiles = (int)ceil_div(a.N, 32 * kFrags);
  const int64_t blocks = a.n_tiles * ceil_div(a.M, kRows);
  hipLaunchKernelGGL((gemm_small<kWaves, kFrags, kAAcross, kBAcross, kSigns>), dim3((unsigned)blocks), dim3(64 * kWaves), lds,
                     stream, a);
  NBLA_HIP_LAUNCH_CHECK("gemm_small");
  return NBLA_HIP_OK;
}

} // namespace

// A round of blocks takes about 4 us and 2 us more for every k tile of a wavefront: 1024^3 (two rounds of four) 29 us as
// x . W, 512 x 2048 x 2048 (two of eight) 46, 4096 x 256 x 1024 (eight of one) 53, past the line: the digits take 43.  `limit` is where
// the digit path's chain takes the same: see the callers.
bool gemm_small_applies(int64_t M, int64_t K, int64_t N, int64_t limit) {
  if (M <= 0 || K <= 0 || N <= 0 || K > (1 << 13) || M > (1 << 24) || N > (1 << 24))
    return false;
  // 32-bit offsets, the rows of the tiles past the ends included
  if ((K + 64) * N * 4 >= (1ll << 31) || (M + kRows) * (K + 64) * 4 >= (1ll << 31) || (K + 64) * M * 4 >= (1ll << 31) ||
      (N + kWideCols) * (K + 64) * 4 >= (1ll << 31))
    return false;
  const int64_t rounds = ceil_div(ceil_div(M, kRows) * ceil_div(N, kWideCols), 256);
  return rounds * (4 + 2 * ceil_div(K, kWavesPerBlock * kTile)) <= limit;
}

int launch_gemm_small(const float *A, bool a_across, const float *B, bool b_across, const float *bias, float *y,
                      int64_t M, int64_t K, int64_t N, bool accumulate, hipStream_t stream, bool signs,
                      const float *kscale, float zero_to) {
  SmallArgs a;
  a.a = A, a.b = B, a.bias = bias, a.y = y;
  a.M = (int)M, a.K = (int)K, a.N = (int)N, a.accumulate = accumulate ? 1 : 0;
  a.a_bytes = (uint32_t)(M * K * 4), a.b_bytes = (uint32_t)(K * N * 4);
  a.kscale = kscale, a.zero_to = zero_to;
  // few blocks: half as wide, so that a block's chain is shorter (20 x 250 x 250: 6.9 -> 4.9 us)
  const bool narrow = ceil_div(M, kRows) * ceil_div(N, kWideCols) <= 128;
  if (a_across)
    return narrow ? run_small<1, true, true>(a, stream) : run_small<2, true, true>(a, stream);
  if (b_across)
    return narrow ? run_small<1, false, true>(a, stream) : run_small<2, false, true>(a, stream);
  if (signs)
    return narrow ? run_small<1, false, false, true>(a, stream) : run_small<2, false, false, true>(a, stream);
  return narrow ? run_small<1, false, false>(a, stream) : run_small<2, false, false>(a, stream);
}

} // namespace nbla_hip
