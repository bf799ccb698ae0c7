// Two-dimensional convolution of real-valued weights on the bf16 matrix cores without an unfolded matrix, forward and
// input gradient:
//     out[n, r, q] = sum over taps t of the class, k of  W_t(r, k) * in[n, k, q * ss + offset_t]        (+ bias[r])
// Forward: r = output channel, k = input channel, ss = stride, one class of all taps (convolution.cpp:185-193).  Input
// gradient: r = input channel, k = output channel, ss = 1; the input positions fall into stride^2 classes by their
// remainders, and of every class only the taps that reach it are taken (convolution.cpp:246-258 scatters the unfolded
// gradient instead).
//
// Arithmetic as in gemm_small.hip: a value is the sum of three bf16 numbers and six of the nine products are taken.  The weights of a row r are scaled by a power of two that puts their
// largest magnitude into [1, 2) (undone at the end), so that products of inputs down to 2^-90 keep all their bits.
//
// Layout.  Block = 64 rows x 64 consecutive positions, counted through the samples.  Its positions' input rows, the rows
// of consecutive samples following each other, are one contiguous run of input positions: a chunk of 16 or 32 channels of
// the run is split and put into LDS as [plane][eight channels][position][8 bf16], so that a lane's operand of
// v_mfma_f32_32x32x16_bf16 under any tap is sixteen bytes at its position plus the tap's displacement, and lanes lie side
// by side; a tap in the padding reads a position of zeros.  The four wavefronts take every fourth (tap, 16 channels) step
// with all of the block's 2 x 2 fragments -- each weight operand, prepared once per call in the lanes' order, is read
// from the L2 once per block and feeds twelve products -- and are added through LDS at the end.
//
// Geometries of at most one block per CU may take blocks of eight wavefronts and chunks of up to 64 channels instead (see
// plan_real): [16,128,28,28] x [256,128,3,3] stride 2 forward 35 -> 30 us, dx of [8,256,14,14] x [256,256,3,3] 46.5 -> 42,
// [4,512,7,7] x [512,512,1,1] 42 -> 34.
//
// What bounds it: a step of 24 MFMAs takes a wavefront 0.56 us (0.32 of the matrix cores alone), a chunk's barriers,
// splitting and stores 0.8, and a block's start and end 7; with few blocks that chain is the time.  Digit operands of the
// unfolded matrix -> this, dx: [16,128,28,28] x [256,128,3,3] stride 2 70 -> 47 us, [32,64,56,56] x [64,64,3,3] 319 -> 91,
// [8,256,56,56] x [128,256,3,3] 275 -> 146; with binary weights at stride 2 61 -> 48; forward with the weights'
// incremental quantization before it: the same three 65 -> 52, 245 -> 103, 163 -> 161.  Off float64 (2-norm): 0.7e-7 to
// 4e-7 for contractions of up to 4608 terms of random signs and 8.2e-7 at 12800 (a wavefront's quarter of them is one chain
// of fp32 sums), the digits 3.5e-7 to 8.4e-7; for terms of one sign 0.5e-7 to 1.3e-7, the digits 0.5e-7 to 0.9e-7.
//
// Positions whose input window holds a NaN, an infinity, a magnitude of 2^100 or more or nothing above 2^-90, and rows of
// weights with a NaN or an infinity, are recomputed one by one in double.
#include "bf16_parts.hpp"
#include "common.hpp"
#include "conv_geom.hpp"
#include "gemm_layout.hpp"
#include "internal.hpp"

#include <cmath>

namespace nbla_hip {
namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256, kWaves = 4;
constexpr int kRows = 64, kPos = 64;
constexpr uint32_t kOutside = 0x80000000u;     // a byte offset past the end of any tensor: such loads give zeros
constexpr int kMaxTaps = 25, kMaxClasses = 9;
constexpr int kLds = 78 * 1024;                // two blocks of four wavefronts to a CU
constexpr int kLdsWide = 150 * 1024;           // one block of eight
constexpr int red_bytes(int waves) { return waves * kRows * kPos * 4; }
constexpr int kMostItems = 5;                  // (position, eight channels) items a thread stages: registers
constexpr uint32_t kLeast = (127u - 90u) << 23, kMost = (127u + 100u) << 23; // magnitudes, as bits
static_assert(kMostItems * kThreads * 48 <= kLds && red_bytes(kWaves) <= kLds, "");
static_assert(4 * 2 * kThreads * 48 <= kLdsWide && red_bytes(2 * kWaves) <= kLdsWide, "");

struct RealClass {
  int first, taps;  // of the taps' table
  int QH, QW, cy, cx;
  int ty_min, ty_max; // displacements along y
  int positions, tiles, tile0; // N * QH * QW, blocks of them, number of blocks of the classes before
};
struct RealArgs {
  const float *in;         // first channel of the group
  const unsigned char *w;  // prepared weights
  const int *shift;        // per row: the scale's exponent, or kBadRow
  const float *weights;    // as stored, for the positions recomputed (value (r, k, t) at r * w_row + k * w_k + t)
  const float *alpha;      // per k, may be null; signs: the weights' signs stand for them
  const float *bias;
  float *out;              // first channel of the group
  int64_t w_row, w_k;
  int N, CS, CD, Kc, R, IH, IW, OH, OW; // channels of the in- and output tensors, contraction channels and rows of the group
  int ss, ds, row_tiles, ksteps, taps_all, chunk, waves, slots, accumulate, signs, transposed;
  float zero_to;
  uint32_t in_bytes; // from `in` to the end of the tensor
  int classes;
  RealClass cls[kMaxClasses];
  signed char ty[kMaxTaps], tx[kMaxTaps], tap[kMaxTaps];
};

// A weight as it takes part: itself or its sign, times alpha.
__device__ __forceinline__ float weight_value(float v, bool scaled, float alpha, int signs, float zero_to) {
  if (signs)
    v = v < 0.0f ? -1.0f : (v > 0.0f ? 1.0f : zero_to);
  return scaled ? v * alpha : v;
}
__device__ __forceinline__ float real_weight(const float *w, int64_t at, int64_t k, const float *alpha, int signs,
                                             float zero_to) {
  return weight_value(w[at], alpha != nullptr, alpha ? alpha[k] : 1.0f, signs, zero_to);
}

constexpr int kFlight = 10; // loads of a row a thread has in flight
// Block = one row r: its largest magnitude, then the three planes in the lanes' order,
// [tap][16 channels][plane][32 rows][lane (half, row)][8 bf16]; rows and channels past the ends are zeros.
__global__ __launch_bounds__(kThreads) void conv_real_weights(const float *__restrict__ W, unsigned char *__restrict__ dst,
                                                              int *__restrict__ shifts, int R, int Kc, int taps, int ksteps,
                                                              int row_frags, int64_t w_row, int64_t w_k,
                                                              const float *__restrict__ alpha, int signs, float zero_to) {
  extern __shared__ __attribute__((aligned(16))) float s_row[]; // [k][tap]
  __shared__ uint32_t s_max[kWaves];
  const int r = blockIdx.x, tid = threadIdx.x, n = Kc * taps;
  uint32_t amax = 0u;
  if (r < R)
    for (int i0 = tid; i0 < n; i0 += kFlight * kThreads) { // (a load a time is a round trip each: 8.4 us, this way 6.2)
      float v[kFlight], sc[kFlight];
#pragma unroll
      for (int j = 0; j < kFlight; ++j) {
        int t;
        const int k = short_divide(min(i0 + j * kThreads, n - 1), taps, t);
        v[j] = W[r * w_row + k * w_k + t];
        sc[j] = alpha ? alpha[k] : 1.0f;
      }
#pragma unroll
      for (int j = 0; j < kFlight; ++j) {
        const int i = i0 + j * kThreads;
        const float q = weight_value(v[j], alpha != nullptr, sc[j], signs, zero_to);
        if (i < n) {
          s_row[i] = q;
          amax = max(amax, __float_as_uint(q) & 0x7fffffffu);
        }
      }
    }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    amax = max(amax, (uint32_t)__shfl_xor((int)amax, off));
  if ((tid & 63) == 0)
    s_max[tid >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
    amax = max(amax, s_max[w]);
  const bool bad = amax >= 0x7f800000u;
  const int shift = amax ? -binade_exponent(binade_of(amax)) : 0;
  if (tid == 0)
    shifts[r] = bad ? kBadRow : shift;
  const int octets = ksteps * 2;
  for (int i = tid; i < octets * taps; i += kThreads) {
    int q;
    const int t = short_divide(i, octets, q), kstep = q >> 1, half = q & 1;
    uint4_t p[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int k = 8 * q + 2 * j + c;
        v[c] = (r < R && k < Kc && !bad) ? ldexpf(s_row[k * taps + t], shift) : 0.0f;
      }
      uint32_t hi, mid, lo;
      split3_pair(v[0], v[1], hi, mid, lo);
      p[0][j] = hi, p[1][j] = mid, p[2][j] = lo;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int64_t at = ((((int64_t)t * ksteps + kstep) * 3 + d) * row_frags + (r >> 5)) * 64 + half * 32 + (r & 31);
      *reinterpret_cast<uint4_t *>(dst + at * 16) = p[d];
    }
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

template <int kItems, int kW> __global__ __launch_bounds__(64 * kW, 2) void conv_real_kernel(RealArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kT = 64 * kW;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[]; // [plane][octet][slots][16 bytes]; the exchange
  __shared__ uint32_t s_max[2][kW];
  __shared__ int s_bad[kPos], s_shift[kRows];
  __shared__ float s_bias[kRows];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t work_all = (uint32_t)xcd_remap(blockIdx.x, gridDim.x);
  const int row_tile = (int)(work_all % (uint32_t)a.row_tiles), work = (int)(work_all / (uint32_t)a.row_tiles);
  int ci = 0;
  while (ci + 1 < a.classes && work >= a.cls[ci + 1].tile0)
    ++ci;
  const RealClass C = a.cls[ci];
  const int m0 = (work - C.tile0) * kPos, q_plane = C.QH * C.QW, in_plane = a.IH * a.IW;
  // the class's taps, one to a lane: displacement along y, x and the weights' tap, a byte each
  const int tap_at = C.first + min(lane, max(C.taps - 1, 0));
  const int taps_of_lanes = C.taps ? (a.ty[tap_at] & 0xff) | ((a.tx[tap_at] & 0xff) << 8) | (a.tap[tap_at] << 16) : 0;
  if (tid < kRows) {
    const int rr = row_tile * kRows + tid;
    s_shift[tid] = a.shift[rr];
    s_bias[tid] = a.bias && rr < a.R ? a.bias[rr] : -0.0f;
  }
  // ---- the run of input positions under the block: rows of consecutive samples one after the other
  const int m_last = min(m0 + kPos, C.positions) - 1;
  const int n_first = (int)((uint32_t)m0 / (uint32_t)q_plane), n_last = (int)((uint32_t)m_last / (uint32_t)q_plane);
  const int qy_first = (int)((uint32_t)(m0 - n_first * q_plane) / (uint32_t)C.QW);
  const int y_first = qy_first * a.ss + C.ty_min;
  const int y_last = (int)((uint32_t)(m_last - n_last * q_plane) / (uint32_t)C.QW) * a.ss + C.ty_max;
  const int run0 = (n_first * a.IH + min(max(y_first, 0), a.IH - 1)) * a.IW;
  const int run1 = (n_last * a.IH + min(max(y_last, 0), a.IH - 1) + 1) * a.IW;
  const int zero_slot = a.slots - 1, run = C.taps ? min(run1 - run0, zero_slot) : 0; // (class_slots: always the first)
  // ---- the lane's positions: the block's first, taken apart above, and at most 63 more.  (Whole divisions by every lane,
  // here, for the items staged, for the outputs and in the weights' pass: training step of [16,128,28,28] x [256,128,3,3]
  // stride 2 116.9 us, this way 115.0)
  const int x_first = m0 - n_first * q_plane - qy_first * C.QW;
  int py[2], px[2], pbase[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    int qx, qy;
    const int line = qy_first + short_divide(x_first + min(32 * f + r, m_last - m0), C.QW, qx);
    const int n = n_first + short_divide(line, C.QH, qy);
    py[f] = qy * a.ss, px[f] = qx * a.ss, pbase[f] = n * in_plane - run0 + py[f] * a.IW + px[f];
  }
  // ---- what the thread stages: item = (octet, slot), slots fastest
  const int octets = a.chunk / 8, items = octets * run, run_off = run0 - n_first * in_plane;
  uint32_t src[kItems]; // byte offset of the item's first channel
  int dst[kItems];      // LDS offset, a multiple of sixteen, plus the octet; negative: no such item
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int it = tid + kT * i;
    int s, at; // (places past the last item are not used)
    const int o = short_divide(it, max(run, 1), s);
    const int n = n_first + short_divide(run_off + s, in_plane, at);
    const bool is = it < items;
    src[i] = is ? (uint32_t)(n * a.CS * in_plane + at + 8 * o * in_plane) * 4 : kOutside;
    dst[i] = is ? (o * a.slots + s) * 16 + o : -1;
  }
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.in), 0, (int)a.in_bytes, 0x00020000);
  float xv[kItems][8];
  auto load_x = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int left = a.Kc - c0 - 8 * (dst[i] & 15);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        // (the range check takes the sum of both offsets; the scalar one stays inside the tensor, so that the sum with
        // kOutside stays below 2^32)
        xv[i][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            xr, (int)(j < left ? src[i] : kOutside), min(c0 + j, a.Kc - 1) * in_plane * 4, 0));
    }
  };
  const int plane_bytes = octets * a.slots * 16;
  if (tid < 3 * octets) {
    const int d = tid / octets, o = tid - d * octets;
    *reinterpret_cast<uint4_t *>(smem + d * plane_bytes + (o * a.slots + zero_slot) * 16) = uint4_t{0u, 0u, 0u, 0u};
  }
  f32x16_t acc[2][2]; // [rows][positions]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[i][f][q] = 0.0f;
  uint32_t amax = 0u, amin = ~0u; // the largest magnitude of the run; the smallest one that is not zero, less one
  const int row_frags = a.row_tiles * 2, sub_shift = a.chunk >> 5, sub = (1 << sub_shift) - 1; // 16, 32 or 64 channels
  const int steps = C.taps << sub_shift;
  const uint4_t *wbase = reinterpret_cast<const uint4_t *>(a.w) + (int64_t)(row_tile * 2) * 64 + lane;
  const int64_t w_plane = (int64_t)row_frags * 64;

  // A wavefront's steps of a chunk in groups of three, the last one filled up with steps that do nothing.  The loads keep
  // one order without branches between them, so that the waits are for a count: three steps' weights are always in
  // flight, and a chunk's inputs are asked for ahead of the last group of the chunk before.
  auto load_w = [&](int kstep0, int s, uint4_t (&w)[2][3]) __attribute__((always_inline)) {
    const int sc = min(s, steps - 1);
    const int t = __builtin_amdgcn_readlane(taps_of_lanes, sc >> sub_shift) >> 16;
    const int ks = min(kstep0, a.ksteps - 1 - sub) + (sc & sub);
    const uint4_t *p = wbase + ((int64_t)t * a.ksteps + ks) * 3 * w_plane;
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        w[i][d] = p[d * w_plane + i * 64];
  };
  auto step = [&](int s, const uint4_t (&w)[2][3]) __attribute__((always_inline)) {
    if (s >= steps) // uniform
      return;
    const int tp = __builtin_amdgcn_readlane(taps_of_lanes, s >> sub_shift);
    const int dy = (signed char)(tp & 0xff), dx = (signed char)((tp >> 8) & 0xff);
    const int o = ((s & sub) * 2 + half) * a.slots;
    uint4_t x[2][3];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int iy = py[f] + dy, ix = px[f] + dx;
      const bool in = (unsigned)iy < (unsigned)a.IH && (unsigned)ix < (unsigned)a.IW;
      const int slot = in ? pbase[f] + (dy * a.IW + dx) : zero_slot;
#pragma unroll
      for (int d = 0; d < 3; ++d)
        x[f][d] = *reinterpret_cast<const uint4_t *>(smem + d * plane_bytes + (o + slot) * 16);
    }
    constexpr int kPairs[6][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}, {0, 0}}; // the smallest products first
#pragma unroll
    for (int p = 0; p < 6; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f)
          acc[i][f] = mma(w[i][kPairs[p][0]], x[f][kPairs[p][1]], acc[i][f]);
  };
  uint4_t w0[2][3], w1[2][3], w2[2][3];
  const int groups = (steps + 3 * kW - 1) / (3 * kW);
  __syncthreads();
  if (steps) {
    load_x(0);
    load_w(0, wave, w0);
    load_w(0, wave + kW, w1);
    load_w(0, wave + 2 * kW, w2);
  }
  for (int c0 = 0; c0 < a.Kc && steps; c0 += a.chunk) {
    __syncthreads(); // the steps of the chunk before have read their operands
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      uint4_t p[3];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t m0 = __float_as_uint(xv[i][2 * j]) & 0x7fffffffu, m1 = __float_as_uint(xv[i][2 * j + 1]) & 0x7fffffffu;
        amax = max(amax, max(m0, m1));
        amin = min(amin, min(m0 - 1u, m1 - 1u));
        uint32_t hi, mid, lo;
        split3_pair(xv[i][2 * j], xv[i][2 * j + 1], hi, mid, lo);
        p[0][j] = hi, p[1][j] = mid, p[2][j] = lo;
      }
      if (dst[i] >= 0)
#pragma unroll
        for (int d = 0; d < 3; ++d)
          *reinterpret_cast<uint4_t *>(smem + d * plane_bytes + (dst[i] & ~15)) = p[d];
    }
    __syncthreads();
    const int kstep0 = c0 >> 4, next = (c0 + a.chunk) >> 4;
    int s = wave;
    for (int grp = 1; grp < groups; ++grp, s += 3 * kW) {
      step(s, w0);
      load_w(kstep0, s + 3 * kW, w0);
      step(s + kW, w1);
      load_w(kstep0, s + 4 * kW, w1);
      step(s + 2 * kW, w2);
      load_w(kstep0, s + 5 * kW, w2);
    }
    load_x(c0 + a.chunk); // (past the last channel: zeros, without an access)
    step(s, w0);
    load_w(next, wave, w0);
    step(s + kW, w1);
    load_w(next, wave + kW, w1);
    step(s + 2 * kW, w2);
    load_w(next, wave + 2 * kW, w2);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    amax = max(amax, (uint32_t)__shfl_xor((int)amax, off));
    amin = min(amin, (uint32_t)__shfl_xor((int)amin, off));
  }
  if (lane == 0)
    s_max[0][wave] = amax, s_max[1][wave] = amin;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kW; ++w)
    amax = max(amax, s_max[0][w]), amin = min(amin, s_max[1][w]);
  // ---- the wavefronts' sums: each finishes its share of the rows, sixteen or (of eight wavefronts) eight
  float *s_red = reinterpret_cast<float *>(smem); // [wave][row][position]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int row = 32 * i + 8 * (q >> 2) + 4 * half + (q & 3);
        s_red[(wave * kRows + row) * kPos + 32 * f + r] = acc[i][f][q];
      }
  __syncthreads();
  const int m = m0 + lane;
  const bool m_in = m < C.positions;
  int qx, qy;
  const int line = qy_first + short_divide(x_first + min(lane, m_last - m0), C.QW, qx);
  const int n = n_first + short_divide(line, C.QH, qy);
  const int out_plane = a.OH * a.OW;
  float *out = a.out + (int64_t)n * a.CD * out_plane + (qy * a.ds + C.cy) * a.OW + (qx * a.ds + C.cx);
  // a window to be recomputed: only blocks whose run holds something out of range look for them
  const bool suspect = amax >= kMost || amin < kLeast - 1u;
  int any_bad = 0;
  if (suspect) {
    uint32_t big = 0u;
    for (int k = wave; k < a.Kc; k += kW)
      for (int t = 0; t < C.taps; ++t) {
        const int iy = qy * a.ss + a.ty[C.first + t], ix = qx * a.ss + a.tx[C.first + t];
        if ((unsigned)iy < (unsigned)a.IH && (unsigned)ix < (unsigned)a.IW)
          big = max(big, __float_as_uint(a.in[((int64_t)n * a.CS + k) * in_plane + iy * a.IW + ix]) & 0x7fffffffu);
      }
    if (tid < kPos)
      s_bad[tid] = 0;
    __syncthreads();
    // (the largest of the window over the wavefronts' channels; magnitudes below 2^31 as unsigned words)
    atomicMax(reinterpret_cast<unsigned int *>(&s_bad[lane]), big);
    __syncthreads();
    const uint32_t all = (uint32_t)s_bad[lane];
    any_bad = all >= kMost || (all != 0u && all < kLeast);
  }
  bool redo = false;
#pragma unroll
  for (int i = 0; i < kRows / kW; ++i) {
    const int row = wave * (kRows / kW) + i, rr = row_tile * kRows + row, shift = s_shift[row];
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < kW; ++w)
      sum += (double)s_red[(w * kRows + row) * kPos + lane];
    const float v = (float)ldexp(sum, -(shift == kBadRow ? 0 : shift)) + s_bias[row];
    float *o = out + (int64_t)rr * out_plane;
    if (m_in && rr < a.R && !any_bad && shift != kBadRow)
      *o = a.accumulate ? *o + v : v;
    redo |= m_in && rr < a.R && (any_bad || shift == kBadRow);
  }
  if (!redo)
    return;
  for (int row = wave * (kRows / kW); row < (wave + 1) * (kRows / kW); ++row) {
    const int rr = row_tile * kRows + row;
    if (rr >= a.R || !(any_bad || s_shift[row] == kBadRow))
      continue;
    double sum = 0.0;
    for (int k = 0; k < a.Kc; ++k)
      for (int t = 0; t < C.taps; ++t) {
        const int iy = qy * a.ss + a.ty[C.first + t], ix = qx * a.ss + a.tx[C.first + t];
        const bool in = (unsigned)iy < (unsigned)a.IH && (unsigned)ix < (unsigned)a.IW;
        // (the padding is a zero that is multiplied: with an infinite weight it makes a NaN, as the unfolded matrix does,
        // in the forward; the gradient's taps outside are no terms at all)
        if (a.transposed && !in)
          continue;
        const float xv = in ? a.in[((int64_t)n * a.CS + k) * in_plane + iy * a.IW + ix] : 0.0f;
        sum += (double)xv * (double)real_weight(a.weights, rr * a.w_row + k * a.w_k + a.tap[C.first + t], k, a.alpha,
                                                a.signs, a.zero_to);
      }
    const float v = (float)sum + s_bias[row];
    float *o = out + (int64_t)rr * out_plane;
    *o = a.accumulate ? *o + v : v;
  }
#endif
}

// The longest run of input positions under any block of a class, and a slot of zeros.
int64_t class_slots(int64_t QH, int64_t QW, int64_t IH, int64_t IW, int64_t N, int ss, int lo, int hi) {
  const int64_t rows = (kPos - 1 + QW - 1) / QW + 1;                    // rows of positions that 64 of them touch
  const int64_t crossings = (kPos - 1 + QH * QW - 1) / (QH * QW);       // samples they step into
  const int64_t extra = IH - QH * ss > 0 ? IH - QH * ss : 0;            // input rows of a step into the next sample
  // (a first row past the tensor's end, or a last one before its start, is moved onto it)
  const int64_t over = (QH - 1) * ss + lo - (IH - 1), under = -(int64_t)hi;
  int64_t vrows = (rows - 1) * ss + crossings * extra + (hi - lo) + 1 + (over > 0 ? over : 0) + (under > 0 ? under : 0);
  if (vrows > N * IH)
    vrows = N * IH;
  return vrows * IW + 1;
}

// What a block's chunks take, in us: a chunk 0.8 and 0.56 for a step of each of four wavefronts, 1.05 of eight (what the
// rounds of both say at [16,128,28,28] x [256,128,3,3] stride 2, 35 -> 30, and [4,96,27,27] x [48,96,5,5], 38 -> 44).
double block_time(const RealArgs &a, int taps) {
  const double rounds = (double)ceil_div(taps * (a.chunk / 16), a.waves);
  return (double)ceil_div(a.Kc, a.chunk) * (0.8 + (a.waves == kWaves ? 0.56 : 1.05) * rounds);
}

// Fills everything but the pointers; false where the form does not cover the geometry.  Rows of positions that only the
// padding reaches are clipped into the tensor by the kernel, which never makes a run longer than class_slots says.
bool plan_real(const ConvGeom &g, bool transposed, RealArgs &a) {
  if (g.in_sp[0] != 1 || g.k[0] != 1 || g.pad[0] != 0 || g.dil[1] != 1 || g.dil[2] != 1)
    return false;
  if (transposed && g.outer > 65535) // (refused, as the unfolded gradient does)
    return false;
  const int s = g.stride[1], KH = g.k[1], KW = g.k[2];
  if (g.stride[2] != s || s < 1 || s > 3 || KH * KW > kMaxTaps || KH > 25 || KW > 25 || g.pad[1] > 12 || g.pad[2] > 12 ||
      g.pad[1] >= KH || g.pad[2] >= KW)
    return false;
  if (g.outer * g.C * g.in_sp_size >= (1ll << 29) || g.outer * g.O * g.out_sp_size >= (1ll << 29))
    return false;
  a.transposed = transposed ? 1 : 0;
  a.N = (int)g.outer, a.ss = transposed ? 1 : s, a.ds = transposed ? s : 1;
  a.CS = (int)(transposed ? g.O : g.C), a.CD = (int)(transposed ? g.C : g.O);
  a.Kc = (int)(transposed ? g.Og : g.Cg), a.R = (int)(transposed ? g.Cg : g.Og);
  a.IH = transposed ? g.out_sp[1] : g.in_sp[1], a.IW = transposed ? g.out_sp[2] : g.in_sp[2];
  a.OH = transposed ? g.in_sp[1] : g.out_sp[1], a.OW = transposed ? g.in_sp[2] : g.out_sp[2];
  a.w_row = transposed ? g.k_size : g.Kg, a.w_k = transposed ? g.Kg : g.k_size;
  a.taps_all = KH * KW;
  a.row_tiles = (int)ceil_div(a.R, kRows);
  a.classes = 0;
  int table = 0, tiles = 0;
  int64_t slots = 0;
  const int cn = transposed ? s : 1;
  for (int cy = 0; cy < cn; ++cy)
    for (int cx = 0; cx < cn; ++cx) {
      if (a.OH <= cy || a.OW <= cx)
        continue;
      RealClass &c = a.cls[a.classes++];
      c.first = table, c.cy = cy, c.cx = cx;
      c.QH = (a.OH - cy + a.ds - 1) / a.ds, c.QW = (a.OW - cx + a.ds - 1) / a.ds;
      int lo = 0, hi = 0;
      for (int ky = 0; ky < KH; ++ky)
        for (int kx = 0; kx < KW; ++kx) {
          const int ny = transposed ? cy + g.pad[1] - ky : ky - g.pad[1], nx = transposed ? cx + g.pad[2] - kx : kx - g.pad[2];
          if (transposed && (ny % s || nx % s))
            continue;
          const int ty = transposed ? ny / s : ny, tx = transposed ? nx / s : nx;
          if (table == c.first)
            lo = hi = ty;
          lo = ty < lo ? ty : lo, hi = ty > hi ? ty : hi;
          a.ty[table] = (signed char)ty, a.tx[table] = (signed char)tx, a.tap[table] = (signed char)(ky * KW + kx);
          ++table;
        }
      c.taps = table - c.first, c.ty_min = lo, c.ty_max = hi;
      c.positions = a.N * c.QH * c.QW;
      c.tiles = (int)ceil_div(c.positions, kPos), c.tile0 = tiles;
      tiles += c.tiles;
      const int64_t n = class_slots(c.QH, c.QW, a.IH, a.IW, a.N, a.ss, lo, hi);
      slots = n > slots ? n : slots;
    }
  if ((int64_t)tiles * a.row_tiles > 0x7fffffff)
    return false;
  int most_taps = 0;
  for (int c = 0; c < a.classes; ++c)
    most_taps = a.cls[c].taps > most_taps ? a.cls[c].taps : most_taps;
  a.waves = kWaves, a.chunk = a.Kc > 16 && slots * 4 <= 4 * kThreads ? 32 : 16;
  if (slots * (a.chunk / 8) > kMostItems * kThreads)
    return false;
  // Where every CU gets one block at most, a block of eight wavefronts may take it: chunks of up to 64 channels leave
  // fewer of a chunk's steps over after whole rounds of the wavefronts, and fewer barriers.
  if ((int64_t)tiles * a.row_tiles <= 256) {
    const int chunk = a.chunk;
    double best = block_time(a, most_taps) - 1.5;
    for (int c = 32; c <= 64; c *= 2) {
      RealArgs wide = a;
      wide.waves = 2 * kWaves, wide.chunk = c;
      if (slots * (c / 8) > 4 * 2 * kThreads || (c > chunk && a.Kc <= c / 2) || block_time(wide, most_taps) >= best)
        continue;
      best = block_time(wide, most_taps), a.waves = 2 * kWaves, a.chunk = c;
    }
  }
  a.slots = (int)slots;
  a.ksteps = (int)ceil_div(a.Kc, a.chunk) * (a.chunk / 16);
  return (int64_t)a.Kc * a.taps_all * 4 <= 150 * 1024; // (a row of weights in LDS)
}

template <int kItems, int kW> int run_real(const RealArgs &a, int64_t blocks, size_t lds, hipStream_t stream) {
  static std::atomic<uint64_t> configured{0};
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(conv_real_kernel<kItems, kW>),
                                   kW == kWaves ? kLds : kLdsWide, configured,
                                   "hipFuncSetAttribute(conv_real_kernel LDS size)");
  if (rc)
    return rc;
  hipLaunchKernelGGL((conv_real_kernel<kItems, kW>), dim3((unsigned)blocks), dim3(64 * kW), lds, stream, a);
  NBLA_HIP_LAUNCH_CHECK("conv_real_kernel");
  return NBLA_HIP_OK;
}

size_t prepared_bytes(const RealArgs &a) {
  return round_up((size_t)a.taps_all * a.ksteps * 3 * a.row_tiles * 2 * 1024, 256) +
         round_up((size_t)a.row_tiles * kRows * sizeof(int), 256);
}

} // namespace

// Where the geometry is covered, by an estimate of both forms in microseconds, from sizes measured on both: here, blocks
// that share a CU add up, launches and weights come on top (dx, [1,512,7,7] x [512,512,3,3] 87 estimated 76, [64,512,7,7] 128 and 133, [32,256,14,14] x [256,256,3,3]
// 71 and 73); on the digit path the unfolded matrix goes through memory (dx: written and gathered, 0.9 MB a microsecond
// with the transposed gradient; forward: 1.8) and six digit products take 2.4 per 10^9 operations.  What the digits win
// are few positions under many channels: [1,512,7,7] dx 44 against 87.
bool conv_real_applies(const ConvGeom &g, bool transposed, bool binary) {
  RealArgs a;
  if (!plan_real(g, transposed, a))
    return false;
  double total = 0.0, longest = 0.0;
  for (int c = 0; c < a.classes; ++c) {
    if (!a.cls[c].taps)
      continue;
    const double block = block_time(a, a.cls[c].taps);
    total += block * a.cls[c].tiles * a.row_tiles;
    longest = block > longest ? block : longest;
  }
  total *= 1.2 / 256.0;
  const double here = 10.5 + 0.0016 * a.Kc * a.taps_all + (total > longest ? total : longest);
  const double M = (double)g.M, col = M * (double)g.Kg * 4e-6;
  const double digits = transposed ? (36.0 + (col + M * (double)g.Og * 8e-6) / 0.9) * (binary ? 0.8 : 1.0)
                                   : 30.0 + col / 1.8 + 2.4e-9 * 2.0 * M * (double)g.Kg * (double)g.Og;
  return here * 1.15 < digits;
}
// The forward's time in microseconds for layers of few channels and maps, where positions staged and started blocks weigh
// more than the steps do (1300 sizes of fewer than 24 channels and at most 64 maps: 6 % off, 27 at the worst; the estimate
// above, made for wide layers against a form that is far off there, says a third too little from 20000 windows on).
double conv_real_forward_time(const ConvGeom &g) {
  RealArgs a;
  if (!plan_real(g, false, a))
    return 0.0;
  const int taps = a.cls[0].taps, threads = 64 * a.waves;
  const double items = (double)(a.slots * (a.chunk / 8)) / threads; // staged by a thread, per chunk
  const double rounds = (double)ceil_div(taps * (a.chunk / 16), a.waves) * (a.waves == kWaves ? 0.48 : 0.86);
  const double block = 3.1 + (double)ceil_div(a.Kc, a.chunk) * (0.42 * items + rounds);
  const double total = block * a.cls[0].tiles * a.row_tiles / 256.0;
  return 9.3 + 0.004 * a.Kc * taps + std::cbrt(block * block * block + total * total * total);
}
size_t conv_real_workspace_bytes(const ConvGeom &g, bool transposed) {
  RealArgs a;
  return plan_real(g, transposed, a) ? prepared_bytes(a) : 0;
}

int launch_conv_real(const float *in, const float *W, const float *bias, float *out, const ConvGeom &g, bool transposed,
                     int64_t grp, bool accumulate, const float *alpha, bool signs, float zero_to, void *workspace,
                     size_t workspace_bytes, hipStream_t stream) {
  RealArgs a;
  if (!plan_real(g, transposed, a))
    return fail(NBLA_HIP_ERR_NOT_IMPLEMENTED, "convolution: geometry not covered by the bf16 form.");
  const size_t need = prepared_bytes(a);
  if (workspace_bytes < need || !aligned256(workspace))
    return fail(NBLA_HIP_ERR_MEMORY, "convolution (bf16 form): workspace too small or misaligned.");
  unsigned char *w = static_cast<unsigned char *>(workspace);
  int *shift = reinterpret_cast<int *>(w + need - round_up((size_t)a.row_tiles * kRows * sizeof(int), 256));
  a.in = in + grp * a.Kc * (int64_t)a.IH * a.IW, a.out = out + grp * a.R * (int64_t)a.OH * a.OW;
  a.in_bytes = (uint32_t)(((int64_t)a.N * a.CS - grp * a.Kc) * a.IH * a.IW * 4);
  a.weights = W, a.alpha = alpha, a.bias = bias, a.w = w, a.shift = shift;
  a.accumulate = accumulate ? 1 : 0, a.signs = signs ? 1 : 0, a.zero_to = zero_to;
  static std::atomic<uint64_t> configured_w{0};
  int rc = allow_dynamic_lds(reinterpret_cast<const void *>(conv_real_weights), 150 * 1024, configured_w,
                             "hipFuncSetAttribute(conv_real_weights LDS size)");
  if (rc)
    return rc;
  hipLaunchKernelGGL(conv_real_weights, dim3((unsigned)(a.row_tiles * kRows)), dim3(kThreads),
                     (size_t)a.Kc * a.taps_all * sizeof(float), stream, W, w, shift, a.R, a.Kc, a.taps_all, a.ksteps,
                     a.row_tiles * 2, a.w_row, a.w_k, alpha, a.signs, zero_to);
  NBLA_HIP_LAUNCH_CHECK("conv_real_weights");
  const RealClass &last = a.cls[a.classes - 1];
  const int64_t slab = (int64_t)a.slots * a.chunk * 6;
  const int64_t blocks = (int64_t)(last.tile0 + last.tiles) * a.row_tiles, items = a.slots * (a.chunk / 8);
  const size_t lds = (size_t)(slab > red_bytes(a.waves) ? slab : red_bytes(a.waves));
  if (a.waves == 2 * kWaves) {
    if (items <= 2 * 2 * kThreads)
      return run_real<2, 2 * kWaves>(a, blocks, lds, stream);
    return run_real<4, 2 * kWaves>(a, blocks, lds, stream);
  }
  if (items <= 2 * kThreads)
    return run_real<2, kWaves>(a, blocks, lds, stream);
  if (items <= 4 * kThreads)
    return run_real<4, kWaves>(a, blocks, lds, stream);
  return run_real<kMostItems, kWaves>(a, blocks, lds, stream);
}

} // namespace nbla_hip
