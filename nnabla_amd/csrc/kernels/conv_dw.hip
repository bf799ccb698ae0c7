// Weight gradient of a two-dimensional convolution on the fp16 matrix cores, without an unfolded matrix:
//     dW[o, c, ky, kx] = sum over (n, oy, ox) of dy[n, o, oy, ox] * x[n, c, oy s - p + ky, ox s - p + kx]
// (convolution.cpp:199-283 unfolds x per sample and multiplies; the contraction here is the same sum over positions).
//
// Arithmetic.  Every fp32 value, scaled by a power of two that puts its channel's largest finite magnitude into
// [2^14, 2^15), is the sum of two fp16 numbers, hi = fp16(v) and lo = fp16(v - hi), exactly or to one unit of its last
// fp32 place (v - hi has at most 12 bits and a sign) for every value within 2^-18 of the channel's largest; below that to
// 2^-39 of the largest.  Three products (hi hi, hi lo, lo hi) accumulate in fp32 inside the matrix instruction; the
// fourth is below 2^-22 of the product.  A block's sums (kDwChain positions at most unless their partial sums would pass
// 2 GiB; half of them in each of two wavefronts) go to memory as fp32 and are added in a fixed order in double, so the error does not grow with the batch.
// With chains as long as 512 places for blocks made them (12544 positions at [64,512,28,28] x [512,512,3,3]) that gradient
// was 1.0e-6 off float64 for random signs and 3.3e-7 for terms of one sign; now 2.9e-7 and 3.8e-8, at 860 -> 970 us.
// Against float64 the gradient of [32,64,56,56] x [64,64,3,3] is off by 2.5e-7 of its norm
// (1.4e-6 with the products of 24-bit digits of the unfolded matrix, 9.4e-7 for fp32 sums in order).  A NaN or an
// infinity makes NaN of every sum it meets (v - hi is then NaN), those included where it only meets the zeros that fill up
// a row, a tile or a step; the sums that are NaN are therefore formed once more, one by one, in the order and with the
// zeros of the reference (convolution.cpp:199-283).
//
// Layout.  A tile is R output rows of one sample (or NS whole samples of a small map), its positions in groups of eight
// along the rows: dy as [group][hi / lo][64 output channels][8 fp16], x as [input row][column phase][group][hi / lo]
// [channel][8 fp16].  A lane's eight k-slots of v_mfma_f32_32x32x16_f16 are one group of one channel, sixteen bytes.
// Under the tap (ky, kx) the positions of a dy group meet the x group of row oy s + ky shifted by floor((kx - p) / s)
// positions inside the column phase (kx - p) mod s: the wavefront reads the x group and a word of either neighbour once
// per (step, ky) and forms the operands of the kx by shifting registers, under the MFMAs.  A group of zeros in front of
// every row is also the end of the row before.  16 bytes of padding behind each group keep writes (lanes along the
// groups) and reads (lanes along the channels) apart in the banks.  Widths 1, 3 and 5 with padding k / 2, strides 1 and 2:
// the shifts are constants of the kernel, and the output row has as many groups as a phase of the input row.
//
// Four wavefronts: two fragments of 32 output channels x two halves of the steps; each holds NKY x KW x NC fragments
// of 32 input channels (nine for 3 x 3: 144 accumulator registers).  Two blocks share a CU (LDS below 80 KB), one
// converting the rows it loaded into registers a tile ahead while the other multiplies.
//
// What bounds it: at 64 channels a tile of 112 positions takes two blocks 12200 cycles, of which their MFMAs are 6000
// and the conversions of either 4000; the maxima of the channels (8.4 us for 51 MB) and the sum over the splits
// (6.4 us) come on top.  The whole weight gradient, in place of unfolding x into a digit matrix chunk by chunk:
// [32,64,56,56] x [64,64,3,3] 400 -> 54 us, [32,256,14,14] x [256,256,3,3] 95 -> 56, [16,128,28,28] x [256,128,3,3]
// stride 2 62 -> 34; and against tiles of fp32 sums on the vector units (few weights, many positions): [64,64,28,28] x
// [64,64,1,1] 117 -> 28, [64,16,28,28] x [64,16,3,3] 125 -> 32.
#include "common.hpp"
#include "conv_geom.hpp"
#include "gemm_layout.hpp"
#include "internal.hpp"

namespace nbla_hip {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));

constexpr int kDwThreads = 256;
constexpr int kDwO = 64;                    // output channels per block
constexpr int kDwLds = 78 * 1024;           // two blocks to a CU
constexpr int kDwTopBit = 14;               // a channel's largest magnitude lands in [2^14, 2^15)
constexpr int kDwChain = 1024;              // positions that a block adds up in fp32
constexpr int kDwMaxSlices = 16;            // partial maxima per channel
constexpr int kDwQStride = 2 * kDwO * 16 + 16;
constexpr uint32_t kDwOutside = 0x80000000u; // a byte offset past the end of any tensor: such loads give zeros

// The kernel's parameters for a kernel width and stride: rows of taps per wavefront, fragments of input channels per
// wavefront, the items of eight positions a thread holds of x and of dy.
template <int KW, int S> struct DwShape {
  static constexpr int nky = KW == 3 ? 3 : 1, nc = KW == 1 ? 4 : 1;
  static constexpr int phases = KW == 1 ? 1 : S;
  static constexpr int mx = KW == 1 ? (S == 1 ? 6 : 4) : (S == 1 ? 4 : 3);
  static constexpr int my = KW == 1 ? 3 : (S == 1 ? 4 : 2);
  static constexpr int row_step = nky == 1 ? 1 : S;      // x rows kept per output row
  static constexpr int lead = KW > 1 ? 1 : 0;            // the group of zeros in front of a row
  static constexpr int rg_stride = 2 * 32 * nc * 16 + 16;
  static constexpr int phase(int kx) { return ((kx - KW / 2) % S + S) % S; }
  static constexpr int shift(int kx) { return (kx - KW / 2 - phase(kx)) / S; }
  // whether a tap of this phase shifts to the left (dir < 0) or to the right
  static constexpr bool shifts(int ph, int dir) {
    for (int kx = 0; kx < KW; ++kx)
      if (phase(kx) == ph && shift(kx) * dir > 0)
        return true;
    return false;
  }
};

// Division of a small non-negative number by a constant of the launch (v < 2^20, d < 2^12: v + 1/2 is at least 1 / (2 d)
// away from a multiple of d, more than the roundings).
struct DwDivide {
  float inv; // (from the host: kept in a scalar register)
  int d;
  void set(int d_) { d = d_, inv = 1.0f / (float)d_; }
  __device__ __forceinline__ int operator()(int v, int &rest) const {
    const int q = (int)(((float)v + 0.5f) * inv);
    rest = v - q * d;
    return q;
  }
};

struct DwPlan {
  int KH, KW, S, nky, nc;
  int items; // runs of eight values that a thread converts per tile
  int G, Gx, R, NS, rows_x, Q, steps, row_tiles; // (G groups per output row; Gx = G and the zeros in front)
  int ot, ct, kg, splits, tiles, per_split;
  int dy_off, tab_off, misc_off, lds;
  int slices;
  DwDivide by_xc, by_rows_x, by_q, by_g, by_r;
  size_t max_off, shift_off, partial_off, sum_off, total;
};

struct DwArgs {
  const float *dy, *x;       // first channel of the group
  const uint32_t *maxima;    // [slice][Cg + Og]
  int32_t *shifts;           // [Cg + Og], written by the first blocks for the last pass
  float *partial;            // [split][tap][Og][Cg]
  int N, C, O, Cg, Og, IH, IW, OH, OW, pad_h;
  uint32_t x_bytes, dy_bytes, partial_bytes; // from the pointers above to the end of the tensors
  DwPlan p;
};

// Largest finite magnitude of every channel of x and dy over slices of the samples: block (slice, channel).  kSum:
// the sums of dy's channels too, for the bias gradient, which had read dy in a pass of its own (two launches, 8 to 12 us).
template <bool kSum>
__global__ __launch_bounds__(256) void conv_dw_maxima(const float *__restrict__ x, const float *__restrict__ dy,
                                                      uint32_t *__restrict__ maxima, float *__restrict__ sums, int N, int C,
                                                      int O, int Cg, int Og, int xplane, int yplane) {
  __shared__ uint32_t s_max[4];
  __shared__ float s_sum[4];
  const int ch = blockIdx.y, slice = blockIdx.x, tid = threadIdx.x;
  const bool is_x = ch < Cg;
  const int plane = is_x ? xplane : yplane;
  const float *src = is_x ? x + (int64_t)ch * xplane : dy + (int64_t)(ch - Cg) * yplane;
  const int64_t sample = is_x ? (int64_t)C * xplane : (int64_t)O * yplane;
  const int per = (N + (int)gridDim.x - 1) / (int)gridDim.x, n0 = slice * per, n1 = min(N, n0 + per);
  uint32_t amax = 0u;
  float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  // (loads past the end repeat the last value)
  auto take = [&](float v, int j, bool in) __attribute__((always_inline)) {
    const uint32_t m = __float_as_uint(v) & 0x7fffffffu;
    amax = max(amax, m < 0x7f800000u ? m : 0u);
    if (kSum)
      sum[j] += in ? v : 0.0f;
  };
  if (plane >= 256) {
    for (int n = n0; n < n1; ++n) {
      const float *p = src + n * sample;
      for (int i = tid; i < plane; i += 1024) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[j] = p[min(i + 256 * j, plane - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          take(v[j], j, i + 256 * j < plane);
      }
    }
  } else { // several samples' planes side by side
    const int total = (n1 - n0) * plane;
    for (int i = tid; i < total; i += 1024) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = min(i + 256 * j, total - 1), n = at / plane;
        v[j] = src[(n0 + n) * sample + (at - n * plane)];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        take(v[j], j, i + 256 * j < total);
    }
  }
  float all = (sum[0] + sum[1]) + (sum[2] + sum[3]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    amax = max(amax, (uint32_t)__shfl_xor((int)amax, off));
  if (kSum) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
      all += __shfl_xor(all, off);
  }
  if ((tid & 63) == 0)
    s_max[tid >> 6] = amax, s_sum[tid >> 6] = all;
  __syncthreads();
  if (tid == 0) {
    maxima[slice * (Cg + Og) + ch] = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
    if (kSum && !is_x)
      sums[slice * Og + (ch - Cg)] = (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]);
  }
}

// The bias gradient from the slices' sums of dy: further blocks of conv_dw_sum.
struct DwBias {
  const float *sums;
  float *db; // null: not wanted
  int slices, accumulate, first_block;
};

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dw_rsrc(const float *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ f32x4_t dw_load4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
#endif

template <int KW, int S>
__global__ __launch_bounds__(kDwThreads, 2) void conv_dw_kernel(DwArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  using T = DwShape<KW, S>;
  constexpr int kNky = T::nky, kNc = T::nc, kPhases = T::phases, kMx = T::mx, kMy = T::my, kRowStep = T::row_step;
  constexpr int kRg = T::rg_stride, kUnits = kNky * KW * kNc, kC = 32 * kNc;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const DwPlan &P = a.p;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wo = wave & 1, wk = wave >> 1;
  // neighbouring blocks share a run of tiles: the channels' tiles fastest
  int work = (int)xcd_remap(blockIdx.x, gridDim.x);
  const int cells = P.ot * P.ct * P.kg, split = work / cells;
  work -= split * cells;
  const int kg = work / (P.ot * P.ct);
  work -= kg * (P.ot * P.ct);
  const int ot = work / P.ct, ct = work - ot * P.ct;
  const int o0 = ot * kDwO, c0 = ct * kC, ky0 = kg * kNky;
  unsigned char *s_dy = smem + P.dy_off;
  uint32_t *s_tab = reinterpret_cast<uint32_t *>(smem + P.tab_off); // x group of every dy group, bytes
  int *s_shift = reinterpret_cast<int *>(smem + P.misc_off);        // [kC] of x, [kDwO] of dy

  // ---- set-up: the channels' scales, the table of groups, zeros where no load ever writes
  for (int i = tid; i < kC + kDwO; i += kDwThreads) {
    const bool is_x = i < kC;
    const int ch = is_x ? c0 + i : o0 + (i - kC);
    int shift = 0;
    if (ch < (is_x ? a.Cg : a.Og)) {
      const int at = is_x ? ch : a.Cg + ch;
      uint32_t m = 0u, part[kDwMaxSlices];
#pragma unroll
      for (int s = 0; s < kDwMaxSlices; ++s)
        part[s] = a.maxima[min(s, P.slices - 1) * (a.Cg + a.Og) + at];
#pragma unroll
      for (int s = 0; s < kDwMaxSlices; ++s)
        m = max(m, part[s]);
      shift = m ? kDwTopBit - binade_exponent(binade_of(m)) : 0;
      if (split == 0 && kg == 0 && (is_x ? ot : ct) == 0)
        a.shifts[at] = shift;
    }
    s_shift[i] = shift;
  }
  for (int q = tid; q <= P.Q; q += kDwThreads) {
    const int row = q / P.G, g = q - row * P.G, ns = row / P.R, rr = row - ns * P.R;
    s_tab[q] = q < P.Q ? (uint32_t)(((ns * P.rows_x + rr * kRowStep) * (kPhases * P.Gx) + T::lead + g) * kRg)
                       : (uint32_t)(T::lead * kRg);
  }
  for (int i = tid * 16; i < kDwQStride; i += kDwThreads * 16) // the group that fills up the last step
    *reinterpret_cast<uint4_t *>(s_dy + P.Q * kDwQStride + i) = uint4_t{0u, 0u, 0u, 0u};
  if (T::lead) {
    const int rows = P.NS * P.rows_x * kPhases, words = kRg / 16;
    for (int i = tid; i < (rows + 1) * words; i += kDwThreads) {
      const int row = i / words;
      *reinterpret_cast<uint4_t *>(smem + row * P.Gx * kRg + (i - row * words) * 16) = uint4_t{0u, 0u, 0u, 0u};
    }
  }
  __syncthreads();

  const __amdgpu_buffer_rsrc_t xr = dw_rsrc(a.x, a.x_bytes), yr = dw_rsrc(a.dy, a.dy_bytes);
  const int x_rows = P.NS * P.rows_x, x_items = kC * x_rows * P.G, y_items = kDwO * P.Q;
  f32x4_t xv[kMx][2 * S], yv[kMy][2];
  // item -> (channel, row inside the tile, group): groups and rows fastest, as they lie in memory.  Computed anew for
  // every tile: kept over the tiles the offsets would spill, and a reload waits for the loads issued before it.
  auto x_item = [&](int m, int &c, int &nsr, int &g) __attribute__((always_inline)) {
    int rest, item = tid + kDwThreads * m;
    asm volatile("" : "+v"(item));
    c = P.by_xc(item, rest);
    nsr = P.by_g(rest, g);
    return item < x_items;
  };
  auto y_item = [&](int m, int &o, int &row, int &g) __attribute__((always_inline)) {
    int rest, item = tid + kDwThreads * m;
    asm volatile("" : "+v"(item));
    o = P.by_q(item, rest);
    row = P.by_g(rest, g);
    return item < y_items;
  };
  auto load_tile = [&](int tile) __attribute__((always_inline)) {
    const int n_part = P.NS > 1 ? tile : tile / P.row_tiles;
    const int n0 = n_part * P.NS, oy0 = P.NS > 1 ? 0 : (tile - n_part * P.row_tiles) * P.R;
#pragma unroll
    for (int m = 0; m < kMx; ++m) {
      int c, nsr, g, rr;
      const bool have = x_item(m, c, nsr, g);
      const int ns = P.by_rows_x(nsr, rr);
      const int iy = kRowStep == 1 && S > 1 ? (oy0 + rr) * S + ky0 - a.pad_h : oy0 * S + rr + ky0 - a.pad_h;
      const bool ok = have && c0 + c < a.Cg && n0 + ns < a.N && (unsigned)iy < (unsigned)a.IH;
      const uint32_t off = (uint32_t)(((((n0 + ns) * a.C + c0 + c) * a.IH + iy) * a.IW + 8 * S * g) * 4);
#pragma unroll
      for (int j = 0; j < 2 * S; ++j)
        xv[m][j] = dw_load4(xr, ok ? off + 16 * j : kDwOutside);
      __builtin_amdgcn_sched_barrier(0); // one item's address arithmetic at a time
    }
#pragma unroll
    for (int m = 0; m < kMy; ++m) {
      int o, row, g, rr;
      const bool have = y_item(m, o, row, g);
      const int ns = P.by_r(row, rr);
      const bool ok = have && o0 + o < a.Og && n0 + ns < a.N && oy0 + rr < a.OH;
      const uint32_t off = (uint32_t)(((((n0 + ns) * a.O + o0 + o) * a.OH + oy0 + rr) * a.OW + 8 * g) * 4);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        yv[m][j] = dw_load4(yr, ok ? off + 16 * j : kDwOutside);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // eight values -> their hi and lo halves; values outside the row (columns before first or from end on) are zeros
  auto split8 = [&](const float (&v)[8], int shift, uint4_t &hi, uint4_t &lo) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x2_t t;
      t.x = ldexpf(v[2 * j], shift), t.y = ldexpf(v[2 * j + 1], shift);
      const half2_t h = __builtin_convertvector(t, half2_t);
      const f32x2_t back = __builtin_convertvector(h, f32x2_t);
      f32x2_t rest;
      rest.x = t.x - back.x, rest.y = t.y - back.y;
      const half2_t l = __builtin_convertvector(rest, half2_t);
      hi[j] = __builtin_bit_cast(uint32_t, h);
      lo[j] = __builtin_bit_cast(uint32_t, l);
    }
  };
  auto store_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < kMx; ++m) {
      __builtin_amdgcn_sched_barrier(0);
      int c, nsr, g;
      if (x_item(m, c, nsr, g)) {
        const int shift = s_shift[c];
#pragma unroll
        for (int ph = 0; ph < kPhases; ++ph) {
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            v[j] = 8 * S * g + S * j + ph < a.IW ? xv[m][(S * j + ph) >> 2][(S * j + ph) & 3] : 0.0f;
          uint4_t hi, lo;
          split8(v, shift, hi, lo);
          unsigned char *dst = smem + ((nsr * kPhases + ph) * P.Gx + T::lead + g) * kRg + c * 16;
          *reinterpret_cast<uint4_t *>(dst) = hi;
          *reinterpret_cast<uint4_t *>(dst + kC * 16) = lo;
        }
      }
    }
#pragma unroll
    for (int m = 0; m < kMy; ++m) {
      __builtin_amdgcn_sched_barrier(0);
      int o, row, g;
      if (y_item(m, o, row, g)) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v[j] = 8 * g + j < a.OW ? yv[m][j >> 2][j & 3] : 0.0f;
        uint4_t hi, lo;
        split8(v, s_shift[kC + o], hi, lo);
        unsigned char *dst = s_dy + (row * P.G + g) * kDwQStride + o * 16;
        *reinterpret_cast<uint4_t *>(dst) = hi;
        *reinterpret_cast<uint4_t *>(dst + kDwO * 16) = lo;
      }
    }
  };

  f32x16_t acc[kUnits];
#pragma unroll
  for (int u = 0; u < kUnits; ++u)
#pragma unroll
    for (int q = 0; q < 16; ++q)
      acc[u][q] = 0.0f;
  const int ky_stride = kPhases * P.Gx * kRg, ph_stride = P.Gx * kRg;
  auto multiply_step = [&](int t) __attribute__((always_inline)) {
    const int q = 2 * t + half;
    const unsigned char *ap = s_dy + (q < P.Q ? q : P.Q) * kDwQStride + (wo * 32 + r) * 16;
    const half8_t ah = *reinterpret_cast<const half8_t *>(ap), al = *reinterpret_cast<const half8_t *>(ap + kDwO * 16);
    const unsigned char *bp = smem + s_tab[q < P.Q ? q : P.Q] + r * 16;
#pragma unroll
    for (int ky = 0; ky < kNky; ++ky) {
      uint32_t w[kPhases][kNc][2][6]; // the last word of the group before, the group, the first word of the next
#pragma unroll
      for (int ph = 0; ph < kPhases; ++ph)
#pragma unroll
        for (int nc = 0; nc < kNc; ++nc)
#pragma unroll
          for (int hl = 0; hl < 2; ++hl) {
            const unsigned char *src = bp + ky * ky_stride + ph * ph_stride + hl * (kC * 16) + nc * 512;
            const uint4_t v = *reinterpret_cast<const uint4_t *>(src);
            w[ph][nc][hl][1] = v.x, w[ph][nc][hl][2] = v.y, w[ph][nc][hl][3] = v.z, w[ph][nc][hl][4] = v.w;
            w[ph][nc][hl][0] = T::shifts(ph, -1) ? *reinterpret_cast<const uint32_t *>(src - kRg + 12) : 0u;
            w[ph][nc][hl][5] = T::shifts(ph, 1) ? *reinterpret_cast<const uint32_t *>(src + kRg) : 0u;
          }
#pragma unroll
      for (int kx = 0; kx < KW; ++kx)
#pragma unroll
        for (int nc = 0; nc < kNc; ++nc) {
          const int ph = T::phase(kx), sh = T::shift(kx);
          uint4_t b[2];
#pragma unroll
          for (int hl = 0; hl < 2; ++hl)
#pragma unroll
            for (int j = 0; j < 4; ++j) // positions sh + 2 j and sh + 2 j + 1 of the group
              b[hl][j] = sh == -1  ? __builtin_amdgcn_alignbit(w[ph][nc][hl][j + 1], w[ph][nc][hl][j], 16)
                         : sh == 1 ? __builtin_amdgcn_alignbit(w[ph][nc][hl][j + 2], w[ph][nc][hl][j + 1], 16)
                                   : w[ph][nc][hl][j + 1 + sh / 2];
          const half8_t bh = __builtin_bit_cast(half8_t, b[0]), bl = __builtin_bit_cast(half8_t, b[1]);
          f32x16_t &d = acc[(ky * KW + kx) * kNc + nc];
          d = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, d, 0, 0, 0);
        }
    }
  };

  // ---- the tiles of this block: a tile's values wait in registers while the one before is multiplied
  const int first = split * P.per_split, last = min(first + P.per_split, P.tiles);
  load_tile(first);
  for (int tile = first; tile < last; ++tile) {
    store_tile();
    __syncthreads();
    if (tile + 1 < last)
      load_tile(tile + 1);
    for (int t = wk; t < P.steps; t += 2)
      multiply_step(t);
    __syncthreads();
  }

  // ---- the two halves of the steps added through LDS: a wavefront finishes the first units (wk = 0) or the rest, and
  // hands its sums of the others to its partner.  Stores outside the channels fall past the buffer's end.
  constexpr int kFirst = (kUnits + 1) / 2;
  float *red = reinterpret_cast<float *>(smem) + wo * (kUnits * 16 * 64) + lane;
#pragma unroll
  for (int u = 0; u < kUnits; ++u)
    if ((u < kFirst) == (wk == 1)) {
#pragma unroll
      for (int q = 0; q < 16; ++q)
        red[(u * 16 + q) * 64] = acc[u][q];
    }
  __syncthreads();
  const int taps = P.KH * KW;
  const __amdgpu_buffer_rsrc_t pr = dw_rsrc(a.partial, a.partial_bytes);
#pragma unroll
  for (int u = 0; u < kUnits; ++u)
    if ((u < kFirst) == (wk == 0)) {
      const int nc = u % kNc, kx = u / kNc % KW, ky = ky0 + u / (kNc * KW);
      const int c = c0 + nc * 32 + r, o = o0 + wo * 32 + 4 * half;
      const uint32_t base = (uint32_t)((((split * taps + ky * KW + kx) * a.Og + o) * a.Cg + c) * 4);
      const bool ok = ky < P.KH && c < a.Cg;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int oq = 8 * (q >> 2) + (q & 3);
        const float v = acc[u][q] + red[(u * 16 + q) * 64];
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), pr,
                                              (int)(ok && o + oq < a.Og ? base + (uint32_t)(oq * a.Cg * 4) : kDwOutside),
                                              0, 0);
      }
    }
#endif
}

// dW[o, c, tap] (+)= 2^-(shifts) * the splits' sums added in double: a thread adds every kRuns-th split of an output,
// 256 / kRuns outputs along c to a block (the launch takes as many runs as give every CU eight blocks: with more, the
// blocks' starts are the time).  Sums that are not finite are formed anew from dy and the unfolded input, by the wavefront
// (the values of a finite x and dy never overflow here).
template <int kRuns>
__global__ __launch_bounds__(256) void conv_dw_sum(const float *__restrict__ partial, const int32_t *__restrict__ shifts,
                                                   float *__restrict__ dW, int Og, int Cg, int taps, int splits,
                                                   int accumulate, const float *__restrict__ x,
                                                   const float *__restrict__ dy, ConvGeom g, int64_t grp, DwBias bias) {
  constexpr int kOuts = 256 / kRuns;
  if (bias.db && (int)blockIdx.x >= bias.first_block) {
    const int o = ((int)blockIdx.x - bias.first_block) * 256 + threadIdx.x;
    if (o < Og) {
      double total = 0.0;
      for (int s = 0; s < bias.slices; ++s)
        total += (double)bias.sums[s * Og + o];
      bias.db[o] = bias.accumulate ? bias.db[o] + (float)total : (float)total;
    }
    return;
  }
  __shared__ double s_sum[kRuns][kOuts];
  const int col = threadIdx.x % kOuts, run = threadIdx.x / kOuts;
  const int64_t outs = (int64_t)taps * Og * Cg, at = (int64_t)blockIdx.x * kOuts + col;
  double sum = 0.0;
  if (at < outs) {
    int s = run;
    for (; s + 3 * kRuns < splits; s += 4 * kRuns) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = partial[(int64_t)(s + kRuns * j) * outs + at];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        sum += (double)v[j];
    }
    for (; s < splits; s += kRuns)
      sum += (double)partial[(int64_t)s * outs + at];
  }
  if (kRuns > 1) {
    s_sum[run][col] = sum;
    __syncthreads();
    if ((int)threadIdx.x >= (kOuts > 64 ? kOuts : 64)) // whole wavefronts
      return;
  }
  bool redo = false;
  if (run == 0 && at < outs) {
#pragma unroll
    for (int j = 1; j < kRuns; ++j)
      sum += s_sum[j][col];
    redo = !__builtin_isfinite(sum);
    const int64_t tap = at / ((int64_t)Og * Cg), oc = at - tap * ((int64_t)Og * Cg);
    const int o = (int)(oc / Cg), c = (int)(oc - (int64_t)o * Cg);
    const float v = (float)ldexp(sum, -(shifts[c] + shifts[Cg + o]));
    float *dst = dW + oc * taps + tap;
    if (!redo)
      *dst = accumulate ? *dst + v : v;
  }
  for (uint64_t left = __ballot(redo); left; left &= left - 1) {
    const int64_t out = (int64_t)blockIdx.x * kOuts + (threadIdx.x & ~63u) + __builtin_ctzll(left), tap = out / ((int64_t)Og * Cg);
    const int64_t oc = out - tap * ((int64_t)Og * Cg), o = oc / Cg, c = oc - o * Cg, L = g.out_sp_size;
    double part = 0.0;
    for (int64_t m0 = 0; m0 < g.M && !__ballot(__builtin_isnan(part)); m0 += 16 * 64) // (nothing brings a NaN back)
      for (int64_t m = m0 + (threadIdx.x & 63); m < g.M && m < m0 + 16 * 64; m += 64) {
        const int64_t n = m / L, l = m - n * L;
        part += (double)dy[(n * g.O + grp * g.Og + o) * L + l] * (double)col_value(x, g, grp, m, c * taps + tap);
      }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
      part += __shfl_xor(part, off);
    if ((threadIdx.x & 63) == 0) {
      float *dst = dW + oc * taps + tap;
      *dst = accumulate ? *dst + (float)part : (float)part;
    }
  }
}

template <int KW, int S> void plan_shape(DwPlan &p, int &mx, int &my, int &row_step, int &phases, int &rg, int &lead) {
  using T = DwShape<KW, S>;
  p.nky = T::nky, p.nc = T::nc;
  mx = T::mx, my = T::my, row_step = T::row_step, phases = T::phases, rg = T::rg_stride, lead = T::lead;
}

bool make_dw_plan(const ConvGeom &g, DwPlan &p) {
  for (int i = 0; i < kMaxSpatial; ++i)
    if (g.dil[i] != 1 && g.k[i] != 1)
      return false;
  if (g.k[0] != 1 || g.in_sp[0] != 1 || g.out_sp[0] != 1 || g.pad[0] != 0)
    return false;
  if (g.outer > 65535) // the unfolded form refuses such calls, with whatever other gradient they want
    return false;
  p.KH = g.k[1], p.KW = g.k[2], p.S = g.stride[2];
  if (g.stride[1] != g.stride[2] || p.KH > 16 || g.pad[2] != p.KW / 2)
    return false;
  int mx, my, row_step, phases, rg, lead;
  switch (p.KW * 4 + p.S) {
  case 1 * 4 + 1: plan_shape<1, 1>(p, mx, my, row_step, phases, rg, lead); break;
  case 1 * 4 + 2: plan_shape<1, 2>(p, mx, my, row_step, phases, rg, lead); break;
  case 3 * 4 + 1: plan_shape<3, 1>(p, mx, my, row_step, phases, rg, lead); break;
  case 3 * 4 + 2: plan_shape<3, 2>(p, mx, my, row_step, phases, rg, lead); break;
  case 5 * 4 + 1: plan_shape<5, 1>(p, mx, my, row_step, phases, rg, lead); break;
  case 5 * 4 + 2: plan_shape<5, 2>(p, mx, my, row_step, phases, rg, lead); break;
  default: return false;
  }
  // a tile of 64 output channels x 32 (1 x 1: 128) input channels should not be mostly padding, and offsets are 32 bits
  if (g.Og < 16 || g.Cg < (p.nc > 1 ? 32 : 8) || g.outer * g.C * g.in_sp_size * 4 >= ((int64_t)1 << 31) ||
      g.outer * g.O * g.out_sp_size * 4 >= ((int64_t)1 << 31) || g.Og * g.Kg >= ((int64_t)1 << 28) || g.Cg + g.Og > 65535)
    return false;
  const int OH = g.out_sp[1], OW = g.out_sp[2], C = 32 * p.nc;
  if (OW > 512)
    return false;
  p.G = (int)ceil_div(OW, 8);
  p.Gx = p.G + lead;
  auto sizes = [&](int R, int NS) {
    p.R = R, p.NS = NS, p.rows_x = (R - 1) * row_step + p.nky, p.Q = R * NS * p.G;
    p.dy_off = (NS * p.rows_x * phases * p.Gx + lead) * rg;
    p.tab_off = p.dy_off + (p.Q + 1) * kDwQStride;
    p.misc_off = (int)round_up((size_t)p.tab_off + 4 * (p.Q + 1), 16);
    p.lds = p.misc_off + 4 * (C + kDwO);
    const int reduce = 2 * p.nky * p.KW * p.nc * 16 * 64 * 4; // the sums two wavefronts exchange
    if (p.lds < reduce)
      p.lds = reduce;
    p.items = (int)(ceil_div(C * NS * p.rows_x * p.G, kDwThreads) * p.S + ceil_div(kDwO * p.Q, kDwThreads));
    return C * NS * p.rows_x * p.G <= mx * kDwThreads && kDwO * p.Q <= my * kDwThreads && p.lds <= kDwLds;
  };
  if (!sizes(1, 1))
    return false;
  int R = 1, NS = 1;
  while (R < OH && sizes(R + 1, 1))
    ++R;
  if (R == OH)
    while (NS < g.outer && sizes(OH, NS + 1))
      ++NS;
  p.row_tiles = (int)ceil_div(OH, R);
  R = (int)ceil_div(OH, p.row_tiles); // as even as possible
  sizes(R, NS);
  p.steps = (p.Q + 1) / 2;
  p.by_xc.set(NS * p.rows_x * p.G), p.by_rows_x.set(p.rows_x), p.by_q.set(p.Q), p.by_g.set(p.G), p.by_r.set(p.R);
  p.ot = (int)ceil_div(g.Og, kDwO), p.ct = (int)ceil_div(g.Cg, C), p.kg = (int)ceil_div(p.KH, p.nky);
  const int64_t tiles = NS > 1 ? ceil_div(g.outer, NS) : g.outer * p.row_tiles;
  if (tiles >= ((int64_t)1 << 30))
    return false;
  p.tiles = (int)tiles;
  // two blocks per CU: as many splits as fill 512 places once -- or several times, where a block would otherwise sum more
  // than kDwChain positions (and the splits' sums stay below 2 GiB) -- each with the same number of tiles (the last fewer)
  const int64_t cells = (int64_t)p.ot * p.ct * p.kg;
  const int64_t most = p.Q * 8 < kDwChain ? kDwChain / (p.Q * 8) : 1; // tiles of a block
  const int64_t rounds = ceil_div(cells * ceil_div(tiles, most), 512);
  int64_t splits = 512 * rounds / cells;
  const int64_t room = (((int64_t)1 << 31) - 1) / (4 * g.Og * g.Kg);
  if (splits > room)
    splits = room;
  if (splits < 1)
    splits = 1;
  if (splits > tiles)
    splits = tiles;
  p.per_split = (int)ceil_div(tiles, splits);
  p.splits = (int)ceil_div(tiles, p.per_split);
  if (cells * p.splits >= ((int64_t)1 << 30) || p.splits * g.Og * g.Kg * 4 >= ((int64_t)1 << 31))
    return false;
  const int64_t channels = g.Cg + g.Og;
  int64_t slices = ceil_div(2048, channels);
  if (slices > g.outer)
    slices = g.outer;
  if (slices > kDwMaxSlices)
    slices = kDwMaxSlices;
  p.slices = (int)ceil_div(g.outer, ceil_div(g.outer, slices));
  p.max_off = 0;
  p.shift_off = round_up((size_t)p.slices * channels * sizeof(uint32_t), 256);
  p.partial_off = p.shift_off + round_up((size_t)channels * sizeof(int32_t), 256);
  p.sum_off = p.partial_off + round_up((size_t)p.splits * g.Og * g.Kg * sizeof(float), 256);
  p.total = p.sum_off + round_up((size_t)p.slices * g.Og * sizeof(float), 256);
  return true;
}

template <int KW, int S> int run_conv_dw(const DwArgs &a, hipStream_t stream) {
  static std::atomic<uint64_t> configured{0};
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(conv_dw_kernel<KW, S>), kDwLds, configured,
                                   "hipFuncSetAttribute(conv_dw LDS size)");
  if (rc)
    return rc;
  const unsigned blocks = (unsigned)(a.p.ot * a.p.ct * a.p.kg * a.p.splits);
  hipLaunchKernelGGL((conv_dw_kernel<KW, S>), dim3(blocks), dim3(kDwThreads), (size_t)a.p.lds, stream, a);
  NBLA_HIP_LAUNCH_CHECK("conv_dw");
  return NBLA_HIP_OK;
}

} // namespace

// Where the geometry is covered, by an estimate of both forms in microseconds, fitted to 110 geometries measured on both
// (1 to 4096 samples of 1 x 1 to 56 x 56 positions, 16 to 512 channels; off by 15 % at the median).  Here: a wavefront's
// MFMAs of a tile at 1.46 times their 32 cycles, 490 cycles for each run of eight values that a thread converts, twice as
// long where blocks share a CU, and the splits' partial sums through memory.  The product of digit operands: x unfolded
// and converted, dy transposed and converted, tiles of 128 x 128 weights.  It wins where a kernel of five rows, whose taps
// take a pass over x for each row, meets many channels on both sides: [32,512,14,14] x [512,512,5,5] 306 us against 530
// here; [64,512,14,14] x [512,512,3,3] 302 against 309, [64,512,2,2] 47 against 48.  A tie goes to this form, the more
// precise one.
bool conv_dw_applies(const ConvGeom &g) {
  DwPlan p;
  if (!make_dw_plan(g, p))
    return false;
  const int64_t blocks = (int64_t)p.ot * p.ct * p.kg * p.splits;
  const double rounds = (double)ceil_div(blocks, 512) * (blocks > 256 ? 2.0 : 1.0);
  const double mfma = 32.0 * 3 * ceil_div(p.steps, 2) * p.nky * p.KW * p.nc, M = (double)g.M;
  const double here = 20.0 + rounds * p.per_split * (1.46 * mfma + 490.0 * p.items) / 2400.0 +
                      1.5e-6 * (double)p.splits * (double)g.Og * (double)g.Kg;
  const double digits = 45.0 + 2.3e-6 * M * (double)g.Kg + 11.5e-6 * M * (double)g.Og +
                        1.2e-9 * M * (double)(ceil_div(g.Kg, 128) * ceil_div(g.Og, 128) * 128 * 128);
  return here <= 1.15 * digits;
}

size_t conv_dw_workspace_bytes(const ConvGeom &g) {
  DwPlan p;
  return conv_dw_applies(g) && make_dw_plan(g, p) ? p.total : 0;
}

int launch_conv_dw(const float *dy, const float *x, float *dW, const ConvGeom &g, int64_t grp, bool accumulate,
                   void *workspace, size_t workspace_bytes, hipStream_t stream, float *db, bool accumulate_db) {
  DwArgs a;
  if (!make_dw_plan(g, a.p))
    return fail(NBLA_HIP_ERR_NOT_IMPLEMENTED, "the weight gradient product does not cover this geometry.");
  if (workspace_bytes < a.p.total || !aligned256(workspace))
    return fail(NBLA_HIP_ERR_MEMORY, "weight gradient workspace too small (%zu < %zu) or misaligned.", workspace_bytes,
                a.p.total);
  char *base = static_cast<char *>(workspace);
  uint32_t *maxima = reinterpret_cast<uint32_t *>(base + a.p.max_off);
  float *sums = reinterpret_cast<float *>(base + a.p.sum_off);
  const int64_t x_first = grp * g.Cg * g.in_sp_size, dy_first = grp * g.Og * g.out_sp_size;
  a.x = x + x_first, a.dy = dy + dy_first;
  a.maxima = maxima;
  a.shifts = reinterpret_cast<int32_t *>(base + a.p.shift_off);
  a.partial = reinterpret_cast<float *>(base + a.p.partial_off);
  a.N = (int)g.outer, a.C = (int)g.C, a.O = (int)g.O, a.Cg = (int)g.Cg, a.Og = (int)g.Og;
  a.IH = g.in_sp[1], a.IW = g.in_sp[2], a.OH = g.out_sp[1], a.OW = g.out_sp[2];
  a.pad_h = g.pad[1];
  a.x_bytes = (uint32_t)((g.outer * g.C * g.in_sp_size - x_first) * 4);
  a.partial_bytes = (uint32_t)(a.p.splits * g.Og * g.Kg * 4);
  a.dy_bytes = (uint32_t)((g.outer * g.O * g.out_sp_size - dy_first) * 4);
  const dim3 max_grid((unsigned)a.p.slices, (unsigned)(g.Cg + g.Og));
  if (db)
    hipLaunchKernelGGL(conv_dw_maxima<true>, max_grid, dim3(256), 0, stream, a.x, a.dy, maxima, sums, a.N, a.C, a.O, a.Cg,
                       a.Og, (int)g.in_sp_size, (int)g.out_sp_size);
  else
    hipLaunchKernelGGL(conv_dw_maxima<false>, max_grid, dim3(256), 0, stream, a.x, a.dy, maxima, sums, a.N, a.C, a.O, a.Cg,
                       a.Og, (int)g.in_sp_size, (int)g.out_sp_size);
  NBLA_HIP_LAUNCH_CHECK("conv_dw_maxima");
  int rc;
  switch (a.p.KW * 4 + a.p.S) {
  case 1 * 4 + 1: rc = run_conv_dw<1, 1>(a, stream); break;
  case 1 * 4 + 2: rc = run_conv_dw<1, 2>(a, stream); break;
  case 3 * 4 + 1: rc = run_conv_dw<3, 1>(a, stream); break;
  case 3 * 4 + 2: rc = run_conv_dw<3, 2>(a, stream); break;
  case 5 * 4 + 1: rc = run_conv_dw<5, 1>(a, stream); break;
  default: rc = run_conv_dw<5, 2>(a, stream); break;
  }
  if (rc)
    return rc;
  const int64_t outs = g.Og * g.Kg;
  DwBias bias{sums, db ? db + grp * g.Og : nullptr, a.p.slices, accumulate_db ? 1 : 0, 0};
  const int64_t bias_blocks = db ? ceil_div(g.Og, 256) : 0;
#define NBLA_DW_SUM(RUNS)                                                                                              \
  do {                                                                                                                 \
    bias.first_block = (int)ceil_div(outs * RUNS, 256);                                                                \
    hipLaunchKernelGGL(conv_dw_sum<RUNS>, dim3((unsigned)(bias.first_block + bias_blocks)), dim3(256), 0, stream,      \
                       a.partial, a.shifts, dW + grp * g.Og * g.Kg, a.Og, a.Cg, (int)g.k_size, a.p.splits,             \
                       accumulate ? 1 : 0, x, dy, g, grp, bias);                                                       \
  } while (0)
  if (outs >= 2048 * 256)
    NBLA_DW_SUM(1);
  else if (outs >= 1024 * 256)
    NBLA_DW_SUM(2);
  else if (outs >= 512 * 256)
    NBLA_DW_SUM(4);
  else
    NBLA_DW_SUM(8);
#undef NBLA_DW_SUM
  NBLA_HIP_LAUNCH_CHECK("conv_dw_sum");
  return NBLA_HIP_OK;
}

} // namespace nbla_hip
