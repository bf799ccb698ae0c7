// Binary convolution forward on the int8 matrix cores with the unfold done by addressing (convolution.cpp:161-197 and
// unfold_to_patches.cpp:103-194 unfold x into a matrix [positions, channels x taps] and multiply it by the weights;
// here that matrix is never formed, not even in LDS).
//
// A block owns up to 32 WM consecutive output positions of one sample and 64 WN output channels.  Every input position
// ("pixel") that one of its windows touches lies in one run [lo, hi] of the flattened input map; the block reads that
// run of all the group's channels once (coalesced along the positions), turns every value into four balanced
// base-256 int8 digits under one power-of-two scale for the whole slab, and keeps the digits in LDS pixel by pixel:
//     slab[pixel 0..npix][channel tile of 32][digit 0..3][32 channels]   (pixel 0 is all zeros: the taps that fall
//                                                                         outside the input)
// The contraction runs over k' = (tap, channel) instead of the reference's (channel, tap): exact integer sums do not
// depend on the order, and in this order the sixteen k-slots of a lane of the i8 MFMA operand are sixteen
// consecutive channels of ONE pixel -- one 16-byte LDS read at (pixel of the lane's window under that tap) + channel
// offset.  So a value is converted once per block (not once per window that holds it: nine times for a 3 x 3 kernel),
// nothing is gathered element by element, and the main loop is LDS reads, one load of packed weight bits per k tile
// and MFMAs, without a barrier.
//
// The weights come as packed bits (gemm_layout.hpp) in the same k order, written by conv_taps_prepare below in its
// one pass over W (Sign(W), the bits, per channel tile the sums of |W| and the counts of weights that are neither
// negative nor positive); the product's set-up adds the partial sums in a fixed order into alpha = mean |W|
// (binary_weight_convolution.cpp:58-69), and its first block writes alpha and the zero count out.  Two launches per
// group make the whole forward.
//
// The forms <WN, WM, WK>: WN x WM x WK wavefronts, each with a tile of 64 output channels x 32 windows (two channel
// fragments x four digits = 128 accumulator registers) and every WK-th k tile.  256 output channels fill <4, 1, 2>; with
// fewer, wavefronts along the channels would multiply padding, so they are laid along the windows instead, and a slab
// that serves 128 windows reads and converts far less per window than one for 32 (64 channels at 56 x 56: the three input
// rows under 32 windows of a 3 x 3 kernel are converted for 32 windows, the four under 112 for 112).  Forms of four
// wavefronts run two blocks to a CU, so one block's set-up and stores lie under the other's MFMAs.  What bounds the
// kernel is those serial phases (a block: 5 to 8 thousand cycles until its loads are back, 450 per 64 x 16 values
// converted, 46 per MFMA of 32 (the matrix clock under the power
// limit), 3 to 7 thousand for the epilogue); slab_form_cost weighs them.  Measured, whole forward
// with the weights' pass, <4, 1, 2> -> the form taken: [32,64,56,56] x [64,64,3,3] 167 -> 44 us, [64,64,28,28] x
// [64,64,1,1] 68 -> 18.5, [32,128,28,28] x [128,128,3,3] 71 -> 30, [32,96,27,27] x [48,96,5,5] 94 -> 33;
// [32,256,14,14] x [256,256,3,3] keeps <4, 1, 2> (26.1 us).  Addresses and the extent as they are found now took these
// from 44.3, 17.9, 30.3, 36.7 (of one day) to 41.2, 16.2, 28.1, 35.5.
//
// Numerics: q = rint(x * 2^s) with s chosen so that the slab's largest finite magnitude lands in [2^29, 2^30); the
// four digit products are accumulated exactly in int32, combined exactly in integers with the windows' sums of q
// (the bits stand for 0 / 1: sum q * (1 - 2 b) = sum q - 2 sum q b) and rounded once to fp32.  The only error is
// the rounding of x to a multiple of 2^-s: at most 2^-30 of the slab's largest magnitude per element.  Windows whose own
// largest value is more than kSlabLevel binades below that are finished by further rounds of the block, each under the
// scale of the largest of the windows left: so an element is off by at most 2^-27 of the largest value of its own window,
// whatever else lies in the slab.  (On inputs of one magnitude no block has a second round, and the window maxima, the test
// for windows left and the second copy of the product cost 2 to 3 %: [32,64,56,56] x [64,64,3,3] 46.8 -> 48.0 us with the
// host's call, [32,256,14,14] x [256,256,3,3] 29.3 -> 29.8; 49.1 and 29.9 with the windows summed behind the product.  One loop around a single copy of the product costs 8 to 11 %:
// the loop's values crowd the product's registers.)  A window that holds a NaN or an
// infinity gives NaN in all its outputs; other windows of the slab are not affected (such values are left out of the
// scale and read as 0).
#include "common.hpp"
#include "conv_geom.hpp"
#include "gemm_layout.hpp"
#include "internal.hpp"

#include <type_traits>

namespace nbla_hip {
namespace {

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));

constexpr int kSlabRows = 32;        // windows per fragment
constexpr int kSlabDigits = 4;
constexpr int kSlabPixPad = 16;      // bytes between two pixels: consecutive pixels start 4 banks apart
constexpr int kSlabMaxTaps = 64;
constexpr int kSlabAhead = 8;        // k tiles of packed words a wavefront holds in registers ahead of its MFMAs
constexpr int kSlabTopBit = 29;      // the slab's largest magnitude lands in [2^29, 2^30): two q add up in 32 bits
constexpr int kSlabLevel = 3;        // windows smaller by more binades than this take a scale of their own
constexpr int kSlabReduceBytes = 2 * 16 * 64 * 4; // per wavefront: one fragment's accumulators, two integers each
constexpr int kSlabHold = 4;         // work items of the set-up a wavefront keeps in registers between its two steps
constexpr int kSlabLdsLimit = 156 * 1024;
constexpr int kPrepThreads = 256;

// Sizes and LDS offsets of one launch (host and device).
struct SlabPlan {
  int form;        // index into kSlabForms
  int tile_rows, tiles_per_sample, wide_groups;
  int col_groups;  // groups of 64 wn output channels
  int ct;          // channel tiles of 32 (channels padded)
  int frags;       // fragments of 32 output channels
  int ct_chunk;    // channel tiles that the slab holds at a time
  int chunks;      // fills of the slab
  bool fits_once;  // some form holds all channels at a time
  int pix_stride;  // bytes per pixel: 128 per channel tile held, and the padding
  int cap;         // pixels a slab may hold (the zero pixel not counted)
  int slab_bytes;
  int k_tiles;     // taps * ct
  int pixsum_off, pixmax_off, rowpix_off, alpha_off, misc_off, total;
  // the prepared weights of one group: packed bits [k tile][wide group][lane], partial |W| sums [ct][frags * 32],
  // partial zero counts [ct][wide groups * 32]
  size_t bits_bytes, wsum_off, zeros_off, prep_bytes;
};

struct ConvSlabArgs {
  const float *x;
  const uint4_t *bits;
  const float *wsum;  // null: no alpha (BinaryConnect)
  const int *zeros;
  float *alpha_out;   // may be null
  int *zero_count;    // may be null
  const float *bias;
  const float *in_scale; // may be null: input channel c of the group is multiplied by in_scale[c] first
  const float *redo_w;   // may be null: Sign(W) of the group [Og, Cg * taps]; windows holding a NaN or an infinity are
                         // then recomputed element by element (else all their outputs are NaN)
  float *y;
  int accumulate;        // add to y instead of overwriting it
  ConvGeom g;
  int grp;
  float inv_k;
  SlabPlan p;
};

// Flattened input offset of output position p's window origin (may be negative).
inline int64_t slab_origin(const ConvGeom &g, int64_t p) {
  const int o2 = (int)(p % g.out_sp[2]);
  p /= g.out_sp[2];
  const int o1 = (int)(p % g.out_sp[1]);
  const int o0 = (int)(p / g.out_sp[1]);
  const int64_t b0 = (int64_t)o0 * g.stride[0] - g.pad[0], b1 = (int64_t)o1 * g.stride[1] - g.pad[1],
                b2 = (int64_t)o2 * g.stride[2] - g.pad[2];
  return (b0 * g.in_sp[1] + b1) * g.in_sp[2] + b2;
}
__host__ __device__ inline int64_t slab_last_tap(const ConvGeom &g) {
  return (((int64_t)(g.k[0] - 1) * g.dil[0]) * g.in_sp[1] + (int64_t)(g.k[1] - 1) * g.dil[1]) * g.in_sp[2] +
         (int64_t)(g.k[2] - 1) * g.dil[2];
}

template <int WN, int WM, int WK, bool kChunked>
__global__ __launch_bounds__(64 * WN * WM * WK, 2) void binary_conv_slab_kernel(ConvSlabArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kWaves = WN * WM * WK, kThreads = 64 * kWaves, kRows = kSlabRows * WM, kCols = 64 * WN;
  static_assert(WK == 1 || WK == 2, "the contraction is split at most in two");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const ConvGeom &g = a.g;
  const SlabPlan &P = a.p;
  int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Blocks go to the eight XCDs round-robin: an XCD takes a contiguous run of tiles, so the tiles of one sample --
  // whose slabs overlap and whose outputs share cache lines -- meet in one L2.
  const uint32_t work = (uint32_t)xcd_remap(blockIdx.x, gridDim.x); // (below 2^31: checked by the host)
  const int cg = (int)(work % (uint32_t)P.col_groups);
  const int wg = cg * kCols / kWideGroup, frag0 = (cg * kCols % kWideGroup) / 32; // first fragment in its wide group
  const int tile_all = (int)(work / (uint32_t)P.col_groups);
  const int n = (int)((uint32_t)tile_all / (uint32_t)P.tiles_per_sample), tile = tile_all - n * P.tiles_per_sample;
  const int p0 = tile * P.tile_rows;
  const int rows = min(P.tile_rows, (int)g.out_sp_size - p0);
  const int taps = (int)g.k_size, plane = (int)g.in_sp_size, Cg = (int)g.Cg, CT = P.ct;
  const int in0 = g.in_sp[0], in1 = g.in_sp[1], in2 = g.in_sp[2];

  long long *s_pixsum = reinterpret_cast<long long *>(smem + P.pixsum_off);
  uint32_t *s_pixmax = reinterpret_cast<uint32_t *>(smem + P.pixmax_off); // largest magnitude, as bits
  uint32_t *s_rowpix = reinterpret_cast<uint32_t *>(smem + P.rowpix_off); // [tap][row]: pixel index
  float *s_alpha = reinterpret_cast<float *>(smem + P.alpha_off), *s_bias = s_alpha + kCols;
  int *s_misc = reinterpret_cast<int *>(smem + P.misc_off); // the wavefronts' maxima, of the slab and of windows left

  // ---- 0. the block's rows and the slab's extent, which every wavefront finds by itself: it can start loading the slab
  // before anything goes through LDS.
  int half = lane >> 5;
  int row = (wave / WN) % WM * kSlabRows + (lane & 31); // the window of this lane in the product
  const bool row_in = row < rows;
  // The block's first position is taken apart once, with whole divisions; a row adds at most 127 to it.  (Divisions for every row
  // and tap, 64-bit addresses for every load and every output, and the extent found by all lanes made a block's set-up and
  // stores 1.5 to 2 us longer: [32,64,56,56] x [64,64,3,3] 17.8 -> 16.1 us per block, [32,256,14,14] x [256,256,3,3]
  // 27.4 -> 26.1 us for the whole forward.)
  const uint32_t line0 = (uint32_t)p0 / (uint32_t)g.out_sp[2], map0 = line0 / (uint32_t)g.out_sp[1];
  const int first2 = p0 - (int)line0 * g.out_sp[2], first1 = (int)(line0 - map0 * (uint32_t)g.out_sp[1]);
  auto decode = [&](int m, int &b0, int &b1, int &b2) __attribute__((always_inline)) {
    int o2, o1; // rows past the tile repeat its first row
    const int line = first1 + short_divide(first2 + (m < rows ? m : 0), g.out_sp[2], o2);
    const int o0 = (int)map0 + short_divide(line, g.out_sp[1], o1);
    b0 = o0 * g.stride[0] - g.pad[0], b1 = o1 * g.stride[1] - g.pad[1], b2 = o2 * g.stride[2] - g.pad[2];
    return (b0 * in1 + b1) * in2 + b2;
  };
  int lo, npix;
  {
    // Origins grow along a line, from line to line of a map at the same place in the line, and from map to map.  So the
    // smallest is that of the first row, of the line after it or of the map after it, as far as the tile has them, and the
    // largest that of the last row, or of the end of the line or of the map before it: scalars, no exchange of lanes.
    auto origin_at = [&](int o0, int o1, int o2) __attribute__((always_inline)) {
      return ((o0 * g.stride[0] - g.pad[0]) * in1 + o1 * g.stride[1] - g.pad[1]) * in2 + o2 * g.stride[2] - g.pad[2];
    };
    const int w = g.out_sp[2], h = g.out_sp[1], last = p0 + rows - 1;
    const int line1 = (int)((uint32_t)last / (uint32_t)w), map1 = (int)((uint32_t)line1 / (uint32_t)h);
    int omin = origin_at((int)map0, first1, first2), omax = origin_at(map1, line1 - map1 * h, last - line1 * w);
    if (line1 > (int)line0) {
      const int after = first1 + 1 < h ? first1 + 1 : 0, before = line1 - map1 * h;
      omin = min(omin, origin_at((int)map0 + (after == 0), after, 0));
      omax = max(omax, origin_at(before > 0 ? map1 : map1 - 1, before > 0 ? before - 1 : h - 1, w - 1));
    }
    if (map1 > (int)map0) {
      omin = min(omin, origin_at((int)map0 + 1, 0, 0));
      omax = max(omax, origin_at(map1 - 1, h - 1, w - 1));
    }
    lo = min(max(omin, 0), plane - 1);
    const int hi = min(max(omax + (int)slab_last_tap(g), 0), plane - 1);
    npix = min(hi - lo + 1, P.cap); // (the host sized the LDS for the exact maximum: the clamp never acts)
  }
  // ---- 1. the slab: largest finite magnitude, then the digits.  A work item is 64 pixels x 16 channels (lanes along
  // the pixels, sixteen loads per lane); wavefront w takes items w, w + kWaves, ...  A slab of at most kSlabHold items
  // per wavefront is loaded once, all loads in flight together, and kept in registers between the two steps; a larger
  // one is read twice.
  const float *xs = a.x + ((int64_t)n * g.C + (int64_t)a.grp * g.Cg) * plane + lo;
  // Where all channels of the slab do not fit the LDS, it is filled a chunk of channel tiles at a time, the accumulators
  // staying in their registers; the scale is that of all channels, found before the first chunk is converted.
  const int pixel_runs = (npix + 63) >> 6;
  int groups16 = 2 * CT, ch_first = 0, items = pixel_runs * groups16; // the items that are walked: all channels, or a chunk
  float per_group = __builtin_amdgcn_rcpf((float)groups16);
  // item -> (first pixel, first channel); fewer than 2^15 items: the quotient of the number plus one half keeps clear of
  // whole numbers by more than the roundings
  auto item_of = [&](int item, int &pix0, int &ch0) __attribute__((always_inline)) {
    const int pc = __builtin_amdgcn_readfirstlane((int)(((float)item + 0.5f) * per_group));
    pix0 = pc * 64, ch0 = ch_first + (item - pc * groups16) * 16;
  };
  auto take_chunk = [&](int chunk) __attribute__((always_inline)) {
    ch_first = chunk * P.ct_chunk * 32;
    groups16 = 2 * min(P.ct_chunk, CT - chunk * P.ct_chunk);
    per_group = __builtin_amdgcn_rcpf((float)groups16);
    items = pixel_runs * groups16;
  };
  // Nothing but loads: a select or a branch on their results here would make a wavefront wait for one item's loads
  // before it issues the next item's.  Channels past the last repeat it, pixels past the slab the first.  The channel's
  // address is a scalar that steps from load to load (a plane is below 2^32 bytes), the pixel's a 32-bit offset.
  auto load_item = [&](int item, float (&v)[16]) __attribute__((always_inline)) {
    int pix0, ch0;
    item_of(item, pix0, ch0);
    const int pix = pix0 + lane;
    const uint32_t off = (uint32_t)(pix < npix ? pix : 0) * 4u;
    const char *src = reinterpret_cast<const char *>(xs + (int64_t)min(ch0, Cg - 1) * plane);
    const int more = Cg - 1 - ch0; // channels after the item's first
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      v[c] = *reinterpret_cast<const float *>(src + off);
      src += c < more ? (uint32_t)plane * 4u : 0u;
    }
  };
  uint32_t amax = 0u;
  auto scan_item = [&](int item, float (&v)[16]) __attribute__((always_inline)) {
    int pix0, ch0;
    item_of(item, pix0, ch0);
    if (a.in_scale) { // one rounded product per element, before anything else
#pragma unroll
      for (int c = 0; c < 16; ++c)
        v[c] = v[c] * a.in_scale[min(ch0 + c, Cg - 1)];
    }
    if (ch0 + 16 > Cg) { // uniform: only the last channel tile can be padded
#pragma unroll
      for (int c = 0; c < 16; ++c)
        v[c] = ch0 + c < Cg ? v[c] : 0.0f;
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const uint32_t m = __float_as_uint(v[c]) & 0x7fffffffu;
      amax = max(amax, m < 0x7f800000u ? m : 0u);
    }
  };
  int shift = 0;
  uint32_t limit = 0u; // magnitudes above it (non-finite ones always) are converted to zeros
  // the item's digits -> LDS: sixteen consecutive channels of a pixel are sixteen consecutive bytes of each digit
  auto convert_item = [&](int item, const float (&v)[16]) __attribute__((always_inline)) {
    uint32_t w[kSlabDigits][4];
    long long psum = 0;
    uint32_t pmax = 0u;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      uint32_t d[4];
      int part[2] = {0, 0}; // two |q| < 2^30 each
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t m = __float_as_uint(v[4 * u + c]) & 0x7fffffffu;
        pmax = max(pmax, m);
        const int q = m <= limit ? (int)rintf(ldexpf(v[4 * u + c], shift)) : 0;
        part[c >> 1] += q;
        // bytes: lowest digit .. top digit (the carries of the balanced form run through the addition)
        d[c] = ((uint32_t)q + 0x808080u) ^ 0x808080u;
      }
      const uint32_t t01 = __builtin_amdgcn_perm(d[1], d[0], 0x05010400u); // d0.b0 d1.b0 d0.b1 d1.b1
      const uint32_t t23 = __builtin_amdgcn_perm(d[3], d[2], 0x05010400u);
      const uint32_t u01 = __builtin_amdgcn_perm(d[1], d[0], 0x07030602u); // d0.b2 d1.b2 d0.b3 d1.b3
      const uint32_t u23 = __builtin_amdgcn_perm(d[3], d[2], 0x07030602u);
      w[3][u] = __builtin_amdgcn_perm(t23, t01, 0x05040100u); // lowest digits of the four channels
      w[2][u] = __builtin_amdgcn_perm(t23, t01, 0x07060302u);
      w[1][u] = __builtin_amdgcn_perm(u23, u01, 0x05040100u);
      w[0][u] = __builtin_amdgcn_perm(u23, u01, 0x07060302u); // top digits
      psum += (long long)part[0] + part[1];
    }
    int pix0, ch0;
    item_of(item, pix0, ch0);
    if (pix0 + lane < npix) {
      // channel tile ch0 / 32 of the chunk, half (ch0 / 16) % 2 of its 32 channels: one byte per channel and digit
      unsigned char *dst = smem + (pix0 + lane + 1) * P.pix_stride + ((ch0 - ch_first) >> 5) * 128 + (ch0 & 16);
#pragma unroll
      for (int dg = 0; dg < kSlabDigits; ++dg) {
        uint4_t o;
        o.x = w[dg][0], o.y = w[dg][1], o.z = w[dg][2], o.w = w[dg][3];
        *reinterpret_cast<uint4_t *>(dst + dg * 32) = o;
      }
      if (psum != 0)
        atomicAdd(reinterpret_cast<unsigned long long *>(&s_pixsum[pix0 + lane + 1]), (unsigned long long)psum);
      if (pmax != 0u)
        atomicMax(&s_pixmax[pix0 + lane + 1], pmax);
    }
  };
  const bool hold = !kChunked && items <= kSlabHold * kWaves; // uniform over the block
  float hv[kSlabHold][16];
  if (hold) {
#pragma unroll
    for (int h = 0; h < kSlabHold; ++h)
      if (wave + h * kWaves < items) // uniform
        load_item(wave + h * kWaves, hv[h]);
  }
  // the partial |W| sums of the block's channels (the first eight channel tiles) and the bias: used in the epilogue
  float av[8], bias_v = -0.0f;
  const int ogp = P.frags * 32, col = cg * kCols + (tid & (kCols - 1));
  if (tid < kCols) {
    if (a.wsum) {
      const float *part = a.wsum + (col < ogp ? col : ogp - 1);
#pragma unroll
      for (int c = 0; c < 8; ++c)
        av[c] = part[(int64_t)(c < CT ? c : CT - 1) * ogp];
    }
    if (a.bias)
      bias_v = a.bias[col < g.Og ? col : g.Og - 1];
  }
  // while the loads are in flight: the tables in LDS
  for (int i = tid; i <= P.cap; i += kThreads) {
    s_pixsum[i] = 0;
    s_pixmax[i] = 0u;
  }
  if (tid < kRows)
    s_rowpix[taps * kRows + tid] = 0u; // the entry of steps past the last k tile: the zero pixel
  for (int i = tid; i < (P.pix_stride >> 2); i += kThreads) // the zero pixel
    *reinterpret_cast<uint32_t *>(smem + 4 * i) = 0u;
  const int trow = tid & (kRows - 1);
  int b0, b1, b2;
  const int origin = decode(trow, b0, b1, b2);
  for (int t = tid / kRows; t < taps; t += kThreads / kRows) { // tap t of row trow: its pixel in the slab, if any
    int k2, k1; // (fewer than kSlabMaxTaps taps)
    const int k0 = short_divide(short_divide(t, g.k[2], k2), g.k[1], k1);
    const int e0 = k0 * g.dil[0], e1 = k1 * g.dil[1], e2 = k2 * g.dil[2];
    const int i0 = b0 + e0, i1 = b1 + e1, i2 = b2 + e2;
    const bool ok = trow < rows && (unsigned)i0 < (unsigned)in0 && (unsigned)i1 < (unsigned)in1 &&
                    (unsigned)i2 < (unsigned)in2;
    const int idx = origin + (e0 * in1 + e1) * in2 + e2 - lo + 1;
    const bool held = ok && idx >= 1 && idx <= npix;
    s_rowpix[t * kRows + trow] = held ? (uint32_t)idx : 0u;
  }
  if (hold) {
#pragma unroll
    for (int h = 0; h < kSlabHold; ++h)
      if (wave + h * kWaves < items)
        scan_item(wave + h * kWaves, hv[h]);
  } else {
    for (int item = wave; item < items; item += kWaves) {
      float v[16];
      load_item(item, v);
      scan_item(item, v);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    amax = max(amax, (uint32_t)__shfl_xor((int)amax, off));
  if (lane == 0)
    s_misc[wave] = (int)amax;
  __syncthreads();
  {
    uint32_t bmax = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      bmax = max(bmax, (uint32_t)s_misc[w]);
    if (bmax != 0u)
      shift = kSlabTopBit - binade_exponent(binade_of(bmax));
    limit = bmax;
  }
  auto convert_chunk = [&]() __attribute__((always_inline)) {
    for (int item = wave; item < items; item += kWaves) {
      float v[16];
      load_item(item, v);
      scan_item(item, v); // (the scale and the padding again; the maximum is not used any more)
      convert_item(item, v);
    }
  };
  if (kChunked)
    take_chunk(0);
  if (hold) {
#pragma unroll
    for (int h = 0; h < kSlabHold; ++h)
      if (wave + h * kWaves < items)
        convert_item(wave + h * kWaves, hv[h]);
  } else {
    convert_chunk();
  }
  if (tid < kCols) { // alpha = (sum of the partial sums, in channel-tile order: every block forms the same bits) / K
    float al = 1.0f;
    if (a.wsum) {
      float acc = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c < CT)
          acc += av[c];
      for (int c = 8; c < CT; ++c)
        acc += a.wsum[(int64_t)c * ogp + (col < ogp ? col : ogp - 1)];
      al = acc * a.inv_k;
      if (tile_all == 0 && a.alpha_out && col < g.Og)
        a.alpha_out[col] = al;
    }
    s_alpha[tid] = al;
    s_bias[tid] = bias_v;
  }
  if (work == 0 && wave == kWaves - 1 && a.zero_count) {
    int z = 0;
    for (int i = lane; i < CT * P.wide_groups * 32; i += 64)
      z += a.zeros[i];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
      z += __shfl_xor(z, off);
    if (lane == 0)
      *a.zero_count = z;
  }
  __syncthreads();
  // ---- 2. the product.  Wavefront (wn, wm, wk): channel fragments 2 wn, 2 wn + 1 of the block's, window fragment wm,
  // k tiles wk, wk + WK, ...
  const int wn = wave % WN, wk = wave / (WN * WM);
  uint32_t frag_mask[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    frag_mask[j] = 0x01010101u << (frag0 + 2 * wn + j);
    asm volatile("" : "+s"(frag_mask[j]));
  }
  const int chunks = kChunked ? P.chunks : 1;
  // One round finishes the windows whose largest magnitude is within 2^-kSlabLevel of the slab's scale -- all of them,
  // for inputs of one magnitude.  Windows much smaller than their slab's largest value are finished by a further round,
  // whose scale is that of the largest among them: it converts the slab again, with zeros for whatever is larger still
  // (no window left holds any of it).  A round finishes the largest window left at least, so the rounds end.
  // Returns the largest magnitude of the windows left, 0 when there is none (the same in every wavefront).
  auto round = [&](auto again) __attribute__((always_inline)) -> uint32_t {
  i32x16_t acc[kSlabDigits][2];
#pragma unroll
  for (int d = 0; d < kSlabDigits; ++d)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        acc[d][j][q] = 0;
  long long rowsum = 0; // the sum of q over the lane's window
  uint32_t left = 0u;
  bool rowbad = false, finish = false; // the window holds a NaN or an infinity; is finished by this round
  for (int chunk = 0; chunk < chunks; ++chunk) {
    if (chunk > 0 || again.value) {
      __syncthreads(); // every wavefront is through with the chunk before
      if (kChunked)
        take_chunk(chunk);
      convert_chunk();
      __syncthreads();
    }
    if (chunk == chunks - 1) {
      // Every wavefront adds up the windows it finishes from the pixels' sums, which are complete since the barrier just
      // passed; its lanes l and l + 32 share a window and take every second tap each, five reads in flight at a time.
      uint32_t rowmax = 0u;
      for (int t0 = half; t0 < taps; t0 += 10) {
        uint32_t idx[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) // (past the last tap: the zero pixel)
          idx[j] = t0 + 2 * j < taps ? s_rowpix[(t0 + 2 * j) * kRows + row] : 0u;
#pragma unroll
        for (int j = 0; j < 5; ++j) {
          rowsum += s_pixsum[idx[j]];
          rowmax = max(rowmax, s_pixmax[idx[j]]);
        }
      }
      rowsum += __shfl_xor(rowsum, 32);
      rowmax = max(rowmax, (uint32_t)__shfl_xor((int)rowmax, 32));
      rowbad = rowmax >= 0x7f800000u;
      const bool todo = row_in && (!again.value || (rowmax != 0u && rowmax <= limit)); // (larger ones are finished)
      // (a window all zero is finished by any scale)
      finish = todo && (rowbad || rowmax == 0u ||
                        binade_exponent(binade_of(rowmax)) + kSlabLevel >= binade_exponent(binade_of(limit)));
      uint32_t mine = todo && !finish ? rowmax : 0u;
      if (__ballot(mine != 0u) != 0) {
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1)
          mine = max(mine, (uint32_t)__shfl_xor((int)mine, off));
      }
      if (lane == 0)
        s_misc[8 + wave] = (int)mine;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kWaves; ++w)
        left = max(left, (uint32_t)s_misc[8 + w]);
      left = __builtin_amdgcn_readfirstlane(left);
    }
    const int ctn = kChunked ? groups16 >> 1 : CT; // channel tiles of the chunk
    const int nk = (taps * ctn - wk + WK - 1) / WK;
    if (nk <= 0)
      continue;
    // (tap, channel tile of the chunk), advanced by WK k tiles per step
    auto normalise = [&](int &tap, int &ct) __attribute__((always_inline)) {
      if (ct >= ctn) {
        ct -= ctn, ++tap;
        if (WK == 2 && ct >= ctn)
          ct -= ctn, ++tap;
      }
    };
    // the words of the next step to load: a uniform pointer that stops at the last step (the k tiles of all channels
    // follow each other; those of a chunk are found by their tap and channel tile)
    int tapw = 0, ctw = wk;
    if (kChunked)
      normalise(tapw, ctw);
    int wleft = nk - 1; // steps the position may still advance
    const uint4_t *wnext = a.bits + ((int64_t)(kChunked ? chunk * P.ct_chunk : wk) * P.wide_groups + wg) * 64;
    const int64_t wstep = (int64_t)WK * P.wide_groups * 64;
    auto load_words = [&]() __attribute__((always_inline)) {
      if constexpr (kChunked) {
        const uint4_t w = wnext[(int64_t)(tapw * CT + ctw) * P.wide_groups * 64 + lane];
        if (wleft > 0) {
          ctw += WK;
          normalise(tapw, ctw);
        }
        --wleft;
        return w;
      } else {
        const uint4_t w = wnext[lane];
        wnext += wleft > 0 ? wstep : 0;
        --wleft;
        return w;
      }
    };
    uint4_t words[kSlabAhead];
#pragma unroll
    for (int u = 0; u < kSlabAhead; ++u)
      words[u] = load_words();
    // position of the k tile two steps ahead
    int tap2 = 0, ct2 = wk;
    normalise(tap2, ct2);
    const uint32_t lane_off = (uint32_t)(half * 16);
    const uint32_t *my_rowpix = s_rowpix + row;
    // LDS offset of the lane's sixteen bytes of step (tap2, ct2); past the last k tile: inside the zero pixel
    auto row_off = [&]() __attribute__((always_inline)) {
      return __umul24(my_rowpix[(tap2 < taps ? tap2 : taps) * kRows], (uint32_t)P.pix_stride) +
             (uint32_t)(ct2 * 128) + lane_off;
    };
    auto advance = [&]() __attribute__((always_inline)) {
      ct2 += WK;
      normalise(tap2, ct2);
    };
    auto read_a = [&](uint32_t off, uint4_t (&af)[kSlabDigits]) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < kSlabDigits; ++d)
        af[d] = *reinterpret_cast<const uint4_t *>(smem + off + d * 32);
    };
    // bits -> bytes in {0, 2^F}: register i of channel fragment F is word_i & (0x01010101 << F)
    auto mma = [&](const uint4_t (&af)[kSlabDigits], const uint4_t &w) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint4_t bf;
        bf.x = w.x & frag_mask[j], bf.y = w.y & frag_mask[j], bf.z = w.z & frag_mask[j], bf.w = w.w & frag_mask[j];
#pragma unroll
        for (int d = 0; d < kSlabDigits; ++d)
          acc[d][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4_t, bf),
                                                            __builtin_bit_cast(i32x4_t, af[d]), acc[d][j], 0, 0, 0);
      }
    };
    uint32_t off_a = row_off(); // step 0
    advance();
    uint32_t off_b = row_off(); // step 1
    advance();
    uint4_t af[2][kSlabDigits];
    read_a(off_a, af[0]);
    // Whole rounds of kSlabAhead steps, without a branch inside a round (the compiler then counts the loads in flight
    // exactly: a word is waited for with the younger loads still outstanding).  Steps past the last k tile
    // multiply the zero pixel.  Inside a step the LDS reads of the next step (the table entry and the four digits) and
    // the load of a later step's words are dealt out one per MFMA of this step (sched_group_barrier: 0x008 = MFMA,
    // 0x100 = LDS read, 0x020 = global load): a wavefront that issues them in a row leaves the matrix pipe waiting.
    for (int i0 = 0; i0 < nk; i0 += kSlabAhead) {
#pragma unroll
      for (int u = 0; u < kSlabAhead; ++u) {
        if (i0 + u >= nk)
          break;
        const uint32_t off_c = row_off(); // step i + 2
        advance();
        read_a(off_b, af[(u + 1) & 1]); // step i + 1
        mma(af[u & 1], words[u]);
        words[u] = load_words();
#pragma unroll
        for (int q = 0; q < kSlabDigits + 1; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, kSlabDigits - 2, 0);
        __builtin_amdgcn_sched_barrier(0);
        off_b = off_c;
      }
    }
  }

  // ---- 3. (WK == 2) the two k groups' accumulators added exactly through LDS (the planes are free once every
  // wavefront has left the loop): a wavefront hands the fragment it does not finish (1 - wk) to its partner in the other
  // k group and adds the partner's copy of fragment wk to its own.  Two digits make one integer before they are handed
  // over (hi = m_0 * 256 + m_1, lo = m_2 * 256 + m_3 as below, |m_d| <= 2^21: sums of both groups stay in 32 bits), so two
  // registers of four cross the LDS, under one barrier instead of one per digit.  Digit by digit this took 4.4 of a block's
  // 22.6 us and 27 registers were spilled; whole forward of [32,256,14,14] x [256,256,3,3] 29.35 -> 27.4 us.
  i32x16_t fin[2]; // hi, lo of the fragment this wavefront finishes
  if constexpr (WK == 2) {
    auto combine = [&](int j, i32x16_t (&out)[2]) __attribute__((always_inline)) {
      const int F = frag0 + 2 * wn + j;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        out[0][q] = ((acc[0][j][q] >> F) << 8) + (acc[1][j][q] >> F);
        out[1][q] = ((acc[2][j][q] >> F) << 8) + (acc[3][j][q] >> F);
      }
    };
    uint4_t *red = reinterpret_cast<uint4_t *>(smem);
    const int mine = wave * 8 * 64 + lane, theirs = (wave ^ (WN * WM)) * 8 * 64 + lane;
    i32x16_t give[2];
    if (wk) // uniform
      combine(0, give), combine(1, fin);
    else
      combine(1, give), combine(0, fin);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      uint4_t v;
      v.x = give[q >> 2][4 * (q & 3) + 0], v.y = give[q >> 2][4 * (q & 3) + 1];
      v.z = give[q >> 2][4 * (q & 3) + 2], v.w = give[q >> 2][4 * (q & 3) + 3];
      red[mine + q * 64] = v;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const uint4_t v = red[theirs + q * 64];
      fin[q >> 2][4 * (q & 3) + 0] += (int)v.x, fin[q >> 2][4 * (q & 3) + 1] += (int)v.y;
      fin[q >> 2][4 * (q & 3) + 2] += (int)v.z, fin[q >> 2][4 * (q & 3) + 3] += (int)v.w;
    }
  }

  // ---- 4. epilogue.  Accumulator register q of lane l: channel 8 (q / 4) + 4 (l / 32) + q % 4 of the fragment,
  // window l % 32.  dot = rowsum - 2 * sum(q * bit); the accumulators carry the factor 2^F of the fragment's byte
  // (-128 for F = 7).  With m_d = acc_d / 2^F:  sum(q * bit) = hi * 2^16 + lo, hi = m_0 * 256 + m_1,
  // lo = m_2 * 256 + m_3 (|m_d| <= 2^21 for the k the host admits), and with rowsum = s_hi * 2^16 + s_lo the result is
  // (s_hi -+ 2 hi) * 2^16 + (s_lo -+ 2 lo) = A * 2^16 + B with 0 <= B < 2^16: one fused multiply-add, rounded once
  // while |A| < 2^24 (sums below 2^40), else twice (2^-24 of the sum).
  if (finish) {
  const int osz = (int)g.out_sp_size;
#pragma unroll
  for (int jj = 0; jj < 3 - WK; ++jj) { // the fragments this wavefront finishes: both, or the one of its k group
  const int jf = WK == 2 ? wk : jj, fb = 2 * wn + jf;
  const int F = frag0 + fb; // the fragment's place in its wide group: the scale of its accumulators
  // (-x - 1 = x ^ -1: for F = 7 the two that 2 * 1 makes go into the windows' sum)
  const int flip = F == 7 ? -1 : 0;
  const int s_hi = (int)(rowsum >> 16) + 2 * flip, s_lo = (int)(rowsum & 0xffff) + 2 * flip;
  // channel of register q: c0 + 8 (q / 4) + q % 4; everything an output needs besides its accumulators is fetched
  // before the stores (the compiler does not move a load across them)
  const int c0 = fb * 32 + 4 * half, og_left = (int)g.Og - cg * kCols - c0; // channels from c0 to the group's last
  if (og_left <= 0)
    break;
  float al[16], bi[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    al[q] = s_alpha[c0 + 8 * (q >> 2) + (q & 3)];
    bi[q] = s_bias[c0 + 8 * (q >> 2) + (q & 3)];
  }
  float *ybase = a.y + (((int64_t)n * g.O + (int64_t)a.grp * g.Og + (int64_t)cg * kCols + c0) * g.out_sp_size + p0 + row);
  // The fragment's outputs as a buffer that ends with the group's last channel: what lies past it is not stored, and an
  // output's address is one 32-bit addition (32 channels are below 2^30 bytes: (Og + 256) * out_sp_size < 2^31).
  const int frag_left = min(32, (int)g.Og - cg * kCols - fb * 32);
  const uint64_t ystart = reinterpret_cast<uint64_t>(ybase - ((int64_t)4 * half * osz + row));
  const __amdgpu_buffer_rsrc_t yrsrc = __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void *>(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(ystart >> 32)) << 32) |
                               (uint32_t)__builtin_amdgcn_readfirstlane((int)ystart)),
      0, __builtin_amdgcn_readfirstlane((frag_left * osz - p0) * 4), 0x00020000);
  const int y_off = (4 * half * osz + row) * 4;
  float prev[16];
  if (a.accumulate) {
#pragma unroll
    for (int q = 0; q < 16; ++q)
      prev[q] = __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(yrsrc, y_off + (8 * (q >> 2) + (q & 3)) * osz * 4, 0, 0));
  }
  const float bad_scale = rowbad ? __uint_as_float(0x7fc00000u) : 65536.0f; // NaN through the multiply-add
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int cq = 8 * (q >> 2) + (q & 3);
    int hi, lo;
    if constexpr (WK == 2)
      hi = fin[0][q], lo = fin[1][q];
    else
      hi = ((acc[0][jj][q] >> F) << 8) + (acc[1][jj][q] >> F), lo = ((acc[2][jj][q] >> F) << 8) + (acc[3][jj][q] >> F);
    int A = s_hi - 2 * (hi ^ flip), B = s_lo - 2 * (lo ^ flip);
    A += B >> 16, B &= 0xffff; // the sum is A * 2^16 + B, 0 <= B < 2^16
    float v = ldexpf(fmaf((float)A, bad_scale, (float)B), -shift);
    if (a.accumulate)
      v = prev[q] + v;
    v = v * al[q];
    v = v + bi[q];
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), yrsrc, y_off + cq * osz * 4, 0, 0);
  }
  // A window holding a NaN or an infinity (rare): the reference's product propagates such values output by output
  // (convolution.cpp:185-193: the row of the unfolded input, zeros where the window leaves the input, times
  // Ws = Wb * alpha, then + b: Inf * w = +-Inf, Inf - Inf = NaN), so the lane recomputes its sixteen outputs as plain
  // fp32 dot products over the materialised signs and replaces the NaN stored above.
  if (rowbad && a.redo_w) {
    int w0, w1, w2;
    decode(row, w0, w1, w2);
    const float *xn = a.x + ((int64_t)n * g.C + (int64_t)a.grp * g.Cg) * plane;
#pragma unroll 1
    for (int q = 0; q < 16; ++q) {
      const int cq = 8 * (q >> 2) + (q & 3);
      if (cq >= og_left)
        continue;
      const float *wrow = a.redo_w + ((int64_t)cg * kCols + c0 + cq) * ((int64_t)Cg * taps);
      const float scale = s_alpha[c0 + cq];
      float acc = 0.0f;
#pragma unroll 1
      for (int c = 0; c < Cg; ++c) {
        int t = 0;
        for (int k0 = 0; k0 < g.k[0]; ++k0)
          for (int k1 = 0; k1 < g.k[1]; ++k1)
            for (int k2 = 0; k2 < g.k[2]; ++k2, ++t) {
              const int i0 = w0 + k0 * g.dil[0], i1 = w1 + k1 * g.dil[1], i2 = w2 + k2 * g.dil[2];
              const bool in = i0 >= 0 && i0 < in0 && i1 >= 0 && i1 < in1 && i2 >= 0 && i2 < in2;
              const float xv = in ? xn[(int64_t)c * plane + (i0 * in1 + i1) * in2 + i2] : 0.0f;
              acc = acc + xv * (wrow[c * taps + t] * scale);
            }
      }
      ybase[cq * osz] = acc + s_bias[c0 + cq];
    }
  }
  }
  }
  return left;
  };
  uint32_t left = round(std::false_type{});
  while (left != 0u) {
    // (opaque: nothing derived from these is kept in registers from one round to the next)
    asm volatile("" : "+v"(tid), "+v"(row));
    tid &= kThreads - 1, row &= kRows - 1, lane = tid & 63, half = lane >> 5; // (the compiler knows their ranges again)
    limit = left;
    __syncthreads(); // every wavefront has read its partner's sums
    shift = kSlabTopBit - binade_exponent(binade_of(left));
    for (int i = tid; i <= P.cap; i += kThreads)
      s_pixsum[i] = 0;
    for (int i = tid; i < (P.pix_stride >> 2); i += kThreads) // the zero pixel: the exchange lies over it
      *reinterpret_cast<uint32_t *>(smem + 4 * i) = 0u;
    left = round(std::true_type{});
  }
#endif
}

// Division of a small non-negative number (below 2^21) by a constant of the launch: the quotient of the number plus one
// half is at least 1 / (2 d) away from a whole number, more than the rounding of the two fp32 operations for
// d <= 2048 (kSlabMaxTaps * 32).
struct SmallDivide {
  float inv;
  __device__ __forceinline__ explicit SmallDivide(int d) : inv(1.0f / (float)d) {}
  __device__ __forceinline__ int operator()(int v) const { return (int)(((float)v + 0.5f) * inv); }
};

// One pass over the weights W [Og, Cg, taps] of a group: Wb = Sign(W) (sign.hpp:48-50), the packed bits of the product
// above in the order k' = tap * (32 ct) + channel, and per channel tile the sums of |W| and the counts of weights that
// are neither negative nor positive.  Block (wide group, channel tile ct, r): the eight output channels
// 256 wg + 32 F + r, F = 0..7 -- the ones whose bits share the packed words of lanes r and r + 32 -- and the 32 input
// channels of the tile: a contiguous run of 32 * taps floats per row.  A negative weight sets its bit of the packed
// words in LDS with an atomic OR (nothing waits for it; assembling a word from 32 bytes in LDS afterwards took as long
// as the rest of the kernel: 8.4 -> 6.0 us for 256 x 256 x 9 weights); |w| goes through LDS so that a row's sum is formed
// by one wavefront in a fixed order.
__global__ __launch_bounds__(kPrepThreads) void conv_taps_prepare(const float *__restrict__ W, float *__restrict__ Wb,
                                                                  uint4_t *__restrict__ bits, float *__restrict__ wsum,
                                                                  int *__restrict__ zeros, int Og, int Cg, int taps,
                                                                  int ct_count, int frags, int wide_groups,
                                                                  float zero_to) {
  // [8 rows][32 * taps] |w|, then the packed words of the block's k tiles: [tap][half][4]
  extern __shared__ __attribute__((aligned(16))) float s_abs[];
  const int seg_full = 32 * taps;
  uint32_t *s_words = reinterpret_cast<uint32_t *>(s_abs + 8 * seg_full);
  __shared__ int s_zero[kPrepThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wg = blockIdx.x / 32, r = blockIdx.x % 32, ct = blockIdx.y;
  const int c0 = ct * 32, cn = min(32, Cg - c0), seg = cn * taps, elems = 8 * seg;
  const int64_t Kg = (int64_t)Cg * taps;
  const SmallDivide by_seg(seg), by_taps(taps);
  for (int i = tid; i < 8 * taps; i += kPrepThreads)
    s_words[i] = 0u; // rows and channels past the end: bit clear (their digits are 0)
  __syncthreads();
  int nzero = 0;
  for (int base = 0; base < elems; base += 12 * kPrepThreads) {
    float w[12];
    int64_t at[12];
#pragma unroll
    for (int m = 0; m < 12; ++m) {
      const int idx = base + tid + kPrepThreads * m;
      const int f = by_seg(idx), kl = idx - f * seg;
      const int n = wg * kWideGroup + 32 * f + r;
      const bool in = idx < elems && n < Og;
      at[m] = in ? (int64_t)n * Kg + (int64_t)c0 * taps + kl : -1;
      w[m] = W[in ? at[m] : 0];
    }
#pragma unroll
    for (int m = 0; m < 12; ++m) {
      const int idx = base + tid + kPrepThreads * m;
      const int f = by_seg(idx), kl = idx - f * seg;
      if (idx < elems)
        s_abs[f * seg_full + kl] = at[m] >= 0 ? fabsf(w[m]) : 0.0f;
      if (at[m] >= 0) {
        const bool is_zero = !(w[m] > 0.0f) && !(w[m] < 0.0f);
        const bool neg = (w[m] < 0.0f) || (is_zero && zero_to < 0.0f);
        if (Wb)
          Wb[at[m]] = (w[m] > 0.0f) ? 1.0f : ((w[m] < 0.0f) ? -1.0f : zero_to);
        const int ch = by_taps(kl), t = kl - ch * taps;
        if (neg)
          atomicOr(&s_words[8 * t + (ch >> 2)], 1u << (f + 8 * (ch & 3)));
        nzero += is_zero ? 1 : 0;
      }
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    nzero += __shfl_xor(nzero, off);
  if (lane == 0)
    s_zero[wave] = nzero;
  __syncthreads();
  // the packed words of lanes r and r + 32 of the block's k tiles (tap, ct): word i, byte c, bit F <- row F, channel
  // c0 + 16 half + 4 i + c
  for (int item = tid; item < 2 * taps; item += kPrepThreads) {
    const int t = item >> 1, g16 = item & 1;
    bits[((int64_t)(t * ct_count + ct) * wide_groups + wg) * 64 + g16 * 32 + r] =
        reinterpret_cast<const uint4_t *>(s_words)[item];
  }
  if (tid == 0)
    zeros[(ct * wide_groups + wg) * 32 + r] = s_zero[0] + s_zero[1] + s_zero[2] + s_zero[3];
  for (int f = wave; f < 8; f += kPrepThreads / 64) {
    float asum = 0.0f;
    for (int kl = lane; kl < seg; kl += 64)
      asum += s_abs[f * seg_full + kl];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
      asum += __shfl_xor(asum, off);
    const int n = wg * kWideGroup + 32 * f + r;
    if (lane == 0 && n < frags * 32)
      wsum[(int64_t)ct * frags * 32 + n] = asum; // rows past Og: zero
  }
}

// The packed bits of the same product run backwards, for the gradient with respect to the input of a convolution of
// unit stride: dx = conv(dy, W') with W'[c][o][t] = Sign(W)[o][c][taps - 1 - t] and the padding (k - 1) dil - pad
// (convolution.cpp:199-283 unfolds dy . W^T and folds it back; here the fold is the contraction over the taps).
// Block (wide group of input channels c, tile of 32 output channels o, r) as in conv_taps_prepare; only the bits are
// written.
__global__ __launch_bounds__(kPrepThreads) void conv_taps_prepare_transposed(const float *__restrict__ W,
                                                                             uint4_t *__restrict__ bits, int Og, int Cg,
                                                                             int taps, int ct_count, int wide_groups,
                                                                             float zero_to) {
  extern __shared__ __attribute__((aligned(16))) uint32_t s_words[]; // [tap, flipped][half][4]
  const int seg_full = 32 * taps;
  const SmallDivide by_taps(taps);
  const int tid = threadIdx.x;
  const int wg = blockIdx.x / 32, r = blockIdx.x % 32, ct = blockIdx.y;
  const int o0 = ct * 32;
  for (int i = tid; i < 8 * taps; i += kPrepThreads)
    s_words[i] = 0u;
  __syncthreads();
  // one output channel o after the other: its rows c = 256 wg + 32 f + r are runs of `taps` floats 32 * taps apart
  for (int base = 0; base < 8 * seg_full; base += 8 * kPrepThreads) {
    float w[8];
    int at[8]; // word * 32 + bit; -1: outside
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int idx = base + tid + kPrepThreads * m;
      const int rest = by_taps(idx), t = idx - rest * taps, f = rest & 7, ol = rest >> 3;
      const int c = wg * kWideGroup + 32 * f + r, o = o0 + ol;
      const bool in = idx < 8 * seg_full && c < Cg && o < Og;
      at[m] = in ? (8 * (taps - 1 - t) + (ol >> 2)) * 32 + f + 8 * (ol & 3) : -1;
      w[m] = W[in ? ((int64_t)o * Cg + c) * taps + t : 0];
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const bool is_zero = !(w[m] > 0.0f) && !(w[m] < 0.0f);
      if (at[m] >= 0 && ((w[m] < 0.0f) || (is_zero && zero_to < 0.0f)))
        atomicOr(&s_words[at[m] >> 5], 1u << (at[m] & 31));
    }
  }
  __syncthreads();
  for (int item = tid; item < 2 * taps; item += kPrepThreads) {
    const int t = item >> 1, g16 = item & 1;
    bits[((int64_t)(t * ct_count + ct) * wide_groups + wg) * 64 + g16 * 32 + r] =
        reinterpret_cast<const uint4_t *>(s_words)[item];
  }
}

// The largest run of input positions a tile's windows span: a window's first position grows along an output row, so
// a tile's lowest origin is at its first position or at the start of a row inside it, its highest at its last
// position or at the end of a row inside it.
int64_t slab_longest_run(const ConvGeom &g, int tile_rows, int tiles_per_sample) {
  const int64_t plane = g.in_sp_size, last = slab_last_tap(g), ow = g.out_sp[2];
  int64_t longest = 1;
  for (int64_t t = 0; t < tiles_per_sample; ++t) {
    const int64_t p0 = t * tile_rows, p1 = (p0 + tile_rows < g.out_sp_size ? p0 + tile_rows : g.out_sp_size) - 1;
    int64_t omin = slab_origin(g, p0), omax = slab_origin(g, p1);
    if (omin > omax) {
      const int64_t s = omin;
      omin = omax, omax = s;
    }
    for (int64_t row = p0 / ow + 1; row * ow <= p1; ++row) {
      const int64_t first = slab_origin(g, row * ow), prev = slab_origin(g, row * ow - 1);
      omin = first < omin ? first : omin, omax = first > omax ? first : omax;
      omin = prev < omin ? prev : omin, omax = prev > omax ? prev : omax;
    }
    const int64_t lo = omin < 0 ? 0 : (omin > plane - 1 ? plane - 1 : omin);
    const int64_t hi_raw = omax + last, hi = hi_raw < 0 ? 0 : (hi_raw > plane - 1 ? plane - 1 : hi_raw);
    if (hi - lo + 1 > longest)
      longest = hi - lo + 1;
  }
  return longest;
}

bool compute_slab_plan(const ConvGeom &g, SlabPlan &p);

// The plan of a geometry is asked for several times per call (does it apply, how much workspace, the launches) and
// sizing the slab walks the tiles of a sample once per width of a tile (5 us at 56 x 56, 60 at 224 x 224): the last answers
// are kept per thread, as many as the layers of a large network have geometries, forward and backward.
bool make_slab_plan(const ConvGeom &g, SlabPlan &p) {
  struct Key {
    int64_t outer, C, O, group;
    int in_sp[kMaxSpatial], k[kMaxSpatial], pad[kMaxSpatial], stride[kMaxSpatial], dil[kMaxSpatial];
    bool operator==(const Key &o) const {
      bool same = outer == o.outer && C == o.C && O == o.O && group == o.group;
      for (int i = 0; i < kMaxSpatial; ++i)
        same = same && in_sp[i] == o.in_sp[i] && k[i] == o.k[i] && pad[i] == o.pad[i] && stride[i] == o.stride[i] &&
               dil[i] == o.dil[i];
      return same;
    }
  };
  constexpr int kKept = 64;
  static thread_local bool kept_ok[kKept];
  static thread_local Key kept_key[kKept];
  static thread_local SlabPlan kept_plan[kKept];
  static thread_local int count = 0, next = 0, last = 0;
  Key key;
  key.outer = g.outer, key.C = g.C, key.O = g.O, key.group = g.group;
  for (int i = 0; i < kMaxSpatial; ++i)
    key.in_sp[i] = g.in_sp[i], key.k[i] = g.k[i], key.pad[i] = g.pad[i], key.stride[i] = g.stride[i],
    key.dil[i] = g.dil[i];
  for (int i = 0; i < count; ++i) { // from the last answer on: a call asks for the same geometry again and again
    const int e = (last + i) % count;
    if (key == kept_key[e]) {
      last = e;
      p = kept_plan[e];
      return kept_ok[e];
    }
  }
  const int e = next;
  next = (next + 1) % kKept;
  kept_ok[e] = compute_slab_plan(g, kept_plan[e]);
  kept_key[e] = key;
  count = count < kKept ? count + 1 : kKept;
  last = e;
  p = kept_plan[e];
  return kept_ok[e];
}

// The forms of the product: WN x WM x WK wavefronts, each with a tile of 64 output channels x 32 windows.
struct SlabForm {
  int wn, wm, wk;
};
constexpr SlabForm kSlabForms[] = {{4, 1, 2}, {4, 2, 1}, {4, 1, 1}, {2, 2, 1}, {1, 4, 2}, {1, 4, 1}};
constexpr int kSlabFormCount = (int)(sizeof(kSlabForms) / sizeof(kSlabForms[0]));

// The longest run of input positions under a tile, by the tile's windows: the forms share a few widths.
struct SlabRuns {
  int tile_rows[3], found = 0;
  int64_t longest[3];
  int64_t operator()(const ConvGeom &g, int rows, int tiles_per_sample) {
    for (int i = 0; i < found; ++i)
      if (tile_rows[i] == rows)
        return longest[i];
    tile_rows[found] = rows;
    return longest[found++] = slab_longest_run(g, rows, tiles_per_sample);
  }
};

// The plan of one form that fills its slab `chunks` times; false when it does not fit the LDS.
bool compute_slab_form(const ConvGeom &g, int form, int chunks, SlabRuns &runs, SlabPlan &p) {
  const SlabForm &f = kSlabForms[form];
  const int waves = f.wn * f.wm * f.wk, rows = kSlabRows * f.wm;
  p.form = form;
  const int64_t cgp = ceil_div(g.Cg, 32) * 32;
  const int64_t ow = g.out_sp[2], map_rows = g.out_sp_size / ow;
  if (ow <= rows) { // whole rows of the output map, evenly
    const int64_t per = rows / ow, tiles = ceil_div(map_rows, per);
    p.tile_rows = (int)(ceil_div(map_rows, tiles) * ow);
  } else {
    p.tile_rows = (int)ceil_div(g.out_sp_size, ceil_div(g.out_sp_size, rows));
  }
  const int64_t tiles = ceil_div(g.out_sp_size, p.tile_rows);
  if (tiles > 16384) // the host walks them to size the slab
    return false;
  p.tiles_per_sample = (int)tiles;
  p.wide_groups = (int)bits_wide_groups(g.Og);
  p.col_groups = (int)ceil_div(g.Og, 64 * f.wn);
  if (g.outer * tiles * p.col_groups >= ((int64_t)1 << 31))
    return false;
  p.ct = (int)(cgp / 32);
  p.frags = (int)ceil_div(g.Og, 32);
  p.ct_chunk = (int)ceil_div(p.ct, chunks);
  p.chunks = (int)ceil_div(p.ct, p.ct_chunk);
  p.pix_stride = kSlabDigits * 32 * p.ct_chunk + kSlabPixPad;
  const int64_t cap = runs(g, p.tile_rows, p.tiles_per_sample);
  const int64_t slab_bytes = (cap + 1) * p.pix_stride;
  if (slab_bytes > kSlabLdsLimit)
    return false;
  p.cap = (int)cap;
  p.slab_bytes = (int)slab_bytes;
  p.k_tiles = (int)(g.k_size * p.ct);
  int64_t off = slab_bytes;
  if (f.wk == 2 && off < waves * kSlabReduceBytes) // the exchange between the k groups
    off = waves * kSlabReduceBytes;
  off = (int64_t)round_up((size_t)off, 16);
  p.pixsum_off = (int)off, off += 8 * (cap + 1);
  off = (int64_t)round_up((size_t)off, 16);
  p.pixmax_off = (int)off, off += 4 * (cap + 1);
  p.rowpix_off = (int)off, off += 4 * rows * (g.k_size + 1);
  p.alpha_off = (int)off, off += 2 * 4 * 64 * f.wn;
  p.misc_off = (int)off, off += 64;
  p.total = (int)off;
  p.bits_bytes = (size_t)p.k_tiles * p.wide_groups * kFragBytes;
  p.wsum_off = round_up(p.bits_bytes, 256);
  p.zeros_off = p.wsum_off + round_up((size_t)p.ct * p.frags * 32 * sizeof(float), 256);
  p.prep_bytes = p.zeros_off + round_up((size_t)p.ct * p.wide_groups * 32 * sizeof(int), 256);
  return off <= kSlabLdsLimit;
}

// Cycles of the launch, roughly: what the phases of a block measured (time stamps in blocks of 64, 256 and 512 input
// channels).  A block starts and waits for its first loads for about 7500 cycles, a work item of the set-up costs
// about 450 (half as much again when the slab is read twice, and 5000 in all for each further fill), an MFMA 46 of which 32 are its own, and the epilogue
// about 2800 per fragment of a wavefront.  Two blocks of four wavefronts share a CU where the LDS holds both slabs:
// each then takes 1.13 times as long, or what their MFMAs and vector instructions add up to, and a third more where all
// CUs do so (memory); tiles one column group wide take a quarter more than this, their loads being the most.
double slab_form_cost(const ConvGeom &g, const SlabPlan &p) {
  const SlabForm &f = kSlabForms[p.form];
  const int waves = f.wn * f.wm * f.wk;
  const double items = (double)ceil_div(p.cap, 64) * 2 * p.ct;
  const double load = items * (p.chunks > 1 || items > kSlabHold * waves ? 700.0 : 450.0) + 5000.0 * (p.chunks - 1);
  const double mma = 46.0 * p.k_tiles * 8 * f.wn * f.wm / 4;
  const double out = 1500.0 + 2800.0 * (f.wk == 2 ? 1 : 2) * (waves == 8 && f.wk == 1 ? 1.3 : 1.0);
  const double one = 7500.0 + load + mma + out;
  const double both = 2 * mma * 0.92 + load + out, pair = 1.3 * (one * 1.13 > both ? one * 1.13 : both);
  const int64_t blocks = g.outer * p.tiles_per_sample * p.col_groups;
  if (waves == 8 || p.total > 79 * 1024)
    return (double)ceil_div(blocks, 256) * one * (waves == 8 && f.wn == 1 ? 1.25 : 1.0);
  const int64_t rest = blocks % 512;
  return (double)(blocks / 512) * pair + (rest > 256 ? pair : rest > 0 ? one : 0.0);
}

bool compute_slab_plan(const ConvGeom &g, SlabPlan &p) {
  if (g.k_size > kSlabMaxTaps || g.Cg < 16 || g.in_sp_size >= ((int64_t)1 << 30) ||
      g.out_sp_size >= ((int64_t)1 << 30) || g.Og >= ((int64_t)1 << 24) ||
      (g.Og + kWideGroup) * g.out_sp_size >= ((int64_t)1 << 31))
    return false;
  const int64_t cgp = ceil_div(g.Cg, 32) * 32;
  if (g.k_size * cgp > kChunkK) // the epilogue's 32-bit steps hold kChunkK terms
    return false;
  // <4, 1, 2> with the slab filled once is for geometries of little padding (padded channels cost as much as real ones)
  SlabRuns runs;
  double best = 0.0;
  bool any = false;
  if (cgp * 3 <= g.Cg * 4 && compute_slab_form(g, 0, 1, runs, p)) {
    best = slab_form_cost(g, p);
    any = true;
  }
  for (int form = 1; form < kSlabFormCount; ++form) {
    SlabPlan q;
    if (!compute_slab_form(g, form, 1, runs, q))
      continue;
    const double cost = slab_form_cost(g, q);
    if (!any || cost < best)
      p = q, best = cost, any = true;
  }
  // The slab filled several times: against the forms that hold all channels at once, or where none does against the
  // product that gathers its operands window by window (912 cycles per k tile of 32 windows x 256 channels), if clearly
  // cheaper by these estimates: [4,512,28,28] x [512,512,3,3] 64 us there and 69 here, [16,512,28,28] x [256,512,3,3]
  // 111 and 76; [8,256,56,56] x [128,256,3,3] 107 filled once and 61 filled several times, [8,200,28,28] x [300,200,5,5]
  // 99 and 120.
  p.fits_once = any;
  best /= 1.3;
  if (!any) {
    const double tiles = (double)ceil_div(ceil_div(g.M, kSlabRows) * bits_wide_groups(g.Og), 256);
    best = tiles * (10000.0 + 912.0 * (double)ceil_div(g.Kg, kTileK)) / 1.3;
  }
  for (int form : {1, 2, 3, 5})
    for (int chunks = 2; chunks <= (int)(cgp / 32); ++chunks) {
      SlabPlan q;
      if (!compute_slab_form(g, form, chunks, runs, q))
        continue;
      const double cost = slab_form_cost(g, q);
      if (cost < best) {
        q.fits_once = p.fits_once;
        p = q, best = cost, any = true;
      }
      if (q.total <= 79 * 1024) // more fills only cost
        break;
    }
  return any;
}

template <int kForm, bool kChunked = false> int run_slab_form(const ConvSlabArgs &a, unsigned blocks, hipStream_t stream) {
  constexpr SlabForm f = kSlabForms[kForm];
  static std::atomic<uint64_t> configured{0};
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(binary_conv_slab_kernel<f.wn, f.wm, f.wk, kChunked>),
                                   kSlabLdsLimit, configured, "hipFuncSetAttribute(binary_conv_slab LDS size)");
  if (rc)
    return rc;
  hipLaunchKernelGGL((binary_conv_slab_kernel<f.wn, f.wm, f.wk, kChunked>), dim3(blocks), dim3(64 * f.wn * f.wm * f.wk),
                     (size_t)a.p.total, stream, a);
  NBLA_HIP_LAUNCH_CHECK("binary_conv_slab");
  return NBLA_HIP_OK;
}

} // namespace

bool conv_slab_applies(const ConvGeom &g) {
  SlabPlan p;
  return make_slab_plan(g, p);
}

// The forward's time in microseconds, the weights' pass included, from slab_form_cost (840 sizes of 16 to 23 channels and 8
// to 64 maps: 9 % off, 32 at the worst); 0 where the form does not cover the geometry.
double conv_slab_time(const ConvGeom &g) {
  SlabPlan p;
  return make_slab_plan(g, p) ? 6.8 + 3.95e-4 * slab_form_cost(g, p) : 0.0;
}

bool conv_slab_plan_summary(const ConvGeom &g, int32_t out[4]) {
  SlabPlan p;
  if (!make_slab_plan(g, p))
    return false;
  out[0] = p.tile_rows, out[1] = p.tiles_per_sample, out[2] = p.cap, out[3] = p.total;
  return true;
}

size_t conv_slab_prepared_bytes(const ConvGeom &g) {
  SlabPlan p;
  return make_slab_plan(g, p) ? p.prep_bytes : 0;
}

int launch_conv_slab_prepare(const float *Wg, float *Wbg, void *prepared, const ConvGeom &g, float zero_to,
                             hipStream_t stream) {
  SlabPlan p;
  if (!make_slab_plan(g, p))
    return fail(NBLA_HIP_ERR_NOT_IMPLEMENTED, "the slab convolution does not cover this geometry.");
  if (!aligned16(prepared))
    return fail(NBLA_HIP_ERR_MEMORY, "prepared-weight buffer must be 16-byte aligned.");
  const size_t lds = (size_t)(8 * 32 + 8) * g.k_size * 4; // |w| and the packed words
  static std::atomic<uint64_t> configured{0};
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(conv_taps_prepare), (8 * 32 + 8) * kSlabMaxTaps * 4,
                                   configured, "hipFuncSetAttribute(conv_taps_prepare LDS size)");
  if (rc)
    return rc;
  char *base = static_cast<char *>(prepared);
  hipLaunchKernelGGL(conv_taps_prepare, dim3((unsigned)p.wide_groups * 32, (unsigned)p.ct), dim3(kPrepThreads), lds,
                     stream, Wg, Wbg, reinterpret_cast<uint4_t *>(base), reinterpret_cast<float *>(base + p.wsum_off),
                     reinterpret_cast<int *>(base + p.zeros_off), (int)g.Og, (int)g.Cg, (int)g.k_size, p.ct, p.frags,
                     p.wide_groups, zero_to);
  NBLA_HIP_LAUNCH_CHECK("conv_taps_prepare");
  return NBLA_HIP_OK;
}

// The convolution that computes the input gradient of `g` (unit stride): dy takes the place of x, the roles of the
// channels are exchanged, the padding becomes (k - 1) dil - pad.  False when `g` has a stride or needs a negative
// padding, or when the slab product does not cover the result.
bool conv_slab_transposed_geom(const ConvGeom &g, ConvGeom &t) {
  t = g;
  for (int i = 0; i < kMaxSpatial; ++i) {
    if (g.stride[i] != 1)
      return false;
    t.pad[i] = (g.k[i] - 1) * g.dil[i] - g.pad[i];
    if (t.pad[i] < 0)
      return false;
    t.in_sp[i] = g.out_sp[i];
    t.out_sp[i] = g.in_sp[i];
  }
  t.C = g.O, t.O = g.C, t.Cg = g.Og, t.Og = g.Cg;
  t.in_sp_size = g.out_sp_size, t.out_sp_size = g.in_sp_size;
  t.Kg = t.Cg * g.k_size;
  t.M = g.outer * t.out_sp_size;
  SlabPlan p; // (a slab that has to be filled several times loses to the unfolded gradient)
  return make_slab_plan(t, p) && p.fits_once;
}

int launch_conv_slab_prepare_transposed(const float *Wg, void *prepared, const ConvGeom &g, float zero_to,
                                        hipStream_t stream) {
  ConvGeom t;
  SlabPlan p;
  if (!conv_slab_transposed_geom(g, t) || !make_slab_plan(t, p))
    return fail(NBLA_HIP_ERR_NOT_IMPLEMENTED, "the slab convolution does not cover this input gradient.");
  if (!aligned16(prepared))
    return fail(NBLA_HIP_ERR_MEMORY, "prepared-weight buffer must be 16-byte aligned.");
  const size_t lds = (size_t)8 * g.k_size * sizeof(uint32_t);
  hipLaunchKernelGGL(conv_taps_prepare_transposed, dim3((unsigned)p.wide_groups * 32, (unsigned)p.ct),
                     dim3(kPrepThreads), lds, stream, Wg, static_cast<uint4_t *>(prepared), (int)g.Og, (int)g.Cg,
                     (int)g.k_size, p.ct, p.wide_groups, zero_to);
  NBLA_HIP_LAUNCH_CHECK("conv_taps_prepare_transposed");
  return NBLA_HIP_OK;
}

int launch_conv_slab(const float *x, const ConvGeom &g, int64_t grp, const void *prepared, float *alpha_out,
                     int *zero_count, const float *bias, float *y, hipStream_t stream, const float *in_scale,
                     bool accumulate, const float *redo_w) {
  ConvSlabArgs a;
  if (!make_slab_plan(g, a.p))
    return fail(NBLA_HIP_ERR_NOT_IMPLEMENTED, "the slab convolution does not cover this geometry.");
  if (!aligned16(prepared))
    return fail(NBLA_HIP_ERR_MEMORY, "prepared-weight buffer must be 16-byte aligned.");
  int rc = ensure_init();
  if (rc)
    return rc;
  const char *base = static_cast<const char *>(prepared);
  a.x = x;
  a.bits = reinterpret_cast<const uint4_t *>(base);
  a.wsum = alpha_out ? reinterpret_cast<const float *>(base + a.p.wsum_off) : nullptr;
  a.zeros = reinterpret_cast<const int *>(base + a.p.zeros_off);
  a.alpha_out = alpha_out;
  a.zero_count = zero_count;
  a.bias = bias;
  a.in_scale = in_scale;
  a.redo_w = (in_scale || accumulate) ? nullptr : redo_w;
  a.accumulate = accumulate ? 1 : 0;
  a.y = y;
  a.g = g;
  a.grp = (int)grp;
  a.inv_k = (float)1 / g.Kg;
  const unsigned blocks = (unsigned)(g.outer * a.p.tiles_per_sample * a.p.col_groups);
  if (a.p.chunks > 1)
    return a.p.form == 1   ? run_slab_form<1, true>(a, blocks, stream)
           : a.p.form == 2 ? run_slab_form<2, true>(a, blocks, stream)
           : a.p.form == 3 ? run_slab_form<3, true>(a, blocks, stream)
                           : run_slab_form<5, true>(a, blocks, stream);
  switch (a.p.form) {
  case 0:
    return run_slab_form<0>(a, blocks, stream);
  case 1:
    return run_slab_form<1>(a, blocks, stream);
  case 2:
    return run_slab_form<2>(a, blocks, stream);
  case 3:
    return run_slab_form<3>(a, blocks, stream);
  case 4:
    return run_slab_form<4>(a, blocks, stream);
  default:
    return run_slab_form<5>(a, blocks, stream);
  }
}

} // namespace nbla_hip
