// Product of two real-valued matrices on the int8 matrix cores: y[m, n] = sum_k A[m, k] * B[n, k] with both
// operands as digit operands (per row a power-of-two scale and three balanced base-256 int8 digits, see
// gemm_layout.hpp).  With qa = a0 * 2^16 + a1 * 2^8 + a2 and qb likewise,
//     qa * qb = a0 b0 * 2^32 + (a0 b1 + a1 b0) * 2^24 + (a0 b2 + a1 b1 + a2 b0) * 2^16 + (lower terms)
// and the six leading digit products are accumulated exactly in three int32 accumulators per output (one per power
// of 256); the dropped terms are below 2^-23 of |row max| * |column max| per k.  The epilogue combines the three
// sums in integer arithmetic, converts once and applies the two scales, so the result does not depend on the order
// of summation.  Used for the weight gradients (x^T . dy), where neither factor is a sign matrix.
//
// Tiling: 128 x 128 outputs per block of four wavefronts (2 x 2, 64 x 64 each: 4 x 4 tiles of
// v_mfma_i32_16x16x64_i8 x 3 accumulators = 192 registers), k in steps of 64 (two k tiles of the operands).  Why the
// 16 x 16 instruction: on large products the part runs at its power limit, and a loop of nothing but these
// instructions sustains 3.9 POP/s on random digits where the 32 x 32 x 32 form, which moves twice the accumulator bytes
// per operation, sustains 3.2 to 3.4.  The weight gradient of 4096 x 4096 x 11008: 870 us with the 32 x 32 x 32 form in
// the same tiles (2.55 POP/s), 760 with this one; 1024 x 4096 x 4096 against one-digit rows: 28.0 and 24.1.
#include "common.hpp"
#include "copy_pipeline.hpp"
#include "gemm_layout.hpp"
#include "internal.hpp"

#include <type_traits>

namespace nbla_hip {
namespace {

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_u __attribute__((ext_vector_type(2), aligned(4))); // a 64-bit access at any multiple of four bytes
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));

struct GemmDigitsArgs {
  const uint4_t *ad, *bd; // [row blocks][k tiles][3][64] uint4 each
  const int32_t *ashift, *bshift, *bshift_narrow, *bflag;
  const float *bias;
  float *y;
  int64_t M, N, a_row_blocks, b_row_blocks, k_tiles, step_begin, step_end, blocks_m, blocks_n;
  int64_t inner, outer_stride, n_stride;
  int accumulate; // add to y instead of overwriting it
  int finish;     // last chunk of the contraction: add the bias
  // contraction split over blockIdx.y (outputs of few tiles): split z multiplies the k tiles
  // [step_begin + z * split_tiles, + split_tiles) and writes its own dense [M, N] partial result at y + z * M * N
  int64_t split_tiles; // 0: no split
};

constexpr int kBM = 128, kBN = 128, kThreads = 256, kWaves = 4;
constexpr int kSegs = 4;              // 32-row fragments per tile side
constexpr int kSegVec = kDigits * 64; // uint4 per fragment and k tile
// A k step is multiplied in phases, each of which needs two parts: one digit of one side (four row blocks x two k
// tiles, 8 KiB).  A phase's two parts lie in one LDS buffer; kStages buffers, so the copies of a phase are issued
// three phases before it (the phases of two k tiles of all digits: 4096 cycles of the matrix pipe with two blocks per
// CU).  64 KiB of LDS per block, two blocks per CU (or two k groups in one).
constexpr int kStages = 4;
constexpr int kPartBytes = kSegs * 2 * kFragBytes, kStageBytes = 2 * kPartBytes;
constexpr int kCopies = kStageBytes / kFragBytes / kWaves; // 1 KiB copies per wavefront and phase, which the loop's wait counts
static_assert(kCopies * kWaves * kFragBytes == kStageBytes, "a phase's copies fill its buffer");
// MFMA tiles along either side of a wavefront's 64 x 64.  Every phase of every form deals its copies out behind the MFMAs
// of one fragment, one copy behind each: as many as the wait counts.
constexpr int kFrags = 4;
static_assert(kFrags == kCopies, "a phase issues the copies that the wait counts");

// Phases per k step: all nine digit pairs' leading six: {a0 b0} {a0 b2, a0 b1} {a1 b0, a1 b1, a2 b0}; one-digit B:
// {a0 b} {a1 b, a2 b}; both one-digit: {a b}.
constexpr int phases_per_step(bool one_a, bool narrow) { return one_a ? 1 : (narrow ? 2 : 3); }

// Workgroup barrier without the memory fence of __syncthreads() (which would wait for every global -> LDS copy in
// flight, including those of later k tiles); the waits that matter are explicit.
#define NBLA_BARRIER()                                                                                                 \
  do {                                                                                                                 \
    asm volatile("" ::: "memory");                                                                                     \
    __builtin_amdgcn_s_barrier();                                                                                      \
    asm volatile("" ::: "memory");                                                                                     \
  } while (0)
// vmcnt(n) with the other counters left alone (gfx9 encoding: vmcnt in bits 3:0 and 15:14).
#define NBLA_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xf) | (((n) >> 4) << 14) | (0x7 << 4) | (0xf << 8))

// Staging: global -> LDS copies bypass the registers (one wavefront instruction moves one 1 KiB fragment of the
// operand).  Two blocks share a CU (256 registers per lane: 192 accumulators, at most 13 operand quads), so one
// block's LDS reads and barrier waits are covered by the other's MFMAs.
//
// A 16 x 64 fragment is put together from the operands' 32 x 32 ones by the LDS address alone: lane l reads row
// l % 16 of half h of a row block, k slots (l / 16) % 2 of k tile l / 32 of the step -- the same 64 k for A and B,
// in an order of their own.  The copy of B sends row 2 r + h of a row block to where half h's row r is read, so a
// lane's accumulators of the two halves are neighbouring columns and are stored as one 64-bit word.
//
// kNarrow: the B operand holds every value in its lowest digit alone (a small integer): three products
// a_t x b2 -> accumulator t, nothing dropped, and only the lowest-digit fragments of B are copied.
// kTopB (a form of kNarrow): every row of the tile's B row blocks is a one-digit row of a row-scaled operand (its value
// sits in the top digit: power-of-two weights once INQ has fixed them): the same three products with b0 in place of
// b2, and the factor 2^16 of the top digit in the epilogue.
// kOneA (only with kNarrow): every row of the tile's A row blocks is a one-digit row (gemm_layout.hpp: its value sits
// in the top digit): a single product a0 x b2 -> accumulator 0, and only the top-digit fragments of A and the
// lowest-digit fragments of B are copied.  Same bits as the other forms: the other digits are zero.
// kGroups = 2 (outputs of at most one tile per CU): eight wavefronts, two groups of four; group g multiplies the k
// steps g, g + 2, ... of the same output tile from stages of its own, so every SIMD has a second wavefront to issue
// from while the first waits.  At the end the groups swap halves of their int32 accumulators through LDS (exactly)
// and group g finishes row block g of each wavefront tile.
template <bool kNarrow, bool kOneA, int kGroups, bool kTopB = false>
__device__ __forceinline__ void gemm_digits_tile(const GemmDigitsArgs &a, unsigned char *smem) {
#if defined(__HIP_DEVICE_COMPILE__) // the host pass only needs the launch stub; the body uses LDS address-space pointers
  static_assert(kGroups == 1 || kGroups == 2, "k groups per block");
  static_assert(!kOneA || kNarrow, "the one-digit A form is implemented for one-digit B operands");
  static_assert(!kTopB || kNarrow, "the top-digit B form is a narrow form");
  constexpr int kBDigit = !kNarrow || kTopB ? 0 : kDigits - 1; // the digit of B that the first phase multiplies
  constexpr int kPhases = phases_per_step(kOneA, kNarrow);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave_all / kWaves, wave = wave_all % kWaves;
  const int wm = wave & 1, wn = wave >> 1;
  int64_t bm, bn;
  band_tile<8>(blockIdx.x, a.blocks_m, a.blocks_n, bm, bn); // two blocks per CU: 64 resident tiles per XCD = 8 x 8

  // This wavefront's copies: of each part the fragments of k tile wave % 2 of the row blocks wave / 2 and wave / 2 + 2.
  // A row block is a buffer resource that starts at the fragment's top digit in the first step of this block's share
  // and ends with the last one: the copies run past the last step, where the range check (it covers the scalar offset
  // too) turns them into zeros in LDS.  Row blocks past the end of the operand are clamped: those rows / columns are
  // not stored.
  constexpr int kStepAdvance = kGroups * 2 * kSegVec * 16; // bytes of a row block between a group's k steps
  __amdgpu_buffer_rsrc_t rsrc[2][2];
#pragma unroll
  for (int side = 0; side < 2; ++side)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      int64_t rb = (side ? bn : bm) * kSegs + (wave >> 1) + 2 * q;
      const int64_t limit = side ? a.b_row_blocks : a.a_row_blocks;
      rb = rb < limit ? rb : limit - 1;
      const int64_t tile = a.step_begin + group * 2 + (wave & 1);
      const uint4_t *src = (side ? a.bd : a.ad) + (rb * a.k_tiles + tile) * kSegVec;
      const int64_t span = (a.step_end - tile) * kSegVec * 16;
      const uint64_t first = reinterpret_cast<uint64_t>(src);
      const uint64_t base = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(first >> 32)) << 32) |
                            (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
      rsrc[side][q] =
          __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(base), 0,
                                            __builtin_amdgcn_readfirstlane(span > 0 ? (int)span : 0), 0x00020000);
    }
  typedef __attribute__((address_space(3))) void lds_void_t;
  unsigned char *ring = smem + group * kStages * kStageBytes;
  const int a_lane = lane * 16;                                                            // rows as they are
  const int b_lane = ((lane >> 5) * 32 + 2 * (lane & 15) + ((lane >> 4) & 1)) * 16;        // columns dealt out in pairs
  // copy c (0..3) of the two parts of phase `ph` of the step at step_off into the buffer at byte offset `dest`
  auto copy_one = [&](auto ph, int c, int step_off, int dest) __attribute__((always_inline)) {
    constexpr int kPh = decltype(ph)::value;
    const int part = c >> 1, q = c & 1;
    const int side = kPh == 0 ? part : (kNarrow || kPh == 2 ? 0 : 1);
    const int digit = kPh == 0 ? (part ? kBDigit : 0) : (side ? 2 - part : 1 + part);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rsrc[side][q],
        (lds_void_t *)(ring + dest + part * kPartBytes + (((wave >> 1) + 2 * q) * 2 + (wave & 1)) * kFragBytes), 16,
        side ? b_lane : a_lane, step_off + digit * kFragBytes, 0, 0);
  };

  i32x4_t acc[4][4][3];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < 3; ++t)
        acc[i][j][t] = i32x4_t{0, 0, 0, 0};

  // The number of most recently issued phases the wait at the top of a phase may leave in flight, from the model of
  // this loop's order of copies, waits, barriers and LDS reads (copy_pipeline.hpp)
  constexpr int kLoopWait = pipeline::one_tile_loop_wait(kStages, kStages - 1);
  static_assert(kLoopWait >= 0 && pipeline::one_tile_safe(kStages, kStages - 1, kLoopWait),
                "the copy pipeline hands a buffer over too early");
  static_assert(pipeline::counter_fits(kLoopWait, kCopies), "vmcnt is a 6-bit counter");

  // fragment f (0..3) of this wavefront's rows (part of side A) or columns (side B) in the part at `part`
  const int a_frag = (wm * 2 * 2 + (lane >> 5)) * kFragBytes + (((lane >> 4) & 1) * 32 + (lane & 15)) * 16;
  const int b_frag = a_frag + (wn - wm) * 4 * kFragBytes;
  auto frag = [&](int lane_off, int part, int f) __attribute__((always_inline)) {
    return __builtin_bit_cast(
        i32x4_t, *reinterpret_cast<const uint4_t *>(ring + part + lane_off + (f >> 1) * 2 * kFragBytes + (f & 1) * 256));
  };
  int buf = 0; // byte offset of the phase's buffer
  auto hand_over = [&]() __attribute__((always_inline)) {
    // this phase's parts have landed (the copies of the two phases after it may still be in flight) and every
    // wavefront is done with the buffer of the phase before it, which the copies issued next take over
    NBLA_WAIT_VMCNT(kLoopWait * kCopies);
    NBLA_BARRIER();
  };
  // Issue order, pinned (sched_barrier): the first two fragments of a phase, then its copies and its other reads dealt
  // out between the MFMAs, each fragment read two fragments' MFMAs before it is used -- a wavefront cannot feed the
  // matrix pipe while it issues a batch of other instructions or waits for LDS.
  auto pin = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
  int ahead = 0; // byte offset of the step that the next copies belong to
  // copy c of the phase three after phase kPh of the current step
  auto copy_ahead = [&](auto ph, int c) __attribute__((always_inline)) {
    constexpr int kPh = decltype(ph)::value, kTarget = kPh + kStages - 1;
    copy_one(std::integral_constant<int, kTarget % kPhases>(), c, ahead + (kTarget / kPhases) * kStepAdvance,
             (buf + (kStages - 1) * kStageBytes) & (kStages * kStageBytes - 1));
  };
  auto advance = [&]() __attribute__((always_inline)) { buf = (buf + kStageBytes) & (kStages * kStageBytes - 1); };
  typedef std::integral_constant<int, 0> P0;
  typedef std::integral_constant<int, 1> P1;
  typedef std::integral_constant<int, 2> P2;
#pragma unroll
  for (int c = 0; c < kCopies; ++c)
    copy_one(P0(), c, 0, 0);
#pragma unroll
  for (int c = 0; c < kCopies; ++c)
    copy_one(std::integral_constant<int, 1 % kPhases>(), c, (1 / kPhases) * kStepAdvance, kStageBytes);
#pragma unroll
  for (int c = 0; c < kCopies; ++c)
    copy_one(std::integral_constant<int, 2 % kPhases>(), c, (2 / kPhases) * kStepAdvance, 2 * kStageBytes);
  auto mma = [&](i32x4_t &c, const i32x4_t &x, const i32x4_t &w) __attribute__((always_inline)) {
    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, w, c, 0, 0, 0);
  };
  const int steps = (int)((a.step_end - a.step_begin) / (2 * kGroups)); // k tiles come in multiples of four
  for (int left = steps; left > 0; --left) {
    i32x4_t a0[4], b0[4];
    hand_over();
    a0[0] = frag(a_frag, buf, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      b0[j] = frag(b_frag, buf + kPartBytes, j);
    a0[1] = frag(a_frag, buf, 1);
    pin();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < kFrags; ++j) {
        mma(acc[i][j][0], a0[i], b0[j]);
        if (i == 0 && (j & 1)) {
          a0[2 + (j >> 1)] = frag(a_frag, buf, 2 + (j >> 1));
          pin();
        }
        if (i == 1) {
          copy_ahead(P0(), j);
          pin();
        }
      }
    pin();
    advance();
    if (kNarrow && !kOneA) {
      hand_over();
      i32x4_t af[8];
      af[0] = frag(a_frag, buf, 0);
      af[1] = frag(a_frag, buf, 1);
      pin();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < kFrags; ++j) {
          mma(acc[i & 3][j][1 + (i >> 2)], af[i], b0[j]);
          if (j == 0 && i + 2 < 8) {
            af[i + 2] = frag(a_frag, buf + ((i + 2) >> 2) * kPartBytes, (i + 2) & 3);
            pin();
          }
          if (i == 0) {
            copy_ahead(P1(), j);
            pin();
          }
        }
        pin();
      }
      advance();
    }
    if (!kNarrow) {
      i32x4_t b1[4];
      {
        hand_over();
        i32x4_t bf[8]; // the third digit's, then the second's
        bf[0] = frag(b_frag, buf, 0);
        bf[1] = frag(b_frag, buf, 1);
        pin();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
#pragma unroll
          for (int i = 0; i < kFrags; ++i) {
            mma(acc[i][j & 3][j < 4 ? 2 : 1], a0[i], bf[j]);
            if (i == 0 && j + 2 < 8) {
              bf[j + 2] = frag(b_frag, buf + ((j + 2) >> 2) * kPartBytes, (j + 2) & 3);
              pin();
            }
            if (j == 0) {
              copy_ahead(P1(), i);
              pin();
            }
          }
          pin();
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          b1[j] = bf[4 + j];
        advance();
      }
      {
        hand_over();
        i32x4_t af[8]; // the second digit's, then the third's
        af[0] = frag(a_frag, buf, 0);
        af[1] = frag(a_frag, buf, 1);
        pin();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
#pragma unroll
          for (int j = 0; j < kFrags; ++j) {
            mma(acc[i & 3][j][i < 4 ? 1 : 2], af[i], b0[j]);
            if (j == 0 && i + 2 < 8) {
              af[i + 2] = frag(a_frag, buf + ((i + 2) >> 2) * kPartBytes, (i + 2) & 3);
              pin();
            }
            if (i == 0) {
              copy_ahead(P2(), j);
              pin();
            }
          }
          if (i < 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              mma(acc[i & 3][j][2], af[i], b1[j]);
          }
          pin();
        }
        advance();
      }
    }
    ahead += kStepAdvance;
  }
  NBLA_WAIT_VMCNT(0);

  if (kGroups == 2) {
    // swap: every wavefront hands the row block it does not finish to its partner in the other group, one accumulator
    // set at a time (8 wavefronts x 2 x 4 tiles x 64 lanes x 16 B = 64 KiB per round)
    i32x4_t *xs = reinterpret_cast<i32x4_t *>(smem);
    const int partner = wave_all ^ kWaves;
#pragma unroll
    for (int t = 0; t < (kOneA ? 1 : 3); ++t) {
      __syncthreads(); // the stages (first round) or the previous round's values have been read
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if ((i >> 1) != group) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            xs[((wave_all * 2 + (i & 1)) * 4 + j) * 64 + lane] = acc[i][j][t];
        }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if ((i >> 1) == group) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j][t] += xs[((partner * 2 + (i & 1)) * 4 + j) * 64 + lane];
        }
    }
  }

  // y = (acc0 * 2^16 + acc1 * 2^8 + acc2) * 2^(16 - sa - sb); the narrow form has no factor 2^16 (b is its low digit)
  // unless b is the top digit of a row-scaled operand.
  // Register r of lane l: row 4 (l / 16) + r of fragment i; columns 2 (l % 16) and the next of row block j / 2 (see the
  // copy of B).  Row by row: the row's offset (one 32-bit division when m is folded into two output indices) and shift
  // are formed once and serve all columns.
  const int32_t *bshift = (kNarrow && !kTopB) ? a.bshift_narrow : a.bshift;
  int64_t n_col[2]; // the even one of a pair
  int32_t sb_n[2][2];
  float bias_n[2][2];
#pragma unroll
  for (int jp = 0; jp < 2; ++jp) {
    n_col[jp] = bn * kBN + (wn * 2 + jp) * 32 + 2 * (lane & 15);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool in = n_col[jp] + h < a.N;
      sb_n[jp][h] = in ? plain_shift(bshift[n_col[jp] + h]) : 0; // one-digit rows store their shift with a bias
      bias_n[jp][h] = (in && a.bias && a.finish) ? a.bias[n_col[jp] + h] : 0.0f;
    }
  }
  const bool add_bias = a.bias && a.finish;
  const uint32_t inner = (uint32_t)a.inner;
  // the wavefront's 64 row shifts: one coalesced load up front (lane l holds row l), handed out by shuffles, instead of
  // a dependent global load per row inside the store loop
  int32_t row_shift;
  {
    const int64_t m = bm * kBM + wm * 64 + lane, last = a.a_row_blocks * kFragRows - 1;
    row_shift = plain_shift(a.ashift[m < last ? m : last]);
  }
  // Copies of the stores with and without reading y back first: with that load anywhere in the loop the compiler waits
  // for all outstanding memory operations before every output, and the stores before it are outstanding memory
  // operations -- each store would wait for the previous one.  Likewise with and without column bounds, for pairs of
  // columns that are neighbours in memory (`pairs`).
  auto store_rows = [&](auto accumulate_c, auto pairs_c) __attribute__((always_inline)) {
    constexpr bool kAcc = decltype(accumulate_c)::value, kPairs = decltype(pairs_c)::value;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (kGroups == 2 && (i >> 1) != group)
        continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = i * 16 + 4 * (lane >> 4) + r;
        const int32_t sa_m = __shfl(row_shift, row);
        const int64_t m = bm * kBM + wm * 64 + row;
        if (m >= a.M)
          continue;
        int64_t off;
        if (inner == 1u) {
          off = m * a.outer_stride;
        } else {
          const uint32_t mu = (uint32_t)m, q = mu / inner; // m < 2^31: operand rows are counted in 32 bits
          off = (int64_t)q * a.outer_stride + (mu - q * inner);
        }
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {
          f32x2_t v;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (sa_m == kBadRow || sb_n[jp][h] == kBadRow) {
              v[h] = __uint_as_float(0x7fc00000u);
            } else {
              // t = acc0 * 2^16 + acc1 * 2^8 + acc2 regrouped as hi * 2^16 + lo with 0 <= lo < 2^17 and |hi| < 2^30
              // (32-bit integer steps only), then one fused multiply-add: exact while |hi| < 2^24, else rounded twice
              // (2^-24 of t)
              const int a0 = acc[i][2 * jp + h][0][r], a1 = acc[i][2 * jp + h][1][r], a2 = acc[i][2 * jp + h][2][r];
              const int hi = a0 + (a1 >> 8) + (a2 >> 16);
              const int lo = ((a1 & 0xff) << 8) + (a2 & 0xffff);
              const float t = fmaf((float)hi, 65536.0f, (float)lo);
              // the two shifts are applied one after the other: each stays inside ldexpf's exponent range
              v[h] = ldexpf(ldexpf(t, ((kNarrow && !kTopB) ? 0 : 16) - sa_m), -sb_n[jp][h]);
            }
          }
          if (kPairs) {
            f32x2_u *dst = reinterpret_cast<f32x2_u *>(a.y + off + n_col[jp]);
            if (kAcc)
              v = *dst + v;
            if (add_bias)
              v[0] += bias_n[jp][0], v[1] += bias_n[jp][1];
            *dst = v;
          } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              if (n_col[jp] + h >= a.N)
                continue;
              float *dst = a.y + off + (n_col[jp] + h) * a.n_stride;
              float w = v[h];
              if (kAcc)
                w = *dst + w;
              if (add_bias)
                w = w + bias_n[jp][h];
              *dst = w;
            }
          }
        }
      }
    }
  };
  const bool pairs = a.n_stride == 1 && (bn + 1) * kBN <= a.N;
  if (a.accumulate) {
    if (pairs)
      store_rows(std::true_type(), std::true_type());
    else
      store_rows(std::true_type(), std::false_type());
  } else {
    if (pairs)
      store_rows(std::false_type(), std::true_type());
    else
      store_rows(std::false_type(), std::false_type());
  }
#endif
}

template <int kGroups>
__global__ __launch_bounds__(kThreads * kGroups, kGroups == 1 ? 2 : 1) void gemm_digits_kernel(GemmDigitsArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  if (a.split_tiles > 0) {
    const int64_t begin = a.step_begin + (int64_t)blockIdx.y * a.split_tiles;
    a.step_end = begin + a.split_tiles < a.step_end ? begin + a.split_tiles : a.step_end;
    a.step_begin = begin;
    a.y += (int64_t)blockIdx.y * a.M * a.N;
  }
  if (*a.bflag == 0) { // uniform over the grid
    // are all rows of this tile's A row blocks one-digit rows?  (rows past the operand clamp to its last row)
    int64_t bm, bn;
    band_tile<8>(blockIdx.x, a.blocks_m, a.blocks_n, bm, bn);
    const int64_t rows = a.a_row_blocks * kFragRows;
    bool one = true;
    for (int r = threadIdx.x; r < kBM; r += kThreads * kGroups) {
      const int64_t m = bm * kBM + r;
      one = one && one_digit_row(a.ashift[m < rows ? m : rows - 1]);
    }
    if (__syncthreads_and(one))
      gemm_digits_tile<true, true, kGroups>(a, smem);
    else
      gemm_digits_tile<true, false, kGroups>(a, smem);
  } else {
    // all rows of this tile's B row blocks one-digit rows (of a row-scaled operand; column-scaled ones never are)?
    int64_t bm, bn;
    band_tile<8>(blockIdx.x, a.blocks_m, a.blocks_n, bm, bn);
    const int64_t arows = a.a_row_blocks * kFragRows, brows = a.b_row_blocks * kFragRows;
    bool one_b = true, one_a = true;
    for (int r = threadIdx.x; r < kBN; r += kThreads * kGroups) {
      const int64_t n = bn * kBN + r;
      one_b = one_b && one_digit_row(a.bshift[n < brows ? n : brows - 1]);
    }
    for (int r = threadIdx.x; r < kBM; r += kThreads * kGroups) {
      const int64_t m = bm * kBM + r;
      one_a = one_a && one_digit_row(a.ashift[m < arows ? m : arows - 1]);
    }
    one_b = __syncthreads_and(one_b);
    one_a = __syncthreads_and(one_a);
    if (one_b && one_a)
      gemm_digits_tile<true, true, kGroups, true>(a, smem);
    else if (one_b)
      gemm_digits_tile<true, false, kGroups, true>(a, smem);
    else
      gemm_digits_tile<false, false, kGroups>(a, smem);
  }
}

// y (+)= sum over the splits of their partial results, in split order, then the bias: what the single-launch epilogue
// does with one value.
__global__ __launch_bounds__(256) void gemm_digits_split_sum(const float *__restrict__ partial, int splits, int64_t M,
                                                             int64_t N, float *__restrict__ y, int64_t inner,
                                                             int64_t outer_stride, int64_t n_stride,
                                                             const float *__restrict__ bias, int accumulate) {
  const int64_t total = M * N;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t m = i / N, n = i - m * N;
    float v = partial[i];
    for (int z = 1; z < splits; ++z)
      v += partial[(int64_t)z * total + i];
    const int64_t q = m / inner;
    float *dst = y + q * outer_stride + (m - q * inner) + n * n_stride;
    if (accumulate)
      v = *dst + v;
    if (bias)
      v = v + bias[n];
    *dst = v;
  }
}

// The same for outputs whose consecutive elements in memory are consecutive rows m (n_stride != 1: convolution
// results [sample, channel, position]): a 32 x 32 tile is read along n and, through LDS, written along m.
__global__ __launch_bounds__(256) void gemm_digits_split_sum_rows(const float *__restrict__ partial, int splits,
                                                                  int64_t M, int64_t N, float *__restrict__ y,
                                                                  int64_t inner, int64_t outer_stride, int64_t n_stride,
                                                                  const float *__restrict__ bias, int accumulate) {
  __shared__ float tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5; // ty: 0..7
  const int64_t n0 = (int64_t)blockIdx.x * 32, m0 = (int64_t)blockIdx.y * 32, total = M * N;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = m0 + ty + 8 * i, n = n0 + tx;
    float v = 0.0f;
    if (m < M && n < N) {
      v = partial[m * N + n];
      for (int z = 1; z < splits; ++z)
        v += partial[(int64_t)z * total + m * N + n];
    }
    tile[ty + 8 * i][tx] = v;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = m0 + tx, n = n0 + ty + 8 * i;
    if (m < M && n < N) {
      float v = tile[tx][ty + 8 * i];
      const int64_t q = m / inner;
      float *dst = y + q * outer_stride + (m - q * inner) + n * n_stride;
      if (accumulate)
        v = *dst + v;
      if (bias)
        v = v + bias[n];
      *dst = v;
    }
  }
}

} // namespace

size_t gemm_digits_split_bytes(int64_t M, int64_t K, int64_t N) {
  const int64_t k_tiles = digit_k_tiles(K) < kChunkK / kTileK ? digit_k_tiles(K) : kChunkK / kTileK;
  const int64_t s = digit_product_splits(ceil_div(M, kBM) * ceil_div(N, kBN), k_tiles);
  return s > 1 ? (size_t)s * M * N * sizeof(float) : 0;
}

int launch_gemm_digits(const void *adigits, const void *bdigits, const float *bias, float *y, int64_t M, int64_t K,
                       int64_t N, int64_t inner, int64_t outer_stride, int64_t n_stride, hipStream_t stream,
                       bool accumulate, void *split_ws, size_t split_ws_bytes) {
  if (M >= ((int64_t)1 << 31) || N >= ((int64_t)1 << 31))
    return fail(NBLA_HIP_ERR_NOT_IMPLEMENTED, "digit product: more than 2^31 - 1 rows or columns.");
  const DigitOperand da = digit_operand(M, K), db = digit_operand(N, K);
  static std::atomic<uint64_t> configured[2];
  int rc = allow_dynamic_lds(reinterpret_cast<const void *>(gemm_digits_kernel<1>), kStages * kStageBytes,
                             configured[0], "hipFuncSetAttribute(gemm_digits LDS size)");
  if (!rc)
    rc = allow_dynamic_lds(reinterpret_cast<const void *>(gemm_digits_kernel<2>), 2 * kStages * kStageBytes,
                           configured[1], "hipFuncSetAttribute(gemm_digits LDS size)");
  if (rc)
    return rc;
  GemmDigitsArgs a;
  a.ad = static_cast<const uint4_t *>(adigits);
  a.bd = static_cast<const uint4_t *>(bdigits);
  a.ashift = reinterpret_cast<const int32_t *>(static_cast<const char *>(adigits) + da.shift_off);
  a.bshift = reinterpret_cast<const int32_t *>(static_cast<const char *>(bdigits) + db.shift_off);
  a.bshift_narrow = reinterpret_cast<const int32_t *>(static_cast<const char *>(bdigits) + db.sum_off);
  a.bflag = reinterpret_cast<const int32_t *>(static_cast<const char *>(bdigits) + db.flag_off);
  a.bias = bias;
  a.y = y;
  a.M = M;
  a.N = N;
  a.a_row_blocks = da.row_blocks;
  a.b_row_blocks = db.row_blocks;
  a.k_tiles = da.k_tiles;
  a.blocks_m = ceil_div(M, kBM);
  a.blocks_n = ceil_div(N, kBN);
  a.inner = inner;
  a.outer_stride = outer_stride;
  a.n_stride = n_stride;
  // chunks of kChunkK contraction elements keep the int32 sums below 2^31; their fp32 results are added up
  const int64_t tiles_per_chunk = kChunkK / kTileK;
  for (int64_t t0 = 0, chunk = 0; t0 < a.k_tiles; t0 += tiles_per_chunk, ++chunk) {
    a.step_begin = t0;
    a.step_end = (t0 + tiles_per_chunk < a.k_tiles) ? t0 + tiles_per_chunk : a.k_tiles;
    a.accumulate = (accumulate || chunk > 0) ? 1 : 0;
    a.finish = a.step_end == a.k_tiles ? 1 : 0;
    // the operands' last k tiles are padding to a multiple of eight: whole rounds of two k groups' steps are enough (20
    // samples, 3777 x 2246, with its operands: 62 -> 47 us)
    const int64_t filled = ceil_div(ceil_div(K, kTileK), 4) * 4, padded_tiles = a.step_end - a.step_begin;
    a.step_end = a.step_end < filled ? a.step_end : filled;
    a.split_tiles = 0;
    const unsigned blocks = (unsigned)(a.blocks_m * a.blocks_n);
    const int64_t chunk_tiles = a.step_end - a.step_begin;
    const int64_t most = split_ws ? (int64_t)(split_ws_bytes / ((size_t)M * N * sizeof(float))) : 1;
    const DigitSplit split = digit_split(blocks, padded_tiles, chunk_tiles, most);
    const int64_t splits = split.count;
    if (splits > 1) {
      // few output tiles, long contraction: every split writes a dense partial result, summed in split order
      GemmDigitsArgs part = a;
      part.split_tiles = split.tiles;
      part.y = static_cast<float *>(split_ws);
      part.inner = 1, part.outer_stride = N, part.n_stride = 1;
      part.accumulate = 0, part.bias = nullptr;
      hipLaunchKernelGGL(gemm_digits_kernel<2>, dim3(blocks, (unsigned)splits), dim3(2 * kThreads),
                         2 * kStages * kStageBytes, stream, part);
      NBLA_HIP_LAUNCH_CHECK("gemm_digits");
      if (n_stride != 1 && ceil_div(M, 32) <= 65535) {
        hipLaunchKernelGGL(gemm_digits_split_sum_rows, dim3((unsigned)ceil_div(N, 32), (unsigned)ceil_div(M, 32)),
                           dim3(256), 0, stream, static_cast<const float *>(split_ws), (int)splits, M, N, y, inner,
                           outer_stride, n_stride, a.finish ? bias : nullptr, a.accumulate);
      } else {
        int64_t sum_blocks = ceil_div(M * N, 256);
        if (sum_blocks > 4096)
          sum_blocks = 4096;
        hipLaunchKernelGGL(gemm_digits_split_sum, dim3((unsigned)sum_blocks), dim3(256), 0, stream,
                           static_cast<const float *>(split_ws), (int)splits, M, N, y, inner, outer_stride, n_stride,
                           a.finish ? bias : nullptr, a.accumulate);
      }
      NBLA_HIP_LAUNCH_CHECK("gemm_digits_split_sum");
      continue;
    }
    if (blocks <= 256) // at most one block per CU: eight wavefronts, two k groups
      hipLaunchKernelGGL(gemm_digits_kernel<2>, dim3(blocks), dim3(2 * kThreads), 2 * kStages * kStageBytes, stream,
                         a);
    else
      hipLaunchKernelGGL(gemm_digits_kernel<1>, dim3(blocks), dim3(kThreads), kStages * kStageBytes, stream, a);
    NBLA_HIP_LAUNCH_CHECK("gemm_digits");
  }
  return NBLA_HIP_OK;
}

} // namespace nbla_hip
