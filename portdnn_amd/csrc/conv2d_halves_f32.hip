// fp32 forward convolution and stride-1 input gradient on the binary16 matrix
// instruction (gfx950): every operand as the sum of two binary16 values, fp32
// accumulation.
//
// The fp32 matrix instruction does 32 multiply-adds per cycle and SIMD, the
// binary16 one 512, of values with 11 significant bits.  A value times a power of two
// that brings it into binary16's range is
//
//   v = hi + 2^-11 lo,   hi = binary16(v),   lo = binary16(2^11 (v - hi)),
//
// with an error below 2^-23 |v| (lo has hi's exponent range, v - hi is exact), and
//
//   v w = hi hi' + 2^-11 (hi lo' + lo hi') + what is left out, below 2^-22 |v w|
//
// (2^-24.7 in the root mean square, of either sign): three instructions' time for what
// takes sixteen with the fp32 one.  The two small products have accumulators of their
// own.  Against 64 bits the sums are closer than those of the fp32 instruction, which rounds
// more often, and than Winograd's; where a launch would otherwise run on tiles of
// three bfloat16 parts, or divide its reductions, this one sums in parts too
// (choose_parts).  A sum of a few products that are not zero is further off than on the
// fp32 instruction, by what the operands are.
//
// Small values beside large ones keep as many bits as those.  The exponents are chosen for
// every 32 channels of a tile's pixels, and of 32 features' filter, from their
// largest value; accumulators follow by multiplying with powers of two.  What is
// smaller than 2^-26 of the largest (one value in 2e7 of normally distributed ones)
// would lose bits: such values are left out of a block's operands, and the block
// is taken once more with these alone, scaled up by 2^26.  Where that is not enough
// (values below 2^-52 of the block's largest, exponents that differ by more than
// 2^30 between blocks, small values in both operands beside sums whose exponent has
// to rise so far that they would overflow, infinities, NaNs in the filter) the tile is
// summed on the fp32 instruction instead, from the same LDS tile.
//
//   * A work-group owns a run of output pixels (images, strips of columns, rows and
//     columns flattened) and up to 128 features.  The input rows the run needs, halo
//     and zero padding included, are taken apart once per block of 32 channels on
//     their way into LDS, [pixel slot][32 hi, 32 lo, 16 bytes of padding], and
//     every filter tap reads the same tile.
//   * The filter is taken apart by a launch in front (packed in the order of the
//     instruction's operand) and streams from L2 into registers.
//
// Whole calls with the filter's launch of 5 us, before / here: 28x28x128 at batch 32,
// 3x3, 44 (Winograd) / 34 us, 64x64x256 at batch 8 161 / 98, 17x27x27 96 -> 256, 5x5,
// 112 (three bfloat16 parts) / 76 in six parts, 62 in three, and its gradient 159 (fp32
// instruction) / 78.  Of the
// 28 us of the first one's kernel the matrix units need 13; the rest is the first
// pixels' way into LDS (6), the last stores (3), 0.85 of their rate in between, and
// 32 compute units without a tile.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <type_traits>

#include "gemm_tile.h"
#include "halves.h"
#include "plan_cache.h"
#include "snn_kernels.h"

namespace snn {
namespace {

using gemm::xcd_remap;

using namespace halves;

constexpr int kKC = 32;                  // channels per LDS tile
constexpr int kSlotBytes = kKC * 4 + 16; // hi and lo, an odd number of pieces
constexpr int kUnitBytes = 2048;         // packed: 16 features x 32 channels
constexpr int kMaxPieces = 16;           // 16-byte pieces of an LDS tile per lane
constexpr int kLoadCoherent = 17;        // (sc0, sc1: from memory's side of L1)

// Images are cut into strips of strip_cols output columns, each with a halo of its
// own, and `padded_rows` is what a strip's output rows need of input rows.
struct Halves {
  int batch, in_rows, in_cols, channels, features;
  int out_rows, out_cols;
  int win_rows, win_cols, pad_rows, pad_cols, step_rows, step_cols;
  int strips, strip_cols;
  int tile_pixels, total_pixels;
  int padded_rows, halo_cols;
  int n_slots;
  int n_fslices, n_fblocks, n_cblocks;
  int part;        // channel blocks whose sums are taken together
  int pause;       // taps of one block that are, or all it has
  int least;       // ... where so many follow
  int headroom;    // powers of two that sums can be scaled up by
  int transposed;  // w[taps - 1 - tap][feature][channel]
  int relu;
  Divisor by_padded_rows, by_halo_cols, by_strip_cols, by_out_rows, by_strips;
};

// N channels of one feature, c ... c + N - 1 of tap `tap`.
template <int N>
__device__ __forceinline__ void load_filter(__amdgpu_buffer_rsrc_t w,
                                            const Halves& g, int tap, int c,
                                            int f, float (&v)[N]) {
  const int taps = g.win_rows * g.win_cols;
  const bool in = f < g.features && tap < taps;
  if (g.transposed != 0) {
    const unsigned at = static_cast<unsigned>(
                            ((taps - 1 - tap) * g.features + f) * g.channels + c) * 4u;
#pragma unroll
    for (int h = 0; h < N / 4; ++h) {
      const float4v four = __builtin_bit_cast(
          float4v, __builtin_amdgcn_raw_buffer_load_b128(
                       w, in && c + 4 * h < g.channels ? at + 16u * h : kOob, 0, 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * h + e] = four[e];
    }
  } else {
    const unsigned at =
        static_cast<unsigned>((tap * g.channels + c) * g.features + f) * 4u;
#pragma unroll
    for (int e = 0; e < N; ++e)
      v[e] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(
                     w, in && c + e < g.channels
                            ? at + static_cast<unsigned>(e * g.features) * 4u
                            : kOob, 0, 0));
  }
}

// Takes the filter apart: channel block, tap, 16 features -> 64 lanes x 8 hi, 64 lanes
// x 8 lo.  A work-group has 32 features and one channel block; their exponent and
// flags go to `head`.
constexpr int kPackWaves = 16;
template <int HELD>
__global__ void __launch_bounds__(64 * kPackWaves)
    halves_pack_kernel(const float* __restrict__ w, char* __restrict__ packed,
                       int* __restrict__ head, Halves g, unsigned w_bytes) {
  __shared__ Range ranges[kPackWaves];
  const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(w, w_bytes);
  const int fb = blockIdx.x, cb = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int units = g.win_rows * g.win_cols * 2;  // (tap, half of the features)
  const int f = fb * 32 + (lane & 15);
  const int c = cb * kKC + 8 * (lane >> 4);
  Range r = {0u, 0xFFFFFFFFu};
  float held[HELD][8];
#pragma unroll
  for (int k = 0; k < HELD; ++k) {
    const int u = wave + kPackWaves * k;
    load_filter(rsrc, g, u >> 1, c, f + 16 * (u & 1), held[k]);
  }
#pragma unroll
  for (int k = 0; k < HELD; ++k)
#pragma unroll
    for (int e = 0; e < 8; ++e) note(r, held[k][e]);
  for (int u = wave + kPackWaves * HELD; u < units; u += kPackWaves) {
    float v[8];
    load_filter(rsrc, g, u >> 1, c, f + 16 * (u & 1), v);
#pragma unroll
    for (int e = 0; e < 8; ++e) note(r, v[e]);
  }
  r = wave_range(r);
  if (lane == 0) ranges[wave] = r;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPackWaves; ++k) {
    r.big = max(r.big, ranges[k].big);
    r.small = min(r.small, ranges[k].small);
  }
  const bool zero = r.big == 0;
  int exponent = zero ? 0 : exponent_for(r.big);
  const int flags = zero ? kZero : loses(r, exponent);
  if ((flags & kBeyond) != 0) exponent = 0;
  if (threadIdx.x == 0)
    head[cb * g.n_fblocks + fb] = (exponent & 0xFFFF) | (flags << 16);
  const float scale = pow2(exponent), scale2048 = scale * 2048.f;
  auto put = [&](int u, float (&v)[8]) {
    if ((flags & kSmall) != 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = __builtin_fabsf(v[e] * scale) < pow2(kLow) ? 0.f : v[e];
    }
    uint4v hi, lo;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const Pair p = take_apart(v[2 * e], v[2 * e + 1], scale, scale2048);
      hi[e] = p.hi;
      lo[e] = p.lo;
    }
    uint4v* const to = reinterpret_cast<uint4v*>(
        packed + (static_cast<size_t>(cb * (units / 2) + (u >> 1)) *
                      g.n_fblocks * 2 + fb * 2 + (u & 1)) * kUnitBytes) + lane;
    to[0] = hi;
    to[64] = lo;
  };
#pragma unroll
  for (int k = 0; k < HELD; ++k)
    if (wave + kPackWaves * k < units) put(wave + kPackWaves * k, held[k]);
  for (int u = wave + kPackWaves * HELD; u < units; u += kPackWaves) {
    float v[8];
    load_filter(rsrc, g, u >> 1, c, f + 16 * (u & 1), v);
    put(u, v);
  }
}

// What a tile of LDS holds.
struct alignas(16) Block {
  int flags;
  int cb;          // channel block
  int unused[2];
  int acc_exp[4];  // exponents of the sums' scale, by feature block
  int by[4];       // ... what they change by in front of this block
  int ex[4];       // the filter's alone
};
// kBand1: the small values alone; kLast: the tile's last block; kPart: the sums of a
// part of the blocks are complete; kPlain: none of the tile's blocks will do;
// kRescale: the sums' scale changes; kSmallFilter << k: feature block k has values
// that are too small for its exponent; kAgain: the filter's operands have to be
// loaded from the block's first.
enum {
  kBand1 = 1, kLast = 2, kPart = 4, kPlain = 8, kRescale = 16, kAgain = 32,
  kSmallFilter = 64, kRare = ~(kLast | kPart)
};
constexpr int kMaxBlocks = 4;  // blocks of 32 features of a work-group

// WF x WP waves that multiply, FA blocks of 16 features x PB blocks of 16 pixels
// each, and as many that load the next block of 32 channels meanwhile and take it
// apart: loads complete in order, so a wave that did both would have to wait for
// pixels from memory in front of every operand of the filter.  Work-groups are
// persistent, so that the first block of a tile is loaded while the tile before is
// multiplied.  PAUSES: parts end inside a block, too (asked about where there are none
// it cost up to 5 %: 95x95x208 -> 28, 3x3, at batch 14 69 -> 72 us).
template <int FA, int PB, int WF, int WP, bool PAUSES>
__global__ void __launch_bounds__(128 * WF * WP)
    __attribute__((amdgpu_waves_per_eu(2, 2)))
    conv_halves_kernel(const float* __restrict__ src,
                       const char* __restrict__ packed,
                       const int* __restrict__ head,
                       const float* __restrict__ w,
                       const float* __restrict__ bias, float* __restrict__ dst,
                       Halves g, unsigned src_bytes, unsigned packed_bytes,
                       unsigned w_bytes, unsigned dst_bytes, unsigned n_groups) {
  constexpr int NW = WF * WP, NT = 64 * NW;  // of either kind
  constexpr int NF = FA * WF / 2;            // blocks of 32 features
  constexpr int ROW = NT / 8;                // slots that a piece per lane covers
  // Registers for the filter's operands of NS units, one block of features and tap
  // each: what is on its way while the others are multiplied has to cover the latency
  // of L2, 500 to 700 cycles; a unit is PB x 3 instructions of 16.
  constexpr int NS = 6;
  static_assert(NF <= kMaxBlocks && NW <= 4, "descriptors and ranges");
  extern __shared__ __align__(16) unsigned char lds[];
  Range* const ranges = reinterpret_cast<Range*>(lds);
  Block* const blocks = reinterpret_cast<Block*>(lds + 64);  // [2]
  unsigned* const table = reinterpret_cast<unsigned*>(lds + 256);
  constexpr int TABLE = kMaxPieces * ROW;  // byte offsets of the slots' pixels
  unsigned char* const tile_lds = lds + 256 + 2 * TABLE * 4;
  const int n_pieces = (g.n_slots + ROW - 1) / ROW;
  const int tile_bytes = n_pieces * ROW * kSlotBytes;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int taps = g.win_rows * g.win_cols;
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(w, w_bytes);
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  // A strip's rows, the strips and the images count as one run of padded rows.
  auto first_padded_of = [&](int pixel0) {
    const int row0 = divide(pixel0, g.by_strip_cols);
    const int strip = divide(row0, g.by_out_rows);
    return strip * g.padded_rows + (row0 - strip * g.out_rows) * g.step_rows;
  };
  unsigned id = blockIdx.x;  // of the tile, in the order of the launch
  // Where the slots' pixels are, kOob: nowhere; by `n` lanes.
  auto fill_table = [&](unsigned tile_id, unsigned* to, int lane_of, int n) {
    const int first_padded = first_padded_of(
        static_cast<int>(xcd_remap(tile_id, n_groups) / g.n_fslices) *
        g.tile_pixels);
#pragma nounroll
    for (int slot = lane_of; slot < n_pieces * ROW; slot += n) {
      const int lrow = divide(slot, g.by_halo_cols);
      const int hx = slot - lrow * g.halo_cols;
      const int row = first_padded + lrow;
      const int strip = divide(row, g.by_padded_rows);
      const int img = divide(strip, g.by_strips);
      const int iy = row - strip * g.padded_rows - g.pad_rows;
      const int ix = (strip - img * g.strips) * g.strip_cols * g.step_cols + hx -
                     g.pad_cols;
      const bool ok =
          slot < g.n_slots && img < g.batch &&
          static_cast<unsigned>(iy) < static_cast<unsigned>(g.in_rows) &&
          static_cast<unsigned>(ix) < static_cast<unsigned>(g.in_cols);
      to[slot] = ok ? static_cast<unsigned>(
                          ((img * g.in_rows + iy) * g.in_cols + ix) * g.channels) *
                          4u
                    : kOob;
    }
  };
  fill_table(id, table, threadIdx.x, 2 * NT);
  __syncthreads();

  if (wave >= NW) {
    const int tid = threadIdx.x - NT;
    const __amdgpu_buffer_rsrc_t src_rsrc = make_rsrc(src, src_bytes);
    const int piece_slot = tid >> 3;
    const unsigned piece_at = static_cast<unsigned>(tid & 7) * 16u;
    float4v v[kMaxPieces];
    const unsigned* now = table;  // of the tile whose blocks are loaded
    int head_now = 0;             // of the feature block lane % 4
    int head_fb = 0;
    bool mine = false;            // whether there is one
    bool plain = false;  // a tile's filter, or one of its blocks, cannot be taken apart
    int spread = 0;      // of the exponents of a tile's filter
    auto load_pieces = [&](int cb) {
      head_now = head[cb * g.n_fblocks + head_fb];
      const unsigned c = static_cast<unsigned>(cb) * (kKC * 4) + piece_at;
      const unsigned past = c < static_cast<unsigned>(g.channels) * 4u ? 0u : kOob;
#pragma unroll
      for (int i = 0; i < kMaxPieces; ++i)
        if (i < n_pieces)
          v[i] = __builtin_bit_cast(
              float4v, __builtin_amdgcn_raw_buffer_load_b128(
                           src_rsrc, (now[piece_slot + i * ROW] + c) | past, 0,
                           0));
    };
    auto start_tile = [&]() {
      const int fslice =
          static_cast<int>(xcd_remap(id, n_groups) % g.n_fslices);
      head_fb = min(fslice * NF + (lane & 3), g.n_fblocks - 1);
      mine = lane < NF && fslice * NF + lane < g.n_fblocks;
      load_pieces(0);
      // The filter's exponents: blocks that cannot be taken apart, and their range.
      bool beyond = false;
      int lowest = 1000, highest = -1000;
#pragma nounroll
      for (int cb = lane >> 2; cb < g.n_cblocks; cb += 16) {
        const int h = head[cb * g.n_fblocks + head_fb];
        beyond |= ((h >> 16) & kBeyond) != 0;
        const int e = static_cast<short>(h);
        lowest = min(lowest, ((h >> 16) & kZero) == 0 ? e : 1000);
        highest = max(highest, ((h >> 16) & kZero) == 0 ? e : -1000);
      }
      plain = __builtin_amdgcn_ballot_w64(beyond) != 0;
      if (!plain) {
        const unsigned up = wave_max(static_cast<unsigned>(highest + 1024));
        const unsigned down = wave_max(static_cast<unsigned>(1024 - lowest));
        spread = max(static_cast<int>(up) + static_cast<int>(down) - 2048, 0);
        plain = spread > 30;
      }
    };
    auto put = [&](int buf, float scale, float scale2048) {
      unsigned char* const to_lane =
          tile_lds + buf * tile_bytes + piece_slot * kSlotBytes + (tid & 7) * 8;
#pragma unroll
      for (int i = 0; i < kMaxPieces; ++i)
        if (i < n_pieces) {
          const Pair p = take_apart(v[i][0], v[i][1], scale, scale2048);
          const Pair q = take_apart(v[i][2], v[i][3], scale, scale2048);
          unsigned char* const to = to_lane + i * ROW * kSlotBytes;
          *reinterpret_cast<uint2v*>(to) = uint2v{p.hi, q.hi};
          *reinterpret_cast<uint2v*>(to + 64) = uint2v{p.lo, q.lo};
        }
    };
    while (id < n_groups) {
      start_tile();
      bool have = false;  // a block that is not zero has set `ex`
      bool empty = true;  // the sums of feature block lane % 4 are zeros
      int ex = 0, ex_low = 0, ex_high = 0, acc_exp = 0;
      int buf = 0, cb = 0, band = 0;
      bool stop = false;
      // A turn prepares a block while the one before is multiplied.
      while (!stop) {
        const bool there = id < n_groups;
        unsigned* const next = now == table ? table + TABLE : table;
        if (cb + 1 >= g.n_cblocks && id + gridDim.x < n_groups)
          fill_table(id + gridDim.x, next, tid, NT);
        Range r = {0u, 0xFFFFFFFFu};
        if (there && band == 0) {
          float most = 0.f;  // (a NaN is none, and makes NaNs of its sums)
#pragma unroll
          for (int i = 0; i < kMaxPieces; ++i)
            if (i < n_pieces) {
#pragma unroll
              for (int e = 0; e < 4; e += 2) {
                most = fmaxf(most, fmaxf(__builtin_fabsf(v[i][e]),
                                         __builtin_fabsf(v[i][e + 1])));
                r.small = min(r.small, min(magnitude(v[i][e]) - 1u,
                                           magnitude(v[i][e + 1]) - 1u));
              }
            }
          r.big = magnitude(most);
          r = wave_range(r);
          if (lane == 0) ranges[wave - NW] = r;
        }
        __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
        barrier();
        if (!there) {
          stop = true;
        } else {
          int flags = 0;
          const int small = static_cast<int>(__builtin_amdgcn_ballot_w64(
              mine && ((head_now >> 16) & kSmall) != 0));
          if (band == 0) {
#pragma unroll
            for (int k = 0; k < NW; ++k) {
              r.big = max(r.big, ranges[k].big);
              r.small = min(r.small, ranges[k].small);
            }
            r.big = __builtin_amdgcn_readfirstlane(r.big);
            r.small = __builtin_amdgcn_readfirstlane(r.small);
            if (r.big != 0) {
              const int want = exponent_for(r.big);
              if (!have) ex_low = ex_high = want;
              if (!have || want < ex || want > ex + 1) ex = want;
              have = true;
              ex_low = min(ex_low, ex);
              ex_high = max(ex_high, ex);
              flags = loses(r, ex);
              plain |= (flags & kBeyond) != 0 || ex_high - ex_low > 30;
            }
            // (sums of larger blocks may lie above this block's by both exponents, and
            // are scaled up for the small values of either operand)
            plain |= ex - ex_low + spread + ((flags & kSmall) != 0 ? kBand : 0) +
                         (small != 0 ? kBand : 0) > g.headroom;
          }
          const bool again = band == 0 && (flags & kSmall) != 0;
          const bool last = !again && cb + 1 >= g.n_cblocks;
          const bool part = !again && (last || (cb + 1) % g.part == 0);
          // (a feature block per lane)
          const int to = mine && ((head_now >> 16) & kZero) == 0
                             ? ex + static_cast<short>(head_now) : acc_exp;
          // (zeros keep their value at any exponent, by however much it changes)
          const int by = (empty ? 0 : to - acc_exp) + (band != 0 ? kBand : 0);
          const bool rescales =
              __builtin_amdgcn_ballot_w64(mine && by != 0) != 0;
          acc_exp = to;
          if (wave == NW) {
            if (lane < kMaxBlocks) {
              blocks[buf].acc_exp[lane] = to;
              blocks[buf].by[lane] = by;
              blocks[buf].ex[lane] = to - ex;
            }
            if (lane == 0) {
              blocks[buf].cb = cb;
              blocks[buf].flags = (band != 0 ? kBand1 | kAgain : 0) |
                                  (plain ? kPlain : 0) | (last ? kLast : 0) |
                                  (part ? kPart : 0) |
                                  (rescales ? kRescale : 0) |
                                  small * kSmallFilter;
            }
          }
          empty &= !(band == 0 && r.big != 0 &&
                     ((head_now >> 16) & kZero) == 0);
          if (plain) {
            stop = true;
          } else {
            const float scale = pow2(ex), scale2048 = scale * 2048.f;
            if (band != 0) {
#pragma unroll
              for (int i = 0; i < kMaxPieces; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const float t = v[i][e] * scale;
                  v[i][e] =
                      __builtin_fabsf(t) < pow2(kLow) ? t * pow2(kBand) : 0.f;
                }
              put(buf, 1.f, 2048.f);
            } else {
              if (again) {
#pragma unroll
                for (int i = 0; i < kMaxPieces; ++i)
#pragma unroll
                  for (int e = 0; e < 4; ++e) {
                    const float t = v[i][e];
                    v[i][e] = __builtin_fabsf(t * scale) < pow2(kLow) ? 0.f : t;
                  }
              }
              put(buf, scale, scale2048);
            }
            buf ^= 1;
            if (again) {
              band = 1;
              load_pieces(cb);
            } else {
              band = 0;
              if (!last) {
                load_pieces(++cb);
              } else {
                cb = 0;
                have = false;
                empty = true;
                acc_exp = 0;
                id += gridDim.x;
                now = next;
                if (id < n_groups) start_tile();
              }
            }
          }
        }
        __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
        barrier();
      }
      if (plain && id < n_groups) {
        // The block's values as they are in the same LDS tile.
        unsigned* const next = now == table ? table + TABLE : table;
        if (id + gridDim.x < n_groups)
          fill_table(id + gridDim.x, next, tid, NT);
        for (cb = 0; cb < g.n_cblocks; ++cb) {
          load_pieces(cb);
#pragma unroll
          for (int i = 0; i < kMaxPieces; ++i)
            if (i < n_pieces)
              *reinterpret_cast<float4v*>(
                  tile_lds + (piece_slot + i * ROW) * kSlotBytes + piece_at) =
                  v[i];
          __syncthreads();
          __syncthreads();
        }
        now = next;
        id += gridDim.x;
      }
    }
    return;
  }

  // (its matrix instructions first: what the loading wave of the SIMD has to do fits in
  // between)
  __builtin_amdgcn_s_setprio(2);
  const int wf = wave / WP, wp = wave % WP;
  const __amdgpu_buffer_rsrc_t packed_rsrc = make_rsrc(packed, packed_bytes);
  const __amdgpu_buffer_rsrc_t dst_rsrc = make_rsrc(dst, dst_bytes);
  float4v acc[FA][PB], low[FA][PB];
  auto rescale = [&](int i, int by) {
    const float s = pow2(by);
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      acc[i][j] *= s;
      low[i][j] *= s;
    }
  };
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < PB; ++j)
        acc[i][j] = low[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  };
  // of a tap, and of a channel block
  const unsigned tap_bytes = static_cast<unsigned>(g.n_fblocks) * 2 * kUnitBytes;
  const unsigned block_bytes = tap_bytes * static_cast<unsigned>(taps);
  half8 a[NS][2];       // [unit][hi, lo]
  half8 b[PB][2];
  int lane_base[PB];    // LDS offset of this lane's pixels
  const unsigned char* cur = tile_lds;
  auto read_b = [&](int j, int offset) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      b[j][h] = *reinterpret_cast<const half8*>(cur + lane_base[j] + offset +
                                                64 * h);
  };
  // (an offset that is asked for lies in the packed filter or, in the lanes' part, past
  // its end)
  const unsigned a_lane = static_cast<unsigned>(lane) * 16u;
  auto fill_a = [&](half8 (&to)[2], int h, unsigned at) {
    to[h] = __builtin_bit_cast(
        half8, __builtin_amdgcn_raw_buffer_load_b128(
                   packed_rsrc, a_lane + at + static_cast<unsigned>(h * 1024), 0,
                   0));
  };
  // (the units of the first taps)
  auto start_filter = [&](unsigned at) {
#pragma unroll
    for (int k = 0; k < NS; ++k)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        fill_a(a[k], h,
               at + static_cast<unsigned>(k / FA) * tap_bytes +
                   static_cast<unsigned>(k % FA) * kUnitBytes);
  };
  // Block i of the features and one tap.  Its operands' registers are loaded again, with
  // those at `next`, as soon as they are free, and behind the last block the pixels'
  // with the next tap's, at LDS offset `offset`: one load behind a matrix instruction,
  // which takes as long as issuing it and its addresses does.
  auto unit = [&](half8 (&x)[2], int i, unsigned next, int offset) {
    const bool last = i == FA - 1;
    auto product = [](const half8& p, const half8& q, const float4v& c) {
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(p, q, c, 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < PB; ++j) low[i][j] = product(x[1], b[j][0], low[i][j]);
    __builtin_amdgcn_sched_barrier(0);
    fill_a(x, 1, next);
    __builtin_amdgcn_sched_barrier(0);
    if (!last) {
#pragma unroll
      for (int j = 0; j < PB; ++j) acc[i][j] = product(x[0], b[j][0], acc[i][j]);
#pragma unroll
      for (int j = 0; j < PB; ++j) low[i][j] = product(x[0], b[j][1], low[i][j]);
      __builtin_amdgcn_sched_barrier(0);
      fill_a(x, 0, next);
    } else {
#pragma unroll
      for (int j = 0; j < PB; ++j) {
        acc[i][j] = product(x[0], b[j][0], acc[i][j]);
        low[i][j] = product(x[0], b[j][1], low[i][j]);
        __builtin_amdgcn_sched_barrier(0);
        read_b(j, offset);
        __builtin_amdgcn_sched_barrier(0);
      }
      fill_a(x, 0, next);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int row_step = (g.halo_cols - g.win_cols) * kSlotBytes;
  int at = 0, col = 0;  // LDS offset and column of the tap
  auto next_tap = [&]() {
    at += kSlotBytes;
    if (++col == g.win_cols) {
      col = 0;
      at += row_step;
    }
  };
  // A tap: units `u` ... of a group of three taps.  `rem` units are left at its start,
  // at `a_at`; after the last ones come the first ones at `a_next`.
  int rem = 0, exchange = 0, pause = 0;
  unsigned a_at = 0, a_next = 0;
  auto one_tap = [&](auto first) {
    constexpr int U = decltype(first)::value;
    next_tap();
#pragma unroll
    for (int i = 0; i < FA; ++i) {
      constexpr int kNs = NS;
      const int ahead = U + i + kNs, set = (U + i) % kNs;
      const unsigned next =
          ahead < rem ? a_at + static_cast<unsigned>(ahead / FA) * tap_bytes +
                            static_cast<unsigned>(ahead % FA) * kUnitBytes
                      : a_next + static_cast<unsigned>(set / FA) * tap_bytes +
                            static_cast<unsigned>(set % FA) * kUnitBytes;
      // (after the last tap nothing of the pixels is used)
      unit(a[set], i, next, at);
    }
  };
  // A lane's number that what follows is worked out from where it is used: the
  // compiler would keep all of it in registers beside the sums.
  auto anew = [](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  // The filter values of a block that are too small for its exponent.
  auto multiply_small_filter = [&](int i, int fb16, int cb, int exponent) {
    const float scale = pow2(exponent);
    const int ln = anew(lane), f = fb16 * 16 + (ln & 15);
    rescale(i, kBand);
    at = col = 0;
    for (int tap = 0; tap < taps; ++tap) {
      float v[8];
      load_filter(w_rsrc, g, tap, cb * kKC + 8 * (ln >> 4), f, v);
      half8 hi, lo;
      bool any = false;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float s = v[e] * scale;
        const float t = __builtin_fabsf(s) < pow2(kLow) ? s * pow2(kBand) : 0.f;
        any |= t != 0.f;
        hi[e] = static_cast<_Float16>(t);
        lo[e] = static_cast<_Float16>((t - static_cast<float>(hi[e])) * 2048.f);
      }
      if (__builtin_amdgcn_ballot_w64(any) != 0) {
#pragma unroll
        for (int j = 0; j < PB; ++j) {
          read_b(j, at);
          low[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, b[j][1],
                                                             low[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, b[j][0],
                                                             acc[i][j], 0, 0, 0);
          low[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, b[j][0],
                                                             low[i][j], 0, 0, 0);
        }
      }
      next_tap();
    }
    rescale(i, -kBand);
  };

  int buf = 0;
  bool restart = true;  // no block of the tile is on its way
  start_filter(static_cast<unsigned>(
                   (static_cast<int>(xcd_remap(id, n_groups) % g.n_fslices) * WF +
                    wf) * FA) * kUnitBytes);
  for (; id < n_groups; id += gridDim.x) {
    const unsigned group = xcd_remap(id, n_groups);
    const int fslice = static_cast<int>(group % g.n_fslices);
    const int fb0 = (fslice * WF + wf) * FA;  // of 16 features
    const int pixel0 = static_cast<int>(group / g.n_fslices) * g.tile_pixels;
    const int n_pixels = min(g.tile_pixels, g.total_pixels - pixel0);
    {
      const int first_padded = first_padded_of(pixel0);
      const int ln = anew(lane);
#pragma unroll
      for (int j = 0; j < PB; ++j) {
        const int q = (wp * PB + j) * 16 + (ln & 15);
        lane_base[j] = (ln >> 4) * 16;
        if (q < n_pixels) {
          const int m = pixel0 + q;
          const int row = divide(m, g.by_strip_cols);
          const int strip = divide(row, g.by_out_rows);
          lane_base[j] += ((strip * g.padded_rows +
                            (row - strip * g.out_rows) * g.step_rows -
                            first_padded) * g.halo_cols +
                           (m - row * g.strip_cols) * g.step_cols) *
                          kSlotBytes;
        }
      }
    }
    // the feature blocks of the tile after this one
    const unsigned id_next = id + gridDim.x < n_groups ? id + gridDim.x : id;
    const int fslice_next =
        static_cast<int>(xcd_remap(id_next, n_groups) % g.n_fslices);
    const unsigned a_slice =
        static_cast<unsigned>(fb0) * kUnitBytes;
    const unsigned a_slice_next =
        static_cast<unsigned>((fslice_next * WF + wf) * FA) * kUnitBytes;
    if (restart) {
      buf = 0;
      barrier();
      barrier();  // the first block is there
      restart = false;
    }
    int flags = 0;
    a_at = a_slice;
    // Parts of the reduction: the sums of all but the last lie in `dst` meanwhile.
    bool inside = false;  // a block goes on behind its part
    for (bool first = true;; first = false) {
      clear();
      for (;; buf ^= 1) {
        if (!inside) {
          cur = tile_lds + buf * tile_bytes;
          at = col = 0;
          flags = __builtin_amdgcn_readfirstlane(blocks[buf].flags);
          rem = taps * FA;
          // (the loading waves exchange their ranges in the middle)
          exchange = rem - taps / 3 / 2 * (3 * FA);
          pause = (flags & kBand1) != 0 ? 0 : rem;
        }
        if constexpr (PAUSES) {
          pause -= g.pause * FA;
          if (pause < g.least * FA) pause = 0;
        }
#pragma unroll
        for (int j = 0; j < PB; ++j) read_b(j, at);
        if ((flags & kRare) != 0 && !inside) {
          if ((flags & kPlain) != 0) break;
          if ((flags & kAgain) != 0) {
            a_at -= block_bytes;
            start_filter(a_at);
          }
          if ((flags & kRescale) != 0) {
#pragma unroll
            for (int i = 0; i < FA; ++i)
              rescale(i, __builtin_amdgcn_readfirstlane(
                             blocks[buf].by[(wf * FA + i) / 2]));
          }
        }
        // (of the block after this one: the tile's next, or the next tile's first)
        if (!inside)
          a_next = (flags & kLast) != 0 ? a_slice_next : a_at + block_bytes;
        const int stop = PAUSES ? max(pause, 3 * FA - 1) : 3 * FA - 1;
        while (rem > stop) {
          if (rem == exchange) barrier();
          one_tap(std::integral_constant<int, 0>{});
          one_tap(std::integral_constant<int, FA>{});
          one_tap(std::integral_constant<int, 2 * FA>{});
          rem -= 3 * FA;
          a_at += 3 * tap_bytes;
        }
        inside = PAUSES && pause > 0;
        if (inside) break;
        if (taps < 3) barrier();
        if (rem >= FA) {
          one_tap(std::integral_constant<int, 0>{});
          a_at += tap_bytes;
          if (rem >= 2 * FA) {
            a_at -= tap_bytes;
            one_tap(std::integral_constant<int, FA>{});
            a_at += 2 * tap_bytes;
          }
        }
        if ((flags & kRare) != 0) {
#pragma unroll
          for (int i = 0; i < FA; ++i) {
            if ((flags & (kSmallFilter << ((wf * FA + i) / 2))) != 0)
              multiply_small_filter(
                  i, fb0 + i, __builtin_amdgcn_readfirstlane(blocks[buf].cb),
                  __builtin_amdgcn_readfirstlane(
                      blocks[buf].ex[(wf * FA + i) / 2]));
            if ((flags & kBand1) != 0) rescale(i, -kBand);
          }
          start_filter(a_next);  // (no registers are kept for it meanwhile)
        }
        barrier();
        if ((flags & kPart) != 0) break;
      }
      const int ln = anew(lane), l16 = ln & 15, q = ln >> 4;
      struct Place { int n, y, x; };  // n < 0: none
      auto place_of = [&](int j) {
        const int in = (wp * PB + j) * 16 + l16;
        const int m = pixel0 + in;
        const int row = divide(m, g.by_strip_cols);
        const int strip = divide(row, g.by_out_rows);
        const int n = divide(strip, g.by_strips);
        const int x =
            (strip - n * g.strips) * g.strip_cols + m - row * g.strip_cols;
        return Place{in < n_pixels && x < g.out_cols ? n : -1,
                     row - strip * g.out_rows, x};
      };
      if ((flags & kPlain) == 0) {
#pragma unroll
        for (int i = 0; i < FA; ++i) {
          const int by = -__builtin_amdgcn_readfirstlane(
              blocks[buf].acc_exp[(wf * FA + i) / 2]);
          // (in two steps: up to 2^226; what is no normal number is rounded by the
          // second)
          const float s = pow2(max(min(by, 100), -100));
#pragma unroll
          for (int j = 0; j < PB; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              acc[i][j][v] =
                  __builtin_fmaf(low[i][j][v], 0x1p-11f, acc[i][j][v]) * s;
          if (by > 100 || by < -100) {
            const float t = pow2(max(min(by - (by > 0 ? 100 : -100), 126), -126));
#pragma unroll
            for (int j = 0; j < PB; ++j) acc[i][j] *= t;
          }
        }
        if (!inside) buf ^= 1;
      } else {
        // The fp32 instruction sums, a block's channels of one tap at a time (in `low`):
        // what it makes of an infinity or NaN in the filter and the zeros of padding is
        // left out, there are no such products.
        restart = true;
        clear();
        int row0[PB], col0[PB];  // of the first tap's pixel
#pragma unroll
        for (int j = 0; j < PB; ++j) {
          const Place place = place_of(j);
          row0[j] = place.y * g.step_rows - g.pad_rows;
          col0[j] = place.x * g.step_cols - g.pad_cols;
        }
        for (int cb = 0; cb < g.n_cblocks; ++cb) {
          __syncthreads();
          at = col = 0;
          for (int tap = 0, row = 0; tap < taps; ++tap) {
#pragma unroll
            for (int i = 0; i < FA; ++i)
#pragma unroll
              for (int j = 0; j < PB; ++j) low[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              float4v y[PB];
#pragma unroll
              for (int j = 0; j < PB; ++j)
                // (16 bytes per quarter of the wave lie in lane_base already)
                y[j] = *reinterpret_cast<const float4v*>(tile_lds + lane_base[j] +
                                                         at + 64 * h);
#pragma unroll
              for (int i = 0; i < FA; ++i) {
                const int f = (fb0 + i) * 16 + l16, c = cb * kKC + 16 * h + 4 * q;
                float x[4];
                load_filter(w_rsrc, g, tap, c, f, x);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                  for (int j = 0; j < PB; ++j)
                    low[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        x[e], y[j][e], low[i][j], 0, 0, 0);
              }
            }
#pragma unroll
            for (int j = 0; j < PB; ++j) {
              const bool there =
                  static_cast<unsigned>(row0[j] + row) <
                      static_cast<unsigned>(g.in_rows) &&
                  static_cast<unsigned>(col0[j] + col) <
                      static_cast<unsigned>(g.in_cols);
#pragma unroll
              for (int i = 0; i < FA; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  acc[i][j][v] += there ? low[i][j][v] : 0.f;
            }
            next_tap();
            row += col == 0 ? 1 : 0;
          }
          __syncthreads();
        }
        start_filter(a_slice_next);
      }

      // (a lane holds four features of a pixel, four lanes 16: runs of 64 bytes)
      const __amdgpu_buffer_rsrc_t bias_rsrc =
          make_rsrc(bias, bias != nullptr ? g.features * 4u : 0u);
      const bool complete = (flags & (kLast | kPlain)) != 0 && !inside;
      const bool act = complete && (bias != nullptr || g.relu != 0);
      unsigned to[PB];
#pragma unroll
      for (int j = 0; j < PB; ++j) {
        const Place place = place_of(j);
        to[j] = place.n >= 0
                    ? static_cast<unsigned>(
                          ((place.n * g.out_rows + place.y) * g.out_cols +
                           place.x) * g.features) * 4u
                    : kOob;
      }
      if (!first && (flags & kPlain) == 0)
        __builtin_amdgcn_s_waitcnt(0);  // (what this lane has stored)
#pragma unroll
      for (int i = 0; i < FA; ++i) {
        const int f = (fb0 + i) * 16 + 4 * q;
        const unsigned past = f < g.features ? static_cast<unsigned>(f) * 4u : kOob;
        auto offset = [&](int j) {
          return to[j] == kOob || past == kOob ? kOob : to[j] + past;
        };
        if (!first && (flags & kPlain) == 0) {
#pragma unroll
          for (int j = 0; j < PB; ++j)
            acc[i][j] += __builtin_bit_cast(
                float4v, __builtin_amdgcn_raw_buffer_load_b128(
                             dst_rsrc, offset(j), 0, kLoadCoherent));
        }
        if (act) {
          const float4v add = __builtin_bit_cast(
              float4v,
              __builtin_amdgcn_raw_buffer_load_b128(bias_rsrc, f * 4, 0, 0));
#pragma unroll
          for (int j = 0; j < PB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float sum = acc[i][j][e] + add[e];
              acc[i][j][e] = g.relu != 0 ? fmaxf(sum, 0.f) : sum;
            }
        }
#pragma unroll
        for (int j = 0; j < PB; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(
              __builtin_bit_cast(uint4v, acc[i][j]), dst_rsrc, offset(j), 0, 0);
      }
      if (complete) break;
    }
  }
}

// Work-groups of eight waves, one to a compute unit: features x pixels, and the slots
// of an LDS tile.
struct Form {
  int fa, pb, wf, wp;
  int features() const { return 16 * fa * wf; }
  int pixels() const { return 16 * pb * wp; }
  int row() const { return 8 * wf * wp; }  // slots that a piece per lane covers
};
constexpr Form kForms[] = {{4, 4, 2, 2}, {4, 4, 1, 4}, {2, 4, 2, 2},
                           {2, 4, 1, 4}, {2, 4, 4, 1}, {2, 2, 2, 2}};
constexpr int kNumForms = sizeof(kForms) / sizeof(kForms[0]);

struct HalvesPlan {
  Halves g;
  int form = -1;  // -1: not for this kernel
  size_t lds_bytes = 0;
  unsigned n_groups = 0;
  size_t packed_bytes = 0;  // of the filter taken apart
  double us = 0;            // estimated, with the launch that takes it apart
  size_t workspace_bytes() const {
    return packed_bytes +
           (static_cast<size_t>(g.n_fblocks) * g.n_cblocks * 4 + 15) / 16 * 16;
  }
};

size_t filter_bytes(const Halves& g) {
  return static_cast<size_t>(g.win_rows) * g.win_cols * g.channels * g.features *
         4;
}

// The convolution that the launch is, if it is one for this kernel.
bool geometry(int direction, const snn_hip_conv2d_params& p, Halves* g) {
  if (p.batch < 1 || p.in_rows < 1 || p.in_cols < 1 || p.out_rows < 1 ||
      p.out_cols < 1 || p.channels < 4 || p.features < 4 ||
      p.channels % 4 != 0 || p.features % 4 != 0 || p.window_rows < 1 ||
      p.window_cols < 1 || p.pad_rows < 0 || p.pad_cols < 0 ||
      p.input_format != 0 || p.filter_format != 0 ||
      static_cast<long>(p.window_rows) * p.window_cols > 256)
    return false;
  const size_t x = static_cast<size_t>(p.batch) * p.in_rows * p.in_cols *
                   p.channels * 4;
  const size_t y = static_cast<size_t>(p.batch) * p.out_rows * p.out_cols *
                   p.features * 4;
  *g = Halves();
  g->batch = p.batch;
  g->win_rows = p.window_rows;
  g->win_cols = p.window_cols;
  if (direction == SNN_HIP_FORWARD) {
    g->in_rows = p.in_rows; g->in_cols = p.in_cols; g->channels = p.channels;
    g->out_rows = p.out_rows; g->out_cols = p.out_cols;
    g->features = p.features;
    g->pad_rows = p.pad_rows; g->pad_cols = p.pad_cols;
    g->step_rows = p.stride_rows; g->step_cols = p.stride_cols;
  } else if (direction == SNN_HIP_INPUT_BACKPROP) {
    if (p.stride_rows != 1 || p.stride_cols != 1 ||
        p.pad_rows >= p.window_rows || p.pad_cols >= p.window_cols)
      return false;
    g->in_rows = p.out_rows; g->in_cols = p.out_cols; g->channels = p.features;
    g->out_rows = p.in_rows; g->out_cols = p.in_cols;
    g->features = p.channels;
    g->pad_rows = p.window_rows - 1 - p.pad_rows;
    g->pad_cols = p.window_cols - 1 - p.pad_cols;
    g->step_rows = g->step_cols = 1;
    g->transposed = 1;
  } else {
    return false;
  }
  g->n_fblocks = ceil_div(g->features, 32);
  g->n_cblocks = ceil_div(g->channels, kKC);
  const size_t packed = static_cast<size_t>(g->n_cblocks) * g->n_fblocks * 2 *
                        g->win_rows * g->win_cols * kUnitBytes;
  return x <= kMaxBufferBytes && y <= kMaxBufferBytes &&
         filter_bytes(*g) <= kMaxBufferBytes && packed <= kMaxBufferBytes;
}

// At most so many padded rows hold the inputs of `pixels` consecutive outputs.
int rows_spanned(const Halves& g, int pixels) {
  int rows = pixels % g.strip_cols == 0 ? pixels / g.strip_cols
                                        : (pixels + g.strip_cols - 2) /
                                                  g.strip_cols + 1;
  const bool aligned = pixels % g.strip_cols == 0 && g.out_rows % rows == 0;
  const int strips_in = aligned ? 0 : (rows - 2 + g.out_rows) / g.out_rows;
  return (rows - 1) * g.step_rows + g.win_rows +
         strips_in * (g.win_rows - g.step_rows > 0 ? g.win_rows - g.step_rows : 0);
}

// What the result is off by against 64 bits, squared and relative in the 2-norm: by the
// operands, by the sums (a root law: parts count by the squares of their products) and
// by adding up the parts.  Fitted to 700 random layers, within a tenth.
double error2(const Halves& g, int* parts) {
  const int taps = g.win_rows * g.win_cols;
  double squares = 0, part = 0;
  *parts = 0;
  for (int cb = 0; cb < g.n_cblocks; ++cb) {
    const int channels = std::min(kKC, g.channels - cb * kKC);
    for (int left = taps; left > 0;) {
      const bool pauses = left - g.pause >= g.least;
      const int now = pauses ? g.pause : left;
      left -= now;
      part += now * channels;
      if (pauses || (left == 0 && ((cb + 1) % g.part == 0 ||
                                   cb + 1 == g.n_cblocks))) {
        squares += part * part;
        part = 0;
        ++*parts;
      }
    }
  }
  return 0.78e-14 + 38.4e-18 * squares / (taps * g.channels) + 0.02e-14 * *parts;
}

// Parts of the reduction whose sums are added up by themselves, so that the result is
// no further from 64 bits than that of the kernel the launch would run on otherwise:
// their number, 0 if that cannot be had.  (17x27x27 96 -> 256, 5x5, 2400 products,
// 1.56e-7 on tiles of three bfloat16 parts with the reduction in two: 3.1e-7 whole,
// 1.98e-7 in three, 1.58e-7 in six.  Winograd's kernel is off by more: 28x28x128
// 3.1e-7, here 2.3e-7 whole.)
int choose_parts(int direction, const snn_hip_conv2d_params& p, bool winograd,
                 Halves* g) {
  const int taps = g->win_rows * g->win_cols;
  int parts = 0;
  g->part = g->n_cblocks;
  g->pause = g->least = taps;
  if (winograd) return 1;
  // (a hundredth is nothing)
  const double most = 1.02 * conv2d_gemm_f32_error2(direction, p);
  for (int n = 1; n <= g->n_cblocks; ++n) {
    const int part = ceil_div(g->n_cblocks, n);
    if (n > 1 && part == g->part) continue;
    g->part = part;
    if (error2(*g, &parts) <= most) return parts;
  }
  for (g->pause = taps / 6 * 3; g->pause > 0; g->pause -= 3) {
    g->least = std::min(g->pause, 6);
    if (error2(*g, &parts) <= most) return parts;
  }
  return 0;
}

int tuned(const char* value, int otherwise) {
  return value != nullptr ? std::atoi(value) : otherwise;
}

HalvesPlan compute_plan(int direction, const snn_hip_conv2d_params& p,
                        bool winograd) {
  HalvesPlan best;
  Halves g;
  if (!geometry(direction, p, &g)) return best;
  const int taps = g.win_rows * g.win_cols;
  const int parts = choose_parts(direction, p, winograd, &g);
  if (parts == 0) return best;
  // (n products below 2^15 * 2^15 each, and fp32 ends at 2^128)
  g.headroom = 97;
  for (long n = static_cast<long>(taps) * g.channels; n > 1; n = (n + 1) / 2)
    --g.headroom;
  const int only = tuned(SNN_TUNING_ENV("SNN_HIP_HALVES_FORM"), -1);
  for (int strips = 1; strips <= 8; ++strips) {
    g.strip_cols = ceil_div(g.out_cols, strips);
    if (strips > 1 && (g.strip_cols < 8 ||
                       ceil_div(g.out_cols, g.strip_cols) != strips))
      continue;
    g.strips = strips;
    const long total = static_cast<long>(g.batch) * strips * g.out_rows *
                       g.strip_cols;
    if (total > (1l << 30)) continue;
    g.total_pixels = static_cast<int>(total);
    g.padded_rows = (g.out_rows - 1) * g.step_rows + g.win_rows;
    g.halo_cols = (g.strip_cols - 1) * g.step_cols + g.win_cols;
    if (static_cast<long>(g.batch) * strips * g.padded_rows > (1l << 30)) continue;
    for (int form = 0; form < kNumForms; ++form) {
      if (only >= 0 && form != only) continue;
      const Form& f = kForms[form];
      const int full = std::min(f.pixels(), g.total_pixels);
      const int most_rows = full / g.strip_cols;
      int tried = 0;
      for (int k = 0; k < 3; ++k) {
        // all pixels; whole rows; whole rows that divide an image's
        int pixels = full;
        if (k > 0) {
          int rows = std::min(most_rows, g.out_rows);
          if (k == 1) rows = most_rows;
          while (k == 2 && rows > 1 && g.out_rows % rows != 0) --rows;
          pixels = rows * g.strip_cols;
        }
        if (pixels < 1 || pixels == tried) continue;
        tried = pixels;
        g.tile_pixels = pixels;
        const long slots = static_cast<long>(rows_spanned(g, pixels)) *
                           g.halo_cols;
        g.n_slots = static_cast<int>(slots);
        const long pieces = (slots + f.row() - 1) / f.row();
        if (pieces > kMaxPieces) continue;
        const size_t lds_bytes = 256 + size_t{2} * kMaxPieces * f.row() * 4 +
                                 size_t{2} * pieces * f.row() * kSlotBytes;
        if (lds_bytes > kMaxLdsBytes) continue;
        g.n_fslices = ceil_div(g.n_fblocks, f.fa * f.wf / 2);
        const long groups = static_cast<long>(ceil_div(g.total_pixels, pixels)) *
                            g.n_fslices;
        if (groups > (1l << 30)) continue;
        // Per work-group and tile: the first block's loads, then for every block the
        // longer of its products and of loading and taking the next one apart, then
        // the stores.  Cycles of a 2.1 GHz clock, fitted to 900 launches of 110 random
        // layers in all forms, within 12 % in the root mean square.  (A tap's
        // FA x PB x 3 instructions of 16 cycles wait for their operands the more the
        // fewer they are.)
        const double wait = f.fa == 4 ? 1.28 : f.pb == 4 ? 1.54 : 2.0;
        const double products = taps * 3.0 * f.fa * f.pb * 16 * wait + 1700;
        const double fill = 900 + 510.0 * pieces;
        const double tile_cycles =
            fill + g.n_cblocks * std::max(products, fill) +
            (2.0 * parts - 1) * f.pixels() * f.features() * 4 / 14.5 +
            1500.0 * (parts - ceil_div(g.n_cblocks, g.part));  // ends inside blocks
        double rounds = static_cast<double>(groups) / kNumCus;
        rounds = rounds < 4 ? std::ceil(rounds) : rounds + 0.5;
        // (the launch that takes the filter apart holds 32 taps in registers)
        const double us = 7.9 + 3.5e-3 * taps * g.n_fblocks * g.n_cblocks +
                          0.17 * std::max(0, taps - 25) +
                          rounds * tile_cycles / 2100;
        if (best.form >= 0 && us >= best.us) continue;
        best.form = form;
        best.g = g;
        best.us = us;
        best.lds_bytes = lds_bytes;
        best.n_groups = static_cast<unsigned>(groups);
      }
    }
  }
  if (best.form < 0) return best;
  Halves& b = best.g;
  b.by_padded_rows = divisor(b.padded_rows);
  b.by_halo_cols = divisor(b.halo_cols);
  b.by_strip_cols = divisor(b.strip_cols);
  b.by_out_rows = divisor(b.out_rows);
  b.by_strips = divisor(b.strips);
  best.packed_bytes = static_cast<size_t>(b.n_cblocks) * b.n_fblocks * 2 * taps *
                      kUnitBytes;
  return best;
}

const HalvesPlan& make_plan(int direction, const snn_hip_conv2d_params& p,
                            bool winograd) {
  thread_local PlanCache<HalvesPlan> cache;
  return cache.get(p, static_cast<unsigned>(direction) * 2 + winograd,
                   [&] { return compute_plan(direction, p, winograd); });
}

struct HalvesOperands {
  const float *src, *w, *bias;
  float* dst;
  char* packed;
};

template <int FORM, bool PAUSES>
void launch_form(const HalvesOperands& ops, const HalvesPlan& plan,
                 const Halves& g, hipStream_t stream) {
  constexpr Form f = kForms[FORM];
  auto kernel = conv_halves_kernel<f.fa, f.pb, f.wf, f.wp, PAUSES>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLdsBytes);
  (void)attr;
  KernelTimer timer(stream);
  hipLaunchKernelGGL(
      kernel, dim3(std::min(plan.n_groups, unsigned{kNumCus})), dim3(128 * f.wf * f.wp), plan.lds_bytes, stream,
      ops.src, ops.packed,
      reinterpret_cast<const int*>(ops.packed + plan.packed_bytes), ops.w,
      ops.bias, ops.dst, g,
      static_cast<unsigned>(static_cast<size_t>(g.batch) * g.in_rows *
                            g.in_cols * g.channels * 4),
      static_cast<unsigned>(plan.packed_bytes),
      static_cast<unsigned>(filter_bytes(g)),
      static_cast<unsigned>(static_cast<size_t>(g.batch) * g.out_rows *
                            g.out_cols * g.features * 4),
      plan.n_groups);
}

}  // namespace

double conv2d_halves_f32_us(int direction, const snn_hip_conv2d_params& p,
                            bool winograd) {
  const HalvesPlan& plan = make_plan(direction, p, winograd);
  return plan.form >= 0 ? plan.us : -1;
}

size_t conv2d_halves_f32_workspace_floats(int direction,
                                          const snn_hip_conv2d_params& p,
                                          bool winograd) {
  const HalvesPlan& plan = make_plan(direction, p, winograd);
  return plan.form >= 0 ? plan.workspace_bytes() / 4 : 0;
}

void conv2d_halves_f32_tile(int direction, const snn_hip_conv2d_params& p,
                            bool winograd, int* pixels, int* features) {
  const HalvesPlan& plan = make_plan(direction, p, winograd);
  *pixels = plan.form >= 0 ? plan.g.tile_pixels : 0;
  *features = plan.form >= 0 ? kForms[plan.form].features() : 0;
}

int launch_conv2d_halves_f32(int direction, const float* input,
                             const float* filter, float* output,
                             const snn_hip_conv2d_params& p, float* workspace,
                             bool winograd, bool prepared, hipStream_t stream,
                             const LaunchOptions* options) {
  const HalvesPlan& plan = make_plan(direction, p, winograd);
  if (plan.form < 0) return SNN_HIP_INVALID_ALGORITHM;
  Halves g = plan.g;
  char* const packed = reinterpret_cast<char*>(workspace);
  if (!prepared) {
    const dim3 grid(g.n_fblocks, g.n_cblocks);
    int* const head = reinterpret_cast<int*>(packed + plan.packed_bytes);
    hipLaunchKernelGGL(g.win_rows * g.win_cols <= kPackWaves
                           ? halves_pack_kernel<2> : halves_pack_kernel<4>,
                       grid, dim3(64 * kPackWaves), 0, stream, filter, packed,
                       head, g, static_cast<unsigned>(filter_bytes(g)));
    if (options != nullptr && options->prepare_only) {
      SNN_HIP_CHECK_LAUNCH();
      return SNN_HIP_OK;
    }
  }
  const bool fuse = direction == SNN_HIP_FORWARD && options != nullptr &&
                    options->wanted();
  g.relu = fuse && options->relu ? 1 : 0;
  const HalvesOperands ops = {input, filter, fuse ? options->bias : nullptr,
                              output, packed};
  const auto launch = [&](auto pauses) {
    constexpr bool P = decltype(pauses)::value;
    switch (plan.form) {
      case 0: launch_form<0, P>(ops, plan, g, stream); break;
      case 1: launch_form<1, P>(ops, plan, g, stream); break;
      case 2: launch_form<2, P>(ops, plan, g, stream); break;
      case 3: launch_form<3, P>(ops, plan, g, stream); break;
      case 4: launch_form<4, P>(ops, plan, g, stream); break;
      default: launch_form<5, P>(ops, plan, g, stream);
    }
  };
  if (g.pause < g.win_rows * g.win_cols)
    launch(std::true_type{});
  else
    launch(std::false_type{});
  if (fuse && options->applied != nullptr) *options->applied = true;
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return report_hip_error(err, "conv_halves_kernel");
  return SNN_HIP_OK;
}

}  // namespace snn
