// Forward convolution and input gradient for every window, stride and channel
// count, as an implicit GEMM on MFMA (gfx950): binary16 or fp32 operands, fp32
// accumulation, one rounding of a binary16 result.
//
//   forward         Y[pixel][f]  = sum over (tap, c) X[pixel o tap][c] * W[tap][c][f]
//   input gradient  dX[pixel][c] = sum over (tap, f) dY[pixel o tap][f] * W[tap'][c][f]
//
// (the Forward and InputBackprop directions of sycldnn::conv2d::launch,
// include/portdnn/conv2d/launch.h:59-118.)  The gradient of a strided
// convolution is split by classes: the dX pixels whose padded row and column
// have one remainder modulo the strides are reached by the same sub-window of
// taps, and form a dense stride-1 convolution of dY with that sub-filter.  All
// classes run in one launch, their tiles side by side and rotated over the
// work-groups (see TileOf), and store their pixels straight into dX; a class that
// no tap reaches stores zeros.
//
// The reduction runs over 16-byte pieces -- eight binary16 or four fp32 channels
// of one tap -- of a pixel, flattened over (tap, piece): a chunk is four pieces,
// which may belong to different taps, so channel counts that are no multiple
// of a chunk's waste nothing but the last chunk's tail.  Source tensors whose
// channel count fills no whole pieces are copied once with the count rounded up.
//
//   * A work-group owns BM pixels x BN features.  Per chunk both tiles, [row][4
//     pieces], arrive in one of three LDS buffers by loads that write LDS
//     directly (1 KB = 16 rows per instruction), two chunks ahead: one barrier
//     per chunk, and no wave waits for more than the loads of the chunk it is
//     about to multiply.  Padding pixels, ragged tails and rows past the last
//     pixel load from out of range, which stores zeros.
//   * Which of its four positions in an LDS row a piece takes is XORed with
//     bits of the row, so that the ds_read_b128 of 8 or 16 consecutive rows
//     touch different banks.
//   * A binary16 forward filter (and a gradient's whose feature count fills no
//     whole pieces) is packed first, [32 features][chunk][row][4 pieces] in the
//     same swizzled order (2-5 us), zeros where channels or features end.  The
//     gradient's is read in place: its reduction index is the contiguous one.
//     So is a forward fp32 filter, whose tile lies in LDS as it does in memory,
//     [16 (tap, channel)][features]: an fp32 instruction wants one value of a
//     lane, which that layout gives it without conflicts.
//   * Features are the MFMA rows and pixels the columns, with the features of
//     a block permuted in the packed filter so that a lane ends with 16
//     consecutive features of one pixel (16-byte stores).
//   * An fp32 instruction (32x32x2) takes as long as a binary16 one but sums two
//     products instead of sixteen: there the matrix units are the bound, and
//     the tap arithmetic of every lane costs nothing beside them.
//   * Larger fp32 tiles (SPLIT) take every operand apart into three bfloat16 parts
//     in registers and sum six of the nine products of parts on the bfloat16
//     instruction, a sixteenth of the time each; the five small ones in
//     accumulators of their own.  What is left out (the second and third parts'
//     products, and that of the third ones) is below 2^-23 of a product, 2^-26 in
//     the root mean square and without a bias; an fp32 sum rounds by as much at
//     every second product.  Against 64 bits the results are closer than the fp32
//     instruction's: on 70 random layers of 36 to 8640 products, with activations of
//     either sign, of one sign and half of them zero, 0.71 of its error in the
//     2-norm and 0.93 in the worst value at the most (17x27x27 96 -> 256, 5x5:
//     2.3e-7 and 6.0e-7).  Two more products take 13 us of 120 and change neither.
//     With the fp32 instruction / here: that layer 144 / 120 us, 28x28x128 at batch
//     128, 3x3, 259 / 215, 147x147x48 -> 64 at batch 8, 5x5, 218 / 208, 56x56x128,
//     3x3 stride 2, at batch 32 80 / 71: 0.15 PFLOP/s, where the matrix units are
//     busy 0.4 of the time and the splitting takes as many cycles of the vector
//     units.  A conversion ahead, into three planes, would move half as many bytes
//     again.
//   * A strided gradient of few channels (a three-channel first layer) would
//     fill 3 of the 32 matrix rows.  Its classes are merged: the pixels of a
//     block of stride x stride share one window of ceil(window / stride) source
//     pixels, and (class, channel) are the rows, with zeros packed for taps that
//     do not reach a class (12 of 32 rows, 49 of 64 taps of a 7x7 stride 2).
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "gemm_tile.h"
#include "plan_cache.h"
#include "snn_kernels.h"

namespace snn {
namespace {

using gemm::float16v;
using gemm::xcd_remap;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int uint2v __attribute__((ext_vector_type(2)));
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr;
template <typename T>
struct PieceOf;
template <> struct PieceOf<_Float16> { typedef half8 type; };
template <> struct PieceOf<float> { typedef float4v type; };
template <typename T>
constexpr int kPiece = 16 / static_cast<int>(sizeof(T));  // channels

// Where the filter operand comes from: packed tiles, the gradient's filter as it
// is (reduction index contiguous), the forward fp32 filter as it is (features
// contiguous).
enum FilterFrom { kPacked, kInPlace, kRows };

constexpr unsigned kOob = 0x7FFFFFF0u;
constexpr size_t kMaxBufferBytes = 0x7FFFFFF0u;
constexpr int kRowBytes = 64;     // one chunk of one row
constexpr int kMaxClasses = 16;
constexpr int kMaxWindow = 12;    // the two tap masks of a pixel share a word

// n / d for 0 <= n < 2^31 by one multiplication: (2 n * magic) >> (32 + shift)
// with magic = ceil(2^(31 + shift) / d), 2^shift >= d.  (Divisions by values
// known at launch only are 35 instructions; a lane has a dozen of them, as long
// as the multiplications of a short reduction.)
struct Divisor {
  unsigned magic, shift;
};
Divisor divisor(int d) {
  unsigned shift = 0;
  while ((1u << shift) < static_cast<unsigned>(d)) ++shift;
  const unsigned long long top = 1ull << (31 + shift);
  return {static_cast<unsigned>((top + d - 1) / d), shift};
}
__device__ __forceinline__ int divide(int n, Divisor d) {
  return static_cast<int>(
      __umulhi(static_cast<unsigned>(n) << 1, d.magic) >> d.shift);
}

struct GatherClass {
  int rows, cols;        // pixels of the class per image
  Divisor by_rows, by_cols;
  int pixels;            // ... and over the batch
  int off_r, off_c;      // source row / column of tap (0, 0) for pixel (0, 0)
  int win_r, win_c;      // taps
  int out_r0, out_c0;    // output row / column of pixel (0, 0)
  int n_chunks;
  unsigned pack_block;   // first 2 KB block of its packed filter
  Divisor by_win_c;
  int tap_r0, tap_rs;    // filter row of tap row t: tap_r0 + t * tap_rs
  int tap_c0, tap_cs;
};

struct Gather {
  int src_rows, src_cols;
  int cp;                // pieces per source pixel
  Divisor by_cp;
  int step_r, step_c;    // source step per class pixel
  int out_rows, out_cols, out_step_r, out_step_c;
  int channels, features;
  int win_rows, win_cols;  // of the whole filter
  int n_tiles_n;
  int n_splits;          // work-groups that share a tile's reduction
  unsigned n_tiles;      // tiles of all classes
  int n_classes;
  int round_shift, turn; // how the classes are rotated, see tile_of
  int mirrored;          // input gradient: w[tap][feature][channel]
  int merged;            // channels per pixel of merged classes, or 0
  int relu;              // of a forward launch with bias and activation
  // A copy to whole pieces that takes every copy_step'th pixel of an image of
  // copy_rows x copy_cols (0: all pixels).
  int copy_rows, copy_cols, copy_step_r, copy_step_c;
  GatherClass cls[kMaxClasses];
};

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p,
                                                   unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x00020000);
}

// Position of piece c in LDS row r: c ^ swz(r % 16).
__host__ __device__ constexpr unsigned swz(unsigned r16) {
  return ((r16 >> 1) ^ (r16 >> 3)) & 3u;
}

// Image, row and column of pixel m of a class.
struct Pixel { int n, y, x; };
__device__ __forceinline__ Pixel pixel_of(int m, const GatherClass& cls) {
  const int t = divide(m, cls.by_cols);
  const int n = divide(t, cls.by_rows);
  return {n, t - n * cls.rows, m - t * cls.cols};
}

// Which feature of its block of 32 an MFMA row holds.  A lane's accumulators are
// rows 8 g + 4 h + i (h = lane / 32): g = 0, 1 become features 8 h ... + 7 and
// g = 2, 3 features 16 + 8 h ... + 7, so that one 16-byte store of the two lanes
// of a pixel covers 32 consecutive bytes.
__host__ __device__ constexpr int feature_of_row(unsigned row) {
  return static_cast<int>(16 * (row >> 4) + 8 * ((row >> 2) & 1) +
                          4 * ((row >> 3) & 1) + (row & 3));
}

// Whether a pixel's sums hold products with zeros that are no taps of theirs.
__device__ __forceinline__ bool window_cut(const Gather& g,
                                           const GatherClass& cls, Pixel px) {
  const int iy = px.y * g.step_r + cls.off_r;
  const int ix = px.x * g.step_c + cls.off_c;
  return g.merged != 0 || iy < 0 || iy + cls.win_r > g.src_rows || ix < 0 ||
         ix + cls.win_c > g.src_cols;
}

// Feature f of a pixel over the taps that exist, with `w` the filter as the
// caller has it; up to the first term that makes it a NaN (a tensor of NaNs
// would otherwise be summed one product at a time).
template <typename T>
__device__ __forceinline__ float exact_sum(const T* __restrict__ src,
                                           const T* __restrict__ w,
                                           const Gather& g,
                                           const GatherClass& cls, Pixel px,
                                           int f) {
  int member_r = 0, member_c = 0, per_tap = g.features;
  if (g.merged != 0) {
    const int member = f / g.merged;
    f -= member * g.merged;
    member_r = member / g.out_step_c;
    member_c = member - member_r * g.out_step_c;
    per_tap = g.merged;
  }
  const size_t stride = g.mirrored ? 1 : static_cast<size_t>(g.features);
  float sum = 0.f;
  for (int tr = 0; tr < cls.win_r; ++tr) {
    const int y = px.y * g.step_r + cls.off_r + tr;
    const int wr = cls.tap_r0 + tr * cls.tap_rs + member_r;
    if (y < 0 || y >= g.src_rows || wr >= g.win_rows) continue;
    for (int ts = 0; ts < cls.win_c; ++ts) {
      const int x = px.x * g.step_c + cls.off_c + ts;
      const int wc = cls.tap_c0 + ts * cls.tap_cs + member_c;
      if (x < 0 || x >= g.src_cols || wc >= g.win_cols) continue;
      const T* const from =
          src + (static_cast<size_t>(px.n * g.src_rows + y) * g.src_cols + x) *
                    g.cp * kPiece<T>;
      const size_t at_tap = static_cast<size_t>(wr * g.win_cols + wc);
      const T* const by = g.mirrored ? w + (at_tap * per_tap + f) * g.channels
                                     : w + at_tap * g.channels * g.features + f;
      for (int c = 0; c < g.channels && sum == sum; ++c)
        sum += static_cast<float>(from[c]) * static_cast<float>(by[c * stride]);
    }
  }
  return sum;
}

// What a bias and an activation make of a sum.
__device__ __forceinline__ float bias_act(float v, float bias, int relu) {
  v += bias;
  return relu != 0 ? fmaxf(v, 0.f) : v;
}

// (a function of its own: the compiler drops the host side of a kernel template
// whose body names the LDS-direct load)
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t rsrc,
                                            char* lds, unsigned offset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)lds, 16, offset, 0, 0,
                                           0);
}

constexpr int vmcnt_imm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

// Tiles run over feature tiles, then classes, then pixels: the classes of one
// piece of dX are written side by side.  (Class after class, every work-group
// in flight wrote the same half of the rows and columns, which are the same
// half of the memory channels: 56x56x256 <- 512, 1x1 stride 2, at batch 128,
// 168 -> 110 us.)  Work-groups go round the 32 compute units of an XCD, so the
// order of the classes is rotated from piece to piece: by one where the tiles of
// a class come round to the units they met before (after 2^round_shift pieces),
// so that the long ones meet every unit, and for two, four or eight classes by one
// per piece (`turn`), which mixes the memory channels.  One per piece alone left
// the long tiles of four classes to eight units (fp32 9x84x84 40 <- 620, 1x1
// stride 2, one class with products: 51 -> 19.5 us; 32x28x28 256 <- 256, 3x3: 86
// -> 79; binary16 32x56x56 128 <- 128, 3x3: 20.6 -> 19.1), without it the largest
// lose (binary16 128x56x56 128 <- 128, 3x3: 53 / 56).
struct TileOf { int m, cls, n; };
__device__ __forceinline__ TileOf tile_of(unsigned tile, const Gather& g) {
  const unsigned n = tile % g.n_tiles_n, t = tile / g.n_tiles_n;
  const unsigned m = t / g.n_classes;
  return {static_cast<int>(m),
          static_cast<int>((t + m * g.turn + (m >> g.round_shift)) %
                           g.n_classes),
          static_cast<int>(n)};
}

// Output element of feature f of a merged block, or -1 outside the image.
__device__ __forceinline__ int merged_element(const Gather& g,
                                              const GatherClass& cls, Pixel px,
                                              int f) {
  const int k = f / g.merged, c = f - k * g.merged;
  const int a = k / g.out_step_c, b = k - a * g.out_step_c;
  const int y = px.y * g.out_step_r + cls.out_r0 + a;
  const int x = px.x * g.out_step_c + cls.out_c0 + b;
  return y >= 0 && y < g.out_rows && x >= 0 && x < g.out_cols &&
                 f < g.features
             ? ((px.n * g.out_rows + y) * g.out_cols + x) * g.merged + c
             : -1;
}

// Filter pack (the first n_pack_groups work-groups, one lane per 16-byte
// piece) and, behind it, the copy of a source tensor to whole pieces.
template <typename T>
__global__ void __launch_bounds__(256)
    gather_prepare_kernel(const T* __restrict__ w, T* __restrict__ wpk,
                          Gather g, unsigned n_pack_lanes,
                          unsigned n_pack_groups, const T* __restrict__ src,
                          T* __restrict__ wide, unsigned n_pieces) {
  constexpr int kE = kPiece<T>;
  typename PieceOf<T>::type v;
  if (blockIdx.x < n_pack_groups) {
    const unsigned idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= n_pack_lanes) return;
    const unsigned block = idx >> 7, row = (idx >> 2) & 31, slot = idx & 3;
    int k = 0;
    while (k + 1 < g.n_classes && block >= g.cls[k + 1].pack_block) ++k;
    const GatherClass& cls = g.cls[k];
    const unsigned local = block - cls.pack_block;
    const unsigned nb = local / cls.n_chunks, chunk = local % cls.n_chunks;
    const int q = static_cast<int>(chunk * 4 + (slot ^ swz(row & 15)));
    const int tap = divide(q, g.by_cp);
    const int c = (q - tap * g.cp) * kE;
    const int tr = divide(tap, cls.by_win_c), ts = tap - tr * cls.win_c;
    int f = nb * 32 + feature_of_row(row), per_tap = g.features;
    bool ok = tr < cls.win_r && f < g.features;
    int wr = cls.tap_r0 + tr * cls.tap_rs, wc = cls.tap_c0 + ts * cls.tap_cs;
    if (g.merged != 0) {
      const int member = f / g.merged;
      f -= member * g.merged;
      per_tap = g.merged;
      wr += member / g.out_step_c;
      wc += member % g.out_step_c;
      ok = ok && wr < g.win_rows && wc < g.win_cols;
    }
    const int valid = ok ? min(kE, g.channels - c) : 0;
    const size_t at_tap = static_cast<size_t>(wr * g.win_cols + wc);
    const T* from = g.mirrored ? w + (at_tap * per_tap + f) * g.channels + c
                               : w + (at_tap * g.channels + c) * g.features + f;
    const size_t stride = g.mirrored ? 1 : static_cast<size_t>(g.features);
#pragma unroll
    for (int e = 0; e < kE; ++e)
      v[e] = e < valid ? from[e * stride] : static_cast<T>(0.f);
    *reinterpret_cast<decltype(v)*>(wpk + static_cast<size_t>(idx) * kE) = v;
    return;
  }
  const unsigned idx = (blockIdx.x - n_pack_groups) * 256 + threadIdx.x;
  if (idx >= n_pieces) return;
  const unsigned pixel = divide(idx, g.by_cp);
  const int c = static_cast<int>(idx - pixel * g.cp) * kE;
  size_t from_pixel = pixel;
  if (g.copy_rows != 0) {  // (the copy's pixels are the output's)
    const Pixel px = pixel_of(static_cast<int>(pixel), g.cls[0]);
    from_pixel = (static_cast<size_t>(px.n) * g.copy_rows +
                  px.y * g.copy_step_r) * g.copy_cols + px.x * g.copy_step_c;
  }
  const T* from = src + from_pixel * g.channels + c;
#pragma unroll
  for (int e = 0; e < kE; ++e)
    v[e] = c + e < g.channels ? from[e] : static_cast<T>(0.f);
  *reinterpret_cast<decltype(v)*>(wide + static_cast<size_t>(idx) * kE) = v;
}

// An fp32 value times 2^24 as the sum of three bfloat16 ones, the first rounded to
// nearest (its remainder then has no bias, nor have the products left out), the
// others cut off: every remainder is exact, and the last one fits.  (Integer
// operations: the conversion instruction takes as long as four of them.)
// The matrix units take operands and sums below 2^-126 for zero.  No part of an
// fp32 value lies below 2^-149, so none of a value times 2^24 is lost, nor is any
// product of parts times 2^48 that an fp32 sum could hold; what grows beyond the
// range by it gives an infinity or a NaN, and such a tile is taken again without
// splitting.  (One instruction per value: 17x27x27 96 -> 256, 5x5, 114.5 -> 119.5
// us; looking for the smallest value on the way takes 125.)
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
struct Parts {
  bf16x8 first, second, third;
};
__device__ __forceinline__ Parts split_parts(const float4v& e,
                                             const float4v& o) {
  uint4v first, second, third;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    unsigned f[2], s[2], t[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = 2 * k + h;
      const float v = (at < 4 ? e[at & 3] : o[at & 3]) * kSplitScale;
      f[h] = (__builtin_bit_cast(unsigned, v) + 0x8000u) & 0xFFFF0000u;
      const float rest = v - __builtin_bit_cast(float, f[h]);
      s[h] = __builtin_bit_cast(unsigned, rest);
      t[h] = __builtin_bit_cast(
          unsigned, rest - __builtin_bit_cast(float, s[h] & 0xFFFF0000u));
    }
    // the upper halves of two values
    first[k] = __builtin_amdgcn_perm(f[1], f[0], 0x07060302u);
    second[k] = __builtin_amdgcn_perm(s[1], s[0], 0x07060302u);
    third[k] = __builtin_amdgcn_perm(t[1], t[0], 0x07060302u);
  }
  return {__builtin_bit_cast(bf16x8, first), __builtin_bit_cast(bf16x8, second),
          __builtin_bit_cast(bf16x8, third)};
}
__device__ __forceinline__ Parts split_parts(const half8&, const half8&) {
  return {};
}

// WM x WN waves of TM x TN blocks of 32 pixels x 32 features.  UNIFORM: whole
// chunks per tap, tap bookkeeping in scalar registers; otherwise every lane
// works out the tap of its own piece.  FROM: what `wpk` is; `w` is the caller's
// filter.
template <typename T, int WM, int WN, int TM, int TN, bool UNIFORM, int FROM,
          bool SPLIT>
__global__ void __launch_bounds__(64 * WM * WN, TM * TN >= 4 ? 2 : 3)
    conv_gather_kernel(const T* __restrict__ src, const T* __restrict__ wpk,
                       const T* __restrict__ w,
                       const float* __restrict__ bias, T* __restrict__ dst,
                       float* __restrict__ part, Gather g, unsigned src_bytes,
                       unsigned wpk_bytes, unsigned dst_bytes,
                       unsigned n_groups) {
  typedef typename PieceOf<T>::type Piece;
  constexpr bool IN_PLACE = FROM == kInPlace;
  constexpr int kE = kPiece<T>;
  constexpr unsigned kSize = sizeof(T);
  static_assert(FROM != kRows || kSize == 4, "one value per lane");
  constexpr int NW = WM * WN;
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  constexpr int LA = BM / 16 / NW;                      // loads per wave, chunk
  constexpr int B_BLOCKS = BN / 16;
  constexpr int LB = B_BLOCKS >= NW ? B_BLOCKS / NW : 1;
  static_assert(LA * NW * 16 == BM && (B_BLOCKS % NW == 0 || NW % B_BLOCKS == 0),
                "whole load instructions per wave");
  constexpr int STAGE = (BM + BN) * kRowBytes;
  // three objects, so that the compiler ties an LDS read to the loads of its
  // own buffer only
  __shared__ __align__(1024) char buf0[STAGE];
  __shared__ __align__(1024) char buf1[STAGE];
  __shared__ __align__(1024) char buf2[STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const unsigned group = xcd_remap(blockIdx.x, n_groups);
  const unsigned tile = group / g.n_splits, split = group % g.n_splits;
  const TileOf at = tile_of(tile, g);
  const GatherClass cls = g.cls[at.cls];
  const int m0 = at.m * BM, n0 = at.n * BN;
  if (m0 >= cls.pixels) return;
  const int per_split = (cls.n_chunks + g.n_splits - 1) / g.n_splits;
  const int chunk0 = min(cls.n_chunks, static_cast<int>(split) * per_split);
  const int n_chunks = min(cls.n_chunks - chunk0, per_split);

  // A class that no tap reaches: zeros, whole runs of features per pixel.
  if (cls.n_chunks == 0 && (g.features & (kE - 1)) == 0) {
    if (split != 0) return;
    const __amdgpu_buffer_rsrc_t out = make_rsrc(dst, dst_bytes);
    for (int i = threadIdx.x; i < BM * (BN / kE); i += 64 * NW) {
      const int m = m0 + i / (BN / kE), f = n0 + i % (BN / kE) * kE;
      const Pixel px = pixel_of(m, cls);
      const unsigned pixel =
          (px.n * g.out_rows + px.y * g.out_step_r + cls.out_r0) * g.out_cols +
          px.x * g.out_step_c + cls.out_c0;
      const uint4v zero = {0u, 0u, 0u, 0u};
      __builtin_amdgcn_raw_buffer_store_b128(
          zero, out, m < cls.pixels && f < g.features
                         ? (pixel * g.features + f) * kSize : kOob, 0, 0);
    }
    return;
  }

  const __amdgpu_buffer_rsrc_t src_rsrc = make_rsrc(src, src_bytes);
  const __amdgpu_buffer_rsrc_t wpk_rsrc = make_rsrc(wpk, wpk_bytes);

  // Rows this lane loads: byte offset of tap (0, 0), the lane's piece included
  // where it is the same for every chunk, and the taps inside the image (rows
  // in the low half of the word, columns in the high half).
  const unsigned piece = (lane & 3u) ^ swz((lane >> 2) & 15u);
  unsigned a_off[LA], a_mask[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int m = m0 + 16 * (wave + NW * i) + (lane >> 2);
    const Pixel px = pixel_of(m, cls);
    const int iy = px.y * g.step_r + cls.off_r;
    const int ix = px.x * g.step_c + cls.off_c;
    // taps r with 0 <= iy + r < src_rows, bits low .. high - 1
    auto bits = [](int low, int high) {
      low = max(low, 0);
      return high > low ? (1u << high) - (1u << low) : 0u;
    };
    const unsigned rows = bits(-iy, min(cls.win_r, g.src_rows - iy));
    const unsigned cols = bits(-ix, min(cls.win_c, g.src_cols - ix));
    a_mask[i] = m < cls.pixels ? rows | cols << 16 : 0u;
    a_off[i] = (static_cast<unsigned>((px.n * g.src_rows + iy) * g.src_cols + ix) *
                    g.cp + (UNIFORM ? piece : 0u)) * 16u;
  }
  unsigned b_off[LB];  // of chunk 0
  int b_block[LB];
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    b_block[i] = (wave + NW * i) % B_BLOCKS;
    if constexpr (IN_PLACE) {
      const int f = n0 + b_block[i] / 2 * 32 +
                    feature_of_row((b_block[i] & 1) * 16 + (lane >> 2));
      // (2^31 stays out of range whatever is added)
      b_off[i] = f < g.features ? static_cast<unsigned>(f * g.channels) * kSize +
                                      (UNIFORM ? piece * 16u : 0u)
                                : 0x80000000u;
    } else if constexpr (FROM == kRows) {
      // 1 KB of the tile: whole runs of BN features of 256 / BN filter rows
      // (columns past the last feature belong to the next row, and to outputs
      // that are not stored; rows past the last one load zeros)
      const int at = b_block[i] * 256 + lane * 4;
      b_off[i] = static_cast<unsigned>((chunk0 * 16 + at / BN) * g.features +
                                       n0 + at % BN) * 4u;
    } else {
      b_off[i] = ((cls.pack_block + static_cast<unsigned>(n0 / 32 + b_block[i] / 2) *
                                        cls.n_chunks) * 2 +
                  (b_block[i] & 1)) * 1024u + lane * 16u;
    }
  }

  const int cp = g.cp, src_cols = g.src_cols, win_c = cls.win_c;
  const Divisor by_cp = g.by_cp, by_win_c = cls.by_win_c;
  int tap_r, tap_c, c4;  // UNIFORM: of the next chunk to load
  int q;                 // otherwise: the lane's next piece
  unsigned b_chunk;
  auto rewind = [&]() {  // to the first chunk
    tap_r = tap_c = c4 = 0;
    q = chunk0 * 4 + piece;
    if (UNIFORM && chunk0 > 0) {
      const int tap = chunk0 * 4 / cp;
      c4 = chunk0 * 4 - tap * cp;
      tap_r = tap / win_c;
      tap_c = tap - tap_r * win_c;
    }
    b_chunk = FROM == kPacked ? chunk0 * 2048u : 0u;
  };
  rewind();
  const unsigned b_step = FROM == kRows ? g.features * 64u : 2048u;
  // IN_PLACE: bytes from a tap to the next column's, the next row's
  const int filter_row = cp * 16, filter_tap = g.features * filter_row;
  const int tap_at = (cls.tap_r0 * g.win_cols + cls.tap_c0) * filter_tap;
  const int tap_dr = cls.tap_rs * g.win_cols * filter_tap;
  const int tap_dc = cls.tap_cs * filter_tap;
  const int win_r = cls.win_r;
  auto issue = [&](char* buf) {
    int tr = tap_r, ts = tap_c;
    unsigned tap_off;
    if constexpr (UNIFORM) {
      if constexpr (IN_PLACE)
        b_chunk = static_cast<unsigned>(tap_at + tr * tap_dr + ts * tap_dc +
                                        c4 * 16);
      tap_off = static_cast<unsigned>((tr * src_cols + ts) * cp + c4) * 16u;
      c4 += 4;
      if (c4 == cp) {
        c4 = 0;
        if (++tap_c == win_c) { tap_c = 0; ++tap_r; }
      }
    } else {
      const int tap = divide(q, by_cp);
      tr = divide(tap, by_win_c);
      ts = tap - tr * win_c;
      tap_off = (static_cast<unsigned>(tr * src_cols + ts) * cp +
                 (q - tap * cp)) * 16u;
      if constexpr (IN_PLACE)
        b_chunk = tr < win_r ? static_cast<unsigned>(tap_at + tr * tap_dr +
                                                     ts * tap_dc +
                                                     (q - tap * cp) * 16)
                             : 0x80000000u;
      q += 4;
    }
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const unsigned ok = (a_mask[i] >> tr) & (a_mask[i] >> (16 + ts)) & 1u;
      load_to_lds(src_rsrc, buf + (wave + NW * i) * 1024,
                  ok != 0 ? a_off[i] + tap_off : kOob);
    }
#pragma unroll
    for (int i = 0; i < LB; ++i)
      load_to_lds(wpk_rsrc, buf + BM * kRowBytes + b_block[i] * 1024,
                  IN_PLACE && !UNIFORM ? (b_off[i] | b_chunk) >= 0x80000000u
                                             ? kOob : b_off[i] + b_chunk
                                       : b_off[i] + b_chunk);
    if constexpr (!IN_PLACE) b_chunk += b_step;
  };

  float16v acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int l32 = lane & 31, khalf = lane >> 5;
  const int in_row =
      static_cast<int>((static_cast<unsigned>(khalf) ^ swz(lane & 15u)) * 16u);
  const int px_at = (wm * TM * 32 + l32) * kRowBytes + in_row;
  const int ft_at = (BM + wn * TN * 32 + l32) * kRowBytes + in_row;
  // Operands of reduction step S (16 channels) of a chunk.  (Step 1 reads
  // pieces 2 and 3: bit 1 of the swizzled position flips.)
  struct Operands { Piece a[TN], b[TM]; };
  const int row_at = BM * kRowBytes + khalf * (4 * BN * 4) +
                     (wn * TN * 32 + feature_of_row(l32)) * 4;
  auto fetch = [&](const char* buf, int s, Operands& o) {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      if constexpr (FROM == kRows) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o.a[i][e] = *reinterpret_cast<const float*>(
              buf + row_at + (8 * s + e) * (BN * 4) + i * 128);
      } else {
        o.a[i] = *reinterpret_cast<const Piece*>(
            buf + (ft_at ^ (32 * s)) + i * 32 * kRowBytes);
      }
    }
#pragma unroll
    for (int j = 0; j < TM; ++j)
      o.b[j] = *reinterpret_cast<const Piece*>(
          buf + (px_at ^ (32 * s)) + j * 32 * kRowBytes);
  };
  // (fp32: element e of the two lane halves is products 4 (2 s) + e and
  // 4 (2 s + 1) + e of the chunk)
  auto multiply = [&](const Operands& o) {
    if constexpr (kSize == 2) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              o.a[i], o.b[j], acc[i][j], 0, 0, 0);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                o.a[i][e], o.b[j][e], acc[i][j], 0, 0, 0);
    }
  };

  // SPLIT: all 16 products of a chunk and lane pair in six instructions.
  float16v low[SPLIT ? TN : 1][SPLIT ? TM : 1];
  auto multiply_split = [&](const Operands& e, const Operands& o) {
    Parts a[TN], b[TM];
#pragma unroll
    for (int i = 0; i < TN; ++i) a[i] = split_parts(e.a[i], o.a[i]);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      b[j] = split_parts(e.b[j], o.b[j]);
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        auto product = [](const bf16x8& p, const bf16x8& q, const float16v& c) {
          return __builtin_amdgcn_mfma_f32_32x32x16_bf16(p, q, c, 0, 0, 0);
        };
        float16v& lo = low[i][j];
        lo = product(a[i].third, b[j].first, lo);
        lo = product(a[i].first, b[j].third, lo);
        lo = product(a[i].second, b[j].second, lo);
        lo = product(a[i].second, b[j].first, lo);
        lo = product(a[i].first, b[j].second, lo);
        acc[i][j] = product(a[i].first, b[j].first, acc[i][j]);
      }
    }
  };

  // One chunk: its step 0 operands are in `even`, the next two chunks are
  // arriving.  Step 1 is read while step 0 multiplies; then every wave is done
  // with the buffer, the load of the chunk after next-but-one goes into it,
  // and the next chunk's step 0 is read while step 1 multiplies.
  Operands even, odd;
  int done = 0;
  auto step = [&](char* cur, const char* next, bool more1, bool more2,
                  bool more3) {
    fetch(cur, 1, odd);
    __builtin_amdgcn_sched_barrier(0);
    multiply(even);
    __builtin_amdgcn_sched_barrier(0);
    if (more1) {
      if (more2)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(LA + LB) & ~0x0F00);  // and LDS
      else
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0) & ~0x0F00);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (more3) issue(cur);
      fetch(next, 0, even);
      __builtin_amdgcn_sched_barrier(0);
    }
    multiply(odd);
    __builtin_amdgcn_sched_barrier(0);
    ++done;
  };
  // SPLIT: a chunk is read whole, and its buffer free once every wave has.
  auto step_split = [&](char* cur, bool more1, bool more2, bool more3) {
    fetch(cur, 0, even);
    fetch(cur, 1, odd);
    if (more1) {
      __builtin_amdgcn_sched_barrier(0);
      if (more2)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(LA + LB) & ~0x0F00);  // and LDS
      else
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0) & ~0x0F00);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (more3) issue(cur);
    }
    multiply_split(even, odd);
    ++done;
  };
  auto multiply_all = [&]() {
    if (n_chunks <= 0) return;
    issue(buf0);
    if (n_chunks > 1) issue(buf1);
    if (n_chunks > 2) issue(buf2);
    // (all three: a wait for the first alone makes the compiler put a full
    // wait into every turn of the loop)
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    fetch(buf0, 0, even);
    while (done + 5 < n_chunks) {
      step(buf0, buf1, true, true, true);
      step(buf1, buf2, true, true, true);
      step(buf2, buf0, true, true, true);
    }
    // at most five chunks are left
    auto last = [&](char* cur, const char* next) {
      if (done < n_chunks)
        step(cur, next, done + 1 < n_chunks, done + 2 < n_chunks,
             done + 3 < n_chunks);
    };
    last(buf0, buf1);
    last(buf1, buf2);
    last(buf2, buf0);
    last(buf0, buf1);
    last(buf1, buf2);
  };
  if constexpr (SPLIT) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) low[i][j][v] = 0.f;
    if (n_chunks > 0) {
      issue(buf0);
      if (n_chunks > 1) issue(buf1);
      if (n_chunks > 2) issue(buf2);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      while (done + 5 < n_chunks) {
        step_split(buf0, true, true, true);
        step_split(buf1, true, true, true);
        step_split(buf2, true, true, true);
      }
      auto last = [&](char* cur) {
        if (done < n_chunks)
          step_split(cur, done + 1 < n_chunks, done + 2 < n_chunks,
                     done + 3 < n_chunks);
      };
      last(buf0);
      last(buf1);
      last(buf2);
      last(buf0);
      last(buf1);
    }
    // A tile with sums that are no numbers (the parts of an infinity are none) is
    // taken again without splitting, by the whole work-group.
    bool again = false;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float sum = (acc[i][j][v] + low[i][j][v]) * kSplitUnscale;
          acc[i][j][v] = sum;
          again |= !(__builtin_fabsf(sum) < __builtin_inff());
        }
    __syncthreads();  // every wave is done with the last chunk
    int* const agains = reinterpret_cast<int*>(buf0);
    again = __builtin_amdgcn_ballot_w64(again) != 0;
    if (lane == 0) agains[wave] = again ? 1 : 0;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) any |= agains[k];
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(any) != 0) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
      rewind();
      done = 0;
      multiply_all();
    }
  } else {
    multiply_all();
  }

  // A shared reduction: the fp32 tile in accumulator order, 1 KB per store.
  if (g.n_splits > 1) {
    float4v* const out =
        reinterpret_cast<float4v*>(part) +
        (static_cast<size_t>(split) * g.n_tiles + tile) * (BM * BN / 4) +
        wave * (TN * TM * 256) + lane;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float4v four = {acc[i][j][4 * v], acc[i][j][4 * v + 1],
                                acc[i][j][4 * v + 2], acc[i][j][4 * v + 3]};
          out[((i * TM + j) * 4 + v) * 64] = four;
        }
    return;
  }

  // A lane holds features f0 .. f0 + 7 and f0 + 16 .. f0 + 23 of one pixel per
  // block.
  // Bit v of strange[..]: sum v of the block is a NaN that may not belong there.
  // It is stored like the others and replaced afterwards, when no sums are held
  // in registers any more.
  unsigned strange[TM * TN] = {};
  {
    // (a maximum that keeps NaNs: two values per instruction)
    float most = 0.f;
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        float block = 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v)
          block = __builtin_elementwise_maximum(block, acc[i][j][v]);
        most = __builtin_elementwise_maximum(most, block);
      }
    if (__builtin_amdgcn_ballot_w64(most != most) != 0) {
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int m = m0 + (wm * TM + j) * 32 + l32;
        const bool cut =
            m < cls.pixels && window_cut(g, cls, pixel_of(m, cls));
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          unsigned bits = 0;
#pragma unroll
          for (int v = 0; v < 16; ++v)
            bits |= acc[i][j][v] != acc[i][j][v] ? 1u << v : 0u;
          strange[j * TN + i] = cut ? bits : 0u;
        }
      }
    }
  }
  auto replace_strange = [&]() {
    unsigned all = 0;
#pragma unroll
    for (int b = 0; b < TM * TN; ++b) all |= strange[b];
    if (__builtin_amdgcn_ballot_w64(all != 0) == 0) return;
    __builtin_amdgcn_s_waitcnt(0);  // the stores of the NaNs
    __builtin_amdgcn_sched_barrier(0);
#pragma nounroll
    for (int b = 0; b < TM * TN; ++b) {
      unsigned bits = 0;
#pragma unroll
      for (int u = 0; u < TM * TN; ++u) bits = u == b ? strange[u] : bits;
      const int j = b / TN, i = b - j * TN;
      const Pixel px = pixel_of(m0 + (wm * TM + j) * 32 + l32, cls);
      while (bits != 0) {
        const int v = __builtin_ctz(bits);
        bits &= bits - 1;
        const int f = n0 + (wn * TN + i) * 32 + 8 * khalf + v + v / 8 * 8;
        if (f >= g.features) continue;
        float sum = exact_sum(src, w, g, cls, px, f);
        if constexpr (kSize == 4) {
          if (bias != nullptr || g.relu != 0)
            sum = bias_act(sum, bias != nullptr ? bias[f] : 0.f, g.relu);
        }
        const int at =
            g.merged != 0
                ? merged_element(g, cls, px, f)
                : ((px.n * g.out_rows + px.y * g.out_step_r + cls.out_r0) *
                       g.out_cols + px.x * g.out_step_c + cls.out_c0) *
                          g.features + f;
        if (at >= 0) dst[at] = static_cast<T>(sum);
      }
    }
  };
  const __amdgpu_buffer_rsrc_t dst_rsrc = make_rsrc(dst, dst_bytes);
  if constexpr (kSize == 4) {
    if (g.merged != 0) {
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int m = m0 + (wm * TM + j) * 32 + l32;
        const Pixel px = pixel_of(m, cls);
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int f = n0 + (wn * TN + i) * 32 + 8 * khalf + v + v / 8 * 8;
            const int at = merged_element(g, cls, px, f);
            // (a variable of its own: a bit_cast of the vector's element takes
            // its first one)
            const float value = acc[i][j][v];
            __builtin_amdgcn_raw_buffer_store_b32(
                __builtin_bit_cast(unsigned, value), dst_rsrc,
                m < cls.pixels && at >= 0 ? at * 4u : kOob, 0, 0);
          }
      }
      replace_strange();
      return;
    }
    if (bias != nullptr || g.relu != 0) {
      const __amdgpu_buffer_rsrc_t bias_rsrc =
          make_rsrc(bias, bias != nullptr ? g.features * 4u : 0u);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int f = n0 + (wn * TN + i) * 32 + 8 * khalf + v + v / 8 * 8;
          const float add = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(bias_rsrc, f * 4u, 0, 0));
#pragma unroll
          for (int j = 0; j < TM; ++j)
            acc[i][j][v] = bias_act(acc[i][j][v], add, g.relu);
        }
    }
  }
  // Features that fill no whole 16-byte pieces (fp32: four, binary16: eight) go
  // out through LDS, block by block, as rows of 32 consecutive features: one
  // store instruction covers two to eight pixels' runs instead of 2 or 4 bytes of
  // 64 pixels each (83x23x23x64 -> 391, 3x3, binary16:
  // 93 -> 47 us; 32x28x28x128 -> 131, 3x3, fp32: 96 -> 92).  Word
  // w of pixel row r lies at w XOR (bits of r), which keeps both the writes of 32
  // rows and the reads along a row off each other's banks.
  const bool by_rows = (g.features & (kPiece<T> - 1)) != 0;
  constexpr int kOutRow = 32 * kSize;
  constexpr int kBlocksPerBuf = STAGE / (32 * kOutRow);
  static_assert(2 * kBlocksPerBuf >= WM * WN,
                "a block of every wave in two buffers of the reduction");
  char* const out_stage =
      wave < kBlocksPerBuf
          ? buf0 + wave * (32 * kOutRow)
          : buf1 + (wave - kBlocksPerBuf) * (32 * kOutRow);
  auto word_at = [&](int row, int word) {
    const int bits = kSize == 4 ? row : row >> 1;
    return reinterpret_cast<unsigned*>(out_stage + row * kOutRow +
                                       (word ^ bits) * 4);
  };
  if (by_rows) __syncthreads();  // every wave is done with the last chunk
  // UNIT: bytes per lane.
  auto store_rows = [&](int n, unsigned at_mine, auto unit) {
    constexpr int UNIT = decltype(unit)::value;
    constexpr int PER_PIXEL = 32 * kSize / UNIT, PIXELS = 64 / PER_PIXEL;
    const int at_lane = lane % PER_PIXEL * UNIT;
    const int f = n + at_lane / kSize;
#pragma unroll 2
    for (int it = 0; it < 32 / PIXELS; ++it) {
      const int row = it * PIXELS + lane / PER_PIXEL;
      const unsigned at = static_cast<unsigned>(
          __shfl(static_cast<int>(at_mine), row));
      const unsigned* const word = word_at(row, at_lane / 4);
      const unsigned off = f < g.features && at != kOob
                               ? at + static_cast<unsigned>(f) * kSize : kOob;
      if constexpr (UNIT == 2) {
        __builtin_amdgcn_raw_buffer_store_b16(
            static_cast<unsigned short>(*word >> (at_lane % 4 * 8)), dst_rsrc,
            off, 0, 0);
      } else if constexpr (UNIT == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(
            *word, dst_rsrc, off, 0, 0);
      } else {
        const uint2v two = {*word, *word_at(row, at_lane / 4 + 1)};
        __builtin_amdgcn_raw_buffer_store_b64(two, dst_rsrc, off, 0, 0);
      }
    }
  };
  // 32-bit words of a block's 16 values of this lane.
  constexpr int kWords = 4 * kSize;
  auto words_of = [&](const float16v& sums, unsigned (&words)[kWords]) {
    if constexpr (kSize == 4) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float value = sums[v];
        words[v] = __builtin_bit_cast(unsigned, value);
      }
    } else {
      half8 lo, hi;
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        lo[v] = static_cast<_Float16>(sums[v]);
        hi[v] = static_cast<_Float16>(sums[8 + v]);
      }
      const uint4v w0 = __builtin_bit_cast(uint4v, lo);
      const uint4v w1 = __builtin_bit_cast(uint4v, hi);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        words[v] = w0[v];
        words[4 + v] = w1[v];
      }
    }
  };
  constexpr int kHalf = kWords / 2;  // words 0 ... kHalf - 1: features f0 ... + 7
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int m = m0 + (wm * TM + j) * 32 + l32;
    const Pixel px = pixel_of(m, cls);
    const int out_y = px.y * g.out_step_r + cls.out_r0;
    const int out_x = px.x * g.out_step_c + cls.out_c0;
    const unsigned at =
        static_cast<unsigned>(((px.n * g.out_rows + out_y) * g.out_cols + out_x) *
                              g.features) * kSize;
    if (by_rows) {
      const unsigned at_mine = m < cls.pixels ? at : kOob;
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        unsigned words[kWords];
        words_of(acc[i][j], words);
#pragma unroll
        for (int v = 0; v < kWords; ++v)
          *word_at(l32, kHalf * khalf + v + v / kHalf * kHalf) = words[v];
        // (LDS operations of a wave are done in order)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int n = n0 + (wn * TN + i) * 32;
        if constexpr (kSize == 4) {
          store_rows(n, at_mine, std::integral_constant<int, 4>{});
        } else {
          if ((g.features & 1) != 0)
            store_rows(n, at_mine, std::integral_constant<int, 2>{});
          else if ((g.features & 3) != 0)
            store_rows(n, at_mine, std::integral_constant<int, 4>{});
          else
            store_rows(n, at_mine, std::integral_constant<int, 8>{});
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      continue;
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int f0 = n0 + (wn * TN + i) * 32 + 8 * khalf;
      const int count = m < cls.pixels ? g.features - f0 : 0;
      const unsigned off = at + static_cast<unsigned>(f0) * kSize;
      unsigned words[kWords];
      words_of(acc[i][j], words);
#pragma unroll
      for (int v = 0; v < kWords / 4; ++v) {
        const int first = kPiece<T> * v + v * 4 / kHalf * 8;
        const uint4v four = {words[4 * v], words[4 * v + 1], words[4 * v + 2],
                             words[4 * v + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(
            four, dst_rsrc, count > first ? off + first * kSize : kOob, 0, 0);
      }
    }
  }
  replace_strange();
}

// Sums the splits of every tile in order and rounds: one float4 -- four
// consecutive features of a pixel -- per lane.
template <typename T, int WM, int WN, int TM, int TN>
__global__ void __launch_bounds__(256)
    gather_reduce_kernel(const float4v* __restrict__ part,
                         const T* __restrict__ src, const T* __restrict__ w,
                         const float* __restrict__ bias, T* __restrict__ dst,
                         Gather g) {
  constexpr unsigned BM = 32 * WM * TM, BN = 32 * WN * TN;
  constexpr unsigned kTileVecs = BM * BN / 4;
  const unsigned at = blockIdx.x * 256 + threadIdx.x;
  const unsigned tile = at / kTileVecs, in = at % kTileVecs;
  if (tile >= g.n_tiles) return;
  const TileOf where = tile_of(tile, g);
  const GatherClass& cls = g.cls[where.cls];
  const unsigned lane = in % 64, v = in / 64 % 4, block = in / 256 % (TN * TM);
  const unsigned wave = in / (256 * TN * TM);
  const unsigned i = block / TM, j = block % TM;
  const int m = where.m * static_cast<int>(BM) +
                static_cast<int>((wave / WN * TM + j) * 32 + lane % 32);
  const int f = where.n * static_cast<int>(BN) +
                static_cast<int>((wave % WN * TN + i) * 32) +
                feature_of_row(8 * v + 4 * (lane / 32));
  if (m >= cls.pixels || f >= g.features) return;
  if (cls.n_chunks == 0 && (g.features & (kPiece<T> - 1)) == 0)
    return;  // stored already
  float4v sum = {0.f, 0.f, 0.f, 0.f};
  const float4v* from = part + at;
#pragma unroll 4
  for (int s = 0; s < g.n_splits; ++s)
    sum += from[static_cast<size_t>(s) * g.n_tiles * kTileVecs];
  const Pixel px = pixel_of(m, cls);
  if ((sum[0] != sum[0] || sum[1] != sum[1] || sum[2] != sum[2] ||
       sum[3] != sum[3]) && window_cut(g, cls, px)) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (sum[e] != sum[e] && f + e < g.features)
        sum[e] = exact_sum(src, w, g, cls, px, f + e);
  }
  if constexpr (sizeof(T) == 4) {
    if (g.merged != 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int to = merged_element(g, cls, px, f + e);
        if (to >= 0) dst[to] = sum[e];
      }
      return;
    }
    if (bias != nullptr || g.relu != 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sum[e] = bias_act(
            sum[e], bias != nullptr && f + e < g.features ? bias[f + e] : 0.f,
            g.relu);
    }
  }
  T* const out =
      dst + (static_cast<size_t>(px.n * g.out_rows + px.y * g.out_step_r +
                                 cls.out_r0) * g.out_cols +
             px.x * g.out_step_c + cls.out_c0) * g.features + f;
  typedef T Four __attribute__((ext_vector_type(4)));
  Four r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = static_cast<T>(sum[e]);
  if ((g.features & 3) == 0) {
    *reinterpret_cast<Four*>(out) = r;
  } else {
    for (int e = 0; e < 4 && f + e < g.features; ++e) out[e] = r[e];
  }
}

struct GatherPlan {
  Gather g;
  bool ok = false;
  int batch = 0;
  size_t src_pixels = 0;
  bool widen = false;       // source channels fill no whole pieces
  size_t out_elems = 0;
  size_t pack_blocks = 0;   // 2 KB blocks of packed filter
  size_t wide_bytes = 0;    // of the widened source
  size_t part_floats = 0;   // of the tiles whose reduction is shared
  int tile = 0;             // index into the tile shapes of the type
  int n_splits = 1;
  double us = 0;            // of the products, by the model of choose_tile
  size_t filter_elems = 0;
  FilterFrom from = kPacked;
  size_t workspace_bytes(bool packs) const {
    return (packs ? pack_blocks * 2048 : 0) + wide_bytes + 4 * part_floats;
  }
};

// Tile shapes, with what one work-group needs per chunk: alone on its CU
// (bound by the time a load takes) and its share of a CU that is full; `split`:
// see kTilesF32.
struct TileShape {
  int pixels, features;
  double alone_us, share_us;
  bool split;
};
constexpr TileShape kTilesF16[] = {
    {256, 128, 0.57, 0.46, false}, {256, 64, 0.34, 0.376, false},
    {128, 128, 0.27, 0.24, false}, {128, 64, 0.245, 0.17, false},
    {128, 32, 0.23, 0.135, false}, {64, 64, 0.22, 0.103, false}};
// (fp32: eight matrix instructions of 64 cycles per chunk and SIMD, in either
// shape, which one wastes fewer columns decides.  128 x 64 and 128 x 128 need
// fewer loads per product but were no faster on any of forty shapes: 17x27x27
// 96 -> 256, 5x5, 158 / 163 us against 162)
// The larger ones split their operands (SPLIT), and a chunk takes `alone_us` and
// `share_us` per work-group on the average CU: the rate hangs on the conversions
// and on power more than on how the tiles fall on compute units.
constexpr TileShape kTilesF32[] = {{128, 32, 0.36, 0.27, false},
                                   {64, 64, 0.36, 0.265, false},
                                   {128, 128, 0.10, 0.88, true},
                                   {128, 64, 0.27, 0.45, true}};
constexpr int kMergedTile = 0;
template <typename T>
struct Tiles;
template <>
struct Tiles<_Float16> {
  static constexpr const TileShape* shapes = kTilesF16;
  static constexpr int count = sizeof(kTilesF16) / sizeof(kTilesF16[0]);
};
template <>
struct Tiles<float> {
  static constexpr const TileShape* shapes = kTilesF32;
  static constexpr int count = sizeof(kTilesF32) / sizeof(kTilesF32[0]);
};
constexpr int kNumCus = 256;
template <typename T>
constexpr int kMaxSplits = sizeof(T) == 4 ? 32 : 16;  // (half the chunk)

int tuned(const char* value, int otherwise) {
  return value != nullptr ? std::atoi(value) : otherwise;
}

// Tile shape and splits of the reduction: the least time by a model of the
// launch, chunks x the fuller of "one chunk after the other" and "every
// work-group's share of its CU", plus what a split reduction adds -- its
// second launch and the partial tiles written and read.  The constants were
// measured; against forced choices the model's was within about 10 % of the
// best on forty shapes from 1x7x7x512 to 16x224x224x64.
template <typename T>
void choose_tile(GatherPlan* plan, bool may_split) {
  const Gather& g = plan->g;
  int pixels = 0;
  double chunks = 0, longest = 0;
  for (int k = 0; k < g.n_classes; ++k) {
    pixels = std::max(pixels, g.cls[k].pixels);
    chunks += g.cls[k].n_chunks;
    longest = std::max(longest, static_cast<double>(g.cls[k].n_chunks));
  }
  double products = 0;  // multiply-adds, in whole chunks
  for (int k = 0; k < g.n_classes; ++k)
    products += static_cast<double>(g.cls[k].pixels) * g.cls[k].n_chunks * 4 *
                kPiece<T> * g.features;
  chunks /= g.n_classes;
  auto tiles_of = [&](const TileShape& t) {
    return static_cast<double>(ceil_div(pixels, t.pixels)) * g.n_classes *
           ceil_div(g.features, t.features);
  };
  double best = 1e30;
  for (int i = 0; i < Tiles<T>::count; ++i) {
    if (g.merged != 0 && i != kMergedTile) continue;
    const TileShape& t = Tiles<T>::shapes[i];
    const double tiles = tiles_of(t);
    // (split operands: from about 2e9 multiply-adds on faster by 10 to 25 % where
    // the estimate is lower; below as often slower, on 80 layers)
    if (t.split && products < 2e9) continue;
    for (int splits = 1; splits <= (may_split ? kMaxSplits<T> : 1); splits *= 2) {
      if (splits > 1 && longest / splits < 4) break;
      const double rounds = std::ceil(tiles * splits / kNumCus);
      const double filled = std::max(0.9, tiles * splits / kNumCus);
      double us =
          t.split ? chunks / longest * std::ceil(longest / splits) *
                            (t.alone_us + t.share_us * filled) + 3.0 * filled
                  : std::max(std::ceil(longest / splits) * t.alone_us,
                             std::ceil(chunks / splits) * rounds * t.share_us) +
                        0.5 * rounds;
      if (splits > 1)
        us += 3.0 + splits * tiles * t.pixels * t.features * 8 /
                        (t.split ? 4.6e6 : 3e6);
      if (us < best) {
        best = us;
        plan->us = us;
        plan->tile = i;
        plan->n_splits = splits;
      }
    }
  }
  plan->tile = tuned(SNN_TUNING_ENV("SNN_HIP_GATHER_TILE"), plan->tile);
  plan->n_splits =
      tuned(SNN_TUNING_ENV("SNN_HIP_GATHER_SPLITS"), plan->n_splits);
  const TileShape& t = Tiles<T>::shapes[plan->tile];
  plan->part_floats =
      plan->n_splits > 1 ? static_cast<size_t>(plan->n_splits * tiles_of(t)) *
                               t.pixels * t.features
                         : 0;
}

// (a workspace may be asked for with parameters that no launch would take)
bool positive(const snn_hip_conv2d_params& p) {
  return p.batch > 0 && p.in_rows > 0 && p.in_cols > 0 && p.channels > 0 &&
         p.features > 0 && p.out_rows > 0 && p.out_cols > 0 &&
         p.window_rows > 0 && p.window_cols > 0 && p.stride_rows > 0 &&
         p.stride_cols > 0 && p.pad_rows >= 0 && p.pad_cols >= 0;
}

template <typename T>
GatherPlan compute_plan(int direction, const snn_hip_conv2d_params& p,
                        bool may_split) {
  constexpr int kE = kPiece<T>;
  GatherPlan plan;
  if (direction != SNN_HIP_FORWARD && direction != SNN_HIP_INPUT_BACKPROP)
    return plan;
  if (!positive(p)) return plan;
  const bool grad = direction == SNN_HIP_INPUT_BACKPROP;
  if (p.window_rows > kMaxWindow || p.window_cols > kMaxWindow) return plan;
  if (grad && p.stride_rows * p.stride_cols > kMaxClasses) return plan;
  Gather& g = plan.g;
  g.src_rows = grad ? p.out_rows : p.in_rows;
  g.src_cols = grad ? p.out_cols : p.in_cols;
  g.out_rows = grad ? p.in_rows : p.out_rows;
  g.out_cols = grad ? p.in_cols : p.out_cols;
  g.channels = grad ? p.features : p.channels;
  g.features = grad ? p.channels : p.features;
  g.cp = (g.channels + kE - 1) / kE;
  g.by_cp = divisor(g.cp);
  g.step_r = grad ? 1 : p.stride_rows;
  g.step_c = grad ? 1 : p.stride_cols;
  g.out_step_r = grad ? p.stride_rows : 1;
  g.out_step_c = grad ? p.stride_cols : 1;
  g.win_rows = p.window_rows;
  g.win_cols = p.window_cols;
  g.mirrored = grad;
  const int strides = p.stride_rows * p.stride_cols;
  // (beyond four channels a class of its own fills more of its matrix rows)
  g.merged = sizeof(T) == 4 && grad && strides > 1 && p.channels <= 4 &&
                     p.channels * strides <= 32 &&
                     p.window_rows >= p.stride_rows &&
                     p.window_cols >= p.stride_cols
                 ? p.channels : 0;
  if (g.merged != 0) g.features = p.channels * strides;
  g.relu = 0;
  // A strided 1x1 window sees one pixel of stride x stride: only those are
  // copied (64x57x57 255 -> 63, stride 2, binary16: 70 -> 30 us).
  g.copy_rows = g.copy_cols = 0;
  if (!grad && g.channels % kE != 0 && strides > 1 && p.window_rows == 1 &&
      p.window_cols == 1 && p.pad_rows == 0 && p.pad_cols == 0 &&
      (p.out_rows - 1LL) * p.stride_rows < p.in_rows &&
      (p.out_cols - 1LL) * p.stride_cols < p.in_cols) {
    g.copy_rows = p.in_rows;
    g.copy_cols = p.in_cols;
    g.copy_step_r = p.stride_rows;
    g.copy_step_c = p.stride_cols;
    g.src_rows = p.out_rows;
    g.src_cols = p.out_cols;
    g.step_r = g.step_c = 1;
  }
  plan.batch = p.batch;
  plan.src_pixels = static_cast<size_t>(p.batch) * g.src_rows * g.src_cols;
  plan.widen = g.channels % kE != 0;
  if (plan.widen) plan.wide_bytes = plan.src_pixels * g.cp * 16;
  plan.out_elems = static_cast<size_t>(p.batch) * g.out_rows * g.out_cols *
                   (grad ? p.channels : p.features);
  if (plan.src_pixels * g.cp * 16 > kMaxBufferBytes ||
      plan.out_elems * sizeof(T) > kMaxBufferBytes)
    return plan;
  g.n_classes = 0;
  if (!grad) {
    GatherClass& c = g.cls[g.n_classes++];
    c.rows = p.out_rows; c.cols = p.out_cols;
    c.off_r = -p.pad_rows; c.off_c = -p.pad_cols;
    c.win_r = p.window_rows; c.win_c = p.window_cols;
    c.out_r0 = 0; c.out_c0 = 0;
    c.tap_r0 = 0; c.tap_rs = 1; c.tap_c0 = 0; c.tap_cs = 1;
  } else if (g.merged != 0) {
    // A block's pixels are first + stride * i + 0 ... stride - 1 along an axis,
    // with padded coordinates stride * (b + i) + 0 ...; tap t of the shared
    // window is source position b + i - (taps - 1) + t and, for member a, filter
    // tap a + stride * (taps - 1 - t).
    auto axis = [](int in, int window, int stride, int pad, int* count,
                   int* first, int* taps, int* off) {
      const int b = pad / stride;
      *first = b * stride - pad;
      *count = (in - 1 + pad) / stride - b + 1;
      *taps = (window + stride - 1) / stride;
      *off = b - (*taps - 1);
    };
    GatherClass& c = g.cls[g.n_classes++];
    axis(p.in_rows, p.window_rows, p.stride_rows, p.pad_rows, &c.rows,
         &c.out_r0, &c.win_r, &c.off_r);
    axis(p.in_cols, p.window_cols, p.stride_cols, p.pad_cols, &c.cols,
         &c.out_c0, &c.win_c, &c.off_c);
    c.tap_r0 = p.stride_rows * (c.win_r - 1);
    c.tap_c0 = p.stride_cols * (c.win_c - 1);
    c.tap_rs = -p.stride_rows;
    c.tap_cs = -p.stride_cols;
  } else {
    // One axis of a class: input positions first, first + stride, ... are
    // reached by taps a, a + stride, ... at source position
    // i + off + (taps - 1 - j) for tap a + stride * j.
    auto axis = [](int a, int in, int window, int stride, int pad, int* count,
                   int* first, int* taps, int* off, int* tap0) {
      *first = ((a - pad) % stride + stride) % stride;
      *count = in > *first ? (in - *first + stride - 1) / stride : 0;
      *taps = window > a ? (window - a + stride - 1) / stride : 0;
      *off = (*first + pad - a) / stride - (*taps - 1);
      *tap0 = a + stride * (*taps - 1);
    };
    for (int a = 0; a < p.stride_rows; ++a)
      for (int b = 0; b < p.stride_cols; ++b) {
        GatherClass c;
        axis(a, p.in_rows, p.window_rows, p.stride_rows, p.pad_rows, &c.rows,
             &c.out_r0, &c.win_r, &c.off_r, &c.tap_r0);
        axis(b, p.in_cols, p.window_cols, p.stride_cols, p.pad_cols, &c.cols,
             &c.out_c0, &c.win_c, &c.off_c, &c.tap_c0);
        c.tap_rs = -p.stride_rows;
        c.tap_cs = -p.stride_cols;
        if (c.rows <= 0 || c.cols <= 0) continue;
        if (c.win_r == 0 || c.win_c == 0) c.win_r = c.win_c = 0;
        g.cls[g.n_classes++] = c;
      }
  }
  const int n_nb = ceil_div(g.features, 32);
  for (int k = 0; k < g.n_classes; ++k) {
    GatherClass& c = g.cls[k];
    c.pixels = p.batch * c.rows * c.cols;
    c.n_chunks = ceil_div(c.win_r * c.win_c * g.cp, 4);
    c.by_win_c = divisor(std::max(c.win_c, 1));
    c.by_rows = divisor(c.rows);
    c.by_cols = divisor(c.cols);
    c.pack_block = static_cast<unsigned>(plan.pack_blocks);
    plan.pack_blocks += static_cast<size_t>(n_nb) * c.n_chunks;
  }
  plan.filter_elems = static_cast<size_t>(p.window_rows) * p.window_cols *
                      p.channels * p.features;
  if (!plan.widen && g.merged == 0 &&
      plan.filter_elems * sizeof(T) <= kMaxBufferBytes / 2) {
    if (grad)
      plan.from = kInPlace;
    else if (sizeof(T) == 4 && p.features % 4 == 0)
      plan.from = kRows;
  }
  choose_tile<T>(&plan, may_split);
  plan.ok = plan.pack_blocks * 2048 <= kMaxBufferBytes / 2 && g.n_classes > 0;
  return plan;
}

template <typename T>
const GatherPlan& make_plan(int direction, const snn_hip_conv2d_params& p,
                            bool may_split = true) {
  thread_local PlanCache<GatherPlan> cache;
  return cache.get(p, static_cast<unsigned>(direction) * 2 + may_split,
                   [&] { return compute_plan<T>(direction, p, may_split); });
}

// A launch's operands: the source as whole pieces, the filter as `from` says.
template <typename T>
struct GatherOperands {
  const T* src;
  const T* filter;
  const T* caller_filter;
  const float* bias;
  T* dst;
  float* part;
  FilterFrom from;
};

template <typename T, int WM, int WN, int TM, int TN, bool UNIFORM, int FROM,
          bool SPLIT>
void launch_kernel(const GatherOperands<T>& ops, const GatherPlan& plan,
                   const Gather& g, hipStream_t stream) {
  const unsigned n_groups = g.n_tiles * static_cast<unsigned>(g.n_splits);
  const unsigned src_bytes = static_cast<unsigned>(plan.src_pixels * g.cp * 16);
  const unsigned filter_bytes = static_cast<unsigned>(
      FROM == kPacked ? plan.pack_blocks * 2048
                      : plan.filter_elems * sizeof(T));
  const unsigned dst_bytes = static_cast<unsigned>(plan.out_elems * sizeof(T));
  KernelTimer timer(stream);
  hipLaunchKernelGGL((conv_gather_kernel<T, WM, WN, TM, TN, UNIFORM, FROM, SPLIT>),
                     dim3(n_groups), dim3(64 * WM * WN), 0, stream, ops.src,
                     ops.filter, ops.caller_filter, ops.bias, ops.dst, ops.part,
                     g, src_bytes, filter_bytes, dst_bytes, n_groups);
}

template <typename T, int WM, int WN, int TM, int TN, bool SPLIT = false>
void launch_tile(const GatherOperands<T>& ops, const GatherPlan& plan,
                 bool relu, hipStream_t stream) {
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  Gather g = plan.g;
  g.relu = relu;
  g.n_tiles_n = ceil_div(g.features, BN);
  int pixels = 0;
  for (int k = 0; k < g.n_classes; ++k)
    pixels = std::max(pixels, g.cls[k].pixels);
  g.n_tiles = static_cast<unsigned>(ceil_div(pixels, BM)) *
              static_cast<unsigned>(g.n_classes * g.n_tiles_n);
  g.n_splits = plan.n_splits;
  // (the tiles of a class are this many work-groups apart)
  const unsigned apart =
      static_cast<unsigned>(g.n_classes * g.n_tiles_n * g.n_splits);
  g.round_shift = std::max(0, 5 - __builtin_ctz(apart));
  g.turn = g.round_shift > 0 && (g.n_classes & (g.n_classes - 1)) == 0;
  if constexpr (sizeof(T) == 4) {
    // (scalar tap bookkeeping where the tap arithmetic of every lane would take
    // vector instructions from the splitting: 3 % of the time)
    const bool uniform = SPLIT && g.cp % 4 == 0;
    if (uniform && ops.from == kInPlace)
      launch_kernel<T, WM, WN, TM, TN, SPLIT, kInPlace, SPLIT>(ops, plan, g, stream);
    else if (uniform && ops.from == kRows)
      launch_kernel<T, WM, WN, TM, TN, SPLIT, kRows, SPLIT>(ops, plan, g, stream);
    else if (ops.from == kInPlace)
      launch_kernel<T, WM, WN, TM, TN, false, kInPlace, SPLIT>(ops, plan, g, stream);
    else if (ops.from == kRows)
      launch_kernel<T, WM, WN, TM, TN, false, kRows, SPLIT>(ops, plan, g, stream);
    else
      launch_kernel<T, WM, WN, TM, TN, false, kPacked, SPLIT>(ops, plan, g, stream);
  } else {
    const bool uniform = g.cp % 4 == 0;
    if (ops.from == kInPlace && uniform)
      launch_kernel<T, WM, WN, TM, TN, true, kInPlace, SPLIT>(ops, plan, g, stream);
    else if (ops.from == kInPlace)
      launch_kernel<T, WM, WN, TM, TN, false, kInPlace, SPLIT>(ops, plan, g, stream);
    else if (uniform)
      launch_kernel<T, WM, WN, TM, TN, true, kPacked, SPLIT>(ops, plan, g, stream);
    else
      launch_kernel<T, WM, WN, TM, TN, false, kPacked, SPLIT>(ops, plan, g, stream);
  }
  if (g.n_splits > 1)
    hipLaunchKernelGGL((gather_reduce_kernel<T, WM, WN, TM, TN>),
                       dim3(g.n_tiles * (BM * BN / 1024)), dim3(256), 0, stream,
                       reinterpret_cast<const float4v*>(ops.part), ops.src,
                       ops.caller_filter, ops.bias, ops.dst, g);
}

// Returns -1 when there is no room for its temporaries.
template <typename T>
int launch_gather(const GatherPlan& plan, const T* input, const T* filter,
                  T* output, T* workspace, size_t workspace_elems,
                  const float* bias, bool relu, hipStream_t stream) {
  const Gather& g = plan.g;
  const FilterFrom from =
      (reinterpret_cast<uintptr_t>(filter) & 15u) == 0 ? plan.from : kPacked;
  const size_t need = plan.workspace_bytes(from == kPacked);
  char* packed = reinterpret_cast<char*>(workspace);
  const bool temporary =
      need != 0 &&
      (workspace == nullptr || workspace_elems < ceil_div(need, sizeof(T)) ||
       (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0);
  if (temporary) {
    void* ptr = nullptr;
    if (temp_malloc_async(&ptr, need, stream) != hipSuccess) {
      (void)hipGetLastError();
      return -1;
    }
    packed = static_cast<char*>(ptr);
  }
  // (every part is a multiple of 16 bytes)
  const size_t pack_blocks = from == kPacked ? plan.pack_blocks : 0;
  T* const wide = reinterpret_cast<T*>(packed + pack_blocks * 2048);
  const unsigned pack_lanes = static_cast<unsigned>(pack_blocks * 128);
  const unsigned pack_groups = ceil_div(pack_lanes, 256u);
  const unsigned pieces =
      plan.widen ? static_cast<unsigned>(plan.src_pixels * g.cp) : 0u;
  const unsigned groups = pack_groups + ceil_div(pieces, 256u);
  if (groups > 0)
    hipLaunchKernelGGL(gather_prepare_kernel<T>, dim3(groups), dim3(256), 0,
                       stream, filter, reinterpret_cast<T*>(packed), g,
                       pack_lanes, pack_groups, input, wide, pieces);
  const GatherOperands<T> ops = {
      plan.widen ? wide : input,
      from == kPacked ? reinterpret_cast<const T*>(packed) : filter,
      filter,
      bias,
      output,
      reinterpret_cast<float*>(packed + pack_blocks * 2048 + plan.wide_bytes),
      from};
  if constexpr (sizeof(T) == 4) {
    switch (plan.tile) {
      case 0: launch_tile<T, 4, 1, 1, 1>(ops, plan, relu, stream); break;
      case 1: launch_tile<T, 2, 2, 1, 1>(ops, plan, relu, stream); break;
      case 2: launch_tile<T, 2, 2, 2, 2, true>(ops, plan, relu, stream); break;
      default: launch_tile<T, 2, 2, 2, 1, true>(ops, plan, relu, stream);
    }
  } else {
    switch (plan.tile) {
      case 0: launch_tile<T, 2, 2, 4, 2>(ops, plan, relu, stream); break;
      case 1: launch_tile<T, 4, 1, 2, 2>(ops, plan, relu, stream); break;
      case 2: launch_tile<T, 2, 2, 2, 2>(ops, plan, relu, stream); break;
      case 3: launch_tile<T, 2, 2, 2, 1>(ops, plan, relu, stream); break;
      case 4: launch_tile<T, 4, 1, 1, 1>(ops, plan, relu, stream); break;
      default: launch_tile<T, 2, 2, 1, 1>(ops, plan, relu, stream);
    }
  }
  const hipError_t err = hipGetLastError();
  if (temporary) temp_free_async(packed, stream);
  if (err != hipSuccess) return report_hip_error(err, "conv_gather_kernel");
  return SNN_HIP_OK;
}

// The input gradient of a stride-1 convolution as a forward convolution of
// dY: channels and features trade places, padding becomes window - 1 - pad.
bool as_forward_of_dy(const snn_hip_conv2d_params& p,
                      snn_hip_conv2d_params* q) {
  if (p.stride_rows != 1 || p.stride_cols != 1) return false;
  if (p.pad_rows > p.window_rows - 1 || p.pad_cols > p.window_cols - 1)
    return false;
  *q = p;
  q->channels = p.features;
  q->features = p.channels;
  q->in_rows = p.out_rows;
  q->in_cols = p.out_cols;
  q->out_rows = p.in_rows;
  q->out_cols = p.in_cols;
  q->pad_rows = p.window_rows - 1 - p.pad_rows;
  q->pad_cols = p.window_cols - 1 - p.pad_cols;
  return true;
}

// 1x1, stride 1, no padding: a plain row-major GEMM over the pixels, X * W for
// the forward and dY * W^T for the gradient.
bool is_pixel_gemm(const snn_hip_conv2d_params& p) {
  return p.window_rows == 1 && p.window_cols == 1 && p.stride_rows == 1 &&
         p.stride_cols == 1 && p.pad_rows == 0 && p.pad_cols == 0 &&
         p.out_rows == p.in_rows && p.out_cols == p.in_cols &&
         static_cast<size_t>(p.batch) * p.in_rows * p.in_cols <=
             static_cast<size_t>(INT_MAX);
}
bool is_short_gemm(int direction, const snn_hip_conv2d_params& p) {
  const bool grad = direction == SNN_HIP_INPUT_BACKPROP;
  return is_pixel_gemm(p) &&
         gemm_short_f16_wanted(p.batch * p.in_rows * p.in_cols,
                               grad ? p.features : p.channels,
                               grad ? p.channels : p.features, grad);
}
bool is_rows_gemm(int direction, const snn_hip_conv2d_params& p) {
  if (!is_pixel_gemm(p)) return false;
  const int m = p.batch * p.in_rows * p.in_cols;
  return direction == SNN_HIP_FORWARD
             ? gemm_rows_f16_supports(m, p.channels, p.features)
             : gemm_nt_f16_supports(m, p.features, p.channels);
}

// What a binary16 launch takes on each of the kernels that take any stride, in
// us back to back.  Fitted to 2060 random layers of 1e4 to 1.5e9 multiply-adds
// (windows 1 to 7, strides 1 to 3, 3 to 1024 channels and features): the middle
// half of the estimates is within 5 % for the gathering kernel and 8 % for the
// other two.  They meet where launches are short.  The gathering one has
// up to two launches in front of its products, the filter's pack and the copy to
// whole pieces (16x55x41 16 -> 12, 1x1: general 5.6, gathering 8.8; 2x24x24
// 52 -> 20, 1x1 stride 2: 5.4 and 7.9), and where the caller brings no workspace a
// call with a temporary takes 22 us of host time, which only longer kernels hide.
constexpr double kNever = 1e30;
constexpr double kTemporaryUs = 22.0;

struct Products {
  double pixels, columns, reduced, macs;
};
Products products_of(int direction, const snn_hip_conv2d_params& p) {
  const bool grad = direction == SNN_HIP_INPUT_BACKPROP;
  const double taps = static_cast<double>(p.window_rows) * p.window_cols;
  const double y = static_cast<double>(p.batch) * p.out_rows * p.out_cols;
  Products r;
  r.pixels = grad ? static_cast<double>(p.batch) * p.in_rows * p.in_cols : y;
  r.columns = grad ? p.channels : p.features;
  r.reduced = taps * (grad ? p.features : p.channels);
  r.macs = y * taps * p.channels * p.features;
  return r;
}

double gather_f16_us(const GatherPlan& plan, bool packs, bool temporary) {
  const double bytes = static_cast<double>(plan.wide_bytes) +
                       (packs ? plan.pack_blocks * 2048.0 : 0.0);
  const double us = 4.0 + 0.8 * plan.us +
                    (bytes > 0 ? 3.0 + bytes / 1.5e6 : 0.0) +
                    plan.out_elems / 2.5e6;
  return temporary ? std::max(us, kTemporaryUs) : us;
}

double general_f16_us(const Products& r) {
  const double chunks = std::ceil(r.reduced / 32);
  const double rounds =
      std::ceil(r.pixels / 64) * std::ceil(r.columns / 64) / kNumCus;
  return 3.0 + 0.9 * chunks + (0.45 * chunks + 0.4) * rounds +
         r.pixels * r.columns / 6e6;
}

// One lane per output, either type.  A gradient's lanes read the filter columns of
// as many channels: with features in multiples of 4 those fall into few banks,
// and other kernels are there.
double direct_us(int direction, const snn_hip_conv2d_params& p,
                 const Products& r, bool half) {
  const double outputs = r.pixels * r.columns;
  if (r.macs >= double(1 << 24)) return kNever;
  if (direction == SNN_HIP_FORWARD)
    return 2.9 + 0.09 * r.reduced + (0.15 * r.reduced + 2.7) * outputs / 1e6;
  const double loop = static_cast<double>(p.features) *
                      ceil_div(p.window_rows, p.stride_rows) *
                      ceil_div(p.window_cols, p.stride_cols);
  const bool small = half && r.reduced <= 32 && outputs <= (1 << 16);
  if (p.features % 4 == 0 || loop > 64 || (small && loop > 16))
    return small ? 5.5 : kNever;
  return (3.1 + 0.05 * loop +
          (half ? 0.11 * loop + 3.3 : 0.06 * loop + 4.3) * outputs / 1e6 +
          0.6 * p.window_rows * p.window_cols /
              (p.stride_rows * p.stride_cols)) *
         (loop <= 16 ? 1.0 : 2.0);  // (longer ones up to three times that)
}

// The forward convolution the LDS-tile kernel would run, if it is wanted.
bool rowtile_params(int direction, const snn_hip_conv2d_params& p,
                    snn_hip_conv2d_params* q) {
  if (direction == SNN_HIP_FORWARD)
    *q = p;
  else if (!as_forward_of_dy(p, q))
    return false;
  double other_us = kNever;
  if (p.window_rows == 3 && p.window_cols == 3 && p.stride_rows == 1 &&
      p.stride_cols == 1 && p.channels % 64 == 0 && p.features % 64 == 0) {
    const GatherPlan& plan = make_plan<_Float16>(direction, p);
    // (the estimate was fitted to shorter layers: 13x198x148 256 -> 64, no padding,
    // takes 227 us there)
    const bool longer = products_of(direction, p).macs > 1.5e9;
    if (plan.ok)
      other_us = gather_f16_us(plan, plan.from == kPacked, false) *
                 (longer ? 1.2 : 1.0);
  }
  return conv2d_rowtile_f16_wanted(*q, other_us);
}

// The same in fp32: this kernel, and the implicit-GEMM one for counts in
// multiples of 4 and stride 1 (or forward), whose shared reductions meet through
// atomics after a launch that clears the output.  (Half of 270 and of 970 layers
// within 5 and 10 %.)
double gather_f32_us(const GatherPlan& plan, bool packs, bool temporary) {
  const double bytes = static_cast<double>(plan.wide_bytes) +
                       (packs ? plan.pack_blocks * 2048.0 : 0.0);
  const double us = 4.4 + 0.87 * plan.us +
                    (bytes > 0 ? 2.9 + bytes / 1.8e6 : 0.0) +
                    plan.out_elems / 5.2e6;
  return temporary ? std::max(us, kTemporaryUs) : us;
}

double igemm_f32_us(const Products& r) {
  const double chunks = std::ceil(r.reduced / 32);
  const double tiles = std::ceil(r.pixels / 64) * std::ceil(r.columns / 64);
  const double splits =
      std::max(1.0, std::min(std::floor(640 / tiles), std::floor(chunks / 2)));
  const bool shared = splits > 1;
  return 4.1 + 0.65 * tiles * chunks / kNumCus +
         0.25 * std::ceil(chunks / splits) + (shared ? 3.5 : 0.0) +
         r.pixels * r.columns * (shared ? 2 : 1) / 2.3e6;
}

bool stream_captures(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) == hipSuccess)
    return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

}  // namespace

namespace {

bool gather_tile_f16(int direction, const snn_hip_conv2d_params& p,
                     GatherTile* tile) {
  snn_hip_conv2d_params q;
  if (is_rows_gemm(direction, p) || rowtile_params(direction, p, &q))
    return false;
  const GatherPlan& plan = make_plan<_Float16>(direction, p);
  if (!plan.ok) return false;
  const Products r = products_of(direction, p);
  if (std::min(conv2d_general_f16_supports(direction, p) ? general_f16_us(r)
                                                         : kNever,
               direct_us(direction, p, r, true)) <
      gather_f16_us(plan, plan.from == kPacked, false))
    return false;
  *tile = {kTilesF16[plan.tile].pixels, kTilesF16[plan.tile].features,
           plan.n_splits};
  return true;
}

}  // namespace

bool conv2d_gather_tile_f16(int direction, const snn_hip_conv2d_params& p,
                            GatherTile* tile) {
  return !is_short_gemm(direction, p) && gather_tile_f16(direction, p, tile);
}

int conv2d_rowtile_form_f16(int direction, const snn_hip_conv2d_params& p) {
  snn_hip_conv2d_params q;
  return !is_short_gemm(direction, p) && !is_rows_gemm(direction, p) &&
                 rowtile_params(direction, p, &q)
             ? conv2d_rowtile_f16_buffers(q) : 0;
}

size_t conv2d_f16_workspace_halves(int direction,
                                   const snn_hip_conv2d_params& p) {
  snn_hip_conv2d_params q;
  if (!is_rows_gemm(direction, p) && rowtile_params(direction, p, &q))
    return static_cast<size_t>(p.window_rows) * p.window_cols * p.channels *
           p.features;
  GatherTile tile;
  // (that of a short product, too, which takes it when an operand is not 16-byte
  // aligned)
  if (!gather_tile_f16(direction, p, &tile)) return 0;
  const GatherPlan& plan = make_plan<_Float16>(direction, p);
  // (with room for the packed filter also where the gradient's is read in
  // place, for one that is not 16-byte aligned; that of a 1x1 layer would take
  // a temporary)
  const bool packs =
      plan.from == kPacked || p.window_rows > 1 || p.window_cols > 1;
  return plan.workspace_bytes(packs) / 2;
}

int launch_conv2d_f16(int direction, const _Float16* input,
                      const _Float16* filter, _Float16* output,
                      const snn_hip_conv2d_params& p, _Float16* workspace,
                      size_t workspace_elems, hipStream_t stream,
                      double otherwise_us) {
  auto aligned = [](const void* ptr) {
    return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0;
  };
  const bool both_aligned = aligned(input) && aligned(filter);
  if (aligned(output) && both_aligned && is_short_gemm(direction, p)) {
    const bool grad = direction == SNN_HIP_INPUT_BACKPROP;
    return launch_gemm_short_f16(input, filter, output,
                                 p.batch * p.in_rows * p.in_cols,
                                 grad ? p.features : p.channels,
                                 grad ? p.channels : p.features, grad, stream);
  }
  if (aligned(output) && is_rows_gemm(direction, p) && both_aligned) {
    const int m = p.batch * p.in_rows * p.in_cols;
    return direction == SNN_HIP_FORWARD
               ? launch_gemm_rows_f16(input, filter, output, m, p.channels,
                                      p.features, stream)
               : launch_gemm_nt_f16(input, filter, output, m, p.features,
                                    p.channels, stream);
  }
  snn_hip_conv2d_params q;
  if (aligned(output) && rowtile_params(direction, p, &q) && both_aligned) {
    const size_t need = static_cast<size_t>(p.window_rows) * p.window_cols *
                        p.channels * p.features;
    _Float16* packed = workspace;
    const bool temporary = workspace == nullptr || workspace_elems < need ||
                           !aligned(workspace);
    if (temporary) {
      // An input gradient needs none on the gathering kernel, which reads its filter
      // in place: recorded launches run there, and those whose temporary cannot be
      // had.
      const GatherPlan& whole = make_plan<_Float16>(direction, p, false);
      const bool without =
          whole.ok && whole.workspace_bytes(whole.from == kPacked) == 0;
      void* ptr = nullptr;
      if ((without && stream_captures(stream)) ||
          temp_malloc_async(&ptr, need * sizeof(_Float16), stream) !=
              hipSuccess) {
        if (!without) return SNN_HIP_ALLOCATION_PROBLEM;
        (void)hipGetLastError();
        return launch_gather<_Float16>(whole, input, filter, output, nullptr, 0,
                                       nullptr, false, stream);
      }
      packed = static_cast<_Float16*>(ptr);
    }
    const int status =
        launch_conv2d_rowtile_f16(input, filter, output, q, packed, stream,
                                  direction == SNN_HIP_INPUT_BACKPROP);
    if (temporary) temp_free_async(packed, stream);
    return status;
  }
  const Products r = products_of(direction, p);
  const GatherPlan* plan = &make_plan<_Float16>(direction, p);
  const bool packs = plan->from == kPacked || !aligned(filter);
  const size_t room = workspace != nullptr && aligned(workspace)
                          ? workspace_elems * sizeof(_Float16) : 0;
  bool able = plan->ok && aligned(output) && (plan->widen || aligned(input));
  bool temporary = able && plan->workspace_bytes(packs) > room;
  // (where the gathering kernel does not apply, large launches are faster
  // through fp32 copies: 2x64x64x64 -> 64, 13x13 stride 2: 53 / 330 us)
  bool general = both_aligned && conv2d_general_f16_supports(direction, p) &&
                 (direction == SNN_HIP_INPUT_BACKPROP || aligned(output)) &&
                 (able || r.macs < double(1 << 24));
  if (temporary) {
    const GatherPlan& whole = make_plan<_Float16>(direction, p, false);
    const bool whole_temporary = whole.workspace_bytes(packs) > room;
    if (stream_captures(stream)) {
      // A launch that is recorded without room for the packed filter or the
      // copy keeps its reduction whole, or takes a kernel that needs no
      // temporary.  (Layers of 64 channels and large ones with counts that no
      // other kernel takes have only kernels with temporaries, or slow ones.)
      plan = &whole;
      temporary = whole_temporary;
      const bool other = otherwise_us < kNever || r.macs < double(1 << 24) ||
                         (general && (direction == SNN_HIP_INPUT_BACKPROP ||
                                      p.channels % 64 != 0));
      able = !temporary || !other;
    } else if (gather_f16_us(whole, packs, whole_temporary) <
               gather_f16_us(*plan, packs, true)) {
      plan = &whole;
      temporary = whole_temporary;
    }
  }
  const double general_us = general ? general_f16_us(r) : kNever;
  const double one_lane_us = direct_us(direction, p, r, true);
  const double gather_us =
      able ? gather_f16_us(*plan, packs, temporary) : kNever;
  if (std::min(otherwise_us, one_lane_us) < std::min(general_us, gather_us))
    return -1;
  if (gather_us <= general_us && able) {
    const int rc = launch_gather<_Float16>(*plan, input, filter, output,
                                           workspace, workspace_elems, nullptr,
                                           false, stream);
    if (rc >= 0) return rc;
  }
  return general ? launch_conv2d_general_f16(direction, input, filter, output,
                                             p, stream)
                 : -1;
}

namespace {

// The kernels with the input rows in LDS take 6 us and 55 multiply-adds per ns at
// their best; tiles with split operands are faster on layers that fill the
// compute units with them.
bool split_beats_rows(int direction, const snn_hip_conv2d_params& p,
                      double macs) {
  const GatherPlan& plan = make_plan<float>(direction, p);
  return plan.ok && kTilesF32[plan.tile].split &&
         gather_f32_us(plan, plan.from == kPacked, false) < 6 + macs / 55e6;
}

// Where the gathering kernel is faster than the other fp32 kernels behind the
// Tiled / Im2col / Matmul tags (times: there / here).
// With a bias and activation (`fused`) those kernels that do not add them on the
// way are followed by a launch of 2 us.  `over_rows`: also in place of the kernels
// with the input rows in LDS, which need no temporary.
bool gather_f32_wanted(int direction, const snn_hip_conv2d_params& p, bool fused,
                       bool over_rows) {
  if (direction == SNN_HIP_FILTER_BACKPROP) return false;
  if (const char* const env = SNN_TUNING_ENV("SNN_HIP_GATHER_F32"))
    return std::atoi(env) != 0;
  const bool grad = direction == SNN_HIP_INPUT_BACKPROP;
  const bool strided = p.stride_rows > 1 || p.stride_cols > 1;
  const long long products = static_cast<long long>(p.window_rows) *
                             p.window_cols * (grad ? p.features : p.channels);
  const double macs = static_cast<double>(p.batch) * p.out_rows * p.out_cols *
                      p.window_rows * p.window_cols * p.channels * p.features;
  const double outputs =
      grad ? static_cast<double>(p.batch) * p.in_rows * p.in_cols * p.channels
           : static_cast<double>(p.batch) * p.out_rows * p.out_cols * p.features;
  // One short loop per output (14x14x33 -> 64, 1x1: 5.3 / 17.8 us).
  if (products <= 64 && outputs <= (1 << 16)) return false;
  // Features of no whole piece: a short loop per output as well, where the
  // filter's pack and the copy would be launches of their own (13x15x19 8 -> 135,
  // 1x1 stride 2: 4.3 / 7.9; gradient of 8x21x21 24 <- 2, 2x2: 4.4 / 7.9; but
  // 24x39x39 50 -> 6, 1x1: 17.2 / 15.5).  The estimate of this kernel's time is
  // within 5 % for half of 262 random layers.
  if (p.features % 4 != 0) {
    const GatherPlan& plan = make_plan<float>(direction, p);
    if (plan.ok &&
        direct_us(direction, p, products_of(direction, p), false) +
                (fused ? 2.0 : 0.0) <
            gather_f32_us(plan, true, false))
      return false;
  }
  // At most one 64 x 64 tile per compute unit and a short reduction in whole
  // pieces: latencies are all there is, and those are shorter there (25x14x18
  // 56 -> 424, 1x1 stride 2: 4.8 / 6.3; 11x14x10 24 -> 88, 1x1: 4.2 / 5.5; gradient
  // of 30x30 441 <- 52, 1x1: 4.7 / 6.3; 0.89 of the time in the middle of 185
  // random layers, four of them up to 9 % slower; but with bias and ReLU 8.0 /
  // 6.0 and 6.2 / 5.2).
  const double tiles = std::ceil(outputs / (grad ? p.channels : p.features) / 64) *
                       ceil_div(grad ? p.channels : p.features, 64);
  if (!fused && p.features % 4 == 0 &&
      (grad ? !strided : p.channels % 4 == 0) && products <= 96 && tiles <= kNumCus)
    return false;
  // Few outputs of a long reduction meet through atomics there, in one pass less
  // (2x19x14 720 -> 80, 3x3 stride 2: 12.5 / 13.7 us; 4x14x14 144 -> 224, 5x5,
  // 24 / 26 and its gradient 24 / 30; but 3x14x14 192 <- 128, 3x3, 12.7 / 12.0).
  const bool whole = p.channels % 4 == 0 && p.features % 4 == 0;
  if (whole && (!grad || !strided) &&
      products >= (grad ? 2000 : 3000) && outputs < (1 << 18))
    return false;
  // 1x1, stride 1: plain products.  The kernels for these want reductions of
  // whole chunks of 32, and tiles of 64 columns that are not mostly padding:
  // 15x213x277 16 -> 84 120 / 101 us, its gradient 126 / 91; 3x201x151
  // 288 -> 80 65 / 55; but 32x56x56 256 -> 64 33 / 41 and 32 / 47.
  const bool plain = p.window_rows == 1 && p.window_cols == 1 && !strided &&
                     p.pad_rows == 0 && p.pad_cols == 0 &&
                     p.out_rows == p.in_rows && p.out_cols == p.in_cols;
  const int reduced = grad ? p.features : p.channels;
  const int columns = grad ? p.channels : p.features;
  if (plain && p.features % 4 == 0 && reduced % 32 == 0) {
    const int padded = (columns + 63) / 64 * 64;
    return macs >= double(1 << 29) && 5 * (padded - columns) > padded;
  }
  if (!grad) {
    if (p.features % 4 != 0) return true;  // nothing else but copies takes it
    // The source is copied to whole pieces first: 5x14x10 166 -> 96, 3x3,
    // 67 / 15 us; 18x168x218 3 -> 32, 7x7 stride 2, 48 / 37; but
    // 8x224x224 3 -> 64, 3x3, 38 / 45 and 3x186x186 3 -> 48, 7x7, 13 / 15.
    // A 1x1 window reads no more than the copy does: 25x43x43 454 -> 176 123 /
    // 115 us, but 8x56x56 257 -> 64 21 / 30, 14x156x156 922 -> 32, stride 2,
    // 151 / 205.
    if (p.channels % 4 != 0 && p.window_rows == 1 && p.window_cols == 1 &&
        p.features <= 128)
      return false;
    if (p.channels % 4 != 0)
      return !conv2d_stem_supports(p) &&
             (products >= 200 || (products >= 100 && macs >= double(1 << 29)));
    // 27x27x96 -> 256, 5x5, at batch 17: 144 / 158 us on the rows-in-LDS
    // kernel; where that does not apply 16x28x28 192 -> 96 146 / 115,
    // 13x95x95 208 -> 28, 3x3, 280 / 140, 64x28x28 32 -> 32 60 / 35.
    if (conv2d_small_supports(p)) return false;
    return !(conv2d_rowtile_supports(p) || conv2d_rowsplit_supports(p)) ||
           (over_rows && split_beats_rows(direction, p, macs));
  }
  if (conv2d_stem_input_backprop_supports(p)) return false;
  if (strided && p.channels <= 4)  // merged classes
    // 37x104x104 3 <- 58, 7x7 stride 2, 1570 / 88 us, 7x111x144 3 <- 36, 3x3,
    // 61 / 12; but 112x112 3 <- 32 at batch 1 8.6 / 11.7 (the filter's pack).
    return macs >= double(1 << 23);
  // (products of dY and the filter per output pixel, gathered: 8x224x224
  // 3 <- 64, 3x3, 66 / 148 us; but 8x64x64 8 <- 32 15.6 / 10.4)
  if (p.channels < 16 && p.features % 32 == 0) return macs < double(1 << 27);
  // (16x28x28 192 <- 96, 5x5, 109 / 118 us and 48 <- 64, 7x7, 58 / 67 on tiles
  // of 64 x 64, where those compute no more columns than tiles of 32 would)
  if (!strided && p.features % 32 == 0 && (p.channels + 31) / 32 % 2 == 0 &&
      macs >= double(1 << 30))
    return over_rows && split_beats_rows(direction, p, macs);
  snn_hip_conv2d_params q;
  if (as_forward_of_dy(p, &q) &&
      (conv2d_rowtile_supports(q) || conv2d_rowsplit_supports(q)))
    return over_rows && split_beats_rows(direction, p, macs);
  // 32x56x56 128 <- 128, 3x3 stride 2, 140 / 92 us; 256 <- 512, 1x1 stride 2,
  // 95 / 90; 17x27x27 96 <- 256, 5x5, 178 / 160; 5x82x107 16 <- 75 129 / 68.
  return true;
}

}  // namespace

bool conv2d_gather_f32_wanted(int direction, const snn_hip_conv2d_params& p,
                              bool fused) {
  return gather_f32_wanted(direction, p, fused, true);
}

namespace {

// Into how many a launch of the implicit-GEMM kernel divides its reductions.
double igemm_splits(const Products& r) {
  const double tiles = std::ceil(r.pixels / 64) * std::ceil(r.columns / 64);
  const double chunks = std::ceil(r.reduced / 32);
  return tiles < 640 ? std::max(1.0, std::min(std::ceil(2048 / tiles),
                                              std::floor(chunks / 8)))
                     : 1.0;
}

// Whether an input gradient that is not for the kernels before it multiplies dY by the
// whole filter per output pixel and folds the taps (the launch's own rule).
bool folds_taps(int direction, const snn_hip_conv2d_params& p) {
  return direction == SNN_HIP_INPUT_BACKPROP && p.channels < 16 &&
         p.features % 32 == 0 && !conv2d_stem_input_backprop_supports(p);
}

}  // namespace

// Fitted to a thousand random layers, from below: the fp32 instruction rounds at every
// few products, 1.2e-8 per root of a sum's; of tiles of three bfloat16 parts the
// gradients are off by more than the forward convolutions, 5.0e-9 and 4.5e-9.
double conv2d_gemm_f32_error2(int direction, const snn_hip_conv2d_params& p) {
  const Products r = products_of(direction, p);
  const auto fp32 = [&](double sums) {
    return 0.3e-14 + 135e-18 * r.reduced / sums;
  };
  if (conv2d_gather_f32_wanted(direction, p, false)) {
    const GatherPlan& plan = make_plan<float>(direction, p);
    if (plan.ok && kTilesF32[plan.tile].split)
      return direction == SNN_HIP_FORWARD
                 ? 20e-18 * r.reduced / plan.n_splits
                 : 0.25e-14 + 25e-18 * r.reduced / plan.n_splits;
    if (plan.ok) return fp32(plan.n_splits);
  }
  snn_hip_conv2d_params q = p;
  if (direction == SNN_HIP_FORWARD || as_forward_of_dy(p, &q)) {
    if (conv2d_rowtile_supports(q)) return fp32(1);
    if (conv2d_rowsplit_supports(q)) return fp32(8);  // waves with sums of their own
  }
  return fp32(folds_taps(direction, p)
                  ? static_cast<double>(p.window_rows) * p.window_cols
                  : igemm_splits(r));
}

double conv2d_gemm_f32_us(int direction, const snn_hip_conv2d_params& p) {
  if (conv2d_gather_f32_wanted(direction, p, false)) {
    const GatherPlan& plan = make_plan<float>(direction, p);
    // (tiles of three parts were under that time on 40 of 42 layers)
    const double more = !kTilesF32[plan.tile].split ? 1.0
                        : plan.n_splits > 1         ? 1.05
                                                    : 1.15;
    if (plan.ok) return more * gather_f32_us(plan, plan.from == kPacked, false);
  }
  const Products r = products_of(direction, p);
  snn_hip_conv2d_params q = p;
  if ((direction == SNN_HIP_FORWARD || as_forward_of_dy(p, &q)) &&
      (conv2d_rowtile_supports(q) || conv2d_rowsplit_supports(q)))
    return 6 + r.macs / 55e6;
  // Both fitted to random layers with windows of 2x2 to 9x9, by the tiles, chunks and
  // splits of the launch: nine of ten within a tenth (412 layers), within a sixth
  // (237 layers of 4 to 12 channels).
  const auto tiles_of = [](double pixels, double columns) {
    return std::ceil(pixels / 64) * std::ceil(columns / 64);
  };
  if (folds_taps(direction, p)) {
    const double taps = static_cast<double>(p.window_rows) * p.window_cols;
    const double pixels = static_cast<double>(p.batch) * p.out_rows * p.out_cols;
    const double columns = taps * p.channels, chunks = p.features / 32;
    const double tiles = tiles_of(pixels, columns);
    // (products beyond what the cache between them and the fold holds)
    const double beyond = std::max(0.0, pixels * columns - double(1 << 24));
    return 9.7 + 0.4 * tiles * chunks / kNumCus +
           0.4 * chunks * std::ceil(tiles / 1024) + 0.22 * taps +
           1.5e-6 * r.pixels * columns + 0.7e-6 * beyond;
  }
  const double tiles = tiles_of(r.pixels, r.columns);
  const double chunks = std::ceil(r.reduced / 32), splits = igemm_splits(r);
  return 3.8 + 0.5 * tiles * chunks / kNumCus +
         0.29 * std::ceil(chunks / splits) * std::ceil(tiles * splits / 1024) +
         (splits > 1 ? 4.3 : 0.0) +
         0.75e-6 * r.pixels * r.columns * (splits > 1 ? 2 : 1);
}

bool conv2d_gather_tile_f32(int direction, const snn_hip_conv2d_params& p,
                            GatherTile* tile) {
  if (!positive(p) || !conv2d_gather_f32_wanted(direction, p, false))
    return false;
  const GatherPlan& plan = make_plan<float>(direction, p);
  *tile = {kTilesF32[plan.tile].pixels, kTilesF32[plan.tile].features,
           plan.n_splits};
  return plan.ok;
}

size_t conv2d_gather_f32_workspace_floats(int direction,
                                          const snn_hip_conv2d_params& p) {
  // (the query does not know of a bias)
  if (!positive(p) ||
      !(conv2d_gather_f32_wanted(direction, p, false) ||
        (direction == SNN_HIP_FORWARD &&
         conv2d_gather_f32_wanted(direction, p, true))))
    return 0;
  const GatherPlan& plan = make_plan<float>(direction, p);
  return plan.ok ? plan.workspace_bytes(plan.from == kPacked) / 4 : 0;
}

int launch_conv2d_gather_f32(int direction, const float* input,
                             const float* filter, float* output,
                             const snn_hip_conv2d_params& p, float* workspace,
                             size_t workspace_elems, hipStream_t stream,
                             const LaunchOptions* epilogue) {
  auto aligned = [](const void* ptr) {
    return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0;
  };
  const GatherPlan* plan = &make_plan<float>(direction, p);
  if (!plan->ok || !aligned(output) || (!plan->widen && !aligned(input)))
    return -1;
  const bool fuse = direction == SNN_HIP_FORWARD && epilogue != nullptr &&
                    epilogue->wanted();
  const bool packs = plan->from == kPacked || !aligned(filter);
  const size_t room =
      workspace != nullptr && aligned(workspace) ? workspace_elems * 4 : 0;
  if (plan->workspace_bytes(packs) > room) {
    if (!gather_f32_wanted(direction, p, fuse, false)) return -1;
    const GatherPlan& whole = make_plan<float>(direction, p, false);
    const bool whole_temporary = whole.workspace_bytes(packs) > room;
    if (stream_captures(stream)) {
      // Recorded without room the reduction stays whole, and what cannot do
      // without a temporary is left to the kernels that need none.
      plan = &whole;
      if (whole_temporary) return -1;
    } else {
      // The host time of a temporary is as much as a short launch: the
      // reduction stays whole, or another kernel that needs none takes over,
      // where that is estimated to be the faster one (18x18x18 36 -> 100,
      // 3x3 stride 2: 21.3 -> 12.3 us).
      const double split_us = gather_f32_us(*plan, packs, true);
      const double whole_us = gather_f32_us(whole, packs, whole_temporary);
      if (whole_us < split_us) plan = &whole;
      const bool all_aligned = aligned(input) && aligned(filter);
      const Products r = products_of(direction, p);
      const double other_us =
          p.features % 4 != 0 ? direct_us(direction, p, r, false)
          : p.channels % 4 == 0 && all_aligned &&
                  (direction == SNN_HIP_FORWARD ||
                   (p.stride_rows == 1 && p.stride_cols == 1))
              ? igemm_f32_us(r)
              : kNever;
      if ((epilogue == nullptr || !epilogue->deterministic) &&
          other_us + (fuse ? 2.0 : 0.0) < std::min(split_us, whole_us))
        return -1;
    }
  }
  const int rc = launch_gather<float>(
      *plan, input, filter, output, workspace, workspace_elems,
      fuse ? epilogue->bias : nullptr, fuse && epilogue->relu, stream);
  if (rc == SNN_HIP_OK && fuse && epilogue->applied != nullptr)
    *epilogue->applied = true;
  return rc;
}

}  // namespace snn
