// Half-precision filter gradient of windowed convolutions on the binary16 matrix
// cores, operands through LDS (gfx950): 3x3 and 5x5 windows at stride 1, 3x3 at
// stride 2, any padding, channel and feature counts in multiples of 8.
//
//   dW[r][s][c][k] = sum over (n, oy, ox) of
//                    X[n][oy sr + r - pr][ox sc + s - pc][c] * dY[n][oy][ox][k]
//
// (the FilterBackprop direction of sycldnn::conv2d::launch,
// include/portdnn/conv2d/launch.h:59-118; products of binary16 values summed
// in fp32 and rounded to binary16 once).
//
// The reduction runs over pixels, which is the slow dimension of both
// operands in memory (NHWC), while v_mfma_f32_32x32x16_f16 wants eight
// consecutive reduction indices per lane.  ds_read_b64_tr_b16 does that
// transposition on the way out of LDS: within 16 lanes, lane 4 j + i supplies
// the address of four consecutive halves (columns 4 i ... 4 i + 3) of row j,
// and lane t receives column t of rows 0 ... 3.  Two such reads make one
// operand.
//
//   * A work-group (8 waves, two per SIMD, one work-group per CU) owns a
//     64-channel x 64-feature tile of dW for a group of taps.  Waves w and
//     w + 4 own the same 32 x 32 quarter of it, one 32 x 32 accumulator block
//     per tap, and every other chunk of the pixels; their sums meet in LDS at
//     the end.  (One wave per SIMD issues a transposing read every 26 cycles,
//     which is slower than LDS answers: four waves read 78 bytes per cycle and
//     CU, eight 125.)
//   * The work-group walks a run of consecutive bands: some output rows of a
//     segment of columns.  A band's input pixels (with halo, zeros for the
//     padding) and dY pixels are loaded into LDS with 16-byte LDS-direct loads,
//     both with the same row pitch (segment + halo columns; dY zeros there), so
//     that the operand of a tap is the run of input pixels m + constant: one
//     flat run of pixels per band, cut into chunks of 16, whatever the image.
//     At stride 2 the input pixels are dealt to 2 x 2 planes by the parity of
//     row and column, each of which holds its taps at such constants again.  Two
//     LDS buffers: the next band arrives while this one is multiplied.
//   * Per chunk and wave: one dY operand (2 transposing reads) + per tap row 12
//     consecutive input pixels (3 reads), whose windows at pixel 0, 1, ... are
//     the row's taps (one funnel shift per register for the odd ones): 3x3 at
//     stride 1 has 11 reads, fetched one chunk ahead, for 9 matrix instructions.
//   * 16-byte pieces of a pixel are XOR-swizzled on the way in so that the 16
//     lanes of a transposing read (4 pixels x 32 bytes) fall into distinct
//     banks.
//   * What it measures: 224x224x64 at batch 16, 3x3, 81 us (73 without the loads of
//     the bands, 23 of them launches, partial tiles and their sum; the kernel with
//     operands straight from memory 158), 56x56x128 at batch 128, 3x3 stride 2, 65
//     (82), 14x14x256 at batch 128, 3x3, 50 (52 with four waves).  The loop runs
//     at 1.0-1.3 PFLOP/s, where matrix instructions alone reach 1.6.
//   * Float atomics retire one lane at a time (measured: 19 M of them cost
//     60 us), so the partial tiles are stored, and a second kernel sums them
//     and rounds to binary16.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "gemm_tile.h"
#include "plan_cache.h"
#include "snn_kernels.h"

namespace snn {

namespace {

using gemm::xcd_remap;

typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));
typedef int int10 __attribute__((ext_vector_type(10)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

constexpr int kWaves = 8;
constexpr int kQuarters = 4;      // 32 x 32 quarters of the tile
constexpr int kTile = 64;         // channels and features per work-group
constexpr int kChunk = 16;        // pixels per matrix instruction
constexpr int kPixelBytes = 128;  // 64 halves
constexpr int kTilePixels = 624;  // LDS pixels of a buffer
constexpr int kBufBytes = kTilePixels * kPixelBytes;  // 78 KB
constexpr int kMaxLoads = 10;     // per band and wave: ceil(624 / 8 / 8)
constexpr int kNumCus = 256;
constexpr int kMaxEntries = 6;    // tap rows of a group
constexpr int kMaxGroups = 5;     // tap groups
constexpr unsigned kOobOffset = 0x7FFFFFF0u;  // beyond every buffer's range
constexpr size_t kMaxBufferBytes = 0x7FFFFFF0u;

// Why a pixel of a band is not loaded: beyond a border of the image that the band
// lies at, or never.
constexpr unsigned kTop = 1, kBottom = 2, kLeft = 4, kRight = 8, kNever = 16;
constexpr int kBorders = 5;
constexpr int kBorderWord = 5;  // loads whose bits share a register

// A run of taps of one filter row whose input pixels lie side by side in a
// plane: read at LDS pixel m + offset, m + offset + 1, ...
struct TapRow {
  int offset;
  int tap;       // first filter tap (row * window columns + column)
  int tap_step;  // ... and the distance to the next
};

// n / d for 0 <= n < 2^16, 0 < d < 2^15: (n * ceil(2^31 / d)) >> 31.
struct Divisor { unsigned magic; };
Divisor divisor(int d) {
  return {static_cast<unsigned>(((1ull << 31) + d - 1) / d)};
}
__device__ __forceinline__ int divide(int n, Divisor d) {
  return static_cast<int>(__umulhi(static_cast<unsigned>(n) << 1, d.magic));
}

struct FbGeom {
  int batch, in_rows, in_cols, channels, out_rows, out_cols, features;
  int win_rows, win_cols, stride_rows, stride_cols, pad_rows, pad_cols;
  int seg_cols;         // output columns per segment
  int segs;             // segments of a row
  int pitch;            // seg_cols + halo columns of a plane
  int band;             // output rows per band
  int plane_rows;       // input rows of a plane that a band needs
  int plane_cols;       // planes per input row: stride_cols (1 or 2)
  int bands_per_image;
  int n_subbands;       // batch * bands_per_image * segs
  int group;            // bands per task (several when small)
  int n_tasks;
  int x_px;             // LDS pixels of a plane
  int y_px;             // LDS pixels of a band's dY rows (multiple of kChunk)
  int sb_px;            // LDS pixels of a band: planes, then dY
  int tap_groups, c_tiles, k_tiles, n_splits;
  Divisor by_pitch, by_x_px;
  int group_row;        // filter rows between tap groups
  int per_split;        // consecutive tasks per work-group
  TapRow rows[kMaxGroups][kMaxEntries];
};

struct FbGeoms { FbGeom g[1]; };  // (see the kernel that sums)

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p,
                                                   size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0,
                                           static_cast<unsigned>(bytes),
                                           0x00020000);
}

constexpr int vmcnt_imm(int n) {
  return 0x0F70 | (n & 15) | ((n >> 4) << 14);
}

// Which 16-byte position of LDS pixel p holds 16-byte piece c: c ^ swz(p).
// Four consecutive pixels get four different piece pairs, and pixels 8 apart
// swap the pairs of even and odd pixels.
__device__ __forceinline__ unsigned swz(unsigned p) {
  return ((p & 3u) ^ ((p >> 3) & 1u)) << 1;
}

__device__ __forceinline__ uint2v read_transposed(const char* at) {
  return __builtin_bit_cast(
      uint2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at)));
}

// (a function of its own: the compiler drops the host side of a kernel template
// whose body names the LDS-direct load)
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t rsrc,
                                            char* lds, unsigned offset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)lds, 16, offset, 0, 0,
                                           0);
}

// A uniform value that stays in a scalar register.
__device__ __forceinline__ int keep(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}

// Taps T of each tap row of a group, in order: at most five of a row (a lane
// holds twelve pixels of it).
template <int... T>
struct TapRows {
  static constexpr int kRows = sizeof...(T);
  static constexpr int kTaps = (T + ...);
  static constexpr int kOf[kRows] = {T...};
};

// The window of eight of a lane's twelve pixels that starts at pixel `at`.
template <int AT>
__device__ __forceinline__ half8 window_of(const uint2v (&w)[3]) {
  const unsigned v[6] = {w[0][0], w[0][1], w[1][0], w[1][1], w[2][0], w[2][1]};
  constexpr int b = AT / 2;
  uint4v r;
  if constexpr (AT % 2 == 0)
    r = uint4v{v[b], v[b + 1], v[b + 2], v[b + 3]};
  else
    r = uint4v{__builtin_amdgcn_alignbit(v[b + 1], v[b], 16),
               __builtin_amdgcn_alignbit(v[b + 2], v[b + 1], 16),
               __builtin_amdgcn_alignbit(v[b + 3], v[b + 2], 16),
               __builtin_amdgcn_alignbit(v[b + 4], v[b + 3], 16)};
  return __builtin_bit_cast(half8, r);
}

// part: [split][unit] tiles of taps x 64 x 64 floats in accumulator order,
// each written once.
template <typename ROWS>
__global__ void __launch_bounds__(64 * kWaves)
    filter_backprop_window_f16_kernel(const _Float16* __restrict__ x,
                                      const _Float16* __restrict__ dy,
                                      float* __restrict__ part, FbGeom g,
                                      unsigned n_groups) {
  constexpr int kRows = ROWS::kRows, kTaps = ROWS::kTaps;
  // two objects, so that the compiler ties an LDS read to the loads of its
  // own buffer only
  __shared__ __align__(1024) char buf0[kBufBytes];
  __shared__ __align__(1024) char buf1[kBufBytes];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned group = xcd_remap(blockIdx.x, n_groups);
  const int n_units = g.tap_groups * g.c_tiles * g.k_tiles;
  const int unit = static_cast<int>(group % n_units);
  const int split = static_cast<int>(group / n_units);
  const int tg = unit % g.tap_groups;
  const int ct = unit / g.tap_groups % g.c_tiles;
  const int kt = unit / g.tap_groups / g.c_tiles;

  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(
      x, static_cast<size_t>(g.batch) * g.in_rows * g.in_cols * g.channels * 2);
  const __amdgpu_buffer_rsrc_t dy_rsrc =
      make_rsrc(dy, static_cast<size_t>(g.batch) * g.out_rows * g.out_cols *
                        g.features * 2);

  const int x_all = keep(g.sb_px - g.y_px);  // LDS pixels of all planes

  // ---- transposing-read offsets, relative to the chunk's first pixel ------
  // v_mfma_f32_32x32x16_f16: lane l holds row (or column) l % 32 at reduction
  // indices 8 (l / 32) ... + 7.  Of lane = 16 gq + 4 j + e, as a source of the
  // transposing read: pixel 8 (gq / 2) + j (+ 4 for the second read), halves
  // 4 e ... 4 e + 3 of the 16-wide block gq % 2 of this wave's 32.
  const unsigned gq = lane >> 4, j = (lane >> 2) & 3, e = lane & 3;
  const unsigned quarter = wave & 3, c32 = quarter & 1, k32 = quarter >> 1;
  const int half = wave >> 2;
  unsigned off_x[kRows][3];
  unsigned off_y[2];
#pragma unroll
  for (int h = 0; h < 3; ++h) {
    const unsigned p0 = 8 * (gq >> 1) + 4 * h + j;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const unsigned p = g.rows[tg][r].offset + p0;
      off_x[r][h] =
          p * kPixelBytes +
          (((4 * c32 + 2 * (gq & 1) + (e >> 1)) ^ swz(p)) << 4) + ((e & 1) << 3);
    }
    if (h < 2) {
      const unsigned p = x_all + p0;
      off_y[h] = p * kPixelBytes +
                 (((4 * k32 + 2 * (gq & 1) + (e >> 1)) ^ swz(p)) << 4) +
                 ((e & 1) << 3);
    }
  }

  // acc[tap][i]: feature 32 k32 + 8 (i / 4) + 4 (lane / 32) + i % 4,
  // channel 32 c32 + lane % 32
  float16v acc[kTaps];
#pragma unroll
  for (int tap = 0; tap < kTaps; ++tap)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[tap][i] = 0.f;

  // A load instruction fetches eight LDS pixels, a lane one 16-byte piece; wave w
  // takes the loads w, w + 8, ... of a band.  Every band has the same shape, and
  // whether a lane's pixel exists depends on which borders of the image the band
  // lies at, so the byte offset from the band's first pixel and five bits (the
  // borders at which the pixel is missing; never there) are worked out once per
  // lane and load.  The bands of a work-group follow one another, so the place of
  // the next takes no divisions either.  A load is then some ten scalar and seven
  // vector instructions between the matrix instructions of a chunk; with the
  // comparisons of rows and columns in each, the matrix units waited for them
  // (224x224x64 at batch 16: 92 us, with this 85).  What the loop needs is kept in
  // registers: a scalar load of an argument there would wait for the operands'
  // reads as well, and with them for the LDS latency.
  const unsigned lane_px = lane >> 3, lane_piece = lane & 7;
  const int n_loads = keep(g.sb_px / 8), x_loads = keep(x_all / 8);
  const int last_oy = (g.bands_per_image - 1) * g.band;
  const int last_ox = (g.segs - 1) * g.seg_cols;
  const int row0 = tg * g.group_row - g.pad_rows;
  int10 load_rel;
  unsigned load_missing[2] = {0, 0};
#pragma unroll
  for (int idx = 0; idx < kMaxLoads; ++idx) {
    const int p = 8 * (wave + kWaves * idx) + static_cast<int>(lane_px);
    const int piece = 8 * static_cast<int>(lane_piece ^ swz(p));
    unsigned missing;
    if (p < x_all) {
      const int plane = divide(p, g.by_x_px);
      const int q = p - plane * g.x_px;
      const int row = divide(q, g.by_pitch), col = q - row * g.pitch;
      const int pr = g.plane_cols == 1 ? plane : plane >> 1;
      const int y = row * g.stride_rows + pr;
      const int xx = col * g.stride_cols + plane - pr * g.plane_cols;
      load_rel[idx] =
          ((y * g.in_cols + xx) * g.channels + ct * kTile + piece) * 2;
      missing = (y + row0 < 0 ? kTop : 0) |
                (last_oy * g.stride_rows + y + row0 >= g.in_rows ? kBottom : 0) |
                (xx - g.pad_cols < 0 ? kLeft : 0) |
                (last_ox * g.stride_cols + xx - g.pad_cols >= g.in_cols ? kRight
                                                                        : 0) |
                (row >= g.plane_rows || ct * kTile + piece >= g.channels ? kNever
                                                                         : 0);
    } else {
      const int q = p - x_all;
      const int row = divide(q, g.by_pitch), col = q - row * g.pitch;
      load_rel[idx] =
          ((row * g.out_cols + col) * g.features + kt * kTile + piece) * 2;
      missing = (last_oy + row >= g.out_rows ? kBottom : 0) |
                (last_ox + col >= g.out_cols ? kRight : 0) |
                (row >= g.band || col >= g.seg_cols ||
                         kt * kTile + piece >= g.features
                     ? kNever : 0);
    }
    load_missing[idx / kBorderWord] |= missing
                                       << (kBorders * (idx % kBorderWord));
  }
  const unsigned missing0 = load_missing[0], missing1 = load_missing[1];
  const int bands = keep(g.group);
  const int band_bytes = keep(g.sb_px * kPixelBytes);
  const int out_rows = keep(g.out_rows), out_cols = keep(g.out_cols);
  const int band_rows = keep(g.band), seg_cols = keep(g.seg_cols);
  const int end_oy = keep(last_oy), end_ox = keep(last_ox);
  // bytes from a band to the next one of its rows, ...
  const int x_seg_bytes = keep(g.seg_cols * g.stride_cols * g.channels * 2);
  const int y_seg_bytes = keep(g.seg_cols * g.features * 2);
  // ... from the first band of a row of bands to the next row's, and from an
  // image's first band to the next image's
  const int x_row_bytes =
      keep(g.band * g.stride_rows * g.in_cols * g.channels * 2);
  const int y_row_bytes = keep(g.band * g.out_cols * g.features * 2);
  const int x_image_bytes = keep(g.in_rows * g.in_cols * g.channels * 2);
  const int y_image_bytes = keep(g.out_rows * g.out_cols * g.features * 2);
  const int task_begin = split * g.per_split;
  const int task_end = min(g.n_tasks, task_begin + g.per_split);
  // The band being loaded: its first output pixel, and its first input and
  // output pixel as bytes (of its image's first, its row's first, its own).
  int load_oy, load_ox, x_image, y_image, x_row, y_row, x_at, y_at;
  {
    const int sb = task_begin * g.group;
    const int rest = sb / g.segs;
    load_ox = (sb - rest * g.segs) * g.seg_cols;
    const int n = rest / g.bands_per_image;
    load_oy = (rest - n * g.bands_per_image) * g.band;
    x_image = n * x_image_bytes +
              (row0 * g.in_cols - g.pad_cols) * g.channels * 2;
    y_image = n * y_image_bytes;
    x_row = x_image + load_oy * g.stride_rows * g.in_cols * g.channels * 2;
    y_row = y_image + load_oy * g.out_cols * g.features * 2;
    x_at = x_row + load_ox * g.stride_cols * g.channels * 2;
    y_at = y_row + load_ox * g.features * 2;
  }
  auto borders = [&]() {
    return kNever | (load_oy == 0 ? kTop : 0u) |
           (load_oy == end_oy ? kBottom : 0u) | (load_ox == 0 ? kLeft : 0u) |
           (load_ox == end_ox ? kRight : 0u);
  };
  unsigned load_borders = borders();
  int load_band = 0, load_idx = 0, load_bands = 0;  // of the task being loaded
  auto issue_one = [&](char* buf) {
    if (load_band >= load_bands) return;
    const int l = wave + kWaves * load_idx;
    if (l < n_loads) {
      const bool is_x = l < x_loads;
      const bool high = load_idx >= kBorderWord;
      const unsigned word = high ? missing1 : missing0;
      const unsigned shift =
          kBorders * (high ? load_idx - kBorderWord : load_idx);
      const unsigned off =
          static_cast<unsigned>(load_rel[load_idx] + (is_x ? x_at : y_at));
      load_to_lds(is_x ? x_rsrc : dy_rsrc, buf + load_band * band_bytes + l * 1024,
                  ((word >> shift) & load_borders) != 0 ? kOobOffset : off);
    }
    if (kWaves * ++load_idx >= n_loads) {
      load_idx = 0;
      ++load_band;
      load_ox += seg_cols;
      x_at += x_seg_bytes;
      y_at += y_seg_bytes;
      if (load_ox >= out_cols) {
        load_ox = 0;
        load_oy += band_rows;
        x_row += x_row_bytes;
        y_row += y_row_bytes;
        if (load_oy >= out_rows) {
          load_oy = 0;
          x_image += x_image_bytes;
          y_image += y_image_bytes;
          x_row = x_image;
          y_row = y_image;
        }
        x_at = x_row;
        y_at = y_row;
      }
      load_borders = borders();
    }
  };
  const int n_subbands = keep(g.n_subbands);
  auto begin_loads = [&](int task) {
    load_band = 0;
    load_bands = min(bands, n_subbands - task * bands);
  };
  auto finish_loads = [&](char* buf) {
    while (load_band < load_bands) issue_one(buf);
  };

  auto fetch = [&](const char* at, uint2v (&ya)[2], uint2v (&xw)[kRows][3]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) ya[h] = read_transposed(at + off_y[h]);
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
      for (int h = 0; h < (ROWS::kOf[r] > 1 ? 3 : 2); ++h)
        xw[r][h] = read_transposed(at + off_x[r][h]);
  };
  // The windows are cut out of the 12 pixels here, a chunk after the reads
  // were issued, so that nothing waits on them.
  auto multiply = [&](const uint2v (&ya)[2], const uint2v (&xw)[kRows][3]) {
    const half8 y = __builtin_bit_cast(
        half8, uint4v{ya[0][0], ya[0][1], ya[1][0], ya[1][1]});
    int tap = 0;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
#define SNN_FILBK_TAP(S)                                          \
  if constexpr (true) {                                           \
    if (S < ROWS::kOf[r]) {                                       \
      acc[tap] = __builtin_amdgcn_mfma_f32_32x32x16_f16(          \
          y, window_of<S>(xw[r]), acc[tap], 0, 0, 0);             \
      ++tap;                                                      \
    }                                                             \
  }
      SNN_FILBK_TAP(0)
      SNN_FILBK_TAP(1)
      SNN_FILBK_TAP(2)
      SNN_FILBK_TAP(3)
      SNN_FILBK_TAP(4)
#undef SNN_FILBK_TAP
    }
  };

  // This wave's chunks of the task's live bands, operands fetched one chunk
  // ahead (the last fetch repeats the last chunk).
  const int n_chunks = keep(g.y_px / kChunk);
  auto multiply_task = [&](int task, const char* buf, char* nxt) {
    const int live = min(bands, n_subbands - task * bands);
    const int total = live * n_chunks;
    uint2v ya0[2], ya1[2], xb0[kRows][3], xb1[kRows][3];
    int fetched = half, in_band = half, px = half * kChunk;
    while (in_band >= n_chunks) {  // (a band of one chunk)
      in_band -= n_chunks;
      px += x_all;
    }
    auto advance = [&]() {
      if (fetched + 2 < total) {
        fetched += 2;
        in_band += 2;
        px += 2 * kChunk;
        while (in_band >= n_chunks) {
          in_band -= n_chunks;
          px += x_all;
        }
      }
    };
    // (The next band's loads are issued at the start by one half and after three
    // chunks by the other, so that one of a SIMD's two waves multiplies
    // meanwhile: 85 -> 81 us on the layer above.)
    if (half >= total) return;
    fetch(buf + px * kPixelBytes, ya0, xb0);
    if (half == 0) finish_loads(nxt);
    for (int f = half; f < total; f += 4) {
      advance();
      fetch(buf + px * kPixelBytes, ya1, xb1);
      multiply(ya0, xb0);
      if (f + 2 >= total) break;
      advance();
      if (f >= 3) finish_loads(nxt);
      fetch(buf + px * kPixelBytes, ya0, xb0);
      multiply(ya1, xb1);
    }
  };

  // ---- bands: load one ahead ------------------------------------------------
  // (past the last task nothing is left to load)
#define SNN_FILBK_STEP(cur, nxt)                              \
  {                                                           \
    if (task >= task_end) break;                              \
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));                 \
    __syncthreads();                                          \
    if (task + 1 < task_end) begin_loads(task + 1);           \
    multiply_task(task, cur, nxt);                            \
    finish_loads(nxt);                                        \
    ++task;                                                   \
  }
  // consecutive bands: the halo rows a band shares with the one before it
  // are still in this XCD's L2
  int task = task_begin;
  if (task < task_end) {
    begin_loads(task);
    finish_loads(buf0);
  }
  for (;;) {
    SNN_FILBK_STEP(buf0, buf1)
    SNN_FILBK_STEP(buf1, buf0)
  }
#undef SNN_FILBK_STEP

  // ---- the two halves meet, four taps of each in one buffer -----------------
  // Tap t is finished by half (t / 4) % 2; what it stores is in accumulator
  // order, [tap][quarter][i4][lane] float4: every store instruction writes 1 KB
  // of consecutive memory.
  float* const out = part + (static_cast<size_t>(split) * n_units + unit) *
                                (kTaps * kTile * kTile);
  auto vec_of = [&](const float16v& a, int i4) {
    return float4v{a[4 * i4], a[4 * i4 + 1], a[4 * i4 + 2], a[4 * i4 + 3]};
  };
  auto place = [&](char* buf, int slot, int i4) {
    return reinterpret_cast<float4v*>(
        buf + (((slot * kQuarters + quarter) * 4 + i4) * 64 + lane) * 16);
  };
#pragma unroll
  for (int t0 = 0; t0 < kTaps; t0 += 8) {
    __syncthreads();
#pragma unroll
    for (int t = t0; t < t0 + 8 && t < kTaps; ++t)
      if (half != ((t >> 2) & 1))
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          *place((t >> 2) & 1 ? buf1 : buf0, t & 3, i4) = vec_of(acc[t], i4);
    __syncthreads();
#pragma unroll
    for (int t = t0; t < t0 + 8 && t < kTaps; ++t)
      if (half == ((t >> 2) & 1))
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          *reinterpret_cast<float4v*>(
              out + (((t * kQuarters + quarter) * 4 + i4) * 64 + lane) * 4) =
              vec_of(acc[t], i4) +
              *place((t >> 2) & 1 ? buf1 : buf0, t & 3, i4);
  }
}

// The sum over the lanes of a wave of value `lane % 16`.
__device__ inline float add_lanes(float16v& sums) {
#pragma nounroll
  for (int m = 1; m < 64; m *= 2)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float other = __shfl_xor(sums[v], m);
      sums[v] += other;
    }
  float mine = sums[0];
#pragma unroll
  for (int v = 1; v < 16; ++v)
    mine = static_cast<int>(threadIdx.x & 15) == v ? sums[v] : mine;
  return mine;
}

// Elements c ... c + 3, k ... k + 3 of dW's tap over the products that exist among
// the pixels of one split, by one wave: number 4 channel + feature for lane % 16;
// `open`: a bit for each that is wanted.  Stops where none of them can be a number
// any more.
__device__ inline float exact_part(const _Float16* __restrict__ x,
                                   const _Float16* __restrict__ dy,
                                   const FbGeom& g, int tap, int c, int k,
                                   int split, unsigned open) {
  const int r = tap / g.win_cols, s = tap - r * g.win_cols;
  const int lane = threadIdx.x & 63;
  const int first = split * g.per_split * g.group;
  const int bands = min(g.n_subbands, first + g.per_split * g.group) - first;
  const int total = bands * g.band * g.seg_cols;
  // A pixel's place, and the digits of 64 pixels more: stepping takes no division.
  struct Place { int col, row, seg, band, n; };
  auto place = [&](int pixel, int first_band) {
    const int rows = pixel / g.seg_cols, in = rows / g.band + first_band;
    const int of_row = in / g.segs, n = of_row / g.bands_per_image;
    return Place{pixel - rows * g.seg_cols, rows % g.band, in - of_row * g.segs,
                 of_row - n * g.bands_per_image, n};
  };
  Place at = place(lane, first);
  const Place more = place(64, 0);
  float16v sums;
#pragma unroll
  for (int v = 0; v < 16; ++v) sums[v] = 0.f;
#pragma nounroll
  for (int i = lane; i - lane < total; i += 64) {
    const int oy = at.band * g.band + at.row;
    const int ox = at.seg * g.seg_cols + at.col;
    const int iy = oy * g.stride_rows + r - g.pad_rows;
    const int ix = ox * g.stride_cols + s - g.pad_cols;
    if (i < total && oy < g.out_rows && ox < g.out_cols && iy >= 0 &&
        iy < g.in_rows && ix >= 0 && ix < g.in_cols) {
      const half4v xs = *reinterpret_cast<const half4v*>(
          x + (static_cast<size_t>(at.n * g.in_rows + iy) * g.in_cols + ix) *
                  g.channels + c);
      const half4v ys = *reinterpret_cast<const half4v*>(
          dy + (static_cast<size_t>(at.n * g.out_rows + oy) * g.out_cols + ox) *
                   g.features + k);
#pragma unroll
      for (int v = 0; v < 16; ++v)
        sums[v] += static_cast<float>(xs[v / 4]) * static_cast<float>(ys[v % 4]);
    }
    auto carry = [](int& digit, int add, int radix, int over) {
      digit += add + over;
      const bool full = digit >= radix;
      if (full) digit -= radix;
      return full ? 1 : 0;
    };
    int over = carry(at.col, more.col, g.seg_cols, 0);
    over = carry(at.row, more.row, g.band, over);
    over = carry(at.seg, more.seg, g.segs, over);
    over = carry(at.band, more.band, g.bands_per_image, over);
    at.n += more.n + over;
    unsigned numbers = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v)
      if (__builtin_amdgcn_ballot_w64(sums[v] != sums[v]) == 0)
        numbers |= 1u << v;
    if ((numbers & open) == 0) break;
  }
  return add_lanes(sums);
}

// Sums the partial tiles and rounds: a work-group is 256 / n_groups
// consecutive float4 of the filter x n_groups groups of splits (a power of two
// up to 16).
// The kernel above multiplies the zeros beside a band's dY and in the padding of X
// with whatever the other operand holds there, which an infinity makes a NaN.  A sum
// that is one has those partial sums that are taken again, over the products that
// exist, one wave per four channels and features, until one is a NaN by these.
// That part keeps to few registers and loads its arguments for itself, as the waves
// in flight bound the rest (122 registers cost 14x14x256 at batch 128 3 us, 69 none).
// 224x224x64 at batch 16, finite 87 us: one infinite dY 137, all infinite 90, an
// infinity in the first row of every image, where the padding meets it, 758; over
// the whole batch and one sum after the other these took 56735, 391 and 69977.
// 56x56x128, 3x3 stride 2, at batch 128, finite 72: 87, 91 and 161.
template <typename ROWS>
__global__ void __launch_bounds__(256)
    filter_backprop_window_f16_reduce_kernel(const float4v* __restrict__ part,
                                             const _Float16* __restrict__ x,
                                             const _Float16* __restrict__ dy,
                                             _Float16* __restrict__ dw,
                                             FbGeoms gs, int n_groups) {
  const FbGeom& g = gs.g[0];
  __shared__ float4v sums[256];
  __shared__ int any_strange;
  __shared__ int strange[64];  // of four channels each, a bit per channel
  constexpr int kTileVecs = ROWS::kTaps * kTile * kTile / 4;
  const int n_units = g.tap_groups * g.c_tiles * g.k_tiles;
  const int width = 256 / n_groups;
  const int lane_o = threadIdx.x % width;
  const int group = threadIdx.x / width;
  const unsigned o = blockIdx.x * width + lane_o;  // float4 of the whole filter
  const unsigned unit = o / kTileVecs;
  const unsigned local = o - unit * kTileVecs;
  float4v sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int sp = group; sp < g.n_splits; sp += n_groups)
    sum += part[(static_cast<size_t>(sp) * n_units + unit) * kTileVecs + local];
  sums[threadIdx.x] = sum;
  if (threadIdx.x < 64) strange[threadIdx.x] = 0;
  if (threadIdx.x == 0) any_strange = 0;
  __syncthreads();
  // accumulator order of the partial tiles: local = ((tap * 4 + quarter) * 4 +
  // i4) * 64 + lane holds channel 32 (quarter & 1) + lane % 32 and features
  // 32 (quarter >> 1) + 8 i4 + 4 (lane / 32) ... + 3
  auto place_of = [](const FbGeom& g, unsigned at, int* tap, int* c, int* k) {
    const unsigned u = at / kTileVecs, l = at - u * kTileVecs;
    const unsigned ln = l & 63, i4 = (l >> 6) & 3, quarter = (l >> 8) & 3;
    const int tg = u % g.tap_groups;
    const int ct = u / g.tap_groups % g.c_tiles;
    const int kt = u / g.tap_groups / g.c_tiles;
    int t = l >> 10, r = 0;
    while (r + 1 < ROWS::kRows && t >= ROWS::kOf[r]) t -= ROWS::kOf[r++];
    *tap = g.rows[tg][r].tap + t * g.rows[tg][r].tap_step;
    *c = ct * kTile + 32 * (quarter & 1) + (ln & 31);
    *k = kt * kTile + 32 * (quarter >> 1) + 8 * i4 + 4 * (ln >> 5);
  };
  if (group == 0) {
    for (int i = 1; i < n_groups; ++i) sum += sums[i * width + lane_o];
    int tap, c, k;
    place_of(g, o, &tap, &c, &k);
    if (c < g.channels && k < g.features) {
      if (sum[0] != sum[0] || sum[1] != sum[1] || sum[2] != sum[2] ||
          sum[3] != sum[3]) {
        atomicOr(&strange[lane_o >> 2], 1 << (lane_o & 3));
        any_strange = 1;
      } else {
        half4v r;
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = static_cast<_Float16>(sum[v]);
        *reinterpret_cast<half4v*>(
            dw + (static_cast<size_t>(tap) * g.channels + c) * g.features + k) = r;
      }
    }
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(any_strange) == 0) return;
  // (an index that is not known before: what follows would load its arguments in
  // front of the sums)
  const FbGeom& h = gs.g[__builtin_amdgcn_readfirstlane(any_strange) - 1];
  const int units = h.tap_groups * h.c_tiles * h.k_tiles;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma nounroll
  for (int i = wave; i < width / 4; i += 4) {
    const int channels = strange[i];
    if (channels == 0) continue;
    const unsigned at = blockIdx.x * width + 4 * i;
    const unsigned u = at / kTileVecs;
    int tap, c, k;
    place_of(h, at, &tap, &c, &k);
    float total = 0.f;  // number 4 channel + feature for lane % 16
    unsigned open = 0;  // sums that may be numbers
#pragma unroll
    for (int ch = 0; ch < 4; ++ch)
      if ((channels >> ch & 1) != 0) open |= 15u << (4 * ch);
#pragma nounroll
    for (int sp0 = 0; sp0 < h.n_splits && open != 0; sp0 += 64) {
      unsigned again = 0;  // sums of this lane's split
      {
        float16v p;
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
          float4v four = {0.f, 0.f, 0.f, 0.f};
          if (sp0 + lane < h.n_splits)
            four = part[(static_cast<size_t>(sp0 + lane) * units + u) * kTileVecs +
                        (at - u * kTileVecs) + ch];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const bool number = four[v] == four[v];
            p[4 * ch + v] = number ? four[v] : 0.f;
            if (!number) again |= 1u << (4 * ch + v);
          }
        }
        total += add_lanes(p);
      }
      unsigned long long left = __builtin_amdgcn_ballot_w64(again != 0);
#pragma nounroll
      for (;;) {
        open &= ~static_cast<unsigned>(
            __builtin_amdgcn_ballot_w64(total != total));
        if (left == 0 || open == 0) break;
        const int from = __builtin_ctzll(left);
        left &= left - 1;
        const unsigned these =
            static_cast<unsigned>(__shfl(static_cast<int>(again), from)) & open;
        if (these == 0) continue;
        const float exact = exact_part(x, dy, h, tap, c, k, sp0 + from, these);
        if ((these >> (lane & 15) & 1u) != 0) total += exact;
      }
    }
    if (lane < 16 && (channels >> (lane >> 2) & 1) != 0)
      dw[(static_cast<size_t>(tap) * h.channels + c + (lane >> 2)) * h.features +
         k + (lane & 3)] = static_cast<_Float16>(total);
  }
}

int round_up(int a, int b) { return ceil_div(a, b) * b; }

enum Shape { kNone, k3x3, k5x5, k3x3s2 };
typedef TapRows<3, 3, 3> Rows3x3;
typedef TapRows<5> Rows5x5;
typedef TapRows<2, 2, 1, 1, 2, 1> Rows3x3s2;

Shape shape_of(const snn_hip_conv2d_params& p) {
  if (p.window_rows == 3 && p.window_cols == 3) {
    if (p.stride_rows == 1 && p.stride_cols == 1) return k3x3;
    if (p.stride_rows == 2 && p.stride_cols == 2) return k3x3s2;
  }
  if (p.window_rows == 5 && p.window_cols == 5 && p.stride_rows == 1 &&
      p.stride_cols == 1)
    return k5x5;
  return kNone;
}

struct WindowPlan {
  Shape shape = kNone;
  double us = 0;  // estimated, beside launches and first loads
  FbGeom g;
};

WindowPlan compute_plan(const snn_hip_conv2d_params& p) {
  WindowPlan plan;
  const Shape shape = shape_of(p);
  if (shape == kNone || p.batch < 1 || p.in_rows < 1 || p.in_cols < 1 ||
      p.out_rows < 1 || p.out_cols < 1 || p.channels < 8 || p.features < 8 ||
      p.channels % 8 != 0 || p.features % 8 != 0 || p.pad_rows < 0 ||
      p.pad_cols < 0 || p.pad_rows >= p.window_rows ||
      p.pad_cols >= p.window_cols)
    return plan;
  const size_t x_bytes = static_cast<size_t>(p.batch) * p.in_rows * p.in_cols *
                         p.channels * 2;
  const size_t y_bytes = static_cast<size_t>(p.batch) * p.out_rows *
                         p.out_cols * p.features * 2;
  if (x_bytes > kMaxBufferBytes || y_bytes > kMaxBufferBytes) return plan;
  FbGeom& g = plan.g;
  std::memset(&g, 0, sizeof g);
  g.batch = p.batch; g.in_rows = p.in_rows; g.in_cols = p.in_cols;
  g.channels = p.channels; g.out_rows = p.out_rows; g.out_cols = p.out_cols;
  g.features = p.features; g.win_rows = p.window_rows;
  g.win_cols = p.window_cols; g.stride_rows = p.stride_rows;
  g.stride_cols = p.stride_cols; g.pad_rows = p.pad_rows;
  g.pad_cols = p.pad_cols;
  g.plane_cols = p.stride_cols;
  const int planes = p.stride_rows * p.stride_cols;
  const int halo_r = (p.window_rows - 1) / p.stride_rows;
  const int halo_c = (p.window_cols - 1) / p.stride_cols;
  g.tap_groups = shape == k5x5 ? 5 : 1;
  g.group_row = 1;
  const int group_halo = shape == k5x5 ? 0 : halo_r;
  const int taps = shape == k5x5 ? 5 : 9;
  g.c_tiles = ceil_div(p.channels, kTile);
  g.k_tiles = ceil_div(p.features, kTile);
  const int n_units = g.tap_groups * g.c_tiles * g.k_tiles;

  // Segments, bands and work-groups per tile: the least estimated time.  A chunk
  // is `taps` matrix instructions of 32 cycles on each SIMD; loads take LDS cycles
  // from the operands' reads, 60 bytes each; a task costs some 500 cycles of
  // barrier and first reads; the clock is 1.7 GHz under this load.  A partial
  // tile is written and read back: 0.42 us per MB.
  const double tile_us = n_units * taps * kTile * kTile * 4 * 0.42e-6;
  // (Only the first and the last band of an image or a row may reach over its
  // border: the kernel knows one set of missing pixels for each border.)
  const int row_reach = shape == k5x5 ? p.window_rows - 1 : 0;
  auto borders_fit = [](int count, int size, int stride, int halo, int reach,
                        int pad, int extent) {
    return count == 1 ||
           (size * stride >= pad &&
            ((count - 2) * size + size - 1 + halo) * stride + stride - 1 +
                    reach - pad < extent);
  };
  double best = -1;
  for (int segs = 1; segs <= p.out_cols; ++segs) {
    const int seg = ceil_div(p.out_cols, segs);
    if (segs > 1 && (ceil_div(p.out_cols, seg) != segs || seg < 4)) continue;
    if (!borders_fit(segs, seg, p.stride_cols, halo_c, 0, p.pad_cols,
                     p.in_cols))
      continue;
    const int pitch = seg + halo_c;
    for (int band = 1; band <= p.out_rows; ++band) {
      const int bands = ceil_div(p.out_rows, band);
      if (band > 1 && ceil_div(p.out_rows, bands) != band) continue;
      if (!borders_fit(bands, band, p.stride_rows, group_halo, row_reach,
                       p.pad_rows, p.in_rows))
        continue;
      const int y_px = round_up(band * pitch, kChunk);
      // (the third read of a row reaches three pixels past the last chunk's
      // last one, from the last tap row's place)
      const int x_px = round_up(y_px + group_halo * pitch + halo_c + 4, 8);
      const int sb_px = planes * x_px + y_px;
      if (sb_px > kTilePixels) break;
      const long subbands = static_cast<long>(p.batch) * bands * segs;
      const int group = static_cast<int>(
          std::max<long>(1, std::min<long>(kTilePixels / sb_px, subbands)));
      const long tasks = (subbands + group - 1) / group;
      const double chunks = static_cast<double>(group) * (y_px / kChunk);
      const double loads = static_cast<double>(group) * sb_px * kPixelBytes;
      const double task_us = (chunks * taps * 32 + loads / 60 + 500) / 1700;
      const long most =
          std::max<long>(1, std::min<long>(tasks, kNumCus / n_units));
      const long fewer = std::lround(std::sqrt(tasks * task_us / tile_us));
      for (const long want : {most, std::max(1l, std::min(most, fewer))}) {
        const long per_split = (tasks + want - 1) / want;
        const long splits = (tasks + per_split - 1) / per_split;
        const long rounds = (splits * n_units + kNumCus - 1) / kNumCus;
        const double cost = rounds * per_split * task_us + splits * tile_us;
        if (best >= 0 && cost >= best) continue;
        best = cost;
        g.segs = segs; g.seg_cols = seg; g.pitch = pitch;
        g.band = band; g.bands_per_image = bands;
        g.plane_rows = band + group_halo;
        g.x_px = x_px; g.y_px = y_px; g.sb_px = sb_px;
        g.group = group;
        g.n_subbands = static_cast<int>(subbands);
        g.n_tasks = static_cast<int>(tasks);
        g.per_split = static_cast<int>(per_split);
        g.n_splits = static_cast<int>(splits);
      }
    }
  }
  if (best < 0) return plan;
  g.by_pitch = divisor(g.pitch);
  g.by_x_px = divisor(g.x_px);
  if (shape == k3x3)
    for (int r = 0; r < 3; ++r) g.rows[0][r] = {r * g.pitch, 3 * r, 1};
  if (shape == k3x3s2) {
    // planes (row parity, column parity) in order
    auto entry = [&](int pr, int pc, int dr) {
      return TapRow{(2 * pr + pc) * g.x_px + dr * g.pitch,
                    3 * (2 * dr + pr) + pc, 2};
    };
    g.rows[0][0] = entry(0, 0, 0);
    g.rows[0][1] = entry(0, 0, 1);
    g.rows[0][2] = entry(0, 1, 0);
    g.rows[0][3] = entry(0, 1, 1);
    g.rows[0][4] = entry(1, 0, 0);
    g.rows[0][5] = entry(1, 1, 0);
  }
  if (shape == k5x5)
    for (int r = 0; r < 5; ++r) g.rows[r][0] = {0, 5 * r, 1};
  plan.shape = shape;
  plan.us = best;
  return plan;
}

// Whether the kernel of conv2d_filter_backprop_direct.hip, which needs no LDS
// bands and a twentieth of the partial tiles, is the faster one: the estimates of
// both (this one's launches and first loads take 10 us) missed 110 random layers
// by a third at most; with them 42 layers of those run here, 0.87 of the time of
// all on that kernel, none slower by more than 5 %.  (Small layers are the
// other's: 4x32x42 32 -> 416, 3x3 stride 2: 28 against 10 us; large ones this
// one's: 4x108x140 32 -> 400, 5x5: 118 against 231.)
// Fewer than 256 output pixels the other one does not take: what those run on
// without this kernel is the faster one up to about 2^24 multiply-adds
// (23x3x3 576 -> 32, stride 2: 16 against 13 us; 16x5x4 256 -> 384: 12 / 20).
WindowPlan wanted_plan(const snn_hip_conv2d_params& p) {
  WindowPlan plan;
  if (shape_of(p) == kNone) return plan;
  plan = compute_plan(p);
  if (plan.shape == kNone) return plan;
  const double macs = static_cast<double>(p.batch) * p.out_rows * p.out_cols *
                      p.window_rows * p.window_cols * p.channels * p.features;
  if (conv2d_filter_backprop_direct_f16_supports(p)
          ? 10 + plan.us >= 0.9 * conv2d_filter_backprop_direct_f16_us(p)
          : macs < 1 << 24)
    plan.shape = kNone;
  return plan;
}

const WindowPlan& make_plan(const snn_hip_conv2d_params& p) {
  thread_local PlanCache<WindowPlan> cache;
  return cache.get(p, 0, [&] { return wanted_plan(p); });
}

template <typename ROWS>
void launch_rows(const _Float16* x, const _Float16* dy, _Float16* dw,
                 float* part, const FbGeom& g, hipStream_t stream) {
  const int n_units = g.tap_groups * g.c_tiles * g.k_tiles;
  const unsigned n_groups = static_cast<unsigned>(n_units * g.n_splits);
  {
    KernelTimer timer(stream);
    hipLaunchKernelGGL(filter_backprop_window_f16_kernel<ROWS>, dim3(n_groups),
                       dim3(64 * kWaves), 0, stream, x, dy, part, g, n_groups);
  }
  const unsigned vecs =
      static_cast<unsigned>(n_units) * (ROWS::kTaps * kTile * kTile / 4);
  int reduce_groups = 1;
  while (reduce_groups < 16 && 2 * reduce_groups <= g.n_splits &&
         vecs / (256 / reduce_groups) < 1024)
    reduce_groups *= 2;
  hipLaunchKernelGGL(filter_backprop_window_f16_reduce_kernel<ROWS>,
                     dim3(vecs / (256 / reduce_groups)), dim3(256), 0, stream,
                     reinterpret_cast<const float4v*>(part), x, dy, dw,
                     FbGeoms{{g}}, reduce_groups);
}

}  // namespace

bool conv2d_filter_backprop_window_f16_supports(
    const snn_hip_conv2d_params& p) {
  return make_plan(p).shape != kNone;
}

int conv2d_filter_backprop_window_f16_splits(const snn_hip_conv2d_params& p) {
  const WindowPlan& plan = make_plan(p);
  return plan.shape != kNone ? plan.g.n_splits : 0;
}

size_t conv2d_filter_backprop_window_f16_partial_floats(
    const snn_hip_conv2d_params& p) {
  const WindowPlan& plan = make_plan(p);
  if (plan.shape == kNone) return 0;
  const FbGeom& g = plan.g;
  return static_cast<size_t>(g.n_splits) * g.tap_groups * g.c_tiles *
         g.k_tiles * (plan.shape == k5x5 ? 5 : 9) * kTile * kTile;
}

int launch_conv2d_filter_backprop_window_f16(const _Float16* x,
                                             const _Float16* dy, _Float16* dw,
                                             float* part,
                                             const snn_hip_conv2d_params& p,
                                             hipStream_t stream) {
  const WindowPlan& plan = make_plan(p);
  if (plan.shape == k3x3)
    launch_rows<Rows3x3>(x, dy, dw, part, plan.g, stream);
  else if (plan.shape == k5x5)
    launch_rows<Rows5x5>(x, dy, dw, part, plan.g, stream);
  else if (plan.shape == k3x3s2)
    launch_rows<Rows3x3s2>(x, dy, dw, part, plan.g, stream);
  else
    return SNN_HIP_INVALID_ALGORITHM;
  return SNN_HIP_OK;
}

}  // namespace snn
