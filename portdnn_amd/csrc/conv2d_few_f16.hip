// Half-precision convolutions of images with one to four channels at stride 2
// (a network's first layer) in all three directions on the binary16 matrix
// cores (gfx950): binary16 operands, fp32 accumulation, binary16 result.  (The
// three directions of sycldnn::conv2d::launch,
// include/portdnn/conv2d/launch.h:59-118.)
//
// With so few channels neither the reduction of the forward direction nor the
// rows of the gradients fill a matrix instruction per filter tap, so each
// direction flattens taps and channels together:
//
//   forward          reduction over runs of eight (column tap, channel) values
//                    of a filter row, which are consecutive in memory;
//   input gradient   the 2 x 2 x C values of dX that share their dY pixels are
//                    the 16 rows of one stride-1 convolution of dY with a
//                    window of half the size, taps that do not exist for a row
//                    being zeros of the filter;
//   filter gradient  the image as 2 x 2 x C planes of half its size, whose
//                    rows times half-size tap rows are the 32 rows of the
//                    product.
//
// All three move little beside dY or Y itself: 224x224x3, 7x7, 64 features at
// batch 128 has 205 MB of it, 44 us at the 4.7 TB/s of a large copy, and 30 GFLOP,
// 26 us at the 1.14 PFLOP/s of a large product.  The step of the three took 1260
// us and takes 247 to 261 from GPU to GPU (traced alone 99, 78 and 97 + 7).
#include <algorithm>
#include <climits>

#include "gemm_tile.h"
#include "snn_kernels.h"

namespace snn {
namespace {

using gemm::float16v;
using gemm::xcd_remap;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

constexpr unsigned kOob = 0x7FFFFFF0u;
constexpr size_t kMaxBufferBytes = 0x7FFFFFF0u;
constexpr int kMaxChannels = 4;
constexpr int kNumCus = 256;

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p,
                                                   size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0,
                                           static_cast<unsigned>(bytes),
                                           0x00020000);
}

__device__ __forceinline__ half8 load_half8(__amdgpu_buffer_rsrc_t rsrc,
                                            unsigned offset) {
  return __builtin_bit_cast(
      half8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0));
}

// Within 16 lanes, lane 4 j + i supplies the address of halves 4 i ... 4 i + 3
// of row j, and lane t receives half t of rows 0 ... 3.
__device__ __forceinline__ half8 read_transposed(const char* rows03,
                                                 const char* rows47) {
  const short4v lo =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(rows03));
  const short4v hi =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(rows47));
  const short8v both =
      __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(half8, both);
}

constexpr int vmcnt_imm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

// Waits for this wave's LDS operations and for the other waves; loads from
// memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

struct FewGeom {
  int batch, in_rows, in_cols, channels;
  int out_rows, out_cols, features;
  int win_rows, win_cols, pad_rows, pad_cols;
  int lo_r, lo_c;      // half-size row / column of tap (0, 0), relative
  int band;            // rows per band
  int bands;           // bands per image
  int col_blocks;      // input gradient: blocks of 32 pixel pairs per row
  int pitch;           // LDS row: halves (forward) or bytes (filter gradient)
  int plane;           // filter gradient: bytes of a plane
  int pixels;          // filter gradient: out_cols, whole chunks of 16
  int lds_rows;        // forward: image rows of a band
  int units, per_group;  // filter gradient: bands, bands per work-group
};

// ---------------------------------------------------------------------------
// Input gradient.  Pixels (2 Y + a, 2 X + b) of dX take dY rows
// (2 Y + a + pad - r) / 2 for the r that make this whole: rows Y + lo ... + T - 1
// for both a, likewise the columns.  So
//   Z[8 a + C b + c][Y][X] = sum over (tr, ts, f) V[8 a + C b + c][tr][ts][f] *
//                            dY[Y + lo_r + tr][X + lo_c + ts][f],
// V = W[r][s][c][f] with r = a + pad - 2 (lo + tr), or zero where r or s is
// outside the window.  (49 of 64 taps of a 7x7 window and 12 of 16 rows are of
// use; at 1.1 PFLOP/s that still is less than the time dY takes to arrive.)
//
//   * Waves are independent: one owns 32 pixel pairs of a row, walks a band of
//     dY rows and keeps V (T * T * KS registers x 4) and T rows of accumulators.
//     A dY row is loaded once, 16 bytes per lane -- exactly the operand of 16
//     pixels x 32 features -- one row ahead, and multiplied into the T rows of
//     Z it belongs to.
//   * The operands of the other column taps are the same registers moved by ts
//     lanes within each 16 (two DPP moves per register, which run while the
//     matrix unit works), so neither LDS nor the L1 sees the T-fold reuse.
//   * A zero of V times an infinity of dY is a NaN that does not belong there:
//     a wave that is about to store a NaN works out those sums term by term.
//
// 128 x 224x224x3 <- 64, 7x7: 529 us through fp32 (409 of it in the fp32
// kernel) -> 78 us.
template <int T, int KS>
__global__ void __launch_bounds__(256, KS < 3 ? 2 : 1)
    few_input_backprop_f16_kernel(const _Float16* __restrict__ dy,
                                  const _Float16* __restrict__ w,
                                  _Float16* __restrict__ dx, FewGeom g,
                                  unsigned n_groups, unsigned n_units) {
  const int lane = threadIdx.x & 63;
  const int l16 = lane & 15, q = lane >> 4;
  const unsigned unit = __builtin_amdgcn_readfirstlane(
      xcd_remap(blockIdx.x, n_groups) * 4 + (threadIdx.x >> 6));
  if (unit >= n_units) return;
  const unsigned bands_at = unit / g.col_blocks;
  const int block = static_cast<int>(unit - bands_at * g.col_blocks);
  const int n = static_cast<int>(bands_at / g.bands);
  const int y0 = static_cast<int>(bands_at - n * g.bands) * g.band;
  const int pair_rows = (g.in_rows + 1) >> 1, pair_cols = (g.in_cols + 1) >> 1;
  const int n_rows = min(g.band, pair_rows - y0);
  const int x0 = 32 * block;

  const __amdgpu_buffer_rsrc_t dy_rsrc =
      make_rsrc(dy, static_cast<size_t>(g.batch) * g.out_rows * g.out_cols *
                        g.features * 2);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      make_rsrc(w, static_cast<size_t>(g.win_rows) * g.win_cols * g.channels *
                       g.features * 2);
  const __amdgpu_buffer_rsrc_t dx_rsrc =
      make_rsrc(dx, static_cast<size_t>(g.batch) * g.in_rows * g.in_cols *
                        g.channels * 2);

  // this lane's row of V
  const int va = l16 >> 3, vb = (l16 & 7) / g.channels;
  const int vc = (l16 & 7) - vb * g.channels;
  half8 v[T][T][KS];
#pragma unroll
  for (int tr = 0; tr < T; ++tr)
#pragma unroll
    for (int ts = 0; ts < T; ++ts) {
      const int r = va + g.pad_rows - 2 * (g.lo_r + tr);
      const int s = vb + g.pad_cols - 2 * (g.lo_c + ts);
      const bool ok = vb < 2 &&
                      static_cast<unsigned>(r) <
                          static_cast<unsigned>(g.win_rows) &&
                      static_cast<unsigned>(s) <
                          static_cast<unsigned>(g.win_cols);
      const unsigned at = static_cast<unsigned>(
          ((r * g.win_cols + s) * g.channels + vc) * g.features * 2);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        v[tr][ts][ks] = load_half8(
            w_rsrc, ok && 32 * ks + 8 * q < g.features
                        ? at + 64u * ks + 16u * q : kOob);
    }

  // Columns this lane loads: 16 j + l16 of the block for j = 0, 1 and the
  // T - 1 behind them.
  unsigned col_at[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int col = x0 + g.lo_c + 16 * j + l16;
    const bool ok = static_cast<unsigned>(col) <
                        static_cast<unsigned>(g.out_cols) &&
                    (j < 2 || l16 < T - 1);
    col_at[j] = ok ? static_cast<unsigned>(col * g.features * 2 + 16 * q) : kOob;
  }
  const bool last_ok = 32 * (KS - 1) + 8 * q < g.features;
  struct Row { half8 at[3][KS]; };
  auto load_row = [&](int k, Row& row) {
    const int yy = y0 + g.lo_r + k;
    const bool ok = static_cast<unsigned>(yy) <
                        static_cast<unsigned>(g.out_rows) &&
                    k < n_rows + T - 1;
    const unsigned row_at = static_cast<unsigned>(n * g.out_rows + yy) *
                            static_cast<unsigned>(g.out_cols * g.features * 2);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const unsigned at = ok && col_at[j] != kOob ? row_at + col_at[j] : kOob;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        row.at[j][ks] = load_half8(
            dy_rsrc, ks < KS - 1 || last_ok ? at + (at == kOob ? 0u : 64u * ks)
                                            : kOob);
    }
  };

  float4v acc[T][2];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[t][j] = float4v{0.f, 0.f, 0.f, 0.f};

  // Lanes 0 ... 15 - S of each 16 take lane + S of `cur`, the others the first
  // S lanes of `next`.
  auto shifted = [](const half8& cur, const half8& next, auto shift) -> half8 {
    constexpr int S = decltype(shift)::value;
    if constexpr (S == 0) {
      return cur;
    } else {
      const uint4v c = __builtin_bit_cast(uint4v, cur);
      const uint4v x = __builtin_bit_cast(uint4v, next);
      uint4v r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int tail = __builtin_amdgcn_update_dpp(
            0, static_cast<int>(x[e]), 0x110 + (16 - S), 0xF, 0xF, false);
        r[e] = static_cast<unsigned>(__builtin_amdgcn_update_dpp(
            tail, static_cast<int>(c[e]), 0x100 + S, 0xF, 0xF, false));
      }
      return __builtin_bit_cast(half8, r);
    }
  };

  const int C = g.channels;
  // Rows 4 q ... 4 q + 3 of Z: values 4 (q & 1) ... of dX row 2 Y + q / 2.
  const int za = q >> 1, zv = 4 * (q & 1);
  auto store = [&](int y, int j, float4v z) {
    const int row = 2 * y + za, x = x0 + 16 * j + l16;
    const int count =
        row < g.in_rows && x < pair_cols
            ? min(2 * C, (g.in_cols - 2 * x) * C) - zv : 0;  // values to store
    const bool strange = (z[0] != z[0]) | (z[1] != z[1]) | (z[2] != z[2]) |
                         (z[3] != z[3]);
    if (__builtin_amdgcn_ballot_w64(strange && count > 0) != 0) {
      if (strange) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (e >= count) continue;
          const int b = (zv + e) / C, c = zv + e - b * C;
          float sum = 0.f;
          for (int r = (za + g.pad_rows) & 1; r < g.win_rows; r += 2) {
            const int oy = (row + g.pad_rows - r) >> 1;
            if (oy < 0 || oy >= g.out_rows) continue;
            for (int s = (b + g.pad_cols) & 1; s < g.win_cols; s += 2) {
              const int ox = (2 * x + b + g.pad_cols - s) >> 1;
              if (ox < 0 || ox >= g.out_cols) continue;
              const _Float16* from =
                  dy + (static_cast<size_t>(n * g.out_rows + oy) * g.out_cols +
                        ox) * g.features;
              const _Float16* by =
                  w + static_cast<size_t>((r * g.win_cols + s) * C + c) *
                          g.features;
              for (int f = 0; f < g.features; ++f)
                sum += static_cast<float>(from[f]) * static_cast<float>(by[f]);
            }
          }
          z[e] = sum;
        }
      }
    }
    const unsigned at = static_cast<unsigned>(
        (((n * g.in_rows + row) * g.in_cols + 2 * x) * C + zv) * 2);
    if ((g.in_cols * C & 1) == 0) {
      // (rows of an even number of values: pairs are 4-byte aligned, and the
      // count is even too)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        typedef _Float16 half2v __attribute__((ext_vector_type(2)));
        const half2v two = {static_cast<_Float16>(z[e]),
                            static_cast<_Float16>(z[e + 1])};
        __builtin_amdgcn_raw_buffer_store_b32(
            __builtin_bit_cast(unsigned, two), dx_rsrc,
            e + 1 < count ? at + 2u * e : kOob, 0, 0);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        __builtin_amdgcn_raw_buffer_store_b16(
            __builtin_bit_cast(unsigned short, static_cast<_Float16>(z[e])),
            dx_rsrc, e < count ? at + 2u * e : kOob, 0, 0);
    }
  };

  // dY row k of the band belongs to rows k - tr of Z; slot (k - tr) % T holds
  // their sums, so that T steps are unrolled.  Rows before and behind the band
  // are summed in part and dropped.
  const bool second = x0 + 16 < pair_cols;
  auto step = [&](int k, auto phase, const Row& row) {
    constexpr int P = decltype(phase)::value;
    auto taps = [&](auto col_tap) {
      constexpr int TS = decltype(col_tap)::value;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (j == 1 && !second) continue;
          const half8 b = shifted(row.at[j][ks], row.at[j + 1][ks], col_tap);
#pragma unroll
          for (int tr = 0; tr < T; ++tr) {
            float4v& a = acc[(P - tr + T) % T][j];
            a = __builtin_amdgcn_mfma_f32_16x16x32_f16(v[tr][TS][ks], b, a, 0,
                                                       0, 0);
          }
        }
    };
    taps(std::integral_constant<int, 0>{});
    taps(std::integral_constant<int, 1>{});
    if constexpr (T > 2) taps(std::integral_constant<int, 2>{});
    if constexpr (T > 3) taps(std::integral_constant<int, 3>{});
    // row k - (T - 1) is complete
    constexpr int D = (P + 1) % T;
    const int done = k - (T - 1);
    if (done >= 0 && done < n_rows) {
      store(y0 + done, 0, acc[D][0]);
      if (second) store(y0 + done, 1, acc[D][1]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[D][j] = float4v{0.f, 0.f, 0.f, 0.f};
  };

  Row even, odd;
  const int n_steps = n_rows + T - 1;
  load_row(0, even);
  for (int k = 0; k < n_steps;) {
    // (T = 3 takes six steps a turn, so that `even` comes first again)
#define SNN_FEW_STEP(P, cur, nxt)                               \
  {                                                             \
    load_row(k + 1, nxt);                                       \
    __builtin_amdgcn_sched_barrier(0);                          \
    step(k, std::integral_constant<int, P>{}, cur);             \
    if (++k >= n_steps) break;                                  \
  }
    SNN_FEW_STEP(0, even, odd)
    SNN_FEW_STEP(1, odd, even)
    if constexpr (T == 3) {
      SNN_FEW_STEP(2, even, odd)
      SNN_FEW_STEP(0, odd, even)
      SNN_FEW_STEP(1, even, odd)
      SNN_FEW_STEP(2, odd, even)
    }
    if constexpr (T == 4) {
      SNN_FEW_STEP(2, even, odd)
      SNN_FEW_STEP(3, odd, even)
    }
#undef SNN_FEW_STEP
  }
}

// ---------------------------------------------------------------------------
// Forward.  The win_cols * C values of a filter row lie side by side in memory,
// 2 C halves further for the next output pixel, so eight of them at a time are
// an operand of v_mfma_f32_16x16x32_f16: instruction (h, i) takes values 8 i ...
// 8 i + 7 of filter rows 4 h ... 4 h + 3, one row per 16 lanes (147 of 192
// products are of use for 7x7x3).
//
//   * A work-group owns a band of output rows and keeps the image rows under it
//     in LDS, from the left padding on.  Where that begins at an odd half the
//     rows sit one half further right, so that every operand is 4-byte aligned.
//   * The filter passes through LDS once, is turned by transposing reads into
//     operands (features as rows, so permuted that a lane ends with eight
//     consecutive features of a pixel) and stays in registers, all features in
//     every wave: a pixel operand serves 2 NP instructions.
//   * Values of an operand outside the filter row belong to other pixels and are
//     cleared, not multiplied by zero: they may be infinite.  Where a window leaves
//     the image an infinite weight meets a zero; sums that are NaN there are
//     worked out term by term.
//
// 128 x 224x224x3 -> 64, 7x7: 153 us with the image widened to eight channels
// -> 99 us.
template <int HS, int G, int NP>
__global__ void __launch_bounds__(256, 2)
    few_forward_f16_kernel(const _Float16* __restrict__ x,
                           const _Float16* __restrict__ w,
                           _Float16* __restrict__ y, FewGeom g,
                           unsigned n_groups) {
  extern __shared__ __align__(16) char lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, q = lane >> 4;
  const unsigned group = xcd_remap(blockIdx.x, n_groups);
  const int n = static_cast<int>(group / g.bands);
  const int oy0 = static_cast<int>(group - n * g.bands) * g.band;
  const int n_rows = min(g.band, g.out_rows - oy0);
  const int C = g.channels, wc = g.win_cols * C;
  const int shift = g.pad_cols * C & 1;

  const __amdgpu_buffer_rsrc_t x_rsrc =
      make_rsrc(x, static_cast<size_t>(g.batch) * g.in_rows * g.in_cols * C * 2);
  const __amdgpu_buffer_rsrc_t y_rsrc =
      make_rsrc(y, static_cast<size_t>(g.batch) * g.out_rows * g.out_cols *
                       g.features * 2);

  // ---- the filter, and behind it a row of zeros ----------------------------
  const int filter_bytes = g.win_rows * wc * g.features * 2;
  for (int i = threadIdx.x * 16; i < filter_bytes + 64 * NP; i += 256 * 16) {
    uint4v piece = {0u, 0u, 0u, 0u};
    if (i < filter_bytes)
      piece = *reinterpret_cast<const uint4v*>(
          reinterpret_cast<const char*>(w) + i);
    *reinterpret_cast<uint4v*>(lds + i) = piece;
  }
  __syncthreads();
  half8 fil[HS][G][NP][2];
#pragma unroll
  for (int h = 0; h < HS; ++h)
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const char* row[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int at = 8 * i + 4 * e + (l16 >> 2) - shift;
        const bool ok = 4 * h + q < g.win_rows && at >= 0 && at < wc;
        row[e] = lds + (ok ? ((4 * h + q) * wc + at) * g.features * 2
                           : filter_bytes) + (l16 & 3) * 16;
      }
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          fil[h][i][p][e] = read_transposed(row[0] + 64 * p + 8 * e,
                                            row[1] + 64 * p + 8 * e);
    }
  __syncthreads();

  // ---- the band's image rows ------------------------------------------------
  const int row_bytes = g.pitch * 2;
  const int row_halves = g.in_cols * C;
  const int before = g.pad_cols * C + shift;  // halves in front of column 0
  const int first_row = 2 * oy0 - g.pad_rows;
  const int rows = 2 * (n_rows - 1) + g.win_rows;
  for (int r = wave; r < rows; r += 4) {
    const int iy = first_row + r;
    const bool live = static_cast<unsigned>(iy) <
                      static_cast<unsigned>(g.in_rows);
    const unsigned from =
        static_cast<unsigned>((n * g.in_rows + iy) * row_halves) * 2u;
    if ((row_halves & 1) == 0) {
#pragma unroll 8
      for (int i = lane; i < g.pitch / 2; i += 64) {
        const int e = 2 * i - before;
        const unsigned two = __builtin_amdgcn_raw_buffer_load_b32(
            x_rsrc, live && e >= 0 && e < row_halves ? from + 2u * e : kOob, 0,
            0);
        *reinterpret_cast<unsigned*>(lds + r * row_bytes + 4 * i) = two;
      }
    } else {
#pragma unroll 8
      for (int i = lane; i < g.pitch; i += 64) {
        const int e = i - before;
        const unsigned short one = __builtin_amdgcn_raw_buffer_load_b16(
            x_rsrc, live && e >= 0 && e < row_halves ? from + 2u * e : kOob, 0,
            0);
        *reinterpret_cast<unsigned short*>(lds + r * row_bytes + 2 * i) = one;
      }
    }
  }
  char* const zeros = lds + g.lds_rows * row_bytes;
  if (threadIdx.x < 16) reinterpret_cast<unsigned*>(zeros)[threadIdx.x] = 0u;

  unsigned keep[G][4];  // halves of operand i that belong to the filter row
#pragma unroll
  for (int i = 0; i < G; ++i)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int at = 8 * i + 2 * d - shift;
      keep[i][d] = (at >= 0 && at < wc ? 0xFFFFu : 0u) |
                   (at + 1 >= 0 && at + 1 < wc ? 0xFFFF0000u : 0u);
    }
  __syncthreads();

  // ---- blocks of 16 pixels ---------------------------------------------------
  const int n_pb = (g.out_cols + 15) >> 4;
  const int n_items = n_rows * n_pb;
  typedef unsigned uint4a4 __attribute__((ext_vector_type(4), aligned(4)));
  struct Pixels { uint4v at[HS][G]; };
  auto fetch = [&](int item, Pixels& px) {
    const int oy = item / n_pb, pb = item - oy * n_pb;
    const char* base = lds + (2 * oy + q) * row_bytes + 4 * C * (16 * pb + l16);
#pragma unroll
    for (int h = 0; h < HS; ++h) {
      const char* from =
          4 * h + q < g.win_rows ? base + 4 * h * row_bytes : zeros;
#pragma unroll
      for (int i = 0; i < G; ++i)
        px.at[h][i] = *reinterpret_cast<const uint4a4*>(from + 16 * i);
    }
  };
  float most = 0.f;  // a NaN once any sum of this lane is
  auto multiply = [&](int item, const Pixels& px) {
    const int oy = item / n_pb, pb = item - oy * n_pb;
    float4v acc[NP][2];
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int e = 0; e < 2; ++e) acc[p][e] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < HS; ++h)
#pragma unroll
      for (int i = 0; i < G; ++i) {
        uint4v b = px.at[h][i];
#pragma unroll
        for (int d = 0; d < 4; ++d) b[d] &= keep[i][d];
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int e = 0; e < 2; ++e)
            acc[p][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                fil[h][i][p][e], __builtin_bit_cast(half8, b), acc[p][e], 0, 0,
                0);
      }
    const int ox = 16 * pb + l16;
    const unsigned at = static_cast<unsigned>(
        ((n * g.out_rows + oy0 + oy) * g.out_cols + ox) * g.features + 8 * q) *
        2u;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          most = __builtin_elementwise_maximum(most, acc[p][e][v]);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      half8 out;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        out[v] = static_cast<_Float16>(acc[p][0][v]);
        out[4 + v] = static_cast<_Float16>(acc[p][1][v]);
      }
      __builtin_amdgcn_raw_buffer_store_b128(
          __builtin_bit_cast(uint4v, out), y_rsrc,
          ox < g.out_cols && 32 * p + 8 * q < g.features ? at + 64u * p : kOob,
          0, 0);
    }
  };
  Pixels even, odd;
  int item = wave;
  if (item < n_items) fetch(item, even);
  while (item < n_items) {
    if (item + 4 < n_items) fetch(item + 4, odd);
    __builtin_amdgcn_sched_barrier(0);
    multiply(item, even);
    item += 4;
    if (item >= n_items) break;
    if (item + 4 < n_items) fetch(item + 4, even);
    __builtin_amdgcn_sched_barrier(0);
    multiply(item, odd);
    item += 4;
  }

  // ---- NaNs of windows that leave the image -----------------------------------
  if (__builtin_amdgcn_ballot_w64(most != most) == 0) return;
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // their stores
  __builtin_amdgcn_sched_barrier(0);
  for (item = wave; item < n_items; item += 4) {
    const int oy = oy0 + item / n_pb, ox = 16 * (item % n_pb) + l16;
    const int iy = 2 * oy - g.pad_rows, ix = 2 * ox - g.pad_cols;
    if (ox >= g.out_cols || (iy >= 0 && iy + g.win_rows <= g.in_rows &&
                             ix >= 0 && ix + g.win_cols <= g.in_cols))
      continue;
    _Float16* const out =
        y + (static_cast<size_t>(n * g.out_rows + oy) * g.out_cols + ox) *
                g.features;
    for (int f = q; f < g.features; f += 4) {
      const _Float16 had = *const_cast<const volatile _Float16*>(out + f);
      if (had == had) continue;
      float sum = 0.f;
      for (int r = max(0, -iy); r < min(g.win_rows, g.in_rows - iy); ++r)
        for (int e = max(0, -ix) * C;
             e < min(g.win_cols, g.in_cols - ix) * C && sum == sum; ++e)
          sum += static_cast<float>(
                     x[(static_cast<size_t>(n * g.in_rows + iy + r) * g.in_cols +
                        ix) * C + e]) *
                 static_cast<float>(w[static_cast<size_t>(r * wc + e) *
                                          g.features + f]);
      out[f] = static_cast<_Float16>(sum);
    }
  }
}

// ---------------------------------------------------------------------------
// Filter gradient.  With the image as 2 x 2 x C planes of half its size,
// plane (a, b, c) at (Y, X) = x[2 Y + a][2 X + b][c], tap r = pad + 2 (lo + tr) +
// a reads plane row oy + lo + tr, the columns likewise:
//   dW[r][s][c][f] = sum over (n, oy, ox) of plane(a, b, c)[oy + lo_r + tr][ox +
//                    lo_c + ts] * dY[n][oy][ox][f].
//
//   * Rows of the product are features (32 per wave), columns pairs of tap rows
//     tr x 16 planes, the reduction 16 pixels of a row: a wave keeps the T sums
//     of the column taps ts.
//   * Planes are written to LDS value by value, eight rows in a ring, so that
//     pixels of a row lie side by side: twelve of them per lane, one 16-byte and
//     one 8-byte read, serve all column taps, cut out at pixel 0 ... 3 (funnel
//     shifts for the odd ones).  dY keeps its layout and passes through
//     transposing reads.
//   * Loads travel through registers two rows ahead; one barrier per row.
//   * Pixels past the end of a row are zeros of dY, and cleared in the planes:
//     a neighbour's infinity must not meet them.
//   * Each wave stores its sums; a second kernel adds those of all work-groups
//     and rounds.
//
// 128 x 224x224x3 -> 64, 7x7: 434 us through fp32 -> 104 us with the sum.
constexpr int kXItems = 4;  // pairs of image values per lane and plane row
constexpr int kYItems = 4;  // 16-byte pieces of dY per lane and row
constexpr int kRing = 8;

template <int T, int NF, int KP>
__global__ void __launch_bounds__(64 * ((T + 1) / 2) * NF * KP, 2)
    few_filter_backprop_f16_kernel(const _Float16* __restrict__ x,
                                   const _Float16* __restrict__ dy,
                                   float4v* __restrict__ part, FewGeom g,
                                   unsigned n_groups) {
  constexpr int RP = (T + 1) / 2;
  constexpr int NT = 64 * RP * NF * KP;
  constexpr int kPixelBytes = 64 * NF;
  extern __shared__ __align__(16) char lds[];
  char* const planes = lds;
  char* const ybuf = lds + 4 * g.channels * g.plane;
  const int y_bytes = g.pixels * kPixelBytes;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kp = wave % KP, rp = wave / KP % RP, nf = wave / (KP * RP);
  const unsigned group = xcd_remap(blockIdx.x, n_groups);
  const int C = g.channels;

  const __amdgpu_buffer_rsrc_t x_rsrc =
      make_rsrc(x, static_cast<size_t>(g.batch) * g.in_rows * g.in_cols * C * 2);
  const __amdgpu_buffer_rsrc_t dy_rsrc =
      make_rsrc(dy, static_cast<size_t>(g.batch) * g.out_rows * g.out_cols *
                        g.features * 2);

  // Which 16-byte position of an LDS pixel of dY holds piece c: c ^ swz.  (At
  // 128 bytes per pixel the four pixels of a transposing read would share
  // banks; 64 and 192 spread them by themselves.)
  auto swz = [](unsigned p) -> unsigned {
    return NF == 2 ? ((p & 3u) ^ ((p >> 3) & 1u)) << 1 : 0u;
  };

  // What this lane loads of a row of dY ...
  unsigned y_from[kYItems], y_to[kYItems];
#pragma unroll
  for (int i = 0; i < kYItems; ++i) {
    const unsigned idx = threadIdx.x + NT * i;
    const unsigned p = idx / (4 * NF), piece = idx % (4 * NF);
    const bool ok = p < static_cast<unsigned>(g.out_cols) &&
                    static_cast<int>(8 * piece) < g.features;
    y_from[i] = ok ? (p * g.features + 8 * piece) * 2u : kOob;
    y_to[i] = p < static_cast<unsigned>(g.pixels)
                  ? p * kPixelBytes + ((piece ^ swz(p)) << 4) : kOob;
  }
  // ... and of the two image rows of a plane row: a pair of values each.
  const int row_halves = g.in_cols * C;
  const int row_pairs = (row_halves + 1) >> 1;
  const bool aligned = (row_halves & 1) == 0;
  unsigned x_from[kXItems], x_to[kXItems][2];
  int x_a[kXItems];
#pragma unroll
  for (int i = 0; i < kXItems; ++i) {
    const int idx = static_cast<int>(threadIdx.x) + NT * i;
    const int a = idx >= row_pairs ? 1 : 0;
    const int e = 2 * (idx - a * row_pairs);
    x_a[i] = a;
    x_from[i] = e < row_halves ? static_cast<unsigned>(e) * 2u : kOob;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int col = (e + u) / C, c = e + u - col * C;
      const int at = (col >> 1) - g.lo_c;
      x_to[i][u] = e + u < row_halves && at < g.out_cols + T - 1
                       ? static_cast<unsigned>(
                             ((2 * a + (col & 1)) * C + c) * g.plane + 2 * at)
                       : kOob;
    }
  }
  struct XRow { unsigned at[kXItems]; };
  struct YRow { uint4v at[kYItems]; };
  auto load_x = [&](int n, int row, XRow& v) {  // row of the planes
#pragma unroll
    for (int i = 0; i < kXItems; ++i) {
      const int iy = 2 * row + x_a[i];
      const bool ok = static_cast<unsigned>(iy) <
                          static_cast<unsigned>(g.in_rows) &&
                      x_from[i] != kOob;
      const unsigned from =
          static_cast<unsigned>((n * g.in_rows + iy) * row_halves) * 2u +
          x_from[i];
      if (aligned) {
        v.at[i] = __builtin_amdgcn_raw_buffer_load_b32(x_rsrc,
                                                       ok ? from : kOob, 0, 0);
      } else {
        const unsigned low = __builtin_amdgcn_raw_buffer_load_b16(
            x_rsrc, ok ? from : kOob, 0, 0);
        const unsigned high = __builtin_amdgcn_raw_buffer_load_b16(
            x_rsrc, ok && x_to[i][1] != kOob ? from + 2u : kOob, 0, 0);
        v.at[i] = (low & 0xFFFFu) | high << 16;
      }
    }
  };
  auto write_x = [&](int slot, const XRow& v) {
    char* const to = planes + slot * g.pitch;
#pragma unroll
    for (int i = 0; i < kXItems; ++i)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (x_to[i][u] != kOob)
          *reinterpret_cast<unsigned short*>(to + x_to[i][u]) =
              static_cast<unsigned short>(v.at[i] >> (16 * u));
  };
  auto load_y = [&](int n, int oy, bool live, YRow& v) {
    const unsigned from = static_cast<unsigned>(n * g.out_rows + oy) *
                          static_cast<unsigned>(g.out_cols * g.features * 2);
#pragma unroll
    for (int i = 0; i < kYItems; ++i)
      v.at[i] = __builtin_amdgcn_raw_buffer_load_b128(
          dy_rsrc, live && y_from[i] != kOob ? from + y_from[i] : kOob, 0, 0);
  };
  auto write_y = [&](int buf, const YRow& v) {
    char* const to = ybuf + buf * y_bytes;
#pragma unroll
    for (int i = 0; i < kYItems; ++i)
      if (y_to[i] != kOob) *reinterpret_cast<uint4v*>(to + y_to[i]) = v.at[i];
  };

  // Operands of chunk 0: dY, features 32 nf + lane % 32 at pixels 8 (lane / 32)
  // ... + 7, and the planes.
  const int half = lane >> 5, gq = lane >> 4, j = (lane >> 2) & 3, e4 = lane & 3;
  unsigned y_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const unsigned p = 8 * half + 4 * h + j;
    const unsigned piece = 4 * nf + 2 * (gq & 1) + (e4 >> 1);
    y_off[h] = p * kPixelBytes + ((piece ^ swz(p)) << 4) + ((e4 & 1) << 3);
  }
  const int m = lane & 31;
  const int my_tr = min(2 * rp + (m >> 4), T - 1);
  const unsigned x_off = min(m & 15, 4 * C - 1) * g.plane + 16 * half;
  const int n_chunks = g.pixels >> 4;
  // halves of the last chunk that are pixels of the row
  unsigned keep[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int p = 16 * (n_chunks - 1) + 8 * half + 2 * d;
    keep[d] = (p < g.out_cols ? 0xFFFFu : 0u) |
              (p + 1 < g.out_cols ? 0xFFFF0000u : 0u);
  }
  const bool ragged = (g.out_cols & 15) != 0;

  float16v acc[T];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;

  struct Operands { half8 y; uint4v lo; uint2v hi; };
  auto multiply_row = [&](int k) {
    const char* const yr = ybuf + (k & 1) * y_bytes;
    const char* const xr =
        planes + ((k + my_tr) & (kRing - 1)) * g.pitch + x_off;
    auto fetch = [&](int c, Operands& o) {
      o.y = read_transposed(yr + y_off[0] + c * (16 * kPixelBytes),
                            yr + y_off[1] + c * (16 * kPixelBytes));
      o.lo = *reinterpret_cast<const uint4v*>(xr + 32 * c);
      o.hi = *reinterpret_cast<const uint2v*>(xr + 32 * c + 16);
    };
    auto multiply = [&](int c, const Operands& o) {
      const unsigned v[6] = {o.lo[0], o.lo[1], o.lo[2], o.lo[3], o.hi[0],
                             o.hi[1]};
      const bool last = ragged && c == n_chunks - 1;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        uint4v b;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          b[d] = (t & 1) != 0
                     ? __builtin_amdgcn_alignbit(v[t / 2 + d + 1], v[t / 2 + d],
                                                 16)
                     : v[t / 2 + d];
        if (last) {
#pragma unroll
          for (int d = 0; d < 4; ++d) b[d] &= keep[d];
        }
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            o.y, __builtin_bit_cast(half8, b), acc[t], 0, 0, 0);
      }
    };
    Operands even, odd;
    int c = kp;
    if (c >= n_chunks) return;
    fetch(c, even);
    for (;;) {
      if (c + KP < n_chunks) fetch(c + KP, odd);
      __builtin_amdgcn_sched_barrier(0);
      multiply(c, even);
      if ((c += KP) >= n_chunks) break;
      if (c + KP < n_chunks) fetch(c + KP, even);
      __builtin_amdgcn_sched_barrier(0);
      multiply(c, odd);
      if ((c += KP) >= n_chunks) break;
    }
  };

  // (columns of the planes outside the image are never written)
  for (int i = threadIdx.x * 4; i < 4 * C * g.plane; i += NT * 4)
    *reinterpret_cast<unsigned*>(planes + i) = 0u;

  const int unit_end = min(g.units, static_cast<int>(group + 1) * g.per_group);
  for (int unit = group * g.per_group; unit < unit_end; ++unit) {
    const int n = unit / g.bands;
    const int oy0 = (unit - n * g.bands) * g.band;
    const int n_rows = min(g.band, g.out_rows - oy0);
    const int row0 = oy0 + g.lo_r;  // of the planes
    XRow xa[T], xe, xo;
    YRow ye, yo;
    load_y(n, oy0, true, ye);
#pragma unroll
    for (int t = 0; t < T; ++t) load_x(n, row0 + t, xa[t]);
    load_y(n, oy0 + 1, 1 < n_rows, yo);
    load_x(n, row0 + T, xo);
    lds_barrier();  // the planes are cleared, the last band is multiplied
    write_y(0, ye);
#pragma unroll
    for (int t = 0; t < T; ++t) write_x(t, xa[t]);
    lds_barrier();
    // (row k in buffer k % 2, plane rows k ... k + T - 1 in their slots; the
    // registers hold what row k + 1 adds)
    int k = 0;
#define SNN_FEW_STEP(ynext, xnext, yafter, xafter)          \
  {                                                         \
    load_y(n, oy0 + k + 2, k + 2 < n_rows, yafter);         \
    load_x(n, row0 + k + T + 1, xafter);                    \
    __builtin_amdgcn_sched_barrier(0);                      \
    multiply_row(k);                                        \
    write_y((k + 1) & 1, ynext);                            \
    write_x((k + T) & (kRing - 1), xnext);                  \
    lds_barrier();                                          \
    if (++k >= n_rows) break;                               \
  }
    for (;;) {
      SNN_FEW_STEP(yo, xo, ye, xe)
      SNN_FEW_STEP(ye, xe, yo, xo)
    }
#undef SNN_FEW_STEP
  }

  float4v* const out =
      part + (static_cast<size_t>(group * KP + kp) * (RP * NF) + rp * NF + nf) *
                 (T * 256) + lane;
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[(t * 4 + i) * 64] = float4v{acc[t][4 * i], acc[t][4 * i + 1],
                                      acc[t][4 * i + 2], acc[t][4 * i + 3]};
}

// Adds the partial sums, 16 consecutive float4 x 16 groups of parts per
// work-group, and rounds.
__global__ void __launch_bounds__(256)
    few_filter_backprop_reduce_kernel(const float4v* __restrict__ part,
                                      _Float16* __restrict__ dw, FewGeom g,
                                      int taps, int nf_count, int n_parts) {
  __shared__ float4v sums[16][16];
  const int part_vecs = (taps + 1) / 2 * nf_count * taps * 256;
  const int at = blockIdx.x * 16 + (threadIdx.x & 15);
  const int from = threadIdx.x >> 4;
  float4v sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int i = from; i < n_parts; i += 16)
    sum += part[static_cast<size_t>(i) * part_vecs + at];
  sums[from][threadIdx.x & 15] = sum;
  __syncthreads();
  if (from != 0) return;
  for (int i = 1; i < 16; ++i) sum += sums[i][threadIdx.x];
  // features 32 nf + 8 i + 4 (lane / 32) ... + 3 of tap row 2 rp + (lane & 16) /
  // 16, column tap ts, plane lane & 15
  const int lane = at & 63, i = (at >> 6) & 3;
  const int ts = (at >> 8) % taps, block = (at >> 8) / taps;
  const int nf = block % nf_count, rp = block / nf_count;
  const int tr = 2 * rp + ((lane >> 4) & 1), plane = lane & 15;
  const int c = plane % g.channels, b = plane / g.channels & 1;
  const int a = plane / g.channels >> 1;
  const int r = g.pad_rows + 2 * (g.lo_r + tr) + a;
  const int s = g.pad_cols + 2 * (g.lo_c + ts) + b;
  const int f = 32 * nf + 8 * i + 4 * (lane >> 5);
  if (a > 1 || tr >= taps || r < 0 || r >= g.win_rows || s < 0 ||
      s >= g.win_cols || f >= g.features)
    return;
  typedef _Float16 half4v __attribute__((ext_vector_type(4)));
  half4v out;
#pragma unroll
  for (int v = 0; v < 4; ++v) out[v] = static_cast<_Float16>(sum[v]);
  *reinterpret_cast<half4v*>(
      dw + ((r * g.win_cols + s) * g.channels + c) * g.features + f) = out;
}

// The half-size taps of one axis of the input gradient: first (relative to the
// pixel pair) and how many.
int gradient_taps(int window, int pad, int* lo) {
  auto floor_half = [](int v) { return v >= 0 ? v / 2 : -((1 - v) / 2); };
  const int hi = floor_half(1 + pad);
  *lo = floor_half(pad - (window - 1) + 1);
  return hi - *lo + 1;
}

// What all three directions ask for.  96 features are three blocks of 32, which
// fill the registers: 351 of 512 for the gradient's filter and accumulators of
// four half-size taps, 237 of 256 for the forward's.  More features take the other
// kernels: 16x224x224x3, 7x7, three directions 20 / 21 / 42 us with 96 features,
// 38 / 189 / 179 with 104.
bool few_shape(const snn_hip_conv2d_params& p) {
  return p.stride_rows == 2 && p.stride_cols == 2 && p.channels >= 1 &&
         p.channels <= kMaxChannels && p.features % 8 == 0 &&
         p.features <= 96 && p.window_rows >= 2 && p.window_cols >= 2 &&
         p.window_rows <= 8 && p.window_cols <= 8 && p.pad_rows >= 0 &&
         p.pad_cols >= 0 && p.pad_rows < p.window_rows &&
         p.pad_cols < p.window_cols && p.batch >= 1 && p.out_rows >= 1 &&
         p.out_cols >= 1 &&
         static_cast<size_t>(p.batch) * p.in_rows * p.in_cols * p.channels * 2 <=
             kMaxBufferBytes &&
         static_cast<size_t>(p.batch) * p.out_rows * p.out_cols * p.features *
                 2 <= kMaxBufferBytes;
}

FewGeom few_geom(const snn_hip_conv2d_params& p) {
  FewGeom g = {};
  g.batch = p.batch; g.in_rows = p.in_rows; g.in_cols = p.in_cols;
  g.channels = p.channels; g.out_rows = p.out_rows; g.out_cols = p.out_cols;
  g.features = p.features; g.win_rows = p.window_rows;
  g.win_cols = p.window_cols; g.pad_rows = p.pad_rows; g.pad_cols = p.pad_cols;
  return g;
}

// Rows per band: the fewest rounds of `slots` bands over the chip, times what
// one band costs -- its rows and `extra` more.
int choose_band(int rows, long bands_of_one_row, long slots, int extra) {
  long best_cost = LONG_MAX;
  int best = rows;
  for (int n = 1; n <= rows; ++n) {
    const int band = ceil_div(rows, n);
    const long units = bands_of_one_row * ceil_div(rows, band);
    const long cost = (units + slots - 1) / slots * (band + extra);
    if (cost < best_cost) {
      best_cost = cost;
      best = band;
    }
  }
  return best;
}

int input_backprop_taps(const snn_hip_conv2d_params& p, FewGeom* g) {
  return std::max({gradient_taps(p.window_rows, p.pad_rows, &g->lo_r),
                   gradient_taps(p.window_cols, p.pad_cols, &g->lo_c), 2});
}

// The same for the filter gradient: plane rows (or columns) of tap 0, relative
// to the output pixel.
int filter_taps(int window, int pad, int* lo) {
  *lo = -((pad + 1) / 2);
  const int last = window - 1 - pad;  // >= 0
  return last / 2 - *lo + 1;
}

struct ForwardPlan {
  FewGeom g;
  int halves = 0, octets = 0, pairs = 0;  // HS, G, NP
  size_t lds_bytes = 0;
};

bool forward_plan(const snn_hip_conv2d_params& p, ForwardPlan* plan) {
  if (!few_shape(p)) return false;
  FewGeom& g = plan->g;
  g = few_geom(p);
  const int wc = p.window_cols * p.channels;
  plan->octets = std::max(2, ceil_div((p.pad_cols * p.channels & 1) + wc, 8));
  plan->halves = p.window_rows > 4 || plan->octets > 2 ? 2 : 1;
  plan->pairs = ceil_div(p.features, 32);
  if (plan->octets > 3) return false;
  const int n_pb = ceil_div(p.out_cols, 16);
  // what the last block of pixels reads, in 16-byte steps
  g.pitch = ceil_div(2 * p.channels * (16 * n_pb - 1) + 8 * plan->octets, 8) * 8;
  const size_t filter_bytes =
      static_cast<size_t>(p.window_rows) * wc * p.features * 2 +
      64 * plan->pairs;
  // Two work-groups per CU, which stage and multiply in turn: 78 KB each.
  const size_t max_lds = 78 * 1024;
  const int max_rows =
      static_cast<int>((max_lds - 64) / (static_cast<size_t>(g.pitch) * 2));
  if (max_rows < p.window_rows + 2 || filter_bytes > max_lds) return false;
  const int max_band = (max_rows - p.window_rows) / 2 + 1;
  // (filter and first rows cost about three rows)
  long best_cost = LONG_MAX;
  for (int n = 1; n <= p.out_rows; ++n) {
    const int band = ceil_div(p.out_rows, n);
    if (band > max_band) continue;
    const long units = static_cast<long>(p.batch) * ceil_div(p.out_rows, band);
    // (a wave takes every fourth block of 16 pixels)
    const long cost = (units + 2 * kNumCus - 1) / (2 * kNumCus) *
                      (ceil_div(band * n_pb, 4) + 6);
    if (cost < best_cost) {
      best_cost = cost;
      g.band = band;
    }
  }
  g.bands = ceil_div(p.out_rows, g.band);
  g.lds_rows = 2 * (g.band - 1) + p.window_rows;
  plan->lds_bytes = std::max(
      filter_bytes, static_cast<size_t>(g.lds_rows) * g.pitch * 2 + 64);
  return true;
}

struct FilterPlan {
  FewGeom g;
  int taps = 0, nf = 0, kp = 0;
  unsigned groups = 0;
  size_t lds_bytes = 0;
  size_t part_floats() const {
    return static_cast<size_t>(groups) * kp * ((taps + 1) / 2 * nf * taps) *
           1024;
  }
};

bool filter_plan(const snn_hip_conv2d_params& p, FilterPlan* plan) {
  if (!few_shape(p)) return false;
  FewGeom& g = plan->g;
  g = few_geom(p);
  plan->taps = std::max({filter_taps(p.window_rows, p.pad_rows, &g.lo_r),
                         filter_taps(p.window_cols, p.pad_cols, &g.lo_c), 2});
  if (plan->taps > 4) return false;
  plan->nf = ceil_div(p.features, 32);
  const int waves = (plan->taps + 1) / 2 * plan->nf;
  // (four or six waves: with fewer, several share the chunks of a row)
  plan->kp = waves == 1 ? 4 : waves < 4 ? 2 : 1;
  const int threads = 64 * waves * plan->kp;
  g.pixels = ceil_div(p.out_cols, 16) * 16;
  if (g.pixels * 4 * plan->nf > kYItems * threads ||
      2 * ((p.in_cols * p.channels + 1) / 2) > kXItems * threads)
    return false;
  // a lane reads twelve halves from each eighth pixel on; planes an odd number
  // of 16-byte steps apart
  g.pitch = ceil_div(2 * (g.pixels + 4), 16) * 16;
  g.plane = kRing * g.pitch + 16;
  plan->lds_bytes = static_cast<size_t>(4 * p.channels) * g.plane +
                    static_cast<size_t>(2) * g.pixels * 64 * plan->nf;
  if (plan->lds_bytes > 80 * 1024) return false;
  // Two work-groups per CU, one band each while there are few.
  const int slots = 2 * kNumCus;
  g.band = choose_band(p.out_rows, p.batch, slots, plan->taps + 4);
  g.bands = ceil_div(p.out_rows, g.band);
  g.units = p.batch * g.bands;
  g.per_group = ceil_div(g.units, slots);
  plan->groups = static_cast<unsigned>(ceil_div(g.units, g.per_group));
  return true;
}

}  // namespace

bool conv2d_few_f16_forward_supports(const snn_hip_conv2d_params& p) {
  ForwardPlan plan;
  return forward_plan(p, &plan);
}

int launch_conv2d_few_f16_forward(const _Float16* x, const _Float16* w,
                                  _Float16* y, const snn_hip_conv2d_params& p,
                                  hipStream_t stream) {
  ForwardPlan plan;
  if (!forward_plan(p, &plan)) return SNN_HIP_INVALID_ALGORITHM;
  const unsigned groups = static_cast<unsigned>(p.batch) * plan.g.bands;
  KernelTimer timer(stream);
#define SNN_FEW_LAUNCH(HS, G, NP)                                             \
  {                                                                           \
    static const hipError_t attr = hipFuncSetAttribute(                       \
        reinterpret_cast<const void*>(few_forward_f16_kernel<HS, G, NP>),     \
        hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);               \
    (void)attr;                                                               \
    hipLaunchKernelGGL((few_forward_f16_kernel<HS, G, NP>), dim3(groups),     \
                       dim3(256), plan.lds_bytes, stream, x, w, y, plan.g,    \
                       groups);                                               \
  }
#define SNN_FEW_LAUNCH_NP(HS, G)                 \
  switch (plan.pairs) {                          \
    case 1: SNN_FEW_LAUNCH(HS, G, 1) break;      \
    case 2: SNN_FEW_LAUNCH(HS, G, 2) break;      \
    default: SNN_FEW_LAUNCH(HS, G, 3)            \
  }
  if (plan.halves == 1) SNN_FEW_LAUNCH_NP(1, 2)
  else if (plan.octets == 2) SNN_FEW_LAUNCH_NP(2, 2)
  else SNN_FEW_LAUNCH_NP(2, 3)
#undef SNN_FEW_LAUNCH_NP
#undef SNN_FEW_LAUNCH
  SNN_HIP_CHECK_LAUNCH();
  return SNN_HIP_OK;
}

size_t conv2d_few_f16_filter_backprop_partial_floats(
    const snn_hip_conv2d_params& p) {
  FilterPlan plan;
  return filter_plan(p, &plan) ? plan.part_floats() : 0;
}

// Returns -1 when there is no room for its partial sums.
int launch_conv2d_few_f16_filter_backprop(const _Float16* x,
                                          const _Float16* dy, _Float16* dw,
                                          const snn_hip_conv2d_params& p,
                                          _Float16* workspace,
                                          size_t workspace_elems,
                                          hipStream_t stream) {
  FilterPlan plan;
  if (!filter_plan(p, &plan)) return SNN_HIP_INVALID_ALGORITHM;
  const FewGeom& g = plan.g;
  const size_t need = 2 * plan.part_floats();
  float4v* part = reinterpret_cast<float4v*>(workspace);
  const bool temporary = workspace == nullptr || workspace_elems < need ||
                         (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0;
  if (temporary) {
    void* ptr = nullptr;
    if (temp_malloc_async(&ptr, need * sizeof(_Float16), stream) !=
        hipSuccess) {
      (void)hipGetLastError();
      return -1;
    }
    part = static_cast<float4v*>(ptr);
  }
  {
    KernelTimer timer(stream);
#define SNN_FEW_LAUNCH(T, NF, KP)                                             \
  {                                                                           \
    static const hipError_t attr = hipFuncSetAttribute(                       \
        reinterpret_cast<const void*>(                                        \
            few_filter_backprop_f16_kernel<T, NF, KP>),                       \
        hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);               \
    (void)attr;                                                               \
    hipLaunchKernelGGL((few_filter_backprop_f16_kernel<T, NF, KP>),           \
                       dim3(plan.groups),                                     \
                       dim3(64 * ((T + 1) / 2) * NF * KP), plan.lds_bytes,    \
                       stream, x, dy, part, g, plan.groups);                  \
  }
    switch (plan.taps * 4 + plan.nf) {
      case 2 * 4 + 1: SNN_FEW_LAUNCH(2, 1, 4) break;
      case 2 * 4 + 2: SNN_FEW_LAUNCH(2, 2, 2) break;
      case 2 * 4 + 3: SNN_FEW_LAUNCH(2, 3, 2) break;
      case 3 * 4 + 1: SNN_FEW_LAUNCH(3, 1, 2) break;
      case 3 * 4 + 2: SNN_FEW_LAUNCH(3, 2, 1) break;
      case 3 * 4 + 3: SNN_FEW_LAUNCH(3, 3, 1) break;
      case 4 * 4 + 1: SNN_FEW_LAUNCH(4, 1, 2) break;
      case 4 * 4 + 2: SNN_FEW_LAUNCH(4, 2, 1) break;
      default: SNN_FEW_LAUNCH(4, 3, 1)
    }
#undef SNN_FEW_LAUNCH
  }
  hipLaunchKernelGGL(
      few_filter_backprop_reduce_kernel,
      dim3((plan.taps + 1) / 2 * plan.nf * plan.taps * 16), dim3(256), 0,
      stream, part, dw, g, plan.taps, plan.nf,
      static_cast<int>(plan.groups) * plan.kp);
  const hipError_t err = hipGetLastError();
  if (temporary) temp_free_async(part, stream);
  if (err != hipSuccess) return report_hip_error(err, "few_filter_backprop");
  return SNN_HIP_OK;
}

bool conv2d_few_f16_input_backprop_supports(const snn_hip_conv2d_params& p) {
  if (!few_shape(p)) return false;
  FewGeom g = few_geom(p);
  return input_backprop_taps(p, &g) <= 4;
}

int launch_conv2d_few_f16_input_backprop(const _Float16* dy, const _Float16* w,
                                         _Float16* dx,
                                         const snn_hip_conv2d_params& p,
                                         hipStream_t stream) {
  FewGeom g = few_geom(p);
  const int taps = input_backprop_taps(p, &g);
  const int ks = ceil_div(p.features, 32);
  const int pair_rows = (p.in_rows + 1) / 2, pair_cols = (p.in_cols + 1) / 2;
  g.col_blocks = ceil_div(pair_cols, 32);
  // (two waves per SIMD; V and the first row cost about three rows)
  g.band = choose_band(pair_rows, static_cast<long>(p.batch) * g.col_blocks,
                       kNumCus * (ks < 3 ? 8 : 4), taps + 2);
  g.bands = ceil_div(pair_rows, g.band);
  const unsigned units = static_cast<unsigned>(p.batch) * g.bands * g.col_blocks;
  const unsigned groups = ceil_div(units, 4u);
  KernelTimer timer(stream);
#define SNN_FEW_LAUNCH(T, KS)                                              \
  hipLaunchKernelGGL((few_input_backprop_f16_kernel<T, KS>), dim3(groups), \
                     dim3(256), 0, stream, dy, w, dx, g, groups, units)
#define SNN_FEW_LAUNCH_KS(T)          \
  switch (ks) {                       \
    case 1: SNN_FEW_LAUNCH(T, 1); break; \
    case 2: SNN_FEW_LAUNCH(T, 2); break; \
    default: SNN_FEW_LAUNCH(T, 3);    \
  }
  switch (taps) {
    case 2: SNN_FEW_LAUNCH_KS(2) break;
    case 3: SNN_FEW_LAUNCH_KS(3) break;
    default: SNN_FEW_LAUNCH_KS(4)
  }
#undef SNN_FEW_LAUNCH_KS
#undef SNN_FEW_LAUNCH
  SNN_HIP_CHECK_LAUNCH();
  return SNN_HIP_OK;
}

}  // namespace snn
