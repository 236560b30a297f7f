// fp32 filter gradient of 3x3 and 5x5 windows at stride 1 on the binary16 matrix
// instruction (gfx950): both operands as the sum of two binary16 values
// (conv2d_halves_f32.hip), fp32 accumulation.
//
//   dW[r][s][c][k] = sum over (n, oy, ox) of
//                    X[n][oy + r - pr][ox + s - pc][c] * dY[n][oy][ox][k]
//
// (the FilterBackprop direction of sycldnn::conv2d::launch,
// include/portdnn/conv2d/launch.h:59-118.)  The reduction runs over pixels, the slow
// dimension of both operands; ds_read_b64_tr_b16 transposes them on the way out of
// LDS: within 16 lanes, lane 4 j + i supplies the address of four consecutive halves
// (columns 4 i ... 4 i + 3) of row j, and lane t receives column t of rows 0 ... 3.
//
//   * A work-group owns a tile of channels x features for a group of taps and a run of
//     bands: some output rows of a segment of columns.  A band's input pixels (with
//     halo) and dY pixels lie in LDS with the same row pitch, zeros in dY's halo
//     columns, so that the operand of a tap is the run of input pixels m + constant.
//   * Four waves multiply, four load the next task's pixels meanwhile and take them
//     apart on their way into LDS, [pixel][hi of all channels, lo, 32 bytes].
//   * The windows of 32 input pixels at pixel 0, 2, ... of a tap row are read; the ones
//     between are put together from these, one funnel shift per register.
//   * Exponents are chosen for a task's pixels of either operand; where a task holds
//     values too small for its exponent it is taken again with these alone, and what
//     that does not hold makes the work-group sum its bands on the fp32 instruction.
//   * The work-groups that share a tile store partial filters, each several where one
//     sum would add too many pixels for its error, which a second launch adds in order.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gemm_tile.h"
#include "halves.h"
#include "plan_cache.h"
#include "snn_kernels.h"

namespace snn {
namespace {

using gemm::xcd_remap;
using namespace halves;

typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

constexpr int kChunk = 32;    // pixels per matrix instruction
constexpr int kNY = 8;        // 16-byte pieces of a task's dY per loading lane
constexpr int kLoaders = 256; // lanes that load

struct FilterHalves {
  int batch, in_rows, in_cols, channels, out_rows, out_cols, features;
  int win_rows, win_cols, pad_rows, pad_cols;
  int seg_cols, segs;          // output columns per segment, segments of a row
  int pitch;                   // seg_cols + halo columns
  int band, bands_per_image;   // output rows per band
  int n_bands;                 // batch * bands_per_image * segs
  int group;                   // bands per task
  int n_tasks, per_split;
  int per_sum, sums;           // tasks that a sum adds up, sums of a split
  int n_slices;                // partial filters
  int x_px, y_px;              // LDS pixels of a band (y_px in whole chunks)
  int tap_groups, c_tiles, f_tiles, n_splits;
  Divisor by_pitch, by_x_px, by_y_px, by_segs, by_bands;
};

// What the barrier in front of a task announces.  kWhole: all its values are in LDS;
// kPass, kLastPass: some of them, the others follow; kPlain: the run of bands has to
// be summed on the fp32 instruction.
enum { kWhole, kPass, kLastPass, kPlain };
struct alignas(16) Task {
  int kind;
  int by;       // the sums' exponent changes by this in front of it ...
  int back;     // ... and by this behind it
  int acc_exp;  // the sums' exponent behind it
};

// Bytes of a pixel in LDS: its channels as hi and lo, and what puts the 32 bytes of
// four pixels that 16 lanes read together into different banks (of 32 a cycle).
constexpr int slot_bytes(int channels) { return channels * 4 + 32; }

__device__ __forceinline__ uint2v read_transposed(const unsigned char* at) {
  return __builtin_bit_cast(
      uint2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at)));
}

// Register `at` of the window of eight pixels between two that start a pixel before
// and a pixel after it.
__device__ __forceinline__ unsigned between(const uint4v& before, const uint4v& after,
                                            int at) {
  return __builtin_amdgcn_alignbit(at < 3 ? before[at + 1] : after[3], before[at],
                                   16);
}

// 17x27x27 96 -> 256, 5x5: 81 us with the launch that adds (179 on the fp32
// instruction); 28x28x128 at batch 32, 3x3: 34 (51 by Winograd's transform),
// 64x64x256 at batch 8: 126 (196).  A chunk's 54 (60) matrix instructions of a wave
// are 864 (960) cycles, half the time: the vector instructions of the SIMD's other
// wave, 22 per piece of 16 bytes for scaling, taking apart and noting the range, take
// turns with them.  So the range of a task is looked at while its values are taken
// apart with the exponents of the one before, and a task that does not fit is taken
// again (a pass of its own over the registers: 6900 -> 15000 cycles a task), slots
// are as many as the template's pieces (a test around each: 7.4 -> 13), and of the
// windows only the odd ones cost instructions.
// TR x TC taps; 2 x 2 waves of CB blocks of 16 channels and FB of 16 features; NX and
// kNY pieces of 16 bytes per loading lane.
template <int TR, int TC, int CB, int FB, int NX>
__global__ void __launch_bounds__(512)
    __attribute__((amdgpu_waves_per_eu(2, 2)))
    filter_halves_kernel(const float* __restrict__ x, const float* __restrict__ dy,
                         float* __restrict__ part, FilterHalves g,
                         unsigned x_bytes, unsigned y_bytes, unsigned n_groups) {
  constexpr int CT = 32 * CB, FT = 32 * FB;  // channels, features of the tile
  constexpr int XS = slot_bytes(CT), YS = slot_bytes(FT);
  constexpr int XP = CT / 4, YP = FT / 4;    // pieces per pixel
  constexpr int XL = kLoaders / XP, YL = kLoaders / YP;  // pixels per piece
  constexpr int XW = XL / 4, YW = YL / 4;                // ... of a wave
  constexpr int kXSlots = NX * XL, kYSlots = kNY * YL;
  constexpr int kEntries = NX * XW + kNY * YW;  // of the table, per wave
  constexpr int kPerLane = (kEntries + 63) / 64;
  constexpr int kYAt = kXSlots * XS, kBufBytes = kYAt + kYSlots * YS;
  constexpr int NU = TR * CB;                // units of a chunk: tap row, channels
  extern __shared__ __align__(16) unsigned char lds[];
  Range* const ranges = reinterpret_cast<Range*>(lds);   // [2][4]
  Task* const tasks = reinterpret_cast<Task*>(lds + 64); // [2]
  uint4v* const bad = reinterpret_cast<uint4v*>(lds + 96);  // [2], a word per wave
  unsigned* const table = reinterpret_cast<unsigned*>(lds + 128);
  unsigned char* const tiles = lds + 128 + (kXSlots + kYSlots) * 4;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned group = xcd_remap(blockIdx.x, n_groups);
  const int n_units = g.tap_groups * g.c_tiles * g.f_tiles;
  const int unit_id = static_cast<int>(group % n_units);
  const int split = static_cast<int>(group / n_units);
  const int tg = unit_id % g.tap_groups;
  const int ct = unit_id / g.tap_groups % g.c_tiles;
  const int ft = unit_id / g.tap_groups / g.c_tiles;
  const int task_begin = split * g.per_split;
  const int task_end = min(g.n_tasks, task_begin + g.per_split);
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto any_bad = [&](int buf) {
    const uint4v v = bad[buf];
    return __builtin_amdgcn_readfirstlane(v[0] | v[1] | v[2] | v[3]) != 0;
  };

  if (wave >= 4) {
    __builtin_amdgcn_s_setprio(2);
    const int tid = threadIdx.x - kLoaders;
    const int w = wave - 4;
    const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, x_bytes);
    const __amdgpu_buffer_rsrc_t y_rsrc = make_rsrc(dy, y_bytes);
    const unsigned x_c = static_cast<unsigned>(ct * CT + tid % XP * 4);
    const unsigned y_f = static_cast<unsigned>(ft * FT + tid % YP * 4);
    const unsigned x_past = x_c < static_cast<unsigned>(g.channels) ? 0u : kOob;
    const unsigned y_past = y_f < static_cast<unsigned>(g.features) ? 0u : kOob;

    // A wave loads the pixels of its own slots, so that it writes the table of where
    // they are (kOob: nowhere) for itself.  Here a lane's entries: the slot, the band
    // of the task, row and column within it.
    int entry_slot[kPerLane], entry_band[kPerLane], entry_row[kPerLane],
        entry_col[kPerLane];
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) {
      const int e = lane + 64 * k;
      const bool is_x = e < NX * XW;
      const int ye = e - NX * XW;
      const int s = is_x ? e / XW * XL + w * XW + e % XW
                         : ye / YW * YL + w * YW + ye % YW;
      const int b = divide(s, is_x ? g.by_x_px : g.by_y_px);
      const int at = s - b * (is_x ? g.x_px : g.y_px);
      const int row = divide(at, g.by_pitch), col = at - row * g.pitch;
      const bool ok =
          e < kEntries && b < g.group &&
          (is_x ? row < g.band + TR - 1 : row < g.band && col < g.seg_cols);
      entry_slot[k] = is_x ? s : kXSlots + s;
      entry_band[k] = ok ? b : -1;
      entry_row[k] = is_x ? row + tg * TR - g.pad_rows : row;
      entry_col[k] = is_x ? col - g.pad_cols : col;
    }
    auto fill_table = [&](int task) {
#pragma unroll
      for (int k = 0; k < kPerLane; ++k) {
        const bool is_x = entry_slot[k] < kXSlots;
        const int gb = task * g.group + entry_band[k];
        const int t = divide(gb, g.by_segs), seg = gb - t * g.segs;
        const int n_img = divide(t, g.by_bands);
        const int row = (t - n_img * g.bands_per_image) * g.band + entry_row[k];
        const int col = seg * g.seg_cols + entry_col[k];
        const int rows = is_x ? g.in_rows : g.out_rows;
        const int cols = is_x ? g.in_cols : g.out_cols;
        const bool ok = entry_band[k] >= 0 && gb < g.n_bands &&
                        static_cast<unsigned>(row) < static_cast<unsigned>(rows) &&
                        static_cast<unsigned>(col) < static_cast<unsigned>(cols);
        const int pixel = (n_img * rows + row) * cols + col;
        const unsigned at =
            static_cast<unsigned>(pixel * (is_x ? g.channels : g.features)) * 4u;
        if (lane + 64 * k < kEntries) table[entry_slot[k]] = ok ? at : kOob;
      }
    };
    float4v vx[NX], vy[kNY];
    auto load_pieces = [&]() {
      unsigned ax[NX], ay[kNY];
#pragma unroll
      for (int i = 0; i < NX; ++i) ax[i] = table[tid / XP + i * XL];
#pragma unroll
      for (int i = 0; i < kNY; ++i) ay[i] = table[kXSlots + tid / YP + i * YL];
#pragma unroll
      for (int i = 0; i < NX; ++i)
        vx[i] = __builtin_bit_cast(
            float4v, __builtin_amdgcn_raw_buffer_load_b128(
                         x_rsrc, (ax[i] + x_c * 4u) | x_past, 0, 0));
#pragma unroll
      for (int i = 0; i < kNY; ++i)
        vy[i] = __builtin_bit_cast(
            float4v, __builtin_amdgcn_raw_buffer_load_b128(
                         y_rsrc, (ay[i] + y_f * 4u) | y_past, 0, 0));
    };
    auto range_of = [&](const float4v* v, int n) {
      Range r = {0u, 0xFFFFFFFFu};
#pragma unroll
      for (int i = 0; i < n; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) note(r, v[i][e]);
      return wave_range(r);
    };
    // The values below 2^kLow alone, scaled up, or the others alone.
    auto mask = [&](float4v* v, int n, float scale, bool small) {
#pragma unroll
      for (int i = 0; i < n; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[i][e] = (__builtin_fabsf(v[i][e] * scale) < pow2(kLow)) == small
                        ? v[i][e] * (small ? pow2(kBand) : 1.f)
                        : 0.f;
    };
    // A piece into LDS; `big`: the largest magnitude so far (or NaN), `low`: the bits of
    // the smallest one that is not zero, sign shifted out, minus one.
    auto put = [&](const float4v& v, unsigned char* to, int lo_at, float scale,
                   float& big, unsigned& low) {
      const Pair p = take_apart(v[0], v[1], scale, scale * 2048.f);
      const Pair q = take_apart(v[2], v[3], scale, scale * 2048.f);
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        big = __builtin_elementwise_maximum(
            __builtin_elementwise_maximum(big, __builtin_fabsf(v[e])),
            __builtin_fabsf(v[e + 1]));
        low = min(min(low, magnitude(v[e]) - 1u), magnitude(v[e + 1]) - 1u);
      }
      *reinterpret_cast<uint2v*>(to) = uint2v{p.hi, q.hi};
      *reinterpret_cast<uint2v*>(to + lo_at) = uint2v{p.lo, q.lo};
    };
    // The exponent of an operand stays while its values fit; else
    // it follows the task's largest.  It rises to 2^10 above the lowest so far at
    // most, so that the sums, which follow both operands', stay finite where they are
    // scaled up for two bands of small values.
    struct Scale {
      int exponent = 0, low = 0, high = 0;
      bool have = false;
      __device__ __forceinline__ int take(Range r) {
        if (r.big == 0) return 0;
        const int want = exponent_for(r.big) - 1;  // (room for the tasks to come)
        if (!have) {
          low = high = exponent = want;
          have = true;
        } else if (want < exponent) {
          exponent = want;
        } else if (want > exponent + 1) {
          exponent = min(want, low + 10);
        }
        low = min(low, exponent);
        high = max(high, exponent);
        return loses(r, exponent) | (high - low > 30 ? kBeyond : 0);
      }
      // (before a first exponent: zeros)
      __device__ __forceinline__ bool fits(float most, unsigned least) const {
        return most * pow2(exponent) < (have ? 0x1p15f : pow2(kLow)) &&
               least >= (static_cast<unsigned>(kLow + 127 - exponent) << 24) - 1u;
      }
    };
    Scale sx, sy;
    unsigned char* const x_to = tiles + tid / XP * XS + tid % XP * 8;
    unsigned char* const y_to = tiles + kYAt + tid / YP * YS + tid % YP * 8;
    auto put_all = [&](int buf) {
      float x_big = 0.f, y_big = 0.f;
      unsigned x_low = ~0u, y_low = ~0u;
      const float x_scale = pow2(sx.exponent), y_scale = pow2(sy.exponent);
      unsigned char* const xt = x_to + buf * kBufBytes;
      unsigned char* const yt = y_to + buf * kBufBytes;
#pragma unroll
      for (int i = 0; i < NX; ++i)
        put(vx[i], xt + i * XL * XS, CT * 2, x_scale, x_big, x_low);
#pragma unroll
      for (int i = 0; i < kNY; ++i)
        put(vy[i], yt + i * YL * YS, FT * 2, y_scale, y_big, y_low);
      const bool is_bad = !sx.fits(x_big, x_low) ||
                          !sy.fits(y_big, y_low);
      const bool any = __builtin_amdgcn_ballot_w64(is_bad) != 0;
      if (lane == 0) reinterpret_cast<unsigned*>(bad + buf)[w] = any ? 1u : 0u;
    };
    bool plain = false;
    int acc_exp = 0;
    fill_table(task_begin);
    load_pieces();
    bool choose = true;  // the exponents, for this task's values
    for (int task = task_begin, buf = 0; task < task_end;) {
      Task announced = {kWhole, 0, 0, acc_exp};
      int small = 0;
      if (choose) {
        const Range rx = range_of(vx, NX), ry = range_of(vy, kNY);
        if (lane == 0) {
          ranges[w] = rx;
          ranges[4 + w] = ry;
        }
        barrier();
        Range tx = ranges[0], ty = ranges[4];
#pragma unroll
        for (int k = 1; k < 4; ++k) {
          tx.big = max(tx.big, ranges[k].big);
          tx.small = min(tx.small, ranges[k].small);
          ty.big = max(ty.big, ranges[4 + k].big);
          ty.small = min(ty.small, ranges[4 + k].small);
        }
        tx.big = __builtin_amdgcn_readfirstlane(tx.big);
        tx.small = __builtin_amdgcn_readfirstlane(tx.small);
        ty.big = __builtin_amdgcn_readfirstlane(ty.big);
        ty.small = __builtin_amdgcn_readfirstlane(ty.small);
        const bool all_zero = !sx.have || !sy.have;  // the sums so far
        const int fx = sx.take(tx), fy = sy.take(ty);
        const int to = sx.exponent + sy.exponent;
        small = ((fx & kSmall) != 0 ? 1 : 0) | ((fy & kSmall) != 0 ? 2 : 0);
        announced.by = all_zero ? 0 : to - acc_exp;
        announced.acc_exp = acc_exp = to;
        if (((fx | fy) & kBeyond) != 0) {
          announced.kind = kPlain;
          if (tid == 0) tasks[buf] = announced;
          barrier();
          plain = true;
          break;
        }
        choose = false;
      }
      if (small == 0) {
        put_all(buf);
        if (tid == 0) tasks[buf] = announced;
        if (task + 1 < task_end) {
          fill_table(task + 1);
          load_pieces();
        }
        barrier();
        if (any_bad(buf)) {
          choose = true;
          fill_table(task);
          load_pieces();
        } else {
          buf ^= 1;
          ++task;
        }
        continue;
      }
      // The subsets of the operands that hold small values, each by its small ones.
#pragma nounroll
      for (int pass = 0; pass < 4; ++pass) {
        if ((pass & ~small) != 0) continue;
        if (pass != 0) load_pieces();
        if ((small & 1) != 0) mask(vx, NX, pow2(sx.exponent), (pass & 1) != 0);
        if ((small & 2) != 0) mask(vy, kNY, pow2(sy.exponent), (pass & 2) != 0);
        put_all(buf);
        announced.kind = pass == small ? kLastPass : kPass;
        announced.back = -kBand * ((pass & 1) + (pass >> 1));
        announced.by -= announced.back;
        if (tid == 0) tasks[buf] = announced;
        announced.by = 0;
        barrier();
        barrier();
      }
      buf ^= 1;
      ++task;
      if (task < task_end) {
        fill_table(task);
        load_pieces();
      }
    }
    if (plain) {
      // The values as they are in the first buffer.
      for (int task = task_begin; task < task_end; ++task) {
        fill_table(task);
        load_pieces();
#pragma unroll
        for (int i = 0; i < NX; ++i)
          *reinterpret_cast<float4v*>(tiles + (tid / XP + i * XL) * XS +
                                      tid % XP * 16) = vx[i];
#pragma unroll
        for (int i = 0; i < kNY; ++i)
          *reinterpret_cast<float4v*>(tiles + kYAt + (tid / YP + i * YL) * YS +
                                      tid % YP * 16) = vy[i];
        barrier();
        barrier();
      }
    }
    return;
  }

  // (its matrix instructions first: what the loading wave of the SIMD has to do fits
  // in between)
  const int wc = wave & 1, wf = wave >> 1;
  const int q = lane >> 4, j4 = (lane >> 2) & 3, e4 = lane & 3;
  const int x_lane = (8 * q + j4) * XS + e4 * 8 + wc * CB * 32;
  const int y_lane = (8 * q + j4) * YS + e4 * 8 + wf * FB * 32;
  const int row_bytes = g.pitch * XS;
  float4v acc[TR * TC][CB][FB], low[TR * TC][CB][FB];
  auto each = [&](auto f) {
#pragma unroll
    for (int t = 0; t < TR * TC; ++t)
#pragma unroll
      for (int i = 0; i < CB; ++i)
#pragma unroll
        for (int k = 0; k < FB; ++k) f(acc[t][i][k], low[t][i][k]);
  };
  auto rescale = [&](int by) {
    const float s = pow2(by);
    each([&](float4v& a, float4v& l) {
      a *= s;
      l *= s;
    });
  };
  each([](float4v& a, float4v& l) { a = l = float4v{0.f, 0.f, 0.f, 0.f}; });

  constexpr int EVEN = (TC + 1) / 2, ODD = TC / 2;
  uint4v xw[EVEN][2];  // the windows at pixels 0, 2, ...: hi, lo
  half8 yr[2][FB][2];  // [chunk's parity][block][hi, lo]
  constexpr int kYReads = FB * 4;
  auto read_x = [&](int e, const unsigned char* at, int n) {
    const int h = n & 1, plane = n >> 1;
    const uint2v v =
        read_transposed(at + x_lane + (2 * e + h * 4) * XS + plane * CT * 2);
    xw[e][plane][2 * h] = v[0];
    xw[e][plane][2 * h + 1] = v[1];
  };
  auto read_y = [&](half8 (&to)[FB][2], const unsigned char* at, int n) {
    const int h = n & 1, plane = (n >> 1) & 1, k = n >> 2;
    const uint2v v = read_transposed(at + y_lane + h * 4 * YS + plane * FT * 2 +
                                     k * 32);
    uint4v whole = __builtin_bit_cast(uint4v, to[k][plane]);
    whole[2 * h] = v[0];
    whole[2 * h + 1] = v[1];
    to[k][plane] = __builtin_bit_cast(half8, whole);
  };
  // A unit: a row's taps and 16 channels of a chunk, the even windows first.  Behind
  // their matrix instructions the odd ones are put together, and then, as the
  // registers become free, what the next unit needs is read.
  auto unit = [&](auto u_, auto parity_, const unsigned char* x_at,
                  const unsigned char* x_next, const unsigned char* y_next) {
    constexpr int U = decltype(u_)::value, P = decltype(parity_)::value;
    const unsigned char* const from =
        U + 1 == NU ? x_next
                    : x_at + (U + 1) / CB * row_bytes + (U + 1) % CB * 32;
    constexpr int r = U / CB, cb = U % CB;
    uint4v odd[ODD][2];
#pragma unroll
    for (int step = 0; step < TC; ++step) {
      const int s = step < EVEN ? 2 * step : 2 * (step - EVEN) + 1;
      const int t = r * TC + s;
      const uint4v* const w = step < EVEN ? xw[step] : odd[step - EVEN];
      const half8 hi = __builtin_bit_cast(half8, w[0]);
      const half8 lo = __builtin_bit_cast(half8, w[1]);
      int slot = 0;
      auto behind = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        if (step < ODD && slot < 3) {
          odd[step][0][slot] = between(xw[step][0], xw[step + 1][0], slot);
          odd[step][1][slot] = between(xw[step][1], xw[step + 1][1], slot);
        } else if (step < ODD && slot == 4) {
          odd[step][0][3] = between(xw[step][0], xw[step + 1][0], 3);
          odd[step][1][3] = between(xw[step][1], xw[step + 1][1], 3);
        }
        const int e = step - ODD;
        if (e >= 0 && slot < 4) {
          read_x(e, from, slot);
        } else if (e >= 0) {
          // (kYReads over the slots 4, 5 of the units' last steps)
          const int n = (U * EVEN + e) * (3 * FB - 4) + slot - 4;
          if (n < kYReads) read_y(yr[P ^ 1], y_next, n);
        }
        ++slot;
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma unroll
      for (int k = 0; k < FB; ++k) {
        acc[t][cb][k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            yr[P][k][0], hi, acc[t][cb][k], 0, 0, 0);
        behind();
      }
#pragma unroll
      for (int k = 0; k < FB; ++k) {
        low[t][cb][k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            yr[P][k][1], hi, low[t][cb][k], 0, 0, 0);
        behind();
      }
#pragma unroll
      for (int k = 0; k < FB; ++k) {
        low[t][cb][k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            yr[P][k][0], lo, low[t][cb][k], 0, 0, 0);
        behind();
      }
    }
  };
  static_assert(FB == 2 && NU * EVEN * (3 * FB - 4) >= kYReads && ODD < EVEN, "slots");
  const int band_chunks = g.y_px / kChunk, n_chunks = g.group * band_chunks;
  const int halo_bytes = (g.x_px - g.y_px) * XS;
  auto multiply_task = [&](const unsigned char* at) {
    const unsigned char* xa = at;
    const unsigned char* ya = at + kYAt;
    int left = band_chunks, total = n_chunks;  // of the band, of the task
#pragma unroll
    for (int n = 0; n < EVEN * 4; ++n) read_x(n / 4, xa, n % 4);
#pragma unroll
    for (int n = 0; n < kYReads; ++n) read_y(yr[0], ya, n);
    auto chunk = [&](auto parity) {
      const unsigned char* xn = xa + kChunk * XS;
      if (--left == 0) {
        left = band_chunks;
        xn += halo_bytes;
      }
      const unsigned char* yn = ya + kChunk * YS;
      if (--total == 0) {  // (nothing to read ahead)
        xn = at;
        yn = at + kYAt;
      }
      unit(std::integral_constant<int, 0>{}, parity, xa, xn, yn);
      if constexpr (NU > 1)
        unit(std::integral_constant<int, 1>{}, parity, xa, xn, yn);
      if constexpr (NU > 2)
        unit(std::integral_constant<int, 2>{}, parity, xa, xn, yn);
      xa = xn;
      ya = yn;
    };
    static_assert(NU <= 3, "units of a chunk");
    for (;;) {
      chunk(std::integral_constant<int, 0>{});
      if (total == 0) break;
      chunk(std::integral_constant<int, 1>{});
      if (total == 0) break;
    }
  };

  // The sums to the next partial filter; rows are features: a lane holds four of a
  // channel.
  const int taps = g.win_rows * g.win_cols;
  int slice = split * g.sums;
  auto store = [&](int exponent) {
    const int a = max(min(-exponent, 100), -100);
    // (in two steps: up to 2^228)
    const float s1 = pow2(a), s2 = pow2(max(min(-exponent - a, 127), -126));
    float* const to =
        part + static_cast<size_t>(slice) * taps * g.channels * g.features;
#pragma unroll
    for (int t = 0; t < TR * TC; ++t)
#pragma unroll
      for (int i = 0; i < CB; ++i)
#pragma unroll
        for (int k = 0; k < FB; ++k) {
          const int c = ct * CT + (wc * CB + i) * 16 + (lane & 15);
          const int f = ft * FT + (wf * FB + k) * 16 + 4 * q;
          float4v sum;
#pragma unroll
          for (int v = 0; v < 4; ++v)
            sum[v] =
                __builtin_fmaf(low[t][i][k][v], 0x1p-11f, acc[t][i][k][v]) * s1 * s2;
          if (c < g.channels && f < g.features)
            *reinterpret_cast<float4v*>(
                to + (static_cast<size_t>(tg * TR * TC + t) * g.channels + c) *
                         g.features + f) = sum;
          acc[t][i][k] = low[t][i][k] = float4v{0.f, 0.f, 0.f, 0.f};
        }
    ++slice;
  };

  bool plain = false;
  int tasks_left = g.per_sum;  // until the sums are stored
  bool choose = true;  // (as the loading waves see it)
  for (int task = task_begin, buf = 0; task < task_end;) {
    if (choose) barrier();
    barrier();
    const Task now = tasks[buf];
    const int kind = __builtin_amdgcn_readfirstlane(now.kind);
    const int by = __builtin_amdgcn_readfirstlane(now.by);
    const int back = __builtin_amdgcn_readfirstlane(now.back);
    if (kind == kPlain) {
      plain = true;
      break;
    }
    choose = kind == kWhole && any_bad(buf);
    if (choose) continue;
    const int acc_exp = __builtin_amdgcn_readfirstlane(now.acc_exp);
    if (by != 0) rescale(by);
    multiply_task(tiles + buf * kBufBytes);
    if (back != 0) rescale(back);
    if (kind != kWhole) barrier();
    if (kind != kPass) {
      buf ^= 1;
      ++task;
      if (--tasks_left == 0 || task == task_end) {
        store(acc_exp);
        tasks_left = g.per_sum;
      }
    }
  }
  if (plain) {
    // The fp32 instruction; both operands are zeros where either pixel does not exist.
    each([](float4v& a, float4v& l) { a = l = float4v{0.f, 0.f, 0.f, 0.f}; });
    tasks_left = g.per_sum;
    slice = split * g.sums;
    const int l16 = lane & 15;
    for (int task = task_begin; task < task_end; ++task) {
      barrier();
      for (int b = 0; b < g.group; ++b)
#pragma nounroll
        for (int m = 0; m < g.y_px; m += 4) {
          const int ym = b * g.y_px + m + q;
          const bool y_ok = table[kXSlots + ym] != kOob;
          float ys[FB];
#pragma unroll
          for (int k = 0; k < FB; ++k)
            ys[k] = *reinterpret_cast<const float*>(
                tiles + kYAt + ym * YS + ((wf * FB + k) * 16 + l16) * 4);
#pragma unroll
          for (int t = 0; t < TR * TC; ++t) {
            const int xm = b * g.x_px + m + q + t / TC * g.pitch + t % TC;
            const bool ok = y_ok && table[xm] != kOob;
#pragma unroll
            for (int i = 0; i < CB; ++i) {
              const float xv = *reinterpret_cast<const float*>(
                  tiles + xm * XS + ((wc * CB + i) * 16 + l16) * 4);
#pragma unroll
              for (int k = 0; k < FB; ++k)
                acc[t][i][k] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                    ok ? ys[k] : 0.f, ok ? xv : 0.f, acc[t][i][k], 0, 0, 0);
            }
          }
        }
      barrier();
      if (--tasks_left == 0 || task + 1 == task_end) {
        store(0);
        tasks_left = g.per_sum;
      }
    }
  }
}

// dw = the sum of the partial filters, in order: 64 float4 per work-group, a quarter of
// the parts per wave.
__global__ void __launch_bounds__(256)
    filter_halves_reduce_kernel(const float4v* __restrict__ part,
                                float4v* __restrict__ dw, unsigned n_vecs,
                                int n_splits) {
  __shared__ float4v sums[256];
  const unsigned o = blockIdx.x * 64 + (threadIdx.x & 63);
  const int wave = threadIdx.x >> 6;
  float4v sum = {0.f, 0.f, 0.f, 0.f};
  if (o < n_vecs) {
#pragma unroll 8
    for (int s = wave; s < n_splits; s += 4)
      sum += part[static_cast<size_t>(s) * n_vecs + o];
  }
  sums[threadIdx.x] = sum;
  __syncthreads();
  if (wave == 0 && o < n_vecs)
    dw[o] = (sum + sums[threadIdx.x + 64]) +
            (sums[threadIdx.x + 128] + sums[threadIdx.x + 192]);
}

enum Shape { kNone, k3x3, k5x5 };
struct FilterHalvesPlan {
  Shape shape = kNone;
  FilterHalves g;
  int nx = 0;
  bool wanted = false;  // against the kernels behind the same tags
};

int round_up(int a, int b) { return ceil_div(a, b) * b; }

FilterHalvesPlan compute_plan(const snn_hip_conv2d_params& p, bool winograd) {
  FilterHalvesPlan plan;
  const bool five = p.window_rows == 5 && p.window_cols == 5;
  if (!five && !(p.window_rows == 3 && p.window_cols == 3)) return plan;
  if (p.stride_rows != 1 || p.stride_cols != 1 || p.input_format != 0 ||
      p.batch < 1 || p.in_rows < 1 || p.in_cols < 1 || p.out_rows < 1 ||
      p.out_cols < 1 || p.channels < 4 || p.features < 4 || p.channels % 4 != 0 ||
      p.features % 4 != 0 || p.pad_rows < 0 || p.pad_cols < 0)
    return plan;
  const size_t x_bytes =
      static_cast<size_t>(p.batch) * p.in_rows * p.in_cols * p.channels * 4;
  const size_t y_bytes =
      static_cast<size_t>(p.batch) * p.out_rows * p.out_cols * p.features * 4;
  if (x_bytes > kMaxBufferBytes || y_bytes > kMaxBufferBytes) return plan;
  FilterHalves& g = plan.g;
  g = FilterHalves();
  g.batch = p.batch; g.in_rows = p.in_rows; g.in_cols = p.in_cols;
  g.channels = p.channels; g.out_rows = p.out_rows; g.out_cols = p.out_cols;
  g.features = p.features; g.win_rows = p.window_rows;
  g.win_cols = p.window_cols; g.pad_rows = p.pad_rows; g.pad_cols = p.pad_cols;
  const int tr = five ? 1 : 3, tc = five ? 5 : 3;
  const int c_tile = five ? 64 : 32, f_tile = 64;
  const int nx_max = five ? 9 : 8;
  g.tap_groups = five ? 5 : 1;
  g.c_tiles = ceil_div(p.channels, c_tile);
  g.f_tiles = ceil_div(p.features, f_tile);
  const int n_units = g.tap_groups * g.c_tiles * g.f_tiles;
  if (n_units > 4096) return plan;
  const double filter_mb = static_cast<double>(p.window_rows) * p.window_cols *
                           p.channels * p.features * 4e-6;
  // Per task the products of four waves, the values' way into LDS, whose vector
  // instructions take turns with these, and a constant, in cycles of a 2.1 GHz clock;
  // a partial filter is written and read back: 0.6 us per MB.  Fitted to 110 random
  // layers of 1e5 ... 2e10 products: nine of ten within a tenth.
  // The error against 64 bits, squared and relative in the 2-norm: of the operands' low
  // parts, by the pixels whose products a sum adds one after another, and by the sums
  // that are added up.  That of the kernel behind the same tags goes by the pixels of
  // one of its waves and by the waves (400 and 870 random layers, normal values, within
  // a tenth).  The sums are stored in time for it to be no larger; reductions that are
  // too short for that stay there, and so do those of fewer pixels than that kernel
  // takes (0.5 ... 0.7e-7), unless one work-group holds all taps and channels (1.3 ...
  // 1.7e-7).  (The Winograd kernel's is above either: 3.6e-7 at 5000 pixels, 2.0e-7
  // here.)
  const double pixels = static_cast<double>(p.batch) * p.out_rows * p.out_cols;
  const double chain = winograd || !conv2d_filter_backprop_direct_f32_wanted(p)
                           ? 0
                           : conv2d_filter_backprop_direct_f32_chain(p);
  const double operands2 = 0.93e-14, pixel2 = 41.5e-18, sum2 = 0.87e-16;
  // (what either is off by more or less than that)
  const double most_error2 =
      chain > 0 ? 0.91 * (0.28e-14 + 151e-18 * chain + 0.435e-16 * pixels / chain)
                : 1.0;
  const double most_pixels =
      std::min(pixels, (most_error2 - operands2) / pixel2);
  const bool few_rows = p.channels < 32 && p.window_rows * p.window_cols *
                                                   p.channels <= 192;
  if (most_pixels < 32 || (!winograd && !few_rows &&
                           !conv2d_filter_backprop_direct_f32_supports(p, true)))
    return plan;
  double best = -1;
  FilterHalves chosen = g;
  for (int segs = 1; segs <= 16; ++segs) {
    g.seg_cols = ceil_div(p.out_cols, segs);
    if (segs > 1 &&
        (g.seg_cols < 8 || ceil_div(p.out_cols, g.seg_cols) != segs))
      continue;
    g.segs = segs;
    g.pitch = g.seg_cols + tc - 1;
    for (int band = 1; band <= p.out_rows; ++band) {
      g.bands_per_image = ceil_div(p.out_rows, band);
      if (ceil_div(p.out_rows, g.bands_per_image) != band) continue;
      g.band = band;
      g.y_px = round_up(band * g.pitch, kChunk);
      // (a row's last window ends three or four pixels past the chunk)
      g.x_px = g.y_px + (tr - 1) * g.pitch + 4;
      if (g.y_px * (f_tile / 4) > kNY * kLoaders) break;
      const long bands = static_cast<long>(p.batch) * g.bands_per_image * segs;
      if (bands > (1l << 28)) continue;
      g.n_bands = static_cast<int>(bands);
      for (int group = 1; group <= 8; group *= 2) {
        if (group > 1 && group / 2 >= bands) break;
        g.group = group;
        const int x_slots = group * g.x_px, y_slots = group * g.y_px;
        const int pieces = ceil_div(x_slots * (c_tile / 4), kLoaders);
        if (pieces > nx_max || y_slots * (f_tile / 4) > kNY * kLoaders) break;
        const int nx = five || pieces > 6 ? nx_max : 6;
        const long tasks = (bands + group - 1) / group;
        const double products =
            static_cast<double>(y_slots) / kChunk * (five ? 5 * 4 : 9 * 2) * 48;
        const double task_us =
            (1.15 * products + 1130 + 63.0 * (nx + kNY)) / 2100;
        const long most = std::max<long>(1, std::min<long>(tasks, kNumCus / n_units));
        const long fewer = std::lround(std::sqrt(tasks * task_us / (filter_mb * 0.6)));
        const long task_pixels = std::max(1l, std::lround(pixels / tasks));
        if (most_pixels < task_pixels) continue;
        for (const long want : {most, std::max(1l, std::min(most, fewer))}) {
          const long per_split = (tasks + want - 1) / want;
          const long splits = (tasks + per_split - 1) / per_split;
          // (as many tasks for each sum of a split as can be)
          const long last = tasks - (splits - 1) * per_split;
          long per_sum = std::min(
              per_split, std::max(1l, std::lround(most_pixels / task_pixels)));
          long sums = 0, slices = 0;
          bool close = false;
          for (;;) {
            sums = (per_split + per_sum - 1) / per_sum;
            slices = (splits - 1) * sums + (last + per_sum - 1) / per_sum;
            const double added2 = operands2 + sum2 * slices;
            close = added2 + pixel2 * per_sum * task_pixels <= most_error2;
            if (close || per_sum == 1 || added2 > most_error2) break;
            per_sum = std::min(per_sum - 1, (per_split + sums) / (sums + 1));
          }
          if (!close || slices * filter_mb > 256) continue;
          const double rounds =
              std::ceil(static_cast<double>(splits) * n_units / kNumCus);
          const double cost = rounds * per_split * task_us + 7.9 +
                              (slices > 1 ? slices * filter_mb * 0.6 : 0);
          if (best >= 0 && cost >= best) continue;
          best = cost;
          g.n_tasks = static_cast<int>(tasks);
          g.per_split = static_cast<int>(per_split);
          g.per_sum = static_cast<int>(per_sum);
          g.sums = static_cast<int>(sums);
          g.n_slices = static_cast<int>(slices);
          g.n_splits = static_cast<int>(splits);
          chosen = g;
          plan.nx = nx;
        }
      }
    }
  }
  if (best < 0) return plan;
  g = chosen;
  g.by_pitch = divisor(g.pitch);
  g.by_x_px = divisor(g.x_px);
  g.by_y_px = divisor(g.y_px);
  g.by_segs = divisor(g.segs);
  g.by_bands = divisor(g.bands_per_image);
  plan.shape = five ? k5x5 : k3x3;
  if (p.channels >= 16 && p.features >= 16)
    plan.wanted = winograd ? pixels >= 1024
                           : !conv2d_filter_backprop_direct_f32_wanted(p) ||
                                 1.05 * best < conv2d_filter_backprop_direct_f32_us(p);
  return plan;
}

const FilterHalvesPlan& make_plan(const snn_hip_conv2d_params& p, bool winograd) {
  thread_local PlanCache<FilterHalvesPlan> cache;
  return cache.get(p, winograd ? 1 : 0, [&] { return compute_plan(p, winograd); });
}

template <int TR, int TC, int CB, int FB, int NX>
void launch_shape(const float* x, const float* dy, float* part,
                  const FilterHalvesPlan& plan, hipStream_t stream) {
  const FilterHalves& g = plan.g;
  auto kernel = filter_halves_kernel<TR, TC, CB, FB, NX>;
  constexpr int kXSlots = NX * kLoaders / (8 * CB);
  constexpr int kYSlots = kNY * kLoaders / (8 * FB);
  constexpr size_t kLds =
      128 + (kXSlots + kYSlots) * 4 +
      2 * (kXSlots * slot_bytes(32 * CB) + kYSlots * slot_bytes(32 * FB));
  static_assert(kLds <= kMaxLdsBytes, "LDS");
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLdsBytes);
  (void)attr;
  const unsigned n_groups = static_cast<unsigned>(g.tap_groups * g.c_tiles *
                                                  g.f_tiles * g.n_splits);
  KernelTimer timer(stream);
  hipLaunchKernelGGL(
      kernel, dim3(n_groups), dim3(512), kLds, stream, x, dy, part, g,
      static_cast<unsigned>(static_cast<size_t>(g.batch) * g.in_rows * g.in_cols *
                            g.channels * 4),
      static_cast<unsigned>(static_cast<size_t>(g.batch) * g.out_rows *
                            g.out_cols * g.features * 4),
      n_groups);
}

}  // namespace

// Behind the Winograd tag from 1024 output pixels on, where the default policy names
// that tag (28x28x128 at batch 32: 34 us instead of 51, 64x64x256 at batch 8: 126
// instead of 196); behind the others in place of the kernel that holds all taps and
// channels (163x212x24 at batch 7 -> 32: 39 us instead of 150) and of the one for tiles
// of 64 where its estimate is higher (17x27x27 96 -> 256, 5x5: 81 us instead of 179;
// 9x9x144 -> 528 at batch 5, below the line: 18.3 here, 11.1 there).
bool conv2d_filter_halves_f32_wanted(const snn_hip_conv2d_params& p, bool winograd) {
  return make_plan(p, winograd).wanted;
}

int conv2d_filter_halves_f32_partials(const snn_hip_conv2d_params& p,
                                      bool winograd) {
  const FilterHalvesPlan& plan = make_plan(p, winograd);
  return plan.shape != kNone ? plan.g.n_slices : 0;
}

size_t conv2d_filter_halves_f32_partial_floats(const snn_hip_conv2d_params& p,
                                               bool winograd) {
  const FilterHalvesPlan& plan = make_plan(p, winograd);
  if (plan.shape == kNone || plan.g.n_slices == 1) return 0;
  return static_cast<size_t>(plan.g.n_slices) * p.window_rows * p.window_cols *
         p.channels * p.features;
}

int launch_conv2d_filter_halves_f32(const float* x, const float* dy, float* dw,
                                    const snn_hip_conv2d_params& p,
                                    bool winograd, float* workspace,
                                    hipStream_t stream) {
  const FilterHalvesPlan& plan = make_plan(p, winograd);
  if (plan.shape == kNone) return SNN_HIP_INVALID_ALGORITHM;
  const bool one = plan.g.n_slices == 1;
  float* const part = one ? dw : workspace;
  if (plan.shape == k5x5)
    launch_shape<1, 5, 2, 2, 9>(x, dy, part, plan, stream);
  else if (plan.nx == 6)
    launch_shape<3, 3, 1, 2, 6>(x, dy, part, plan, stream);
  else
    launch_shape<3, 3, 1, 2, 8>(x, dy, part, plan, stream);
  if (!one) {
    const unsigned n_vecs = static_cast<unsigned>(
        static_cast<size_t>(p.window_rows) * p.window_cols * p.channels *
        p.features / 4);
    hipLaunchKernelGGL(filter_halves_reduce_kernel, dim3(ceil_div(n_vecs, 64u)),
                       dim3(256), 0, stream,
                       reinterpret_cast<const float4v*>(workspace),
                       reinterpret_cast<float4v*>(dw), n_vecs, plan.g.n_slices);
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return report_hip_error(err, "filter_halves_kernel");
  return SNN_HIP_OK;
}

}  // namespace snn
