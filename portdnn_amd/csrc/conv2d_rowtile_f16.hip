// Half-precision stride-1 forward convolution on MFMA (gfx950) with the
// input tile resident in LDS: binary16 operands, fp32 accumulation, binary16
// result.
//
// The gathering kernel in conv2d_gather.hip loads every input pixel once
// per filter tap and passes both operands through LDS; at 32x32x16 f16 MFMA
// rates that makes LDS and the loads the limit, not the matrix cores.  Here a work-group owns a run
// of consecutive output pixels (images, rows and columns flattened, so a tile
// may start inside a row and run over an image boundary) and a slice of the
// features:
//
//   * the input rows those outputs need (the tile plus its halo, zero padding
//     included as explicit zero pixels) are loaded into LDS once per block of
//     KC channels, [pixel slot][KC halves + 16 bytes of padding], by buffer
//     loads that write LDS directly; every filter tap then reads the same LDS
//     tile at a slot offset of r * Wh + s;
//   * the filter never touches LDS: it is pre-packed in MFMA A-operand order,
//     [k-step][feature block of 32][lane][8 halves], and streams from global
//     memory (L2-resident) straight into registers, prefetched two units of
//     16 MFMAs ahead;
//   * features are the MFMA rows and pixels the columns, with the 32 feature
//     rows permuted in the packed filter so that a lane ends up holding 16
//     consecutive features of one pixel: the epilogue is two 16-byte stores
//     per lane per 32x32 block.
//
// Each wave owns 2 feature blocks x 4 pixel blocks (64 features x 128
// pixels, 128 accumulator registers): per 16-deep reduction step it reads
// 4 KB from LDS and 2 KB of filter for 8 MFMAs; or, where that balances the
// compute units better, 2 x 2 blocks.  224x224x64 at batch 16, 3x3: 85 us (69
// without the stores, 71 without the loads, 55 with neither).
//
// portDNN's half build accumulates in half (e.g. `DataType out_val{0}` with
// T = cl::sycl::half in src/conv2d/direct/kernels_nhwc.h:92); accumulating in
// fp32 is more accurate and stays inside the 1e-2 relative bar against it.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <numeric>

#include "gemm_tile.h"
#include "plan_cache.h"
#include "snn_kernels.h"

namespace snn {
namespace {

using gemm::float16v;
using gemm::xcd_remap;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
constexpr unsigned kOob = 0x7FFFFFF0u;
constexpr int kStoreAux = 2;  // the output is written once: stream it (slc)
constexpr size_t kMaxBufferBytes = 0x7FFFFFF0u;
constexpr int kNumCus = 256;
constexpr int kFA = 2;  // feature blocks (of 32) per wave
constexpr size_t kMaxLdsBytes = 160 * 1024;

struct RowTile {
  int batch, in_rows, in_cols, channels, features;
  int out_rows, out_cols;
  int win_rows, win_cols, pad_rows, pad_cols;
  int tile_pixels;   // output pixels (flattened n, y, x) per work-group
  int total_pixels;  // batch * out_rows * out_cols
  int padded_rows;  // Hp = out_rows + win_rows - 1: padded input rows per image
  int halo_cols;    // Wh = out_cols + win_cols - 1
  int n_slots;      // LDS pixel slots per tile = lds rows * Wh
  int n_fslices;    // features / (64 * WF)
};

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p,
                                                   unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x00020000);
}

// wpk[step][fb][lane][e] = w[tap][c][f] with step = (chunk * taps + tap) *
// (KC / 16) + ks, c = chunk * KC + ks * 16 + 8 * (lane / 32) + e and, for
// MFMA row rho = lane % 32, f = fb * 32 + 16 * ((rho / 4) % 2) + 4 * (rho / 8)
// + rho % 4: the accumulator rows 8g + 4h + i a lane holds (h = lane / 32)
// are then features 16h + 4g + i, 16 consecutive ones.  `transposed`: the
// input gradient's filter, w[taps - 1 - tap][f][c] of the HWCF tensor of a
// convolution with `features` input channels and `channels` features
// (mirrored taps, channel and feature roles swapped).
//
// A launch this short is its own latency: a work-group's place in the grid says
// which 32 channels x 64 features of which tap it packs, so nothing is divided, and
// the transposed filter's eight channels come in one load (the caller's filter is
// aligned to 16 bytes).  Input gradients of 14x14x256 and 28x28x128 at batch 128,
// whole calls: 36.9 -> 35.0 and 38.3 -> 37.0 us (three divisions and eight loads of
// 2 bytes from 64 rows before); forward launches and other layers level.
template <bool TRANSPOSED>
__global__ void __launch_bounds__(256)
    pack_filter_rowtile_kernel(const _Float16* __restrict__ w,
                               _Float16* __restrict__ wpk, int channels,
                               int features, int kc_log2) {
  // Wave: 16 channels x 32 features; lane: eight channel values of one feature.
  // The 32 lanes of a half-wave read 32 permuted but adjacent features.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tap = blockIdx.z, taps = gridDim.z;
  const int fb = blockIdx.x * 2 + (wave & 1), n_fb = gridDim.x * 2;
  const int c0 = blockIdx.y * 32 + (wave >> 1) * 16;
  const int chunk = c0 >> kc_log2, ks = (c0 & ((1 << kc_log2) - 1)) >> 4;
  const int step = (chunk * taps + tap) * (1 << (kc_log2 - 4)) + ks;
  const int c = c0 + 8 * (lane >> 5);
  const int rho = lane & 31;
  const int f = fb * 32 + 16 * ((rho >> 2) & 1) + 4 * (rho >> 3) + (rho & 3);
  const _Float16* src =
      TRANSPOSED
          ? w + (static_cast<size_t>(taps - 1 - tap) * features + f) * channels + c
          : w + (static_cast<size_t>(tap) * channels + c) * features + f;
  half8 v;
  if constexpr (TRANSPOSED) {
    v = *reinterpret_cast<const half8*>(src);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = src[static_cast<size_t>(e) * features];
  }
  *reinterpret_cast<half8*>(
      wpk + ((static_cast<size_t>(step) * n_fb + fb) * 64 + lane) * 8) = v;
}

// s_waitcnt immediates that wait on the vector-memory counter only.
constexpr int kWaitVm0 = 0x0F70;
constexpr int kWaitLgkm0 = 0xC07F;  // (LDS reads)
constexpr int kWaitVm4 = 0x0F74;
constexpr int kWaitVm8 = 0x0F78;

// WF x WP waves: WF feature groups of 64, WP pixel groups of PB * 32.  KC =
// channels per LDS tile.  BUFS: 1, one channel block; 2, more than one and two LDS
// tiles, the next one loading while the current one is multiplied; 3, more than
// one and one LDS tile, so that two work-groups fit a CU and one loads while the
// other multiplies (3x3 windows only).  WIN3: 3x3
// window, whose reduction loop is unrolled over a filter row with all tap
// bookkeeping resolved at compile time.
//
// LDS tile: [pixel slot][KC halves + one 16-byte pad piece].  A slot is then
// an odd number of 16-byte pieces (5 or 9), so the ds_read_b128 of 16
// consecutive slots at the same piece touch 16 different bank groups, and a
// slot's address is linear in its index: the three taps of a filter row and
// the reduction steps of a tap are compile-time offsets of one address per
// pixel block, which leaves the reduction loop without address arithmetic.
// Tiles are filled by buffer loads that write LDS directly (64 lanes x 16
// bytes = 1 KB of consecutive LDS per instruction; the lanes that fall on pad
// pieces load from out of range), so a whole tile is in flight without
// holding registers; out-of-range offsets (padding pixels) store zeros.
template <int WF, int WP, int PB, int KC, int BUFS, bool WIN3>
__global__ void __launch_bounds__(64 * WF * WP)
    __attribute__((amdgpu_waves_per_eu(2, 2)))
    conv_rowtile_f16_kernel(const _Float16* __restrict__ src,
                            const _Float16* __restrict__ wpk,
                            _Float16* __restrict__ dst, RowTile g,
                            unsigned src_bytes, unsigned wpk_bytes,
                            unsigned dst_bytes, unsigned n_groups) {
  constexpr int NT = 64 * WF * WP;
  constexpr int NW = WF * WP;
  constexpr bool MULTI = BUFS != 1;  // more than one channel block
  constexpr bool AHEAD = BUFS == 2;  // the next one loads meanwhile
  constexpr int KS = KC / 16;        // MFMA reduction steps per tap
  constexpr int UPT = KS / 2;        // units of two steps per tap
  constexpr int PPS = KC / 8;        // 16-byte pieces of data per slot
  constexpr int SLOTB = KC * 2 + 16; // bytes per LDS pixel slot (one pad piece)
  extern __shared__ __align__(16) unsigned char lds[];
  typedef __attribute__((address_space(3))) void* lds_ptr;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wf = wave / WP, wp = wave % WP;
  const unsigned group = xcd_remap(blockIdx.x, n_groups);
  const int tile = static_cast<int>(group / g.n_fslices);
  const int fslice = static_cast<int>(group % g.n_fslices);

  const int pixel0 = tile * g.tile_pixels;  // first flattened output pixel
  const int n_pixels = min(g.tile_pixels, g.total_pixels - pixel0);
  // Padded-row coordinate of the first LDS row: image * Hp + padded row.
  const int row0 = pixel0 / g.out_cols;  // flattened (image, row)
  const int first_padded =
      (row0 / g.out_rows) * g.padded_rows + row0 % g.out_rows;

  // 1 KB blocks per tile, and the slots they reach into
  const int n_blocks = (g.n_slots * SLOTB + 1023) / 1024;
  const int n_table = n_blocks * 1024 / SLOTB + 1;
  const int buf_bytes = n_blocks * 1024;
  unsigned char* const bufs = lds;
  unsigned* const table =
      reinterpret_cast<unsigned*>(lds + (AHEAD ? 2 : 1) * buf_bytes);

  // Global byte offset of channel 0 of every pixel slot (kOob for padding
  // and for the slots that only fill up the last block).
  for (int slot = tid; slot < n_table; slot += NT) {
    const int lrow = slot / g.halo_cols;
    const int hx = slot - lrow * g.halo_cols;
    const int padded = first_padded + lrow;
    const int n = padded / g.padded_rows;
    const int iy = padded - n * g.padded_rows - g.pad_rows;
    const int ix = hx - g.pad_cols;
    const bool ok = slot < g.n_slots && n < g.batch &&
                    static_cast<unsigned>(iy) <
                        static_cast<unsigned>(g.in_rows) &&
                    static_cast<unsigned>(ix) < static_cast<unsigned>(g.in_cols);
    table[slot] =
        ok ? static_cast<unsigned>(((n * g.in_rows + iy) * g.in_cols + ix) *
                                   g.channels) * 2u
           : kOob;
  }
  __syncthreads();

  const __amdgpu_buffer_rsrc_t src_rsrc = make_rsrc(src, src_bytes);
  const __amdgpu_buffer_rsrc_t wpk_rsrc = make_rsrc(wpk, wpk_bytes);

  // Starts the loads of one channel block into an LDS tile: wave w takes the
  // 1 KB blocks w, w + NW, ...; lane l fills bytes 16 l .. 16 l + 15 of its
  // block, which belong to piece (position % SLOTB) / 16 of slot position /
  // SLOTB; the pad piece of a slot loads from out of range (zeros).  `soff`
  // (in range by construction) selects the channel block; padding pixels go
  // out of range through the vector offset, the only one the hardware
  // range-checks.
  auto start_tile = [&](unsigned char* buf, unsigned soff) {
    for (int block = wave; block < n_blocks; block += NW) {
      const int pos = block * 1024 + lane * 16;
      const int slot = pos / SLOTB;
      const int piece = (pos - slot * SLOTB) >> 4;
      const unsigned voff =
          piece < PPS ? table[slot] + static_cast<unsigned>(piece) * 16u : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          src_rsrc, (lds_ptr)(buf + block * 1024), 16, voff, soff, 0, 0);
    }
  };
  start_tile(bufs, 0);

  // LDS slot (tap (0,0)) of this lane's pixel in each of its pixel blocks,
  // and the flattened output pixel (-1: none).
  const int l32 = lane & 31;
  const int khalf = lane >> 5;
  int b_slot[PB];
  int out_pixel[PB];
#pragma unroll
  for (int j = 0; j < PB; ++j) {
    const int q = (wp * PB + j) * 32 + l32;
    b_slot[j] = 0;
    out_pixel[j] = -1;
    if (q < n_pixels) {
      const int m = pixel0 + q;
      const int orow = m / g.out_cols;
      const int x = m - orow * g.out_cols;
      const int n = orow / g.out_rows;
      const int lrow = n * g.padded_rows + (orow - n * g.out_rows) -
                       first_padded;
      b_slot[j] = lrow * g.halo_cols + x;
      out_pixel[j] = m;
    }
  }

  const int n_fb = g.features / 32;
  const int fb0 = (fslice * WF + wf) * kFA;
  const unsigned a_voff = static_cast<unsigned>(fb0 * 64 + lane) * 16u;
  const unsigned a_step_bytes = static_cast<unsigned>(n_fb) * 1024u;
  // The reduction runs in units of two MFMA steps (32 channels of one tap).
  // Filter fragments: DEPTH buffers of one unit each in rotation.  Unit u
  // multiplies out of buffer u % DEPTH while the buffer unit u - 1 used is
  // refilled with the fragments of unit u + DEPTH - 1, so a load has
  // DEPTH - 1 units of MFMAs to arrive and no register copies wait on it.
  // The smaller wave tile has half the MFMAs per unit and registers to
  // spare: it prefetches twice as far.  Reads past the end of the packed
  // filter return zeros.
  constexpr int DEPTH = (PB == 2 && !WIN3) ? 5 : 3;
  half8 a_buf[DEPTH][2][kFA];
  auto load_a = [&](half8 (&frag)[2][kFA], unsigned first_step) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < kFA; ++i)
        frag[ks][i] = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(
                       wpk_rsrc,
                       a_voff + static_cast<unsigned>(i) * 1024u +
                           (first_step + static_cast<unsigned>(ks)) *
                               a_step_bytes,
                       0, 0));
  };
#pragma unroll
  for (int d = 0; d + 1 < DEPTH; ++d)
    load_a(a_buf[d], static_cast<unsigned>(2 * d));

  float16v acc[kFA][PB];
#pragma unroll
  for (int i = 0; i < kFA; ++i)
#pragma unroll
    for (int j = 0; j < PB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // The first tile has landed once no vector-memory load is outstanding.
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  __syncthreads();

  const int taps = g.win_rows * g.win_cols;
  const int n_chunks = g.channels / KC;
  const int units_per_chunk = taps * UPT;
  const int total_units = n_chunks * units_per_chunk;
  unsigned step = 0;  // first reduction step of the unit
  half8 b_even[PB], b_odd[PB];  // pixel fragments of even / odd steps
  auto mfma_step = [&](const half8 (&a)[kFA], const half8 (&b)[PB]) {
#pragma unroll
    for (int i = 0; i < kFA; ++i)
#pragma unroll
      for (int j = 0; j < PB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[j],
                                                           acc[i][j], 0, 0, 0);
  };
  if constexpr (WIN3) {
    // Scalar and branch instructions between MFMAs leave the matrix pipe
    // idle, so this path has none per unit: the loop runs over filter rows
    // with the three taps of a row (UPT units each) unrolled, which also
    // keeps the rotation of the three filter buffers static.
    int cur_off = 0, nxt_off = AHEAD ? buf_bytes : 0;
    // Byte offset inside a tile of this lane's fragment of tap (0, 0), step 0.
    // Slots are SLOTB bytes apart, so the taps of a filter row and the steps
    // of a tap are compile-time offsets from the row's address.
    int lane_base[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) lane_base[j] = b_slot[j] * SLOTB + khalf * 16;
    const int row_step = g.halo_cols * SLOTB;
    auto read_b = [&](half8 (&b)[PB], const int (&rb)[PB], int offset) {
#pragma unroll
      for (int j = 0; j < PB; ++j)
        b[j] = *reinterpret_cast<const half8*>(bufs + rb[j] + offset);
    };
    int rb[PB];  // filter row r of the current tile
#pragma unroll
    for (int j = 0; j < PB; ++j) rb[j] = cur_off + lane_base[j];
    read_b(b_even, rb, 0);
#pragma unroll 1
    for (int c = 0; c < n_chunks; ++c) {
#pragma unroll 1
      for (int r = 0; r < 3; ++r) {
        // the next filter row (after the last one the tiles swap and the
        // fragment is read again; the tile's first row will do here)
        int rb_next[PB];
#pragma unroll
        for (int j = 0; j < PB; ++j)
          rb_next[j] = r < 2 ? rb[j] + row_step : cur_off + lane_base[j];
#pragma unroll
        for (int sc = 0; sc < 3; ++sc) {
#pragma unroll
          for (int u = 0; u < UPT; ++u) {
            constexpr int kRot = 3;
            const int v = sc * UPT + u;  // unit within the filter row
            half8 (&a_use)[2][kFA] = a_buf[v % kRot];
            half8 (&a_fill)[2][kFA] = a_buf[(v + 2) % kRot];
            if constexpr (AHEAD) {
              if (sc == 0 && u == 0) {
                if (r == 0 && c + 1 < n_chunks)
                  start_tile(bufs + nxt_off,
                             static_cast<unsigned>((c + 1) * KC * 2));
              }
            }
            read_b(b_odd, rb, sc * SLOTB + (2 * u + 1) * 32);
            __builtin_amdgcn_sched_barrier(0);
            // The filter prefetch issues in the shadow of the MFMAs.
            load_a(a_fill, step + 4);
            step += 2;
            mfma_step(a_use[0], b_even);
            __builtin_amdgcn_sched_barrier(0);
            if (u + 1 < UPT)
              read_b(b_even, rb, sc * SLOTB + (2 * u + 2) * 32);
            else if (sc < 2)
              read_b(b_even, rb, (sc + 1) * SLOTB);
            else
              read_b(b_even, rb_next, 0);
            __builtin_amdgcn_sched_barrier(0);
            mfma_step(a_use[1], b_odd);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int j = 0; j < PB; ++j) rb[j] = rb_next[j];
      }
      if constexpr (MULTI) {
        // End of the channel block.  Vector-memory loads complete in order:
        // the next tile was issued at the block's start, so it has landed
        // once only the filter loads of the last two units (2 * kFA each)
        // can still be outstanding.  No fence: this tile's pixel fragments
        // have all been read into registers, and the barrier alone makes
        // every wave's part of the next tile visible.
        if constexpr (AHEAD) {
          __builtin_amdgcn_s_waitcnt(0x0F70 | (4 * kFA));
        } else if (c + 1 < n_chunks) {
          // One buffer: once every wave is done with this tile the next one is
          // loaded in its place (the CU's other work-group multiplies meanwhile).
          __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
          start_tile(bufs, static_cast<unsigned>((c + 1) * KC * 2));
          __builtin_amdgcn_s_waitcnt(kWaitVm0);
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const int t = cur_off;
        cur_off = nxt_off;
        nxt_off = t;
#pragma unroll
        for (int j = 0; j < PB; ++j) rb[j] = cur_off + lane_base[j];
        read_b(b_even, rb, 0);
      }
    }
  } else {
    const unsigned char* cur = bufs;
    unsigned char* nxt = bufs + buf_bytes;
    int chunk = 0, tap = 0, tap_r = 0, tap_c = 0, sub = 0;
    int tap_slots = 0;  // slot offset of the current tap: r * Wh + s
    // Pixel fragments of reduction step `ks` (0 .. KS-1) of a tap.
    auto load_b = [&](half8 (&b)[PB], int slots, int ks) {
      const int offset = slots * SLOTB + (2 * ks + khalf) * 16;
#pragma unroll
      for (int j = 0; j < PB; ++j)
        b[j] = *reinterpret_cast<const half8*>(cur + b_slot[j] * SLOTB + offset);
    };
    load_b(b_even, 0, 0);

    // One unit.  Pixel fragments of a reduction step are read from LDS while
    // the MFMAs of the step before run; the loads of the next channel block's
    // tile start in the first unit of a block.  The scheduling barriers keep
    // the compiler from sinking these prefetches below the MFMAs that hide
    // their latency.
    auto do_unit = [&](half8 (&a_use)[2][kFA], half8 (&a_fill)[2][kFA]) {
      const int slots = tap_slots;
      const int ks0 = 2 * sub;
      const bool tap_ends = sub + 1 == UPT;
      const bool last = tap_ends && tap + 1 == taps;
      int next_ks = ks0 + 2;
      if (tap_ends) {
        if (++tap_c == g.win_cols) { tap_c = 0; ++tap_r; }
        // After the last tap the tiles swap and the fragment is read again;
        // any slot inside the tile will do here.
        tap_slots = last ? 0 : tap_r * g.halo_cols + tap_c;
        next_ks = 0;
      }
      load_a(a_fill, step + 2 * (DEPTH - 1));
      if constexpr (AHEAD) {
        if (tap == 0 && sub == 0 && chunk + 1 < n_chunks) {
          __builtin_amdgcn_sched_barrier(0);
          start_tile(nxt, static_cast<unsigned>((chunk + 1) * KC * 2));
        }
      }
      load_b(b_odd, slots, ks0 + 1);
      __builtin_amdgcn_sched_barrier(0);
      mfma_step(a_use[0], b_even);
      __builtin_amdgcn_sched_barrier(0);
      load_b(b_even, tap_slots, next_ks);
      __builtin_amdgcn_sched_barrier(0);
      mfma_step(a_use[1], b_odd);
      __builtin_amdgcn_sched_barrier(0);
      step += 2;
      if (last) {
        if constexpr (MULTI) {
          // End of the channel block.  Vector-memory loads complete in order:
          // the next tile was issued before the filter loads of all units but
          // the first, so it has landed once only the last two units' filter
          // loads (four each) can still be outstanding.  No fence: this
          // tile's pixel fragments have all been read into registers, and
          // the barrier alone makes every wave's part of the next tile
          // visible.
          if (units_per_chunk >= 3)
            __builtin_amdgcn_s_waitcnt(kWaitVm8);
          else if (units_per_chunk == 2)
            __builtin_amdgcn_s_waitcnt(kWaitVm4);
          else
            __builtin_amdgcn_s_waitcnt(kWaitVm0);
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
          unsigned char* const t = const_cast<unsigned char*>(cur);
          cur = nxt;
          nxt = t;
          ++chunk;
          load_b(b_even, 0, 0);
        }
        tap = 0;
        tap_r = 0;
        tap_c = 0;
        sub = 0;
      } else if (tap_ends) {
        ++tap;
        sub = 0;
      } else {
        ++sub;
      }
    };

    int done = 0;
    for (; done + DEPTH <= total_units; done += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d)
        do_unit(a_buf[d], a_buf[(d + DEPTH - 1) % DEPTH]);
    }
#pragma unroll
    for (int d = 0; d + 1 < DEPTH; ++d)
      if (done + d < total_units)
        do_unit(a_buf[d], a_buf[(d + DEPTH - 1) % DEPTH]);

  }

  const __amdgpu_buffer_rsrc_t dst_rsrc = make_rsrc(dst, dst_bytes);
  const unsigned row_bytes = static_cast<unsigned>(g.features) * 2u;
#pragma unroll
  for (int j = 0; j < PB; ++j) {
    const unsigned pix_off =
        out_pixel[j] >= 0 ? static_cast<unsigned>(out_pixel[j]) * row_bytes
                          : kOob;
#pragma unroll
    for (int i = 0; i < kFA; ++i) {
      const unsigned off =
          pix_off + static_cast<unsigned>((fb0 + i) * 32 + 16 * khalf) * 2u;
      half8 lo, hi;
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        lo[v] = static_cast<_Float16>(acc[i][j][v]);
        hi[v] = static_cast<_Float16>(acc[i][j][8 + v]);
      }
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, lo),
                                             dst_rsrc, off, 0, kStoreAux);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, hi),
                                             dst_rsrc, off + 16u, 0, kStoreAux);
    }
  }
}

struct RowTilePlan {
  RowTile g;
  int wf = 0;            // feature groups of 64 per work-group
  int wp = 0;            // pixel groups of PB * 32 per work-group
  int pb = 0;            // pixel blocks of 32 per wave
  int kc = 0;            // channels per LDS tile
  int bufs = 0;          // see BUFS
  size_t lds_bytes = 0;  // 0: shape not supported
  long score = 0;
  double us = 0;         // estimated
  unsigned n_groups = 0;
};

// Padded rows a tile of `tile_pixels` consecutive output pixels spans: from the
// padded row of its first pixel to the padded row of its last pixel plus the
// window, the largest over all tiles (their position inside an image repeats every
// image / gcd tiles).
int rows_spanned(const snn_hip_conv2d_params& p, int tile_pixels) {
  const int total = p.batch * p.out_rows * p.out_cols;
  const int padded_rows = p.out_rows + p.window_rows - 1;
  const int image = p.out_rows * p.out_cols;
  const int period = std::min(ceil_div(total, tile_pixels),
                              image / std::gcd(image, tile_pixels) + 1);
  auto padded_row = [&](int pixel) {
    const int row = pixel / p.out_cols;
    return row / p.out_rows * padded_rows + row % p.out_rows;
  };
  int rows = 0;
  for (int t = 0; t < period; ++t) {
    const int first = t * tile_pixels;
    const int last = std::min(total - first, tile_pixels) + first - 1;
    rows = std::max(rows,
                    padded_row(last) - padded_row(first) + p.window_rows);
  }
  return rows;
}

// Geometry for work-groups of `tile_pixels` consecutive output pixels;
// lds_bytes == 0 when the tile does not fit.  The score estimates the useful
// pixels resident on a compute unit: work-groups that fit its LDS (at most two
// waves per SIMD) times the pixels of a tile, discounted by the unused part
// of the wave tiles.
RowTilePlan plan_tile(const snn_hip_conv2d_params& p, int wf, int wp, int pb,
                      int kc, int bufs, int tile_pixels, int lds_rows) {
  RowTilePlan plan;
  RowTile& g = plan.g;
  g.batch = p.batch; g.in_rows = p.in_rows; g.in_cols = p.in_cols;
  g.channels = p.channels; g.features = p.features;
  g.out_rows = p.out_rows; g.out_cols = p.out_cols;
  g.win_rows = p.window_rows; g.win_cols = p.window_cols;
  g.pad_rows = p.pad_rows; g.pad_cols = p.pad_cols;
  g.total_pixels = p.batch * p.out_rows * p.out_cols;
  g.tile_pixels = tile_pixels;
  g.padded_rows = p.out_rows + p.window_rows - 1;
  g.halo_cols = p.out_cols + p.window_cols - 1;
  g.n_slots = lds_rows * g.halo_cols;
  g.n_fslices = p.features / (64 * wf);
  const size_t slot_bytes = static_cast<size_t>(kc) * 2 + 16;
  const size_t n_blocks = ceil_div(g.n_slots * slot_bytes, size_t{1024});
  const size_t n_table = n_blocks * 1024 / slot_bytes + 1;
  const size_t lds_bytes =
      (bufs == 2 ? 2 : 1) * n_blocks * 1024 + n_table * 4;
  if (lds_bytes > kMaxLdsBytes) return plan;
  plan.wf = wf; plan.wp = wp; plan.pb = pb; plan.kc = kc; plan.bufs = bufs;
  plan.lds_bytes = lds_bytes;
  const long resident =
      std::min<long>(kMaxLdsBytes / lds_bytes, 8 / (wf * wp));
  plan.score = resident * tile_pixels * tile_pixels / (wp * pb * 32);
  plan.n_groups = static_cast<unsigned>(ceil_div(g.total_pixels, tile_pixels)) *
                  static_cast<unsigned>(g.n_fslices);
  // The estimated time: rounds of the work-groups that fit the compute units, each
  // its products (faster per wave with two on a SIMD), then loads at 18 and stores
  // at 10 bytes per cycle and CU -- on 200 layers the estimates that took a part of
  // these as hidden behind the products were the worse ones, with one buffer and
  // with two.
  const int here =
      std::min<int>(static_cast<int>(resident),
                    std::max(1, ceil_div(static_cast<int>(plan.n_groups), kNumCus)));
  const int n_chunks = p.channels / kc;
  const int per_simd = ceil_div(here * wf * wp, 4);
  const double products = n_chunks * p.window_rows * p.window_cols * (kc / 16) *
                          64.0 * pb * (pb == 2 ? 1.12 : 1.0) *
                          (per_simd == 1 ? 1.44 : 0.805 * per_simd);
  const double memory =
      here * (n_chunks * static_cast<double>(g.n_slots) * kc * 2 / 17.9 +
              tile_pixels * 128.0 * wf / 10.0);
  double rounds = static_cast<double>(plan.n_groups) / (kNumCus * here);
  rounds = rounds < 4 ? std::ceil(rounds) : rounds + 0.5;
  plan.us = 5.2 + rounds * (products + memory + 2340) / 2000;
  return plan;
}

RowTilePlan compute_plan(const snn_hip_conv2d_params& p) {
  const int total = p.batch * p.out_rows * p.out_cols;
  const bool win3 = p.window_rows == 3 && p.window_cols == 3;
  // rows spanned by tiles of 64, 128, 256, 512 pixels and of 1, 2, ... rows
  int of_pixels[4] = {0, 0, 0, 0};
  std::array<int, 65> of_rows{};
  // Of the tile sizes -- the full capacity of the work-group (tiles then start
  // anywhere in a row), and every whole number of rows below it -- the one of the
  // best score.
  auto best_tile = [&](int wf, int wp, int pb, int kc, int bufs) {
    const int full = wp * pb * 32;
    const int capacity = std::min(full, total);
    int& spanned = of_pixels[full == 64 ? 0 : full == 128 ? 1 : full == 256 ? 2 : 3];
    if (spanned == 0) spanned = rows_spanned(p, capacity);
    RowTilePlan best = plan_tile(p, wf, wp, pb, kc, bufs, capacity, spanned);
    for (int rows = std::min(64, capacity / p.out_cols); rows >= 1; --rows) {
      // (not even a tile that lies in one image fits)
      if (static_cast<size_t>(rows + p.window_rows - 1) *
              (p.out_cols + p.window_cols - 1) * (kc * 2 + 16) *
              (bufs == 2 ? 2 : 1) > kMaxLdsBytes)
        continue;
      if (of_rows[rows] == 0) of_rows[rows] = rows_spanned(p, rows * p.out_cols);
      const RowTilePlan plan = plan_tile(p, wf, wp, pb, kc, bufs,
                                         rows * p.out_cols, of_rows[rows]);
      if (plan.lds_bytes != 0 && plan.score > best.score) best = plan;
    }
    return best;
  };
  // Work-groups of two or four waves, 64 features x 64 or 128 pixels each, on 64
  // (all of them) or 32 channels at a time: the least estimated time.  On 200
  // layers of 1e9 to 1.2e11 operations the estimates were within 10 % and the one
  // taken 1.6 % slower than the fastest, on the average.  (By counting wave tiles
  // and work-groups instead, images of some widths were left with two waves per
  // CU: 149x149x64 at batch 8 76 us, now 34; 150x150x64 -> 128 at batch 8 94, now
  // 45; and 224x224x64 at batch 16 with one work-group, whose loads, products and
  // stores took turns: 99, with two that share the LDS 85.)
  RowTilePlan best;
  for (int wf = 1; wf <= (p.features % 128 == 0 ? 2 : 1); ++wf)
    for (int waves = 2; waves <= 4; waves += 2)
      for (int pb = 2; pb <= 4; pb += 2)
        for (int bufs = 1; bufs <= 3; ++bufs) {
          if ((bufs == 1) != (p.channels == 64) && bufs == 1) continue;
          if (bufs == 3 && (waves != 4 || !win3)) continue;
          const RowTilePlan plan =
              best_tile(wf, waves / wf, pb, bufs == 1 ? 64 : 32, bufs);
          if (plan.lds_bytes != 0 && (best.lds_bytes == 0 || plan.us < best.us))
            best = plan;
        }
  return best;
}

bool takes(const snn_hip_conv2d_params& p) {
  const size_t x = static_cast<size_t>(p.batch) * p.in_rows * p.in_cols *
                   p.channels;
  const size_t y = static_cast<size_t>(p.batch) * p.out_rows * p.out_cols *
                   p.features;
  // (1x1 windows have no taps to reuse an LDS tile over)
  return p.stride_rows == 1 && p.stride_cols == 1 && p.channels % 64 == 0 &&
         p.features % 64 == 0 && p.channels > 0 && p.features > 0 &&
         p.batch > 0 && p.out_rows > 0 && p.out_cols > 0 && p.in_rows > 0 &&
         p.in_cols > 0 && p.window_rows * p.window_cols > 1 &&
         (x > y ? x : y) * 2 <= kMaxBufferBytes;
}

const RowTilePlan& make_plan(const snn_hip_conv2d_params& p) {
  thread_local PlanCache<RowTilePlan> cache;
  return cache.get(p, 0, [&] { return takes(p) ? compute_plan(p) : RowTilePlan(); });
}

template <int WF, int WP, int PB, int KC, int BUFS, bool WIN3>
void launch_plan(const _Float16* input, const _Float16* wpk, _Float16* output,
                 const snn_hip_conv2d_params& p, const RowTilePlan& plan,
                 size_t wgt_elems, hipStream_t stream) {
  auto kernel = conv_rowtile_f16_kernel<WF, WP, PB, KC, BUFS, WIN3>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLdsBytes);
  (void)attr;
  const size_t x = static_cast<size_t>(p.batch) * p.in_rows * p.in_cols *
                   p.channels;
  const size_t y = static_cast<size_t>(p.batch) * p.out_rows * p.out_cols *
                   p.features;
  KernelTimer timer(stream);
  hipLaunchKernelGGL(kernel, dim3(plan.n_groups), dim3(64 * WF * WP),
                     plan.lds_bytes, stream, input, wpk, output, plan.g,
                     static_cast<unsigned>(x * 2),
                     static_cast<unsigned>(wgt_elems * 2),
                     static_cast<unsigned>(y * 2), plan.n_groups);
}

template <int WF, int WP, int PB>
bool launch_shape(const _Float16* input, const _Float16* wpk,
                  _Float16* output, const snn_hip_conv2d_params& p,
                  const RowTilePlan& plan, size_t wgt_elems,
                  hipStream_t stream) {
  if (plan.wf != WF || plan.wp != WP || plan.pb != PB) return false;
  const bool win3 = p.window_rows == 3 && p.window_cols == 3;
#define SNN_ROWTILE_CASE(KC, BUFS, WIN3)                                      \
  if (plan.kc == KC && plan.bufs == BUFS && win3 == WIN3) {                   \
    launch_plan<WF, WP, PB, KC, BUFS, WIN3>(input, wpk, output, p, plan,      \
                                            wgt_elems, stream);               \
    return true;                                                              \
  }
  SNN_ROWTILE_CASE(64, 1, true)
  SNN_ROWTILE_CASE(32, 2, true)
  if constexpr (WF * WP == 4) {
    SNN_ROWTILE_CASE(32, 3, true)
  }
  SNN_ROWTILE_CASE(64, 1, false)
  SNN_ROWTILE_CASE(32, 2, false)
#undef SNN_ROWTILE_CASE
  return false;
}

}  // namespace

// Where this kernel is faster than the gathering one (conv2d_gather.hip,
// which shares a reduction between work-groups where there are few tiles), whose
// estimate is `other_us`: 3x3 windows by the estimates of both.  Other windows:
// short reductions at every size, and long ones with at least 1.5 wave tiles per
// SIMD that leave two waves on each.  Windows beyond 12 x 12 the other one does
// not take (gradient of 2x64x64x64 <- 64, 13x13: 89 us, through fp32 136).
bool conv2d_rowtile_f16_wanted(const snn_hip_conv2d_params& p,
                               double other_us) {
  const RowTilePlan& plan = make_plan(p);
  if (plan.lds_bytes == 0) return false;
  if (p.window_rows == 3 && p.window_cols == 3) return plan.us < other_us;
  if (p.window_rows * p.window_cols * p.channels <= 576 ||
      p.window_rows > 12 || p.window_cols > 12)
    return true;
  const size_t pixels = static_cast<size_t>(p.batch) * p.out_rows * p.out_cols;
  return ceil_div(pixels, size_t{64}) * static_cast<size_t>(p.features / 64) >=
             1536 &&
         (plan.pb == 4 || 2 * plan.lds_bytes <= kMaxLdsBytes);
}

int conv2d_rowtile_f16_buffers(const snn_hip_conv2d_params& p) {
  const RowTilePlan& plan = make_plan(p);
  return plan.lds_bytes != 0 ? plan.bufs : 0;
}

int launch_conv2d_rowtile_f16(const _Float16* input, const _Float16* filter,
                              _Float16* output, const snn_hip_conv2d_params& p,
                              _Float16* packed, hipStream_t stream,
                              bool transposed_filter) {
  const RowTilePlan& plan = make_plan(p);
  if (plan.lds_bytes == 0) return SNN_HIP_INVALID_ALGORITHM;
  static const bool print_plan = SNN_TUNING_ENV("SNN_HIP_F16_PLAN") != nullptr;
  if (print_plan)
    fprintf(stderr,
            "rowtile f16: waves %dx%d, %d pixel blocks, %d channels/tile, "
            "%d pixels/tile, %u work-groups, %zu B LDS\n",
            plan.wf, plan.wp, plan.pb, plan.kc, plan.g.tile_pixels,
            plan.n_groups, plan.lds_bytes);
  const int taps = p.window_rows * p.window_cols;
  const size_t wgt_elems =
      static_cast<size_t>(taps) * p.channels * p.features;
  // (channels and features are multiples of 64, kc is 32 or 64)
  hipLaunchKernelGGL(
      transposed_filter ? pack_filter_rowtile_kernel<true>
                        : pack_filter_rowtile_kernel<false>,
      dim3(static_cast<unsigned>(p.features / 64),
           static_cast<unsigned>(p.channels / 32), static_cast<unsigned>(taps)),
      dim3(256), 0, stream, filter, packed, p.channels, p.features,
      plan.kc == 64 ? 6 : 5);
  const bool launched =
      launch_shape<1, 2, 2>(input, packed, output, p, plan, wgt_elems, stream) ||
      launch_shape<1, 2, 4>(input, packed, output, p, plan, wgt_elems, stream) ||
      launch_shape<1, 4, 2>(input, packed, output, p, plan, wgt_elems, stream) ||
      launch_shape<1, 4, 4>(input, packed, output, p, plan, wgt_elems, stream) ||
      launch_shape<2, 1, 2>(input, packed, output, p, plan, wgt_elems, stream) ||
      launch_shape<2, 1, 4>(input, packed, output, p, plan, wgt_elems, stream) ||
      launch_shape<2, 2, 2>(input, packed, output, p, plan, wgt_elems, stream) ||
      launch_shape<2, 2, 4>(input, packed, output, p, plan, wgt_elems, stream);
  if (!launched) return SNN_HIP_INVALID_ALGORITHM;
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return report_hip_error(err, "conv_rowtile_f16_kernel");
  return SNN_HIP_OK;
}

}  // namespace snn
