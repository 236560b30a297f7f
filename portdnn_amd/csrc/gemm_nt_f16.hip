// Half-precision GEMM with both operands contiguous along the reduction on MFMA
// (gfx950): y[m][n] = sum_k x[m][k] w[n][k], binary16 operands, fp32
// accumulation, binary16 result.  The input gradient of a stride-1 unpadded 1x1
// convolution is this product (x = dY, w = the HWCF filter, read in place), and
// so is a row-major A * B^T.
//
// A work-group owns a BM x BN tile and walks the reduction in chunks of 64
// halves -- one 128-byte line of every row, which is what these products, bound
// by the bytes they move, want: the gathering kernel of conv2d_gather.hip,
// whose chunks are half a line, takes 58 us where this one takes 55.8
// (401408x64x256, 257 MB) and 15.0 against 12.4 at a quarter of the rows.  Both
// tiles pass through registers into two LDS stages; lane l supplies
// A[row = l % 32][k = 8 * (l / 32) .. + 7] and the matching B values, exactly
// one ds_read_b128 per operand per v_mfma_f32_32x32x16_f16.
#include <algorithm>

#include "gemm_tile.h"
#include "snn_kernels.h"

namespace snn {
namespace {

using gemm::float16v;
using gemm::kThreads;
using gemm::xcd_remap;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
constexpr int kBKh = 64;             // halves per reduction chunk
constexpr int kRowH = kBKh + 8;      // halves per LDS tile row (16-byte pad)
constexpr unsigned kOob = 0x7FFFFFF0u;
constexpr size_t kMaxBufferBytes = 0x7FFFFFF0u;

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p,
                                                   unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x00020000);
}

template <int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__(kThreads)
    gemm_nt_f16_kernel(const _Float16* __restrict__ x,
                       const _Float16* __restrict__ w,
                       _Float16* __restrict__ y, int m, int k, int n,
                       unsigned n_tiles_n, unsigned n_tiles) {
  static_assert(WM * WN == 4, "four waves per work-group");
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int A_HALVES = BM * kRowH;
  constexpr int STAGE_HALVES = (BM + BN) * kRowH;
  extern __shared__ __align__(16) _Float16 lds_h[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wave_m = wave / WN, wave_n = wave % WN;
  const unsigned tile = xcd_remap(blockIdx.x, n_tiles);
  const int m0 = static_cast<int>(tile / n_tiles_n) * BM;
  const int n0 = static_cast<int>(tile % n_tiles_n) * BN;
  const int n_chunks = k / kBKh;

  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(x, 2u * m * k);
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(w, 2u * n * k);

  constexpr int A_PASSES = BM / 32;
  constexpr int B_PASSES = BN / 32;
  const int cc = tid & 7;   // 16-byte column of the 128-byte tile row
  const int r0 = tid >> 3;  // tile row of pass 0
  unsigned a_voff[A_PASSES], b_voff[B_PASSES];
#pragma unroll
  for (int i = 0; i < A_PASSES; ++i) {
    const int row = m0 + r0 + 32 * i;
    a_voff[i] = row < m ? static_cast<unsigned>(row * k + 8 * cc) * 2u : kOob;
  }
#pragma unroll
  for (int i = 0; i < B_PASSES; ++i) {
    const int col = n0 + r0 + 32 * i;
    b_voff[i] = col < n ? static_cast<unsigned>(col * k + 8 * cc) * 2u : kOob;
  }

  int chunk = 0;
  uint4v a_reg[A_PASSES], b_reg[B_PASSES];
  auto load_global = [&]() {
    if (chunk >= n_chunks) return;
    const unsigned soff = static_cast<unsigned>(chunk * kBKh) * 2u;
#pragma unroll
    for (int i = 0; i < A_PASSES; ++i)
      a_reg[i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, a_voff[i], soff, 0);
#pragma unroll
    for (int i = 0; i < B_PASSES; ++i)
      b_reg[i] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, b_voff[i], soff, 0);
    ++chunk;
  };
  _Float16* const a_store = lds_h + r0 * kRowH + 8 * cc;
  _Float16* const b_store = lds_h + A_HALVES + r0 * kRowH + 8 * cc;
  auto store_tiles = [&](int stage) {
#pragma unroll
    for (int i = 0; i < A_PASSES; ++i)
      *reinterpret_cast<uint4v*>(a_store + stage * STAGE_HALVES +
                                 32 * i * kRowH) = a_reg[i];
#pragma unroll
    for (int i = 0; i < B_PASSES; ++i)
      *reinterpret_cast<uint4v*>(b_store + stage * STAGE_HALVES +
                                 32 * i * kRowH) = b_reg[i];
  };

  float16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int l32 = lane & 31;
  const int k_half = 8 * (lane >> 5);
  auto compute = [&](int stage) {
    const _Float16* a_tile = lds_h + stage * STAGE_HALVES;
    const _Float16* b_tile = a_tile + A_HALVES;
    half8 a[kBKh / 16][TM], b[kBKh / 16][TN];
#pragma unroll
    for (int s = 0; s < kBKh / 16; ++s) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
        a[s][i] = *reinterpret_cast<const half8*>(
            a_tile + (wave_m * WTM + 32 * i + l32) * kRowH + 16 * s + k_half);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        b[s][j] = *reinterpret_cast<const half8*>(
            b_tile + (wave_n * WTN + 32 * j + l32) * kRowH + 16 * s + k_half);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < kBKh / 16; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              a[s][i], b[s][j], acc[i][j], 0, 0, 0);
  };

  load_global();
  store_tiles(0);
  __syncthreads();
  for (int done = 0;; done += 2) {
    load_global();
    compute(0);
    if (done + 1 >= n_chunks) break;
    store_tiles(1);
    __syncthreads();
    load_global();
    compute(1);
    if (done + 2 >= n_chunks) break;
    store_tiles(0);
    __syncthreads();
  }

  const __amdgpu_buffer_rsrc_t y_rsrc = make_rsrc(y, 2u * m * n);
  const unsigned row_bytes = static_cast<unsigned>(n) * 2u;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wave_n * WTN + 32 * j + l32;
      const int m_base = m0 + wave_m * WTM + 32 * i + 4 * (lane >> 5);
      const unsigned voff =
          (col < n && m_base < m)
              ? static_cast<unsigned>(m_base) * row_bytes +
                    static_cast<unsigned>(col) * 2u
              : kOob;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const unsigned off =
            voff + static_cast<unsigned>(8 * (v >> 2) + (v & 3)) * row_bytes;
        const _Float16 h = static_cast<_Float16>(acc[i][j][v]);
        __builtin_amdgcn_raw_buffer_store_b16(
            __builtin_bit_cast(unsigned short, h), y_rsrc, off, 0, 0);
      }
    }
  }
}

template <int BM, int BN, int WM, int WN>
void launch_tile(const _Float16* x, const _Float16* w, _Float16* y, int m,
                 int k, int n, hipStream_t stream) {
  const unsigned tiles_n = static_cast<unsigned>(ceil_div(n, BN));
  const unsigned n_tiles = static_cast<unsigned>(ceil_div(m, BM)) * tiles_n;
  constexpr size_t kLdsBytes = 2 * sizeof(_Float16) * (BM + BN) * kRowH;
  auto kernel = gemm_nt_f16_kernel<BM, BN, WM, WN>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
  (void)attr;
  KernelTimer timer(stream);
  hipLaunchKernelGGL(kernel, dim3(n_tiles), dim3(kThreads), kLdsBytes, stream,
                     x, w, y, m, k, n, tiles_n, n_tiles);
}

}  // namespace

bool gemm_nt_f16_supports(int m, int k, int n) {
  const size_t x = static_cast<size_t>(m) * k, w = static_cast<size_t>(n) * k,
               y = static_cast<size_t>(m) * n;
  return k % kBKh == 0 &&
         std::max(std::max(x, y), w) * sizeof(_Float16) <= kMaxBufferBytes;
}

// x and w 16-byte aligned.
int launch_gemm_nt_f16(const _Float16* x, const _Float16* w, _Float16* y, int m,
                       int k, int n, hipStream_t stream) {
  if (n > 64 && static_cast<long>(ceil_div(m, 128)) * ceil_div(n, 128) >= 512)
    launch_tile<128, 128, 2, 2>(x, w, y, m, k, n, stream);
  else
    launch_tile<64, 64, 2, 2>(x, w, y, m, k, n, stream);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return report_hip_error(err, "gemm_nt_f16_kernel");
  return SNN_HIP_OK;
}

}  // namespace snn
