// Row-major binary16 GEMM of few tiles (gfx950):
//   Y[m][n] = sum_k X[m][k] W[k][n]    (1x1 stride-1 convolution, matmul)
//   Y[m][n] = sum_k X[m][k] W[n][k]    (its input gradient, matmul with B
//                                       transposed)
// with fp32 accumulation on v_mfma_f32_32x32x16_f16 (portDNN runs both through
// its matmul kernel, src/matmul/kernels.h:26-133).
//
// A small batch through a channel-reducing layer (1568 pixels, 1024 -> 256) has
// 196 tiles of 32 x 64, fewer than compute units, and a reduction that a single
// wave takes 64 dependent steps for.  Here the eight waves of a work-group share
// the reduction of one such tile: a wave loads its share of both operands at once
// -- one round trip to memory for the whole product, which is what bounds the
// launch -- multiplies it without a barrier, and the eight sums meet in LDS, in a
// fixed order.  The operand whose reduction index is contiguous goes straight to
// registers, 16 bytes per lane; W[k][n] goes through the wave's own part of LDS,
// whence transposing reads fetch four rows of a column at a time
// (ds_read_b64_tr_b16, 16-byte pieces swizzled as the LDS-direct loads write them).
// 1568 x 1024 x 256: 10.9 -> 6.1 us a launch among others (one column group of the
// filter-in-LDS kernel, gemm_rows_f16.hip, is the work of a single wave there).
#include "snn_kernels.h"

namespace snn {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef unsigned int uint2v __attribute__((ext_vector_type(2)));
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

constexpr int kWaves = 8;    // shares of the reduction
constexpr int kRows = 32;    // rows of Y per work-group
constexpr int kCols = 64;    // columns
constexpr int kRowBytes = 2 * kCols;  // of W in LDS
constexpr int kSumPitch = kCols + 4;  // floats
constexpr int kSumBytes = kWaves * kRows * kSumPitch * 4;
constexpr unsigned kOob = 0x7FFFFFF0u;
constexpr size_t kMaxBufferBytes = 0x7FFFFFF0u;

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p,
                                                   unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x00020000);
}

// (a function of its own: the compiler drops the host side of a kernel template
// whose body names the LDS-direct load)
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t rsrc,
                                            char* lds, unsigned offset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)lds, 16, offset, 0, 0,
                                           0);
}

__device__ __forceinline__ uint4v load16(__amdgpu_buffer_rsrc_t rsrc,
                                         unsigned offset) {
  return __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0);
}

// Which 16-byte position of row r of W holds 16-byte piece c: c ^ swz(r) (four
// consecutive rows get four different pairs, rows 8 apart swap the pairs of even
// and odd rows: the 16 lanes of a transposing read fall into distinct banks).
__device__ __forceinline__ unsigned swz(unsigned r) {
  return ((r & 3u) ^ ((r >> 3) & 1u)) << 1;
}

// STEPS matrix-instruction steps of 16 reduction indices per wave and block of
// the reduction (blocks of 128 * STEPS).
template <int STEPS, bool NT>
__global__ void __launch_bounds__(64 * kWaves)
    gemm_short_f16_kernel(const _Float16* __restrict__ x,
                          const _Float16* __restrict__ w,
                          _Float16* __restrict__ y, int m_total, int k_total,
                          int n_total, int col_tiles) {
  extern __shared__ __align__(1024) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (column tiles side by side: the work-groups of one XCD share rows of X every
  // 8 / col_tiles, and W lies in every XCD's L2)
  const int m0 = static_cast<int>(blockIdx.x) / col_tiles * kRows;
  const int n0 = static_cast<int>(blockIdx.x) % col_tiles * kCols;
  const __amdgpu_buffer_rsrc_t x_rsrc =
      make_rsrc(x, static_cast<unsigned>(m_total) * k_total * 2u);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      make_rsrc(w, static_cast<unsigned>(n_total) * k_total * 2u);
  constexpr int kShare = 16 * STEPS;  // reduction indices of a wave
  char* const mine = lds + wave * (kShare * kRowBytes);
  const int l32 = lane & 31, khalf = lane >> 5;
  const unsigned gq = lane >> 4, j = (lane >> 2) & 3, e = lane & 3;

  float16v acc[2];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[c][i] = 0.f;

  for (int k0 = wave * kShare; k0 < k_total; k0 += kWaves * kShare) {
    uint4v xb[STEPS], wb[NT ? STEPS : 1][2];
    if constexpr (!NT) {
      // a load instruction fetches 8 rows of W (128 bytes each)
#pragma unroll
      for (int i = 0; i < 2 * STEPS; ++i) {
        const unsigned r = 8u * i + (lane >> 3);
        const unsigned piece = (lane & 7u) ^ swz(r);
        const bool ok = k0 + static_cast<int>(r) < k_total &&
                        n0 + 8 * static_cast<int>(piece) < n_total;
        load_to_lds(w_rsrc, mine + i * 1024,
                    ok ? ((k0 + r) * n_total + n0 + 8u * piece) * 2u : kOob);
      }
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = k0 + 16 * s + 8 * khalf;
      xb[s] = load16(x_rsrc, m0 + l32 < m_total && k < k_total
                                 ? static_cast<unsigned>(
                                       (m0 + l32) * k_total + k) * 2u
                                 : kOob);
      if constexpr (NT)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          wb[s][c] = load16(w_rsrc, n0 + 32 * c + l32 < n_total && k < k_total
                                        ? static_cast<unsigned>(
                                              (n0 + 32 * c + l32) * k_total + k) *
                                              2u
                                        : kOob);
    }
    if constexpr (!NT) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        half8 a;
        if constexpr (NT) {
          a = __builtin_bit_cast(half8, wb[s][c]);
        } else {
          // of lane = 16 gq + 4 j + e, as a source of the transposing read: row
          // 8 (gq / 2) + j (+ 4 for the second), halves 4 e ... + 3 of the
          // 16-wide block gq % 2 of the 32 columns
          uint2v part[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const unsigned r = 16u * s + 8 * (gq >> 1) + 4 * h + j;
            const char* const at =
                mine + r * kRowBytes +
                (((4u * c + 2 * (gq & 1) + (e >> 1)) ^ swz(r)) << 4) +
                ((e & 1) << 3);
            part[h] = __builtin_bit_cast(
                uint2v,
                __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at)));
          }
          a = __builtin_bit_cast(half8, uint4v{part[0][0], part[0][1],
                                               part[1][0], part[1][1]});
        }
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            a, __builtin_bit_cast(half8, xb[s]), acc[c], 0, 0, 0);
      }
    }
  }

  // acc[c][i]: row l32 of the tile, column 32 c + 8 (i / 4) + 4 khalf + i % 4
  __syncthreads();  // (W in LDS is done with)
  float* const sums = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4v*>(sums + (wave * kRows + l32) * kSumPitch +
                                  32 * c + 8 * g + 4 * khalf) =
          float4v{acc[c][4 * g], acc[c][4 * g + 1], acc[c][4 * g + 2],
                  acc[c][4 * g + 3]};
  __syncthreads();
  const int row = threadIdx.x >> 4, col = 4 * (threadIdx.x & 15);
  float4v sum = *reinterpret_cast<const float4v*>(sums + row * kSumPitch + col);
#pragma unroll
  for (int s = 1; s < kWaves; ++s)
    sum += *reinterpret_cast<const float4v*>(
        sums + (s * kRows + row) * kSumPitch + col);
  if (m0 + row < m_total && n0 + col < n_total) {
    half4v r;
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = static_cast<_Float16>(sum[v]);
    *reinterpret_cast<half4v*>(y + static_cast<size_t>(m0 + row) * n_total + n0 +
                               col) = r;
  }
}

template <int STEPS, bool NT>
int launch_as(const _Float16* x, const _Float16* w, _Float16* y, int m, int k,
              int n, hipStream_t stream) {
  constexpr int kLds =
      !NT && kWaves * 16 * STEPS * kRowBytes > kSumBytes
          ? kWaves * 16 * STEPS * kRowBytes : kSumBytes;
  auto kernel = gemm_short_f16_kernel<STEPS, NT>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kernel),
      hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (attr != hipSuccess) return report_hip_error(attr, "gemm_short_f16_kernel");
  const int col_tiles = ceil_div(n, kCols);
  KernelTimer timer(stream);
  hipLaunchKernelGGL(kernel,
                     dim3(static_cast<unsigned>(ceil_div(m, kRows) * col_tiles)),
                     dim3(64 * kWaves), kLds, stream, x, w, y, m, k, n,
                     col_tiles);
  SNN_HIP_CHECK_LAUNCH();
  return SNN_HIP_OK;
}

template <bool NT>
int launch_steps(const _Float16* x, const _Float16* w, _Float16* y, int m,
                 int k, int n, hipStream_t stream) {
  if (k <= 128) return launch_as<1, NT>(x, w, y, m, k, n, stream);
  if (k <= 256) return launch_as<2, NT>(x, w, y, m, k, n, stream);
  if (k <= 512) return launch_as<4, NT>(x, w, y, m, k, n, stream);
  return launch_as<8, NT>(x, w, y, m, k, n, stream);
}

}  // namespace

// Where it is the faster one, by 150 random products (us, back to back): X W up
// to 512 tiles (1568 x 1024 x 256, 196 tiles: 6.1 against 10.9; 1728 x 320 x 640,
// 540: 7.2 / 7.8; 3380 x 1600 x 512, 848: 32 / 20, as every tile reads all its
// operands by itself).  X W^T has a kernel that needs no transposition where k is
// a multiple of 64 and loses to it from about 128 tiles or 512 reduction indices
// on (2205 x 128 x 64, 69 tiles: 3.5 / 3.6; 392 x 896 x 576, 117: 7.4 / 6.7;
// 2916 x 192 x 128, 184: 4.0 / 3.6); other k ran on the gathering kernel (1008 x 216
// x 456, 256: 3.6 / 5.3; 1944 x 24 x 1592, 1525: 7.5 / 5.5).
bool gemm_short_f16_wanted(int m, int k, int n, bool transpose_w) {
  if (m < 1 || k < 8 || n < 8 || k % 8 != 0 || n % 8 != 0) return false;
  if (static_cast<size_t>(m) * k * 2 > kMaxBufferBytes ||
      static_cast<size_t>(n) * k * 2 > kMaxBufferBytes)
    return false;
  const size_t tiles = ceil_div(static_cast<size_t>(m), size_t{kRows}) *
                       ceil_div(static_cast<size_t>(n), size_t{kCols});
  if (transpose_w && k % 64 == 0) return tiles <= 128 && k <= 512;
  return tiles <= 512;
}

int launch_gemm_short_f16(const _Float16* x, const _Float16* w, _Float16* y,
                          int m, int k, int n, bool transpose_w,
                          hipStream_t stream) {
  return transpose_w ? launch_steps<true>(x, w, y, m, k, n, stream)
                     : launch_steps<false>(x, w, y, m, k, n, stream);
}

}  // namespace snn
