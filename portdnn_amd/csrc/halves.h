// fp32 operands as two binary16 values each: v = hi + 2^-11 lo times a power of two
// that a block of values shares (conv2d_halves_f32.hip says what is lost and what
// happens where that is too much).
#ifndef PORTDNN_AMD_CSRC_HALVES_H_
#define PORTDNN_AMD_CSRC_HALVES_H_

#include <hip/hip_runtime.h>

namespace snn {
namespace halves {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
typedef unsigned int uint2v __attribute__((ext_vector_type(2)));
constexpr unsigned kOob = 0x7FFFFFF0u;
constexpr size_t kMaxBufferBytes = 0x7FFFFFF0u;
constexpr int kNumCus = 256;
constexpr size_t kMaxLdsBytes = 160 * 1024;
constexpr int kWaitLgkm0 = 0xC07F;       // s_waitcnt: LDS operations only

// n / d for 0 <= n < 2^31 by one multiplication: (2 n * magic) >> (32 + shift)
// with magic = ceil(2^(31 + shift) / d), 2^shift >= d.
struct Divisor {
  unsigned magic, shift;
};
inline Divisor divisor(int d) {
  unsigned shift = 0;
  while ((1u << shift) < static_cast<unsigned>(d)) ++shift;
  const unsigned long long top = 1ull << (31 + shift);
  return {static_cast<unsigned>((top + d - 1) / d), shift};
}
__device__ __forceinline__ int divide(int n, Divisor d) {
  return static_cast<int>(
      __umulhi(static_cast<unsigned>(n) << 1, d.magic) >> d.shift);
}

__device__ inline __amdgpu_buffer_rsrc_t make_rsrc(const void* p,
                                                   unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x00020000);
}

// The exponents of a block's scale.  A value's magnitude bits are shifted left by
// one (`big`: the largest; `small`: the smallest one that is not zero, minus one).
constexpr int kTop = 14;    // the largest scaled value is in [2^14, 2^15)
constexpr int kLow = -12;   // and values below 2^-12 lose bits
constexpr int kBand = 26;   // by which these are scaled up
enum { kSmall = 1, kBeyond = 2, kZero = 4 };
struct Range {
  unsigned big, small;
};
__device__ __forceinline__ unsigned magnitude(float v) {
  return __builtin_bit_cast(unsigned, v) << 1;
}
__device__ __forceinline__ void note(Range& r, float v) {
  const unsigned u = magnitude(v);
  r.big = max(r.big, u);
  r.small = min(r.small, u - 1u);
}
__device__ __forceinline__ int exponent_for(unsigned big) {
  return kTop + 127 - static_cast<int>(big >> 24);
}
// What scaling by 2^exponent does to a block: kSmall, kBeyond.
__device__ __forceinline__ int loses(Range r, int exponent) {
  int flags = 0;
  if ((r.big >> 24) == 255u || exponent > 100) flags |= kBeyond;
  if (r.small != 0xFFFFFFFFu) {
    const int low = static_cast<int>((r.small + 1u) >> 24) + exponent - 127;
    if (low < kLow) flags |= kSmall;
    if (low < kLow - kBand || (low < kLow && (r.small + 1u) >> 24 == 0))
      flags |= kBeyond;
  }
  return flags;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned max_from(unsigned v) {
  return max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(
                    0, static_cast<int>(v), CTRL, ROWS, 0xF, false)));
}
__device__ __forceinline__ unsigned wave_max(unsigned v) {
  v = max_from<0x111, 0xF>(v);  // lanes 1, 2, 4, 8 to the left in a row of 16
  v = max_from<0x112, 0xF>(v);
  v = max_from<0x114, 0xF>(v);
  v = max_from<0x118, 0xF>(v);
  v = max_from<0x142, 0xA>(v);  // the last lane of a row to the next row
  v = max_from<0x143, 0xC>(v);  // lane 31 to the upper half
  return static_cast<unsigned>(
      __builtin_amdgcn_readlane(static_cast<int>(v), 63));
}
__device__ __forceinline__ Range wave_range(Range r) {
  return {wave_max(r.big), ~wave_max(~r.small)};
}

__device__ __forceinline__ float pow2(int exponent) {
  return __builtin_bit_cast(float, static_cast<unsigned>(exponent + 127) << 23);
}

// Two values times `scale` as two binary16 ones each.
struct Pair {
  unsigned hi, lo;
};
__device__ __forceinline__ Pair take_apart(float a, float b, float scale,
                                           float scale2048) {
  typedef _Float16 half2 __attribute__((ext_vector_type(2)));
  typedef float float2v __attribute__((ext_vector_type(2)));
  unsigned hi = __builtin_bit_cast(
      unsigned, __builtin_convertvector(float2v{a * scale, b * scale}, half2));
  // (else every value is converted a second time, by itself, for the difference)
  asm("" : "+v"(hi));
  const half2 h = __builtin_bit_cast(half2, hi);
  half2 lo;
  lo[0] = static_cast<_Float16>(
      __builtin_fmaf(static_cast<float>(h[0]), -2048.f, a * scale2048));
  lo[1] = static_cast<_Float16>(
      __builtin_fmaf(static_cast<float>(h[1]), -2048.f, b * scale2048));
  return {hi, __builtin_bit_cast(unsigned, lo)};
}

}  // namespace halves
}  // namespace snn

#endif  // PORTDNN_AMD_CSRC_HALVES_H_
