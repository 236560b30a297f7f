// Launches whose stream-ordered temporary cannot be had: the allocation is made to
// fail here, on the host, and the launch takes a kernel that needs none.
#include <portdnn/backend/hip_backend.h>

#include <cstdint>
#include <cstring>
#include <vector>

#include "check.h"
#include "snn_hip.h"

// (the library's calls bind to these, the program's own first)
static int g_refused = 0;
extern "C" hipError_t hipMallocFromPoolAsync(void** ptr, size_t, hipMemPool_t,
                                             hipStream_t) {
  ++g_refused;
  *ptr = nullptr;
  return hipErrorOutOfMemory;
}
extern "C" hipError_t hipMallocAsync(void** ptr, size_t, hipStream_t) {
  ++g_refused;
  *ptr = nullptr;
  return hipErrorOutOfMemory;
}

namespace {

float half_value(std::uint16_t h) {
  const int exponent = h >> 10 & 31, mantissa = h & 1023;
  float v = exponent == 0 ? mantissa / 1024.f : 1.f + mantissa / 1024.f;
  for (int e = exponent == 0 ? 1 : exponent; e > 15; --e) v *= 2.f;
  for (int e = exponent == 0 ? 1 : exponent; e < 15; ++e) v /= 2.f;
  return h & 0x8000 ? -v : v;
}

// -1, 0 or 1: every sum of up to 2048 products is exact.
std::vector<std::uint16_t> values(size_t n, unsigned seed) {
  const std::uint16_t of[3] = {0xBC00, 0, 0x3C00};
  std::vector<std::uint16_t> v(n);
  for (auto& e : v) {
    seed = seed * 1664525u + 1013904223u;
    e = of[(seed >> 24) % 3];
  }
  return v;
}

void* on_device(const std::vector<std::uint16_t>& v) {
  void* p = nullptr;
  CHECK(hipMalloc(&p, v.size() * 2) == hipSuccess);
  CHECK(hipMemcpy(p, v.data(), v.size() * 2, hipMemcpyHostToDevice) ==
        hipSuccess);
  return p;
}

// A 5x5 layer of fewer than 256 output pixels on the kernel with bands in LDS, with
// a workspace that holds the filter in fp32 but not the partial tiles.
void test_filter_gradient() {
  constexpr int kRows = 15, kCols = 16, kC = 64, kK = 64, kW = 5;
  snn_hip_conv2d_params p{};
  p.channels = kC;
  p.features = kK;
  p.batch = 1;
  p.in_rows = p.out_rows = kRows;
  p.in_cols = p.out_cols = kCols;
  p.window_rows = p.window_cols = kW;
  p.stride_rows = p.stride_cols = 1;
  p.pad_rows = p.pad_cols = kW / 2;
  p.dilation_rows = p.dilation_cols = p.groups = 1;
  int form = 0;
  CHECK(snn_hip_conv2d_lds_form_f16(&p, SNN_HIP_FILTER_BACKPROP, &form) == SNN_HIP_OK && form > 1);
  const auto x = values(kRows * kCols * kC, 1), dy = values(kRows * kCols * kK, 2);
  std::vector<std::uint16_t> dw(kW * kW * kC * kK, 0xFFFF);
  void* const d_x = on_device(x);
  void* const d_dy = on_device(dy);
  void* const d_dw = on_device(dw);
  void* workspace = nullptr;
  const size_t elems = 2 * dw.size();
  CHECK(hipMalloc(&workspace, elems * 2) == hipSuccess);
  g_refused = 0;
  CHECK_EQ(snn_hip_conv2d_filter_backprop_f16(d_x, d_dy, d_dw, &p,
                                              SNN_HIP_ALGO_IM2COL, workspace,
                                              elems, nullptr),
           SNN_HIP_OK);
  CHECK(g_refused > 0);
  CHECK(hipMemcpy(dw.data(), d_dw, dw.size() * 2, hipMemcpyDeviceToHost) ==
        hipSuccess);
  int wrong = 0;
  for (int r = 0; r < kW; ++r)
    for (int s = 0; s < kW; ++s)
      for (int c = 0; c < kC; ++c)
        for (int k = 0; k < kK; ++k) {
          float sum = 0;
          for (int y = 0; y < kRows; ++y)
            for (int z = 0; z < kCols; ++z) {
              const int iy = y + r - kW / 2, ix = z + s - kW / 2;
              if (iy < 0 || iy >= kRows || ix < 0 || ix >= kCols) continue;
              sum += half_value(x[(iy * kCols + ix) * kC + c]) *
                     half_value(dy[(y * kCols + z) * kK + k]);
            }
          wrong += half_value(dw[((r * kW + s) * kC + c) * kK + k]) != sum;
        }
  CHECK_EQ(wrong, 0);
  // without that workspace there is no kernel for it, and the call says so
  CHECK_EQ(snn_hip_conv2d_filter_backprop_f16(d_x, d_dy, d_dw, &p,
                                              SNN_HIP_ALGO_IM2COL, nullptr, 0,
                                              nullptr),
           SNN_HIP_ALLOCATION_PROBLEM);
  for (void* ptr : {d_x, d_dy, d_dw, workspace})
    CHECK(hipFree(ptr) == hipSuccess);
}

// An input gradient on the row-tile kernel, whose packed filter has no room.
void test_input_gradient() {
  constexpr int kBatch = 11, kRows = 108, kCols = 37, kC = 64, kK = 64;
  snn_hip_conv2d_params p{};
  p.channels = kC;
  p.features = kK;
  p.batch = kBatch;
  p.in_rows = p.out_rows = kRows;
  p.in_cols = p.out_cols = kCols;
  p.window_rows = p.window_cols = 3;
  p.stride_rows = p.stride_cols = 1;
  p.pad_rows = p.pad_cols = 1;
  p.dilation_rows = p.dilation_cols = p.groups = 1;
  int form = 0;
  CHECK(snn_hip_conv2d_lds_form_f16(&p, SNN_HIP_INPUT_BACKPROP, &form) ==
        SNN_HIP_OK);
  const auto dy = values(size_t{kBatch} * kRows * kCols * kK, 3);
  const auto w = values(9 * kC * kK, 4);
  std::vector<std::uint16_t> dx(size_t{kBatch} * kRows * kCols * kC, 0xFFFF);
  void* const d_dy = on_device(dy);
  void* const d_w = on_device(w);
  void* const d_dx = on_device(dx);
  g_refused = 0;
  CHECK_EQ(snn_hip_conv2d_input_backprop_f16(d_dy, d_w, d_dx, &p,
                                             SNN_HIP_ALGO_IM2COL, nullptr, 0,
                                             nullptr),
           SNN_HIP_OK);
  CHECK(g_refused > 0);
  CHECK(hipMemcpy(dx.data(), d_dx, dx.size() * 2, hipMemcpyDeviceToHost) ==
        hipSuccess);
  int wrong = 0;
  for (int pixel = 0; pixel < kBatch * kRows * kCols; pixel += 97) {
    const int n = pixel / (kRows * kCols), y = pixel / kCols % kRows;
    const int x = pixel % kCols;
    for (int c = 0; c < kC; ++c) {
      float sum = 0;
      for (int r = 0; r < 3; ++r)
        for (int s = 0; s < 3; ++s) {
          const int oy = y + 1 - r, ox = x + 1 - s;
          if (oy < 0 || oy >= kRows || ox < 0 || ox >= kCols) continue;
          const size_t at = (size_t{1} * (n * kRows + oy) * kCols + ox) * kK;
          for (int k = 0; k < kK; ++k)
            sum += half_value(dy[at + k]) *
                   half_value(w[((r * 3 + s) * kC + c) * kK + k]);
        }
      wrong += half_value(dx[static_cast<size_t>(pixel) * kC + c]) != sum;
    }
  }
  CHECK_EQ(wrong, 0);
  for (void* ptr : {d_dy, d_w, d_dx}) CHECK(hipFree(ptr) == hipSuccess);
}

}  // namespace

int main() {
  test_filter_gradient();
  test_input_gradient();
  return report("gpu_no_temporary_test");
}
