// The per-thread cache of launch plans on the layers that a network has: channel
// counts and image sizes in multiples of powers of two must not displace each other.
#include "../../portdnn_amd/csrc/plan_cache.h"

#include <vector>

#include "check.h"

namespace {

struct Plan {
  int channels, rows;
  unsigned form;
};

snn_hip_conv2d_params layer(int batch, int size, int channels, int features,
                            int window, int stride) {
  snn_hip_conv2d_params p{};
  p.batch = batch;
  p.in_rows = p.in_cols = size;
  p.channels = channels;
  p.features = features;
  p.window_rows = p.window_cols = window;
  p.stride_rows = p.stride_cols = stride;
  p.out_rows = p.out_cols = size / stride;
  p.pad_rows = p.pad_cols = window / 2;
  p.dilation_rows = p.dilation_cols = p.groups = 1;
  return p;
}

struct Counting {
  snn::PlanCache<Plan> cache;
  int computed = 0;
  Plan ask(const snn_hip_conv2d_params& p, unsigned form) {
    return cache.get(p, form, [&] {
      ++computed;
      return Plan{p.channels, p.in_rows, form};
    });
  }
};

void test_layers_of_a_network() {
  std::vector<snn_hip_conv2d_params> layers;
  const int sizes[] = {56, 28, 14, 7};
  for (int k = 0; k < 4; ++k) {
    const int c = 64 << k, size = sizes[k];
    layers.push_back(layer(128, size, 4 * c, c, 1, 1));
    layers.push_back(layer(128, size, c, c, 3, 1));
    layers.push_back(layer(128, size, c, 4 * c, 1, 1));
    layers.push_back(layer(128, 2 * size, c, c, 3, 2));
    layers.push_back(layer(128, 4 * size, c, c, 3, 1));
    layers.push_back(layer(128, 4 * size, c / 2, c, 3, 1));
  }
  Counting plans;
  for (int step = 0; step < 3; ++step)
    for (const auto& p : layers)
      for (unsigned form = 0; form < 4; ++form) {
        const Plan plan = plans.ask(p, form);
        CHECK(plan.channels == p.channels && plan.rows == p.in_rows &&
              plan.form == form);
      }
  CHECK(plans.computed == static_cast<int>(layers.size()) * 4);
}

// More layers than it holds: every answer is right, the one asked for last time
// is kept, and so is a reference while another plan is looked up.
void test_more_layers_than_it_holds() {
  Counting plans;
  constexpr int kMany = 3 * snn::PlanCache<Plan>::kCapacity;
  for (int round = 0; round < 2; ++round)
    for (int k = 1; k <= kMany; ++k) {
      const auto p = layer(k, 8, 16 * k, 64, 3, 1);
      const Plan& first = plans.cache.get(
          p, 0, [&] { return Plan{p.channels, p.in_rows, 0}; });
      const Plan& second = plans.cache.get(
          p, 1, [&] { return Plan{p.channels, p.in_rows, 1}; });
      CHECK(first.channels == 16 * k && first.form == 0);
      CHECK(second.channels == 16 * k && second.form == 1);
      const int before = plans.computed;
      plans.ask(p, 0);
      plans.ask(p, 1);
      CHECK(plans.computed == before);
    }
}

}  // namespace

int main() {
  test_layers_of_a_network();
  test_more_layers_than_it_holds();
  return report("plan_cache_test");
}
