// The launch plans of a network's layers, kept per thread: a launch asks for its plan
// several times, and a network comes round to the same layers with every step.
// A plan takes 5-100 us to compute, a kept one is found in 0.1 us.
#ifndef SNN_PLAN_CACHE_H_
#define SNN_PLAN_CACHE_H_

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <new>
#include <type_traits>

#include "snn_hip.h"

namespace snn {

// Fully associative, so that no set of up to kCapacity layers has two that displace
// each other; the one asked for longest ago makes room.  A reference stays valid
// until kCapacity - 1 other plans have been asked for.
template <typename Plan>
class PlanCache {
  static_assert(std::is_trivially_copyable<Plan>::value &&
                    std::is_trivially_destructible<Plan>::value,
                "plans live in raw memory");

 public:
  static constexpr int kCapacity = 128;  // (the deepest networks have as many)

  PlanCache() = default;
  PlanCache(const PlanCache&) = delete;
  PlanCache& operator=(const PlanCache&) = delete;
  ~PlanCache() { std::free(entries_); }

  // The plan of (p, form), from compute() where it is not kept.
  template <typename F>
  const Plan& get(const snn_hip_conv2d_params& p, unsigned form, F compute) {
    ++now_;
    if (latest_ < used_ && matches(latest_, p, form)) return hit(latest_);
    const std::uint64_t hash = hash_of(p, form);
    for (int k = 0; k < used_; ++k)
      if (hashes_[k] == hash && matches(k, p, form)) return hit(k);
    const Plan plan = compute();
    if (entries_ == nullptr)
      entries_ = static_cast<Entry*>(std::malloc(kCapacity * sizeof(Entry)));
    if (entries_ == nullptr) {
      // (no memory: the last two plans, so that a launch can compare two)
      spare_[now_ & 1] = plan;
      return spare_[now_ & 1];
    }
    int at = used_;
    if (used_ < kCapacity) {
      ++used_;
    } else {
      at = 0;
      for (int k = 1; k < kCapacity; ++k)
        if (asked_[k] < asked_[at]) at = k;
    }
    hashes_[at] = hash;
    new (&entries_[at]) Entry{p, form, plan};
    return hit(at);
  }

 private:
  struct Entry {
    snn_hip_conv2d_params params;
    unsigned form;
    Plan plan;
  };

  static std::uint64_t hash_of(const snn_hip_conv2d_params& p, unsigned form) {
    constexpr int kWords = (sizeof p + 7) / 8;
    std::uint64_t words[kWords] = {};
    std::memcpy(words, &p, sizeof p);
    std::uint64_t h = form;
    for (const std::uint64_t word : words) {
      h = (h ^ word) * 0x9E3779B97F4A7C15ull;
      h ^= h >> 32;
    }
    return h;
  }
  bool matches(int k, const snn_hip_conv2d_params& p, unsigned form) const {
    return entries_[k].form == form &&
           std::memcmp(&entries_[k].params, &p, sizeof p) == 0;
  }
  const Plan& hit(int k) {
    asked_[k] = now_;
    latest_ = k;
    return entries_[k].plan;
  }

  Entry* entries_ = nullptr;
  int used_ = 0, latest_ = 0;
  std::uint64_t now_ = 0;
  std::uint64_t hashes_[kCapacity] = {};
  std::uint64_t asked_[kCapacity] = {};
  Plan spare_[2] = {};
};

}  // namespace snn

#endif  // SNN_PLAN_CACHE_H_
