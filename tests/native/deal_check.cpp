// yx::Deal against a sort and a heap: the same busiest slot for random lists, longest first and
// in order, one object for all lists. Prints a JSON line with both times of large lists.
#include <chrono>
#include <cstdio>
#include <functional>
#include <random>

#include "../../yaxus_amd/csrc/deal.hpp"

static uint32_t by_heap(std::vector<uint32_t> lens, size_t slots, bool sorted) {
  if (sorted) std::sort(lens.begin(), lens.end(), std::greater<uint32_t>());
  std::vector<uint32_t> load(slots, 0);
  uint32_t most = 0;
  for (uint32_t n : lens) {
    std::pop_heap(load.begin(), load.end(), std::greater<uint32_t>());
    load.back() += n;
    most = std::max(most, load.back());
    std::push_heap(load.begin(), load.end(), std::greater<uint32_t>());
  }
  return most;
}

int main() {
  std::mt19937 rng(7);
  const auto pick = [&](uint32_t lo, uint32_t hi) { return lo + rng() % (hi - lo + 1); };
  yx::Deal deal;
  std::vector<uint32_t> lens, out;
  for (int round = 0; round < 4000; ++round) {
    const size_t slots = pick(1, round % 2 ? 600 : 8);
    const uint32_t longest = pick(1, round % 3 ? 40 : 5000);
    const bool sorted = round % 5 != 0;
    lens.clear();
    deal.clear();
    uint64_t sum = 0;
    for (uint32_t i = pick(round % 7 != 0, 900); i > 0; --i) {
      const uint32_t len = pick(1, longest), n = sorted ? pick(0, 4) : 1;
      lens.insert(lens.end(), n, len);
      sum += static_cast<uint64_t>(len) * n;
      sorted ? deal.add(len, n) : deal.add_in_order(len);
    }
    if (deal.items() != lens.size() || deal.sum() != sum) return std::puts("items or sum differ"), 1;
    if (deal.busiest(slots) != by_heap(lens, slots, sorted)) return std::puts("busiest slot differs"), 1;
    if (sorted) {
      deal.sorted(out);
      std::sort(lens.begin(), lens.end(), std::greater<uint32_t>());
      if (out != lens) return std::puts("order differs"), 1;
    }
  }
  // 1400 items over 256 slots, as a pass of several hundred sequences has them.
  lens.clear();
  for (int i = 0; i < 1400; ++i) lens.push_back(pick(20, 300));
  double us[2] = {1e30, 1e30};
  uint32_t most[2];
  for (int rep = 0; rep < 50; ++rep)
    for (int k = 0; k < 2; ++k) {
      const auto t0 = std::chrono::steady_clock::now();
      if (k == 0) {
        most[k] = by_heap(lens, 256, true);
      } else {
        deal.clear();
        for (uint32_t n : lens) deal.add(n, 1);
        most[k] = deal.busiest(256);
      }
      us[k] = std::min(us[k], std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count());
    }
  if (most[0] != most[1]) return std::puts("busiest slot differs"), 1;
  std::printf("{\"heap_us\": %.1f, \"deal_us\": %.1f}\n", us[0], us[1]);
  return 0;
}
