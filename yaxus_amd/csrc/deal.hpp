// The load of a number of slots (CUs, or workgroup slots of CUs) that take a work list's items
// one after the other: what the chunk searches of the work lists estimate their time from.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace yx {

// The busiest of a number of slots once items are dealt, each to the least loaded slot:
// longest first, or in the order they were added. A step costs one slot group of equal load
// instead of a sort and two heap operations per item (the whole list of 48 ragged sequences
// 21 -> 11 us on the host, of 521 on one KV head 439 -> 60; without a search 2 and 17).
class Deal {
 public:
  void clear() {
    std::fill(count_.begin(), count_.begin() + std::min<size_t>(longest_ + 1, count_.size()), 0u);
    order_.clear();
    longest_ = 0;
    items_ = 0;
    sum_ = 0;
  }
  // n items of len > 0, to be dealt longest first.
  void add(uint32_t len, uint32_t n) {
    if (n == 0) return;
    if (len >= count_.size()) count_.resize(std::max<size_t>(len + 1, 2 * count_.size()), 0u);
    count_[len] += n;
    note(len, n);
  }
  // An item to be dealt in order (all of a list, or none).
  void add_in_order(uint32_t len) {
    order_.push_back(len);
    note(len, 1);
  }
  size_t items() const { return items_; }
  uint64_t sum() const { return sum_; }
  uint32_t busiest(size_t slots) {
    size_t n = 1;
    while (n <= longest_) n *= 2;
    at_.assign(n, 0);  // slots per load, modulo n: loads differ by the longest item at most
    mask_ = static_cast<uint32_t>(n - 1);
    at_[0] = static_cast<uint32_t>(slots);
    low_ = most_ = 0;
    if (!order_.empty())
      for (uint32_t len : order_) give(len, 1);
    else
      for (uint32_t len = longest_; len > 0; --len)
        if (count_[len]) give(len, count_[len]);
    return most_;
  }
  // The lengths, longest first.
  void sorted(std::vector<uint32_t>& out) const {
    out.clear();
    for (uint32_t len = longest_; len > 0; --len) out.insert(out.end(), count_[len], len);
  }

 private:
  void note(uint32_t len, uint32_t n) {
    longest_ = std::max(longest_, len);
    items_ += n;
    sum_ += static_cast<uint64_t>(len) * n;
  }
  void give(uint32_t len, uint32_t n) {
    while (n > 0) {
      while (at_[low_ & mask_] == 0) ++low_;
      uint32_t& from = at_[low_ & mask_];
      const uint32_t k = std::min(n, from);
      from -= k;
      at_[(low_ + len) & mask_] += k;
      most_ = std::max(most_, low_ + len);
      n -= k;
    }
  }
  std::vector<uint32_t> count_, order_, at_;
  uint32_t longest_ = 0, mask_ = 0, low_ = 0, most_ = 0;
  size_t items_ = 0;
  uint64_t sum_ = 0;
};

}  // namespace yx
