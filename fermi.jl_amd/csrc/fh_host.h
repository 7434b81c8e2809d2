// Host code without HIP types: compiled into the library, and by itself in the CPU tests.
#pragma once
#include <algorithm>
#include <cstdint>

namespace fh {

// Workgroups of `threads` threads that a launch may have along x: HIP refuses gridDim.x blockDim.x >= 2^32.
inline int64_t max_workgroups(int threads) { return (((int64_t)1 << 32) - 1) / threads; }

// f(first, count) for `items` cut into launches of `each` workgroups an item
template <typename F>
void for_launches(int64_t items, int64_t each, int threads, F&& f) {
  const int64_t per = std::max<int64_t>(1, max_workgroups(threads) / each);
  for (int64_t i = 0; i < items; i += per) f(i, std::min(per, items - i));
}

}  // namespace fh
