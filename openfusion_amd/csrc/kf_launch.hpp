// kf_launch.hpp — launches of one thread per item, at any number of items.
#pragma once

#include <stddef.h>

namespace kf {

constexpr unsigned kItemThreads = 256;  // block size
// HIP takes grids of fewer than 2^32 threads; a volume of 2048^3 FP32 voxels has 2^32
// 16-byte vectors.
constexpr size_t kMaxLaunchItems = (size_t)1 << 31;

// launch(first, count, blocks) for consecutive parts of `items`, each a launch of
// `blocks` blocks of kItemThreads.  Stops at the first result that is not 0 and returns it.
template <typename Launch>
inline auto launch_items(size_t items, const Launch& launch) -> decltype(launch(items, items, 0u)) {
  decltype(launch(items, items, 0u)) st{};
  for (size_t first = 0; first < items; first += kMaxLaunchItems) {
    const size_t left = items - first, count = left < kMaxLaunchItems ? left : kMaxLaunchItems;
    st = launch(first, count, (unsigned)((count + kItemThreads - 1) / kItemThreads));
    if (st != decltype(st){}) return st;
  }
  return st;
}

}  // namespace kf
