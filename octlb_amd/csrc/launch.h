// Long runs of workgroups as several launches.
#pragma once

#include <algorithm>
#include <cstdint>

namespace octlb {

// One launch holds fewer than 2^32 threads: a grid beyond that wraps to a
// smaller one without an error and leaves the rest of its work undone.
constexpr int64_t kMaxLaunchThreads = (int64_t{1} << 32) - 1;

// launch(first, count) for consecutive ranges that cover workgroups [0, groups)
// of `threads` threads each.
template <typename F>
void ForLaunches(int64_t groups, int threads, F&& launch) {
  const int64_t most = kMaxLaunchThreads / threads;
  for (int64_t first = 0; first < groups; first += most) launch(first, std::min(most, groups - first));
}

}  // namespace octlb
