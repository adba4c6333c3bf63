// Independent host work over the host's threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace octlb {

// Threads that ParallelFor takes for `count` bodies, this one among them: one for
// every `each` bodies beyond the first, at most 16.
inline int ParallelThreads(int count, int each) {
  return std::max(1, std::min({16, static_cast<int>(std::thread::hardware_concurrency()), 1 + (count - 1) / each}));
}

// body(k) for k in [0, count), spread over the host's threads; what a body throws
// is thrown here.  `each`: bodies that are worth a thread, which takes about 25 us
// to start.
template <typename F>
void ParallelFor(int count, int each, F&& body) {
  const int want = ParallelThreads(count, each);
  const int chunk = std::max(1, std::min(16, count / (8 * want)));
  std::atomic<int> next{0};
  std::exception_ptr failed;
  std::mutex failed_mu;
  auto run = [&] {
    try {
      for (int k0; (k0 = next.fetch_add(chunk)) < count;)
        for (int k = k0; k < std::min(k0 + chunk, count); ++k) body(k);
    } catch (...) {
      std::lock_guard<std::mutex> lock(failed_mu);
      if (!failed) failed = std::current_exception();
      next = count;
    }
  };
  std::vector<std::thread> threads;
  try {
    threads.reserve(want - 1);
    while (static_cast<int>(threads.size()) + 1 < want) threads.emplace_back(run);
  } catch (...) {
    // no memory or no thread for more: those there are, and this one, do the
    // work; leaving without joining them would end the process
  }
  run();
  for (std::thread& th : threads) th.join();
  if (failed) std::rethrow_exception(failed);
}

}  // namespace octlb
