// Independent host work over the host's threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace octlb {

// body(k) for k in [0, count), spread over the host's threads (at most 16);
// what a body throws is thrown here.
template <typename F>
void ParallelFor(int count, F&& body) {
  constexpr int kChunk = 16;
  const int want = std::min({16, static_cast<int>(std::thread::hardware_concurrency()), count / kChunk});
  std::atomic<int> next{0};
  std::exception_ptr failed;
  std::mutex failed_mu;
  auto run = [&] {
    try {
      for (int k0; (k0 = next.fetch_add(kChunk)) < count;)
        for (int k = k0; k < std::min(k0 + kChunk, count); ++k) body(k);
    } catch (...) {
      std::lock_guard<std::mutex> lock(failed_mu);
      if (!failed) failed = std::current_exception();
      next = count;
    }
  };
  std::vector<std::thread> threads;
  try {
    threads.reserve(want > 1 ? want - 1 : 0);
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
