// Host threads of the planners.
#pragma once

#include <algorithm>
#include <atomic>
#include <thread>
#include <vector>

namespace tfqx {

inline int HostThreads() {
  unsigned n = std::thread::hardware_concurrency();
  return int(std::max(1u, std::min(n, 16u)));  // one GPU's share of host cores
}

template <typename F>
void ParallelFor(int n, F f) {
  const int T = std::min(HostThreads(), n);
  if (T <= 1) {
    for (int i = 0; i < n; ++i) f(i);
    return;
  }
  std::atomic<int> next(0);
  std::vector<std::thread> pool;
  for (int t = 0; t < T; ++t)
    pool.emplace_back([&]() {
      while (true) {
        int i = next.fetch_add(1);
        if (i >= n) break;
        f(i);
      }
    });
  for (auto& th : pool) th.join();
}

}  // namespace tfqx
