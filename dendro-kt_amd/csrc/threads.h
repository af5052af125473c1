// Host threads of plan construction.
#pragma once
#include <algorithm>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace dkt {

// Threads worth starting on this host, at most 16.
inline int host_threads() { return (int)std::clamp(std::thread::hardware_concurrency(), 1u, 16u); }

// Runs work() on up to n threads, the caller's among them; work takes its share from
// what all of them see.  Where the system grants fewer threads, those do it all.
// The first exception of a thread is thrown here once all have ended.
template <typename F>
void on_threads(int n, F &&work) {
  std::exception_ptr err;
  std::mutex mu;
  auto body = [&]() {
    try {
      work();
    } catch (...) {
      std::lock_guard<std::mutex> g(mu);
      if (!err) err = std::current_exception();
    }
  };
  std::vector<std::thread> pool;
  try {
    pool.reserve((size_t)std::max(0, n - 1));
    for (int i = 1; i < n; i++) pool.emplace_back(body);
  } catch (...) {  // no more threads
  }
  body();
  for (auto &th : pool) th.join();
  if (err) std::rethrow_exception(err);
}

}  // namespace dkt
