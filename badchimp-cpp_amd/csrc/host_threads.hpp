// Host loops of the set-up split over threads: node-list passes that read
// shared input and write disjoint output ranges.
#pragma once
#include <algorithm>
#include <cstdint>
#include <exception>
#include <thread>
#include <utility>
#include <vector>

namespace lbamd {

// Threads a host pass may use: the host's cores, at most kMaxHostThreads (the
// host share of one GPU on the machines this runs on).
constexpr int kMaxHostThreads = 16;

inline int host_threads() {
  const unsigned hw = std::thread::hardware_concurrency();
  return std::max(1, std::min(kMaxHostThreads, static_cast<int>(hw ? hw : 1)));
}

// Starts f on a thread of its own in the pool; false where the system has none
// to give (a process or container limit), which the callers, C entry points
// among them, take as having fewer threads.
template <class F>
bool start_thread(std::vector<std::thread>& pool, F&& f) {
  try {
    pool.emplace_back(std::forward<F>(f));
  } catch (const std::exception&) {
    return false;
  }
  return true;
}

// f(begin, end, t) over contiguous chunks of [0, n), chunk t on thread t
// (t < host_threads()) or on the caller's, at least min_items each: a thread
// costs about 25 us, an item of a light pass (some loads and stores) a
// nanosecond or less.  f must not throw.
template <class F>
void parallel_ranges(int64_t n, F&& f, int64_t min_items = int64_t{1} << 16) {
  const int T = static_cast<int>(std::min<int64_t>(host_threads(), std::max<int64_t>(1, n / min_items)));
  if (T <= 1) {
    f(int64_t{0}, n, 0);
    return;
  }
  const int64_t chunk = (n + T - 1) / T;
  auto run = [&f, n, chunk](int t) {
    const int64_t b = std::min(n, t * chunk);
    f(b, std::min(n, b + chunk), t);
  };
  std::vector<std::thread> pool;
  pool.reserve(T - 1);
  int next = 1;
  while (next < T && start_thread(pool, [&run, next] { run(next); })) ++next;
  run(0);
  for (; next < T; ++next) run(next);
  for (auto& th : pool) th.join();
}

}  // namespace lbamd
