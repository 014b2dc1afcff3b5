// Host loops over several threads.
#ifndef APCOST_PARALLEL_H
#define APCOST_PARALLEL_H

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace apc_internal {

// ------------------------------------------------------------------------------------------
// Work over [0, n) on up to `threads` threads, in chunks handed out as they are finished.  A thread
// costs about 20 us to start and join: callers ask for one thread per megabyte of work or so.
// ------------------------------------------------------------------------------------------
constexpr int kMaxThreads = 8;

template <typename F>
void in_parallel(int64_t n, int threads, F &&body) {
  threads = std::max(1, std::min<int>(threads, kMaxThreads));
  if (threads == 1 || n < 2) {
    body((int64_t)0, n);
    return;
  }
  const int64_t chunk = std::max<int64_t>(1, n / (threads * 8));
  std::atomic<int64_t> next{0};
  std::mutex first;
  std::exception_ptr error;  // (of any thread: thrown again in the caller, once all have ended)
  auto work = [&] {
    try {
      for (;;) {
        const int64_t b = next.fetch_add(chunk, std::memory_order_relaxed);
        if (b >= n) return;
        body(b, std::min(n, b + chunk));
      }
    } catch (...) {
      next.store(n, std::memory_order_relaxed);
      std::lock_guard<std::mutex> lock(first);
      if (!error) error = std::current_exception();
    }
  };
  std::vector<std::thread> team;
  try {
    for (int i = 1; i < threads; ++i) team.emplace_back(work);
  } catch (...) {  // (no thread to be had: the ones that started, and this one, do it)
  }
  work();
  for (auto &t : team) t.join();
  if (error) std::rethrow_exception(error);
}

inline int threads_for(int64_t bytes) { return (int)std::min<int64_t>(kMaxThreads, 1 + (bytes >> 20)); }

}  // namespace apc_internal

#endif
