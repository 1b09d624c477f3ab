// evp1d_par.hpp - host threads for the planner.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <exception>
#include <thread>
#include <vector>

namespace evp1d {

// Host threads for the planner and its check: the machine's, at most 16.
inline int plan_threads() {
  const unsigned hw = std::thread::hardware_concurrency();
  return (int)std::max(1u, std::min(hw ? hw : 1u, 16u));
}

// Run body(w) for w = 0..T-1, on T-1 new threads and the caller; when a
// thread cannot be started (a process thread limit) its share runs on the
// caller, so the work is always done.  An exception thrown by a share (a
// host allocation failure) is caught on its thread and the first one is
// rethrown on the caller after every thread has joined; the C entry points
// turn it into a status code (no_throw).
template <class B>
void run_workers(int T, B body) {
  std::vector<std::exception_ptr> err((size_t)T);
  auto guarded = [&body, &err](int w) {
    try {
      body(w);
    } catch (...) {
      err[(size_t)w] = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  std::vector<int> left;
  try {
    th.reserve((size_t)T);
    left.reserve((size_t)T);
  } catch (...) {
    for (int w = 0; w < T; ++w) guarded(w);   // no room for the bookkeeping: all on the caller
    for (const auto &e : err)
      if (e) std::rethrow_exception(e);
    return;
  }
  for (int w = 1; w < T; ++w) {
    try {
      th.emplace_back([&guarded, w] { guarded(w); });
    } catch (...) {
      left.push_back(w);
    }
  }
  guarded(0);
  for (int w : left) guarded(w);
  for (auto &t : th) t.join();
  for (const auto &e : err)
    if (e) std::rethrow_exception(e);
}

// f(lo, hi, w) over [0, n) in contiguous chunks, one per worker w, in order.
template <class F>
void par_chunks(int64_t n, int64_t grain, F f) {
  const int T = (int)std::max<int64_t>(1, std::min<int64_t>(plan_threads(), n / std::max<int64_t>(grain, 1)));
  if (T <= 1) {
    f((int64_t)0, n, 0);
    return;
  }
  run_workers(T, [&](int w) { f(n * w / T, n * (w + 1) / T, w); });
}

// f(i, w) for every i in [0, n), items handed out dynamically (uneven work);
// work: the points of them all (fewer than 1024 a thread take less time than
// its start: a first run's planning of 64x48 0.5 ms in place of 0.6
// to 1.0)
template <class F>
void par_items(int n, int64_t work, F f) {
  const int T = (int)std::max<int64_t>(1, std::min<int64_t>(std::min(plan_threads(), n / 4), work / 1024));
  if (T <= 1) {
    for (int i = 0; i < n; ++i) f(i, 0);
    return;
  }
  std::atomic<int> next{0};
  run_workers(T, [&](int w) {
    for (int i = next.fetch_add(8); i < n; i = next.fetch_add(8))
      for (int j = i; j < std::min(n, i + 8); ++j) f(j, w);
  });
}

}  // namespace evp1d
