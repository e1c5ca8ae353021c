// Loops over host threads for the planning of device structures.  Host code
// only: no HIP in here.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <exception>
#include <thread>
#include <vector>

namespace psbhip {

constexpr int kHostThreads = 8;

// f(k, lo, hi) over [0, n) in up to kHostThreads ranges, one host thread each
// (one range below min_n).  Ranges whose thread cannot be created (the process
// is at its limit of threads or memory) run on the caller's.  An exception of f
// is rethrown here once all threads have ended.
template <typename F>
void host_parallel(int n, int min_n, F f) {
  const int hw = (int)std::thread::hardware_concurrency();
  const int nt = n < min_n ? 1 : std::max(1, std::min({hw, kHostThreads, n}));
  std::exception_ptr err[kHostThreads];
  auto run = [&](int k) {
    try {
      f(k, (int)((int64_t)n * k / nt), (int)((int64_t)n * (k + 1) / nt));
    } catch (...) {
      err[k] = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  th.reserve(nt);
  try {
    while ((int)th.size() < nt - 1) th.emplace_back(run, (int)th.size() + 1);
  } catch (...) {   // no more threads
  }
  run(0);
  for (int k = (int)th.size() + 1; k < nt; k++) run(k);
  for (std::thread& t : th) t.join();
  for (const std::exception_ptr& e : err)
    if (e) std::rethrow_exception(e);
}

}  // namespace psbhip
