// Runs a piece of host work on several threads, the caller's among them.
#pragma once

#include <exception>
#include <thread>
#include <vector>

namespace tpx {

// work(0) on the calling thread and work(1..threads - 1) on helpers, all ended
// on return.  Where a helper cannot be started (no more threads, no memory) the
// others do without it: `work` has to take its items from a common counter.
// `work` must not throw on a helper; what it throws on the caller is passed on
// after the helpers have ended.
template <class F>
void run_team(int threads, F &&work) {
  struct Helpers {
    std::vector<std::thread> t;
    ~Helpers() {  // also when the caller's share throws: they use its frame
      for (auto &h : t) h.join();
    }
  } helpers;
  try {
    if (threads > 1) helpers.t.reserve((size_t)threads - 1);  // a growing vector may throw with helpers running
    for (int i = 1; i < threads; ++i) helpers.t.emplace_back([&work, i] { work(i); });
  } catch (const std::exception &) {
  }
  work(0);
}

}  // namespace tpx
