// spark_workers.hpp -- helper threads of one call (host code).
#pragma once
#include <exception>
#include <thread>
#include <vector>

namespace spark {

// work(0) on the calling thread beside work(1) .. work(n - 1) on threads of
// their own; returns when all are done.  Where a thread cannot be started (no
// thread or no memory for one) the rest are left out, so the work has to be
// shared by whoever runs.  work itself must not throw.
template <class Work> void run_workers(int n, const Work& work) {
  std::vector<std::thread> threads;
  try {
    threads.reserve(n > 1 ? n - 1 : 0);
    for (int w = 1; w < n; w++) threads.emplace_back([work, w]() { work(w); });
  } catch (const std::exception&) {
  }
  work(0);
  for (auto& t : threads) t.join();
}

}  // namespace spark
