// Checks spark::run_workers: every item of a shared queue is done once for 1
// to 8 workers, also when starting the k-th thread fails for want of memory
// (the work's copy throws std::bad_alloc): the call ends, with the threads
// that did start joined.  Prints "ok <cases>" or the first mismatch.
#include <atomic>
#include <cstdio>
#include <new>

#include "spark_workers.hpp"

struct Work {
  std::atomic<int>* next;
  std::atomic<int>* done;
  std::atomic<int>* busy;
  int* copies_left;  // copies until one fails
  Work(std::atomic<int>* n, std::atomic<int>* d, std::atomic<int>* b, int* c) : next(n), done(d), busy(b), copies_left(c) {}
  Work(const Work& o) : next(o.next), done(o.done), busy(o.busy), copies_left(o.copies_left) {
    if ((*copies_left)-- == 0) throw std::bad_alloc();
  }
  Work(Work&& o) noexcept = default;
  void operator()(int) const {
    (*busy)++;
    while (next->fetch_add(1) < 1000) (*done)++;
    (*busy)--;
  }
};

int main() {
  long cases = 0;
  for (int workers = 1; workers <= 8; workers++)
    for (int fails = 0; fails <= 8; fails++) {
      std::atomic<int> next{0}, done{0}, busy{0};
      int left = fails;
      const Work w(&next, &done, &busy, &left);
      spark::run_workers(workers, w);
      if (done != 1000 || busy != 0) {
        std::printf("%d workers, copy %d fails: %d items done, %d still busy\n", workers, fails, (int)done, (int)busy);
        return 1;
      }
      cases++;
    }
  std::printf("ok %ld\n", cases);
  return 0;
}
