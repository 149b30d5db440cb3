// run_workers with the allocation of the k-th thread's start refused, k = 1 .. n:
// every share runs exactly once and no exception leaves.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>

#include "workers.hpp"

static std::atomic<int> countdown{-1};  // allocations until one is refused (-1: none is)

void *operator new(std::size_t n) {
  if (countdown.load() >= 0 && countdown.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main() {
  constexpr int kMax = 4;
  for (int n = 1; n <= kMax; ++n)
    for (int refused = -1; refused < n; ++refused) {
      std::atomic<int> ran[kMax] = {};
      countdown = refused;
      e2d::run_workers<kMax>(n, [&](int t) { ran[t].fetch_add(1); });
      countdown = -1;
      for (int t = 0; t < kMax; ++t)
        if (ran[t] != (t < n ? 1 : 0)) {
          std::printf("n %d refused %d: share %d ran %d times\n", n, refused, t, ran[t].load());
          return 1;
        }
    }
  std::printf("every share ran once\n");
  return 0;
}
