// workers.hpp -- one call's work on a few host threads
#pragma once
#include <exception>
#include <thread>

namespace e2d {

// work(0) .. work(n - 1), n <= MAX, side by side: 0 on the caller's thread, each other
// on a thread of its own, which has ended when this returns.  The shares for which no
// thread can be started (std::system_error: too many; std::bad_alloc: no memory for its
// start) are the caller's too: an exception that passed threads still running would
// end the process.  `work` must not throw.
template <int MAX, class F>
void run_workers(int n, F &&work) {
  std::thread helpers[MAX];
  int started = 1;
  try {
    for (; started < n; ++started) helpers[started] = std::thread([&work, t = started] { work(t); });
  } catch (const std::exception &) {
  }
  work(0);
  for (int t = started; t < n; ++t) work(t);
  for (std::thread &h : helpers)
    if (h.joinable()) h.join();
}

}  // namespace e2d
