// Host threads that help with a copy.
#pragma once

#include <thread>

namespace ufx {

// Starts `n` threads of f into th; how many there are, fewer where one cannot
// be had.  A thread's start fails with std::system_error or, finding no memory
// for its state, std::bad_alloc; neither may leave a function that has threads
// running (nor a C entry).
template <typename F>
int start_threads(std::thread* th, int n, const F& f) noexcept {
  int k = 0;
  try {
    for (; k < n; ++k) th[k] = std::thread(f);
  } catch (...) {
  }
  return k;
}

}  // namespace ufx
