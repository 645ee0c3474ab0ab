// start_threads where the memory for a thread's state runs out: no exception
// leaves it, and the threads that started finish.
#include "helper_threads.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <system_error>

static std::atomic<int> allocations_left{-1};  // -1: any number

void* operator new(std::size_t n) {
  if (allocations_left.load() == 0) throw std::bad_alloc();
  if (allocations_left.load() > 0) --allocations_left;
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
  for (int want = 0; want <= 7; ++want) {
    std::thread th[7];
    std::atomic<int> ran{0};
    auto f = [&] { ++ran; };
    allocations_left = want;
    const int got = ufx::start_threads(th, 7, f);
    allocations_left = -1;
    for (int i = 0; i < got; ++i) th[i].join();
    if (got != want || ran != want) {
      std::printf("%d threads of %d, %d ran\n", got, want, ran.load());
      return 1;
    }
  }
  std::puts("ok");
}
