// operator new that fails on request: linked into a build of csrc/q4host.cpp whose own allocations take it (-Bsymbolic).
#include <cstdlib>
#include <new>

static long allowed = -1;   // allocations that succeed before one fails; negative: all

extern "C" __attribute__((visibility("default"))) void fail_after(long n) { allowed = n; }

void *operator new(std::size_t size) {
  if (allowed == 0) {
    allowed = -1;
    throw std::bad_alloc();
  }
  if (allowed > 0) --allowed;
  void *p = std::malloc(size ? size : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }
