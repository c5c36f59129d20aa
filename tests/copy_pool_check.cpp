// CopyPool (p2z-tests_amd/host/p2z_copy.cpp) whose construction runs out of
// memory: allocation i of the constructor fails, for every i it makes.  Built
// and run by tests/test_copy_pool.py.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "p2z_copy.hpp"

static std::atomic<long> g_left{-1};  // allocations until the one that fails; below 0: none fails

void* operator new(std::size_t n) {
  if (g_left.load() >= 0 && g_left.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
  // rows of 600 of 900 bytes into a packed buffer, several pieces of work
  const size_t rows = 5000, in = 900, out = 600;
  std::vector<char> src(rows * in), dst(rows * out);
  for (size_t i = 0; i < src.size(); ++i) src[i] = (char)(i * 31 + i / in);
  for (long fail = 0;; ++fail) {
    dst.assign(dst.size(), 0);
    g_left.store(fail);
    p2z::CopyPool pool;
    const bool failed = g_left.exchange(-1) < 0;
    pool.rows(dst.data(), out, src.data(), in, out, rows);
    for (size_t r = 0; r < rows; ++r)
      for (size_t c = 0; c < out; ++c)
        if (dst[r * out + c] != src[r * in + c]) return 2;
    if (!failed) {
      std::printf("%ld allocations\n", fail);
      return 0;
    }
  }
}
