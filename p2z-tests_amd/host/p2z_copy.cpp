#include "p2z_copy.hpp"

#include <emmintrin.h>
#include <sched.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <system_error>

namespace p2z {
namespace {

constexpr int kMaxHelpers = 15;
constexpr size_t kPieceBytes = 256 << 10;
constexpr int kSpins = 4000;  // about 100 us: the next chunk of the same call

int processors() {
  cpu_set_t set;
  if (sched_getaffinity(0, sizeof set, &set) == 0) return CPU_COUNT(&set);
  return (int)std::thread::hardware_concurrency();
}

void copy_row(char* dst, const char* src, size_t bytes) {
  size_t i = 0;
  for (; i + 64 <= bytes; i += 64) {
    const auto* s = reinterpret_cast<const __m128i*>(src + i);
    auto* d = reinterpret_cast<__m128i*>(dst + i);
    const __m128i a = _mm_loadu_si128(s), b = _mm_loadu_si128(s + 1), c = _mm_loadu_si128(s + 2),
                  e = _mm_loadu_si128(s + 3);
    _mm_stream_si128(d, a);
    _mm_stream_si128(d + 1, b);
    _mm_stream_si128(d + 2, c);
    _mm_stream_si128(d + 3, e);
  }
  if (i < bytes) std::memcpy(dst + i, src + i, bytes - i);
}

}  // namespace

CopyPool::CopyPool() {
  const int n = std::min(kMaxHelpers, processors() - 1);
  // no exception leaves the constructor: it would destroy running threads
  try {
    if (n > 0) helpers_.reserve(n);
    for (int i = 0; i < n; ++i) helpers_.emplace_back([this] { helper(); });
  } catch (const std::system_error&) {
    // no more threads to be had: the caller and those there are do the work
  } catch (const std::bad_alloc&) {  // or no memory for one
  }
}

CopyPool::~CopyPool() {
  {
    std::lock_guard<std::mutex> lock(mu_);
    stop_.store(true);
  }
  cv_.notify_all();
  for (auto& t : helpers_) t.join();
}

void CopyPool::helper() {
  uint64_t seen = 0;
  for (;;) {
    for (int i = 0; i < kSpins && posted_.load(std::memory_order_acquire) == seen && !stop_.load(); ++i) _mm_pause();
    {
      std::unique_lock<std::mutex> lock(mu_);
      cv_.wait(lock, [&] { return stop_.load() || posted_.load() != seen; });
      if (stop_.load()) return;
      seen = posted_.load();
    }
    work();
  }
}

// Takes pieces of the current job until none is left to take.
void CopyPool::work() {
  for (;;) {
    Job j;
    size_t piece;
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (next_ >= pieces_) return;
      piece = next_++;
      j = job_;
    }
    const size_t r1 = std::min(j.rows, (piece + 1) * j.grain);
    const bool stream = ((uintptr_t)j.dst | j.dst_pitch) % 16 == 0;
    for (size_t r = piece * j.grain; r < r1; ++r) {
      char* d = j.dst + r * j.dst_pitch;
      const char* s = j.src + r * j.src_pitch;
      if (stream)
        copy_row(d, s, j.row_bytes);
      else
        std::memcpy(d, s, j.row_bytes);
    }
    _mm_sfence();
    left_.fetch_sub(1, std::memory_order_release);
  }
}

void CopyPool::rows(void* dst, size_t dst_pitch, const void* src, size_t src_pitch, size_t row_bytes, size_t rows) {
  if (rows == 0 || row_bytes == 0) return;
  const size_t grain = std::max<size_t>(1, kPieceBytes / row_bytes);
  const size_t pieces = (rows + grain - 1) / grain;
  {
    // the previous job is done (left_ is 0): no thread is between taking a
    // piece and copying it
    std::lock_guard<std::mutex> lock(mu_);
    job_ = Job{static_cast<char*>(dst), static_cast<const char*>(src), dst_pitch, src_pitch, row_bytes, rows, grain};
    next_ = 0;
    pieces_ = pieces;
    left_.store(pieces);
    if (pieces > 1) posted_.fetch_add(1);
  }
  if (pieces > 1) cv_.notify_all();
  work();
  while (left_.load(std::memory_order_acquire) != 0) _mm_pause();
}

}  // namespace p2z
