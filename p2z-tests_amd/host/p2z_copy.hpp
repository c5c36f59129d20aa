// Copies between host buffers by several threads, for the staging of pageable
// buffers (plain C++, no HIP).
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <thread>
#include <vector>

namespace p2z {

// One thread copies about 10 GB/s, the link to the GPU takes 57.  The helpers
// belong to the pool's owner and sleep while nothing is copied; a copy is cut
// into pieces that the caller and whichever helpers are awake take in turn, so
// that it ends with its last piece and not with the slowest thread's start (a
// parallel region that waits for all of its threads took 6 ms instead of 1.4
// where the processors were also held by another library's spinning threads).
// Used by one thread at a time.
class CopyPool {
 public:
  CopyPool();   // as many helpers as there are other processors, at most 15
  ~CopyPool();
  CopyPool(const CopyPool&) = delete;
  CopyPool& operator=(const CopyPool&) = delete;

  // Copies rows of row_bytes, dst_pitch and src_pitch bytes apart; stores
  // bypass the caches where dst is aligned to 16 bytes.  Returns when done.
  void rows(void* dst, size_t dst_pitch, const void* src, size_t src_pitch, size_t row_bytes, size_t rows);

 private:
  struct Job {
    char* dst;
    const char* src;
    size_t dst_pitch, src_pitch, row_bytes, rows, grain;  // grain: rows per piece
  };
  void helper();
  void work();

  std::mutex mu_;
  std::condition_variable cv_;
  Job job_{};                          // under mu_, as are the two below
  size_t next_ = 0, pieces_ = 0;       // pieces handed out, pieces of the job
  std::atomic<size_t> left_{0};        // pieces not yet copied
  std::atomic<uint64_t> posted_{0};    // jobs so far
  std::atomic<bool> stop_{false};
  std::vector<std::thread> helpers_;
};

}  // namespace p2z
