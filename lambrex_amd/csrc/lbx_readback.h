// lbx_readback.h -- copies of device memory into ordinary host memory.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

struct lbx_ctx;

namespace lbx {

// hipMemcpyAsync into pageable memory is one thread's copy out of the
// runtime's own staging (10 GB/s into fresh memory, 17 GB/s into touched
// memory; the link moves 57 GB/s).  Here the link fills a ring of pinned
// chunks and a few threads empty it: 512 MB of fresh memory 50.5 -> 11.8 ms,
// 64 MB 6.4 -> 1.8 ms, 16 MB 1.6 -> 0.6 ms.
class ReadBack {
 public:
  // The ring from 2 MB on: below, the threads' start costs what they bring.  Us
  // into memory already touched, directly and so: 2.2 MB 142 and 120, 3.5 MB 219
  // and 194, 4.5 MB 282 and 235, 6.9 MB 405 and 289, 8.4 MB 481 and 317; 1 MB
  // would lose 30.
  static constexpr size_t kFrom = (size_t)2 << 20;
  struct Part {
    void* dst;
    const void* src;
    size_t bytes;
  };
  // Copies parts[0 .. n) behind the work on `st` (of `device`, the current
  // one) and returns when they have arrived.
  hipError_t copy(int device, const Part* parts, int n, hipStream_t st);
  // Frees the ring; the next copy that wants it allocates it again.
  void release();

 private:
  static constexpr int kSlots = 8;
  static constexpr size_t kRing = (size_t)32 << 20;
  bool ready();
  std::mutex mutex_;  // one copy at a time
  char* ring_ = nullptr;
  hipEvent_t arrived_[kSlots] = {};
};

// A context's (lbx_abi.cpp).
ReadBack& ctx_readback(lbx_ctx* ctx);

}  // namespace lbx
