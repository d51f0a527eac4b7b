// lbx_readback.cpp -- ReadBack: device memory to host memory through a ring
// of pinned chunks (see lbx_readback.h).
#include "lbx_readback.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

namespace lbx {

namespace {

// Larger chunks as the copy grows: a chunk's fixed cost (17 us) against the
// time until the first one has arrived (512 MB: 11.8 ms in 4 MB, 13.3 in 2 MB;
// 2.2 MB 178 us in 512 KB, more than directly; a served run of 60^3 with 6.9 MB
// of fields 1.29 ms in 1 MB, 1.78 in 512 KB).
size_t chunk_bytes(size_t total) {
  return total >= (size_t)64 << 20 ? (size_t)4 << 20 : total >= (size_t)8 << 20 ? (size_t)2 << 20 : (size_t)1 << 20;
}
// Copying threads, the caller included: four fill fresh memory as fast as the
// link (two reach 26 GB/s); for a few chunks more than two cost their start.
int copiers(size_t total) { return total >= (size_t)8 << 20 ? 4 : 2; }
constexpr int kMaxCopiers = 4;

// Memory that HIP knows (pinned, managed, a device's) is copied into directly.
bool ordinary(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

bool ReadBack::ready() {
  if (ring_) return true;
  bool ok = hipHostMalloc((void**)&ring_, kRing) == hipSuccess;
  if (!ok) ring_ = nullptr;
  for (int s = 0; ok && s < kSlots; ++s)
    if (!arrived_[s]) ok = hipEventCreateWithFlags(&arrived_[s], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    release();
    (void)hipGetLastError();
  }
  return ok;
}

void ReadBack::release() {
  for (hipEvent_t& e : arrived_)
    if (e) {
      (void)hipEventDestroy(e);
      e = nullptr;
    }
  if (ring_) (void)hipHostFree(ring_);
  ring_ = nullptr;
}

hipError_t ReadBack::copy(int device, const Part* parts, int n, hipStream_t st) {
  const std::lock_guard<std::mutex> lock(mutex_);
  size_t total = 0;
  bool direct = false;
  for (int p = 0; p < n; ++p) total += parts[p].bytes;
  if (total >= kFrom)
    for (int p = 0; p < n; ++p) direct |= !ordinary(parts[p].dst);
  if (total < kFrom || direct || !ready()) {
    hipError_t e = hipSuccess;
    for (int p = 0; p < n && e == hipSuccess; ++p)
      e = hipMemcpyAsync(parts[p].dst, parts[p].src, parts[p].bytes, hipMemcpyDeviceToHost, st);
    const hipError_t w = hipStreamSynchronize(st);
    return e == hipSuccess ? w : e;
  }
  // The threads below spin for their chunks: the work ahead is waited for here.
  if (const hipError_t e = hipStreamSynchronize(st)) return e;
  const size_t chunk = chunk_bytes(total);
  size_t chunks = 0;
  for (int p = 0; p < n; ++p) chunks += (parts[p].bytes + chunk - 1) / chunk;
  // chunk c: its part and its bytes there
  auto piece = [&](size_t c, size_t& at, size_t& bytes) -> const Part& {
    int p = 0;
    for (size_t k; c >= (k = (parts[p].bytes + chunk - 1) / chunk); ++p) c -= k;
    at = c * chunk;
    bytes = std::min(chunk, parts[p].bytes - at);
    return parts[p];
  };
  // Chunk c goes through slot c % kSlots; issued[slot] is 1 + the last chunk
  // sent there.  Whoever has emptied a slot sends the next chunk into it.
  std::atomic<size_t> issued[kSlots] = {}, next{0};
  std::atomic<int> error{hipSuccess};
  auto send = [&](size_t c) {
    const int s = int(c % kSlots);
    size_t at, bytes;
    const Part& p = piece(c, at, bytes);
    hipError_t e = hipMemcpyAsync(ring_ + s * chunk, (const char*)p.src + at, bytes, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(arrived_[s], st);
    if (e != hipSuccess) error = e;
    issued[s].store(c + 1, std::memory_order_release);
  };
  auto empty = [&]() {
    for (size_t c; (c = next.fetch_add(1)) < chunks;) {
      const int s = int(c % kSlots);
      while (issued[s].load(std::memory_order_acquire) != c + 1) std::this_thread::yield();
      if (error == hipSuccess) {
        const hipError_t e = hipEventSynchronize(arrived_[s]);
        if (e != hipSuccess) error = e;
      }
      size_t at, bytes;
      const Part& p = piece(c, at, bytes);
      if (error == hipSuccess) std::memcpy((char*)p.dst + at, ring_ + s * chunk, bytes);
      if (c + kSlots < chunks) send(c + kSlots);
    }
  };
  for (size_t c = 0; c < std::min(chunks, (size_t)kSlots); ++c) send(c);
  std::thread helpers[kMaxCopiers - 1];
  for (int t = 0; t < copiers(total) - 1; ++t) {
    try {
      helpers[t] = std::thread([&] {
        if (hipSetDevice(device) == hipSuccess) empty();
      });
    } catch (...) {  // no thread to be had: the others do its share
      break;
    }
  }
  empty();
  for (std::thread& t : helpers)
    if (t.joinable()) t.join();
  if (error != hipSuccess) (void)hipStreamSynchronize(st);
  return (hipError_t)error.load();
}

}  // namespace lbx
