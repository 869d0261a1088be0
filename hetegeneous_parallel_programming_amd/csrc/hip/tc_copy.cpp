// Large copies from the device to pageable host memory.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <thread>

#include "tc_internal.hpp"

namespace tcr {

hipError_t Stager::ring() {
  if (mem) return hipSuccess;
  hipError_t e = hipHostMalloc((void**)&mem, kBufs * kChunk, hipHostMallocDefault);
  for (int i = 0; i < kBufs && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
  if (e != hipSuccess) release();
  return e;
}

void Stager::release() {
  for (hipEvent_t& x : ev) {
    if (x) (void)hipEventDestroy(x);
    x = nullptr;
  }
  if (mem) (void)hipHostFree(mem);
  mem = nullptr;
}

hipError_t Stager::to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes < kLeast) return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  if (ring() != hipSuccess) {
    (void)hipGetLastError();
    return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  }
  const int64_t n = (int64_t)((bytes + kChunk - 1) / kChunk);
  // Chunk c passes through buffer c mod kBufs.  open: chunks that have arrived
  // in theirs; done[c]: slices of chunk c that the threads have copied out.
  std::atomic<int64_t> next{0}, open{0};
  std::atomic<bool> stop{false};
  std::unique_ptr<std::atomic<int>[]> done(new std::atomic<int>[(size_t)n]);
  for (int64_t c = 0; c < n; ++c) done[(size_t)c].store(0, std::memory_order_relaxed);
  auto work = [&]() {
    for (;;) {
      const int64_t t = next.fetch_add(1, std::memory_order_relaxed), c = t / kSlices;
      if (c >= n) return;
      while (open.load(std::memory_order_acquire) <= c) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      const size_t slice = kChunk / kSlices, a = (size_t)(t % kSlices) * slice, at = (size_t)c * kChunk + a;
      if (at < bytes) {
        std::memcpy((char*)dst + at, mem + (size_t)(c % kBufs) * kChunk + a, std::min(slice, bytes - at));
      }
      done[(size_t)c].fetch_add(1, std::memory_order_release);
    }
  };
  std::vector<std::thread> threads;
  try {
    threads.reserve(kThreads);
    for (int i = 0; i < kThreads; ++i) threads.emplace_back(work);
  } catch (...) {  // fewer threads than asked for
  }
  if (threads.empty()) return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  hipError_t e = hipSuccess;
  auto start = [&](int64_t c) {
    const size_t at = (size_t)c * kChunk;
    if (e == hipSuccess)
      e = hipMemcpyAsync(mem + (size_t)(c % kBufs) * kChunk, (const char*)src + at, std::min(kChunk, bytes - at),
                         hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(ev[c % kBufs], s);
  };
  for (int64_t c = 0; c < std::min<int64_t>(kBufs, n); ++c) start(c);
  for (int64_t c = 0; c < n && e == hipSuccess; ++c) {
    e = hipEventSynchronize(ev[c % kBufs]);
    if (e != hipSuccess) break;
    open.store(c + 1, std::memory_order_release);
    if (c > 0 && c - 1 + kBufs < n) {  // the buffer before this one takes its next chunk
      while (done[(size_t)c - 1].load(std::memory_order_acquire) < kSlices) std::this_thread::yield();
      start(c - 1 + kBufs);
    }
  }
  if (e != hipSuccess) stop.store(true);
  for (std::thread& t : threads) t.join();
  const hipError_t e2 = hipStreamSynchronize(s);  // the ring is free again
  return e != hipSuccess ? e : e2;
}

}  // namespace tcr
