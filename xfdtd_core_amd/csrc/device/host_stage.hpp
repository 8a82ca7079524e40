// Device-to-host reads through pinned memory.
//
// A copy to pageable memory goes through the runtime's own staging on one host
// thread: 16 GB/s here, and 30 us for the smallest.  Here chunks cross into
// pinned slots (a kernel's stores or a copy, whatever the caller enqueues) while
// host threads move earlier ones to the caller's array, widening FP32 on the
// way, so half the bytes cross the bus.  Measured, six 384^3 FP32 fields (1.4 GB
// to 2.7 GB): 165 -> 31 ms.
//
// The slots are shared by every context of the process, one read at a time, and
// freed with the last context.
#pragma once

#include <emmintrin.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace xfd {

class HostStage {
 public:
  static constexpr size_t kSlotBytes = size_t(2) << 20;
  static constexpr size_t kSlots = 16;
  static constexpr size_t kMinItems = size_t(64) << 10;  // per chunk, where a read is split
  static constexpr size_t kThreads = 8;

  // One per context: the slots live while any does.
  struct User {
    User() {
      std::lock_guard<std::mutex> lock(mu());
      ++users();
    }
    ~User() {
      std::lock_guard<std::mutex> lock(mu());
      if (--users() == 0 && base()) {
        (void)hipHostFree(base());
        base() = nullptr;
      }
    }
    User(const User&) = delete;
    User& operator=(const User&) = delete;
  };

  // Reads `items` of `item` bytes: enqueue(first, count, slot) puts items on
  // `stream` for the slot, take(first, count, slot) moves them on (host threads,
  // any order).  `check` throws on a HIP error.  Returns with everything taken.
  template <class Check, class Enqueue, class Take>
  static void read(hipStream_t stream, size_t items, size_t item, Check check, Enqueue enqueue, Take take) {
    if (items == 0) return;
    check(hipStreamSynchronize(stream));  // what came before, without holding the slots
    std::lock_guard<std::mutex> lock(mu());
    if (!base()) {
      void* p = nullptr;
      check(hipHostMalloc(&p, kSlotBytes * kSlots, hipHostMallocPortable));
      base() = static_cast<unsigned char*>(p);
    }
    const size_t most = kSlotBytes / item;
    const size_t per = std::min(most, std::max(kMinItems, (items + kSlots - 1) / kSlots));
    const size_t chunks = (items + per - 1) / per;
    auto slot = [&](size_t c) { return base() + (c % kSlots) * kSlotBytes; };
    auto count = [&](size_t c) { return std::min(per, items - c * per); };
    if (chunks == 1) {
      enqueue(size_t(0), items, slot(0));
      check(hipStreamSynchronize(stream));
      take(size_t(0), items, slot(0));
      return;
    }
    // This thread makes every HIP call; the others wait for `ready` chunks.
    std::vector<hipEvent_t> done(std::min(chunks, kSlots), nullptr);
    std::vector<std::atomic<size_t>> taken(kSlots);  // chunks taken from each slot
    for (auto& t : taken) t = 0;
    std::atomic<size_t> ready{0}, next{0};
    std::atomic<bool> stop{false};
    auto work = [&] {
      for (;;) {
        const size_t c = next.fetch_add(1);
        if (c >= chunks) return;
        while (ready.load(std::memory_order_acquire) <= c) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        take(c * per, count(c), slot(c));
        taken[c % kSlots].fetch_add(1, std::memory_order_release);
      }
    };
    std::vector<std::thread> threads;
    std::exception_ptr failure;
    try {
      for (auto& e : done) check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      const size_t n = std::min(kThreads, chunks);
      for (size_t w = 0; w < n; ++w) threads.emplace_back(work);
      size_t sent = 0;
      for (size_t c = 0; c < chunks; ++c) {
        for (; sent < chunks && sent < c + kSlots; ++sent) {
          if (taken[sent % kSlots].load(std::memory_order_acquire) < sent / kSlots) {
            if (sent > c) break;  // still being taken, and earlier chunks are on their way
            while (taken[sent % kSlots].load(std::memory_order_acquire) < sent / kSlots) std::this_thread::yield();
          }
          enqueue(sent * per, count(sent), slot(sent));
          check(hipEventRecord(done[sent % kSlots], stream));
        }
        check(hipEventSynchronize(done[c % kSlots]));
        ready.store(c + 1, std::memory_order_release);
      }
    } catch (...) {
      failure = std::current_exception();
      stop = true;
    }
    for (auto& t : threads) t.join();
    for (auto& e : done)
      if (e) (void)hipEventDestroy(e);
    if (failure) {
      (void)hipStreamSynchronize(stream);
      std::rethrow_exception(failure);
    }
  }

  // Moves n values to dst as doubles; past the caches, which a large read would
  // only sweep.
  template <class T>
  static void widen(const T* src, double* dst, size_t n) {
    size_t q = 0;
    if (n >= 4096) {
      for (; q < n && reinterpret_cast<uintptr_t>(dst + q) % 16; ++q) dst[q] = static_cast<double>(src[q]);
      for (; q + 2 <= n; q += 2) _mm_stream_pd(dst + q, pairAt(src + q));
      _mm_sfence();
    }
    for (; q < n; ++q) dst[q] = static_cast<double>(src[q]);
  }

 private:
  static __m128d pairAt(const double* p) { return _mm_loadu_pd(p); }
  static __m128d pairAt(const float* p) { return _mm_set_pd(static_cast<double>(p[1]), static_cast<double>(p[0])); }
  static std::mutex& mu() {
    static std::mutex m;
    return m;
  }
  static int& users() {
    static int n = 0;
    return n;
  }
  static unsigned char*& base() {
    static unsigned char* p = nullptr;
    return p;
  }
};

}  // namespace xfd
