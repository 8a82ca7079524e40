// Device-to-host reads through pinned memory.
//
// A copy to pageable memory goes through the runtime's own staging on one host
// thread: 16 GB/s here, and 30 us for the smallest.  Here chunks cross into
// pinned slots (a kernel's stores or a copy, whatever the caller enqueues) while
// host threads move earlier ones to the caller's array, widening FP32 on the
// way, so half the bytes cross the bus.  Measured, six 384^3 FP32 fields (1.4 GB
// to 2.7 GB): 165 -> 31 ms.
//
// The slots are shared by every context of the process: up to kSets reads at a
// time, each with slots of its own, made for the first read that finds none free,
// grown to the largest read (at most 32 MB) and freed with the last context.
// Reads of several contexts at once, us each over all of 1 / 4 / 8 threads, FP64:
// pageable copies 64^3 215 / 125 / 105, 100^3 560 / 310 / 280; one read at a time
// with eight host threads 164 / 145 / 154 and 376 / 365 / 381; four with eight 165 /
// 115 / 117 and 375 / 288 / 283; four with four, as here, 152 / 97 / 90 and 320 / 203
// / 183.  Two host threads are faster still into memory in use (64^3 135 / 65 / 57)
// but not into fresh memory, whose pages they touch first (300^3 FP32 50 ms against
// 30; pageable 59).
#pragma once

#include <emmintrin.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
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
  static constexpr size_t kThreads = 4;
  static constexpr size_t kSets = 4;

  // One per context: the slots live while any does.
  struct User {
    User() {
      std::lock_guard<std::mutex> lock(pool().mu);
      ++pool().users;
    }
    ~User() {
      std::lock_guard<std::mutex> lock(pool().mu);
      if (--pool().users > 0) return;
      for (Set& set : pool().sets) set.release();
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
    check(hipStreamSynchronize(stream));  // what came before, without holding slots
    const size_t most = kSlotBytes / item;
    const size_t per = std::min(most, std::max(kMinItems, (items + kSlots - 1) / kSlots));
    const size_t chunks = (items + per - 1) / per;
    const size_t pitch = (per * item + 255) / 256 * 256;
    const Lease slots(std::min(chunks, kSlots) * pitch, check);
    auto slot = [&](size_t c) { return slots.base() + (c % kSlots) * pitch; };
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
  // The slots of one read.
  struct Set {
    unsigned char* p = nullptr;
    size_t bytes = 0;
    bool busy = false;
    void release() {
      if (p) (void)hipHostFree(p);
      p = nullptr;
      bytes = 0;
    }
  };
  struct Pool {
    std::mutex mu;
    std::condition_variable freed;
    int users = 0;
    Set sets[kSets];
  };
  static Pool& pool() {
    static Pool& p = *new Pool;  // outlives contexts that live until the process ends
    return p;
  }

  // A set for the time of a read: a free one that is large enough, else the
  // largest free one, grown, so that reads one after the other share a set.
  class Lease {
   public:
    template <class Check>
    Lease(size_t need, Check check) {
      size_t bytes = size_t(64) << 10;
      while (bytes < need) bytes *= 2;
      Pool& P = pool();
      {
        std::unique_lock<std::mutex> lock(P.mu);
        auto pick = [&]() -> Set* {
          Set* best = nullptr;
          for (Set& s : P.sets)
            if (!s.busy && (!best || (best->bytes < bytes ? s.bytes > best->bytes
                                                          : s.bytes >= bytes && s.bytes < best->bytes)))
              best = &s;
          return best;
        };
        P.freed.wait(lock, [&] { return (set_ = pick()) != nullptr; });
        set_->busy = true;
      }
      if (set_->bytes >= bytes) return;
      try {
        set_->release();
        void* p = nullptr;
        check(hipHostMalloc(&p, bytes, hipHostMallocPortable));
        set_->p = static_cast<unsigned char*>(p);
        set_->bytes = bytes;
      } catch (...) {
        giveBack();
        throw;
      }
    }
    ~Lease() { giveBack(); }
    Lease(const Lease&) = delete;
    Lease& operator=(const Lease&) = delete;
    unsigned char* base() const { return set_->p; }

   private:
    void giveBack() {
      {
        std::lock_guard<std::mutex> lock(pool().mu);
        set_->busy = false;
      }
      pool().freed.notify_one();
    }
    Set* set_ = nullptr;
  };
};

}  // namespace xfd
