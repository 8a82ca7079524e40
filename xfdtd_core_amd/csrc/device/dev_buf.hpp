// An owned device allocation, cleared when made.  `bytes` is what `p` holds, also
// after an allocation that failed: buffers that outlive a call grow by it.
//
// XFD_HIP (throws on a HIP error) and the HIP functions come from the includer.
#pragma once

#include <cstddef>

struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept : p(o.p), bytes(o.bytes) {
    o.p = nullptr;
    o.bytes = 0;
  }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) {
      reset();
      p = o.p;
      bytes = o.bytes;
      o.p = nullptr;
      o.bytes = 0;
    }
    return *this;
  }
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  void reset() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  void alloc(size_t b) {
    reset();
    if (b == 0) return;
    void* q = nullptr;
    XFD_HIP(hipMalloc(&q, b));
    p = q;
    bytes = b;
    XFD_HIP(hipMemset(p, 0, b));
  }
  template <class T>
  T* as() const {
    return static_cast<T*>(p);
  }
};
