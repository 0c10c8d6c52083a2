// kept_pool.h -- one idle buffer per device, kept between calls for the static
// queries' workspace (capi.cpp) and given up whenever memory is short.  Shared
// with the host-side test harness, which runs it over a memory of its own.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <mutex>

namespace c2a {

constexpr size_t kKeepBytes = (size_t)512 << 20;   // the largest buffer kept
constexpr int kKeepDevices = 64;

// M::alloc(void**, size_t) allocates on the current device (0 = done) and
// M::free(void*) frees.
template <class M>
class KeptPool {
  struct Buf {
    void* p;
    size_t bytes;
  };
  std::mutex mu_;
  Buf kept_[kKeepDevices] = {};
  int64_t holders_ = 0;

  static bool dev_ok(int dev) { return dev >= 0 && dev < kKeepDevices; }

  Buf take_out(int dev) {
    std::lock_guard<std::mutex> lock(mu_);
    const Buf k = kept_[dev];
    kept_[dev] = {};
    return k;
  }

 public:
  // Frees every kept buffer; whether there was one.
  bool drop() {
    bool any = false;
    for (int d = 0; d < kKeepDevices; d++)
      if (void* p = take_out(d).p) {
        M::free(p);
        any = true;
      }
    return any;
  }

  // Nothing is kept without a holder.
  void hold() {
    std::lock_guard<std::mutex> lock(mu_);
    holders_++;
  }
  void release() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (--holders_ > 0) return;
    }
    drop();
  }

  // Bytes kept on a device: free memory to a caller that allocates here.
  size_t kept(int dev) {
    std::lock_guard<std::mutex> lock(mu_);
    return dev_ok(dev) && kept_[dev].p ? kept_[dev].bytes : 0;
  }

  // An allocation of any other use: it gets the kept memory when it does not
  // fit beside it.
  int alloc(void** p, size_t n) {
    const int rc = M::alloc(p, n);
    return rc && drop() ? M::alloc(p, n) : rc;
  }

  // A buffer of at least n bytes of the current device, `dev`.  A kept one that
  // is too small goes first: the two never stand side by side.
  int take(int dev, size_t n, void** p, size_t* bytes) {
    if (dev_ok(dev)) {
      const Buf k = take_out(dev);
      if (k.p && k.bytes >= n) {
        *p = k.p;
        *bytes = k.bytes;
        return 0;
      }
      if (k.p) M::free(k.p);
    }
    *bytes = n;
    return alloc(p, n);
  }

  // Hands a buffer of take() back; idle: no work that uses it is in flight.
  void give(int dev, void* p, size_t bytes, bool idle) {
    if (idle && bytes <= kKeepBytes && dev_ok(dev)) {
      std::lock_guard<std::mutex> lock(mu_);
      Buf& k = kept_[dev];
      if (holders_ > 0 && (!k.p || k.bytes < bytes)) {
        void* old = k.p;
        k = {p, bytes};
        p = old;
      }
    }
    if (p) M::free(p);
  }
};

}  // namespace c2a
