// host_task.h -- host work beside the device's (capi.cpp: the hierarchy build
// and refit).  Shared with the host-side test harness.
#pragma once

#include <exception>
#include <thread>

namespace c2a {

// One task on its own thread (in place when no thread or no memory for one can
// be had: nothing is thrown), waited for on every path.  The task itself must
// not throw.
struct HostTask {
  std::thread t;
  ~HostTask() { wait(); }
  template <class F>
  void start(const F& f) {
    try {
      t = std::thread(f);
    } catch (const std::exception&) {
      f();
    }
  }
  void wait() {
    if (t.joinable()) t.join();
  }
};

}  // namespace c2a
