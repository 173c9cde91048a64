// Copies of whole device fields into a caller's memory (host code only).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace ilbm {

struct HipError {
  hipError_t e;
};
#define HIPCHK(x)                                   \
  do {                                              \
    hipError_t e_ = (x);                            \
    if (e_ != hipSuccess) throw ::ilbm::HipError{e_}; \
  } while (0)

// Device-to-host copies of whole fields into a caller's ordinary memory.
// hipMemcpy stages such a copy through one buffer and one core, and the
// destination is usually fresh memory whose pages the copy touches first
// (134 MB of macros: 14 ms, 10 GB/s).  Here up to kWorkers threads each own a
// pinned buffer: a thread queues the transfer of its next slice, waits for it
// and copies it out, so that transfers run behind each other while the cores
// share the page faults and the copying: 134 MB in 3.3 ms, 537 MB 51 -> 11.8
// ms (45 GB/s).  The buffers live with the level (allocated by its first
// large copy in 2.3 ms, given back with it).  Copies below kDirect bytes
// (1.8 ms plain) are plain, and so is one that finds the buffers in use by
// another thread's copy of the same level or cannot have them (the runtime's
// last error, which the next launch check would report, is then cleared).
struct HostCopy {
  static constexpr int kWorkers = 8;
  static constexpr size_t kSlice = (size_t)4 << 20;
  static constexpr size_t kDirect = (size_t)32 << 20;
  char* pinned = nullptr;
  hipEvent_t ev[kWorkers] = {};
  std::mutex busy;   // held while the buffers are in use

  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (pinned) (void)hipHostFree(pinned);
  }

  // The device of stream s as the calling thread's, while the copy runs: its
  // events must be of the stream's device, whichever is current.
  struct OnDevice {
    int dev = 0, prev = 0;
    explicit OnDevice(hipStream_t s) {
      HIPCHK(hipGetDevice(&prev));
      HIPCHK(hipStreamGetDevice(s, &dev));
      if (dev != prev) HIPCHK(hipSetDevice(dev));
    }
    ~OnDevice() {
      if (dev != prev) (void)hipSetDevice(prev);
    }
  };

  // ordered behind the work of stream s; returns when dst is complete
  void copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
    const OnDevice on(s);
    std::unique_lock<std::mutex> lock(busy, std::defer_lock);
    if (bytes < kDirect || !lock.try_lock() || !ready()) {
      HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
      HIPCHK(hipStreamSynchronize(s));
      return;
    }
    const size_t slices = (bytes + kSlice - 1) / kSlice;
    std::atomic<size_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int w) {
      hipError_t e = hipSetDevice(on.dev);
      char* buf = pinned + (size_t)w * kSlice;
      while (e == hipSuccess) {
        const size_t i = next.fetch_add(1);
        if (i >= slices) return;
        const size_t off = i * kSlice, n = std::min(kSlice, bytes - off);
        e = hipMemcpyAsync(buf, static_cast<const char*>(src) + off, n, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev[w], s);
        if (e == hipSuccess) e = hipEventSynchronize(ev[w]);
        if (e == hipSuccess) std::memcpy(static_cast<char*>(dst) + off, buf, n);
      }
      failed = (int)e;
    };
    std::thread th[kWorkers];
    const int want = (int)std::min<size_t>(kWorkers, slices);
    for (int w = 1; w < want; ++w) {
      try {
        th[w] = std::thread(work, w);
      } catch (const std::exception&) {   // no thread, or no memory for one
        break;                             // the threads there are take every slice
      }
    }
    work(0);
    for (std::thread& t : th)
      if (t.joinable()) t.join();
    HIPCHK((hipError_t)failed.load());
  }

 private:
  bool ready() {
    if (pinned) return true;
    bool ok = true;
    for (hipEvent_t& e : ev)
      ok = ok && (e || hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess);
    void* p = nullptr;
    ok = ok && hipHostMalloc(&p, kWorkers * kSlice, hipHostMallocDefault) == hipSuccess;
    if (ok) pinned = static_cast<char*>(p);
    else (void)hipGetLastError();
    return ok;
  }
};

}  // namespace ilbm
