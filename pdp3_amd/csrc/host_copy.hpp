// Device memory to pageable host memory.
#pragma once

#include <hip/hip_runtime.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <cstring>
#include <thread>

namespace pdp3 {

// pinned buffers for copies to the host, allocated by the first that needs them
struct HostStage {
  static constexpr int kSlots = 8;
  static constexpr size_t kSlot = 512 << 10;
  void *mem = nullptr;
  hipEvent_t ev[kSlots] = {};
  bool ensure() {
    if (mem) return true;
    if (hipHostMalloc(&mem, kSlots * kSlot, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      mem = nullptr;
      return false;
    }
    for (auto &e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        e = nullptr;
        free_all();
        return false;
      }
    return true;
  }
  void free_all() {
    for (auto &e : ev) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
  }
};

// whether most of a host range's pages are in memory (mincore, some pages at a time)
inline bool resident(const void *p, size_t bytes) {
  const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
  const uintptr_t a = (uintptr_t)p & ~(page - 1), b = ((uintptr_t)p + bytes + page - 1) & ~(page - 1);
  const size_t pages = (b - a) / page;
  std::array<unsigned char, 4096> vec;
  size_t in = 0;
  for (size_t at = 0; at < pages; at += vec.size()) {
    const size_t n = std::min(vec.size(), pages - at);
    if (mincore((void *)(a + at * page), n * page, vec.data()) != 0) return true;
    for (size_t j = 0; j < n; j++) in += vec[j] & 1;
  }
  return 8 * in >= 7 * pages;
}

// a device made current for a scope
struct OnDevice {
  int device, before = -1;
  bool ok;
  explicit OnDevice(int d) : device(d) {
    ok = hipGetDevice(&before) == hipSuccess && (before == d || hipSetDevice(d) == hipSuccess);
  }
  ~OnDevice() {
    if (ok && before != device) (void)hipSetDevice(before);
  }
};

// the copy through the slots of `hs` (see copy_to_host), the stream's device current
inline hipError_t copy_staged(HostStage &hs, int device, hipStream_t stream, void *dst, const void *src,
                              size_t bytes) {
  constexpr size_t kSlot = HostStage::kSlot, kThreadsFrom = 1 << 20;
  constexpr int kThreads = 4;
  static_assert(HostStage::kSlots == 2 * kThreads, "two slots a thread");
  const size_t chunks = (bytes + kSlot - 1) / kSlot;
  const int nt = bytes >= kThreadsFrom ? kThreads : 1;
  std::array<hipError_t, kThreads> err{};
  // thread t copies chunks t, t + nt, ..: one on its way into a slot while the
  // one before is copied out of the other
  auto work = [&](int t, bool helper) {
    hipError_t e = helper ? hipSetDevice(device) : hipSuccess;
    auto issue = [&](size_t j, int s) {
      const size_t at = j * kSlot;
      if (e == hipSuccess)
        e = hipMemcpyAsync((char *)hs.mem + (2 * t + s) * kSlot, (const char *)src + at, std::min(kSlot, bytes - at),
                           hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipEventRecord(hs.ev[2 * t + s], stream);
    };
    if ((size_t)t < chunks) issue(t, 0);
    int s = 0;
    for (size_t j = t; j < chunks; j += nt, s ^= 1) {
      if (j + nt < chunks) issue(j + nt, s ^ 1);
      if (e == hipSuccess) e = hipEventSynchronize(hs.ev[2 * t + s]);
      if (e != hipSuccess) break;
      const size_t at = j * kSlot;
      std::memcpy((char *)dst + at, (char *)hs.mem + (2 * t + s) * kSlot, std::min(kSlot, bytes - at));
    }
    err[t] = e;
  };
  std::array<std::thread, kThreads> helpers;
  int started = 1;
  try {
    for (; started < nt; started++) helpers[started] = std::thread(work, started, true);
  } catch (...) {
    // fewer threads than wanted (no thread or no memory for one): this one
    // takes their shares
  }
  work(0, false);
  for (int t = 1; t < started; t++) helpers[t].join();
  for (int t = started; t < nt; t++) work(t, false);
  for (hipError_t e : err)
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(stream);  // no copy into the slots is left in flight
      return e;
    }
  return hipSuccess;
}

// Complete on return.  The runtime pins the destination for a copy like this,
// which is fast for memory in use (228 us for 4.2 MB) but takes each page fault
// of fresh memory on the way: 1083 us for a newly allocated 4.2 MB array, 8.7 ms
// for 34 MB.  Such a destination is filled from pinned buffers, by several
// threads that share its page faults (522 us, 3.9 ms).  Threads pay from 1 MiB;
// below kStageFrom the runtime's own staging is used, and throughout where
// nothing may be allocated (stage false), and where the staged copy fails.
// device: the stream's, of which the slots' events have to be (the caller's
// current device may be another)
inline hipError_t copy_to_host(HostStage &hs, int device, hipStream_t stream, void *dst, const void *src,
                               size_t bytes, bool stage) {
  constexpr size_t kStageFrom = 192 << 10;
  if (stage && bytes >= kStageFrom && !resident(dst, bytes)) {
    OnDevice on(device);
    if (on.ok && hs.ensure() && copy_staged(hs, device, stream, dst, src, bytes) == hipSuccess) return hipSuccess;
    (void)hipGetLastError();
  }
  const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
  return e == hipSuccess ? hipStreamSynchronize(stream) : e;
}

}  // namespace pdp3
