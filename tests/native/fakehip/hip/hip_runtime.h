// A HIP runtime of two devices in host memory, for tests of host code: an event
// belongs to the device that was current when it was made and can be recorded
// on that device's streams only, as in the real one.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };

namespace fakehip {
inline thread_local int current = 0;
inline std::atomic<int> copies{0}, bytes_max{0}, live_events{0}, live_pinned{0};
inline std::atomic<int> records_left{1 << 30};  // records that succeed
inline std::atomic<bool> no_pinned{false};
struct Object {
  int device;
};
}  // namespace fakehip
using hipStream_t = fakehip::Object *;
using hipEvent_t = fakehip::Object *;

inline hipError_t hipGetDevice(int *d) {
  *d = fakehip::current;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  if (d < 0 || d > 1) return hipErrorInvalidDevice;
  fakehip::current = d;
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (fakehip::no_pinned) return hipErrorOutOfMemory;
  fakehip::live_pinned++;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  fakehip::live_pinned--;
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  fakehip::live_events++;
  *e = new fakehip::Object{fakehip::current};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  fakehip::live_events--;
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return e->device == s->device && fakehip::records_left-- > 0 ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  fakehip::copies++;
  if ((int)n > fakehip::bytes_max) fakehip::bytes_max = (int)n;
  std::memcpy(d, s, n);
  return hipSuccess;
}
