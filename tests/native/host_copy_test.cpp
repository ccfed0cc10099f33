// Copies of the library's host_copy.hpp on the fake runtime of fakehip/: one
// case by name, exit status 0 where it holds.
#include "host_copy.hpp"

#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <new>
#include <string>

static std::atomic<bool> g_no_threads{false}, g_no_memory{false}, g_no_memory_in_copy{false};

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
  using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
  static const Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
  return g_no_threads ? EAGAIN : real(t, a, f, arg);
}
void *operator new(size_t n) {
  void *p = g_no_memory ? nullptr : std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// one copy of `bytes` into memory that was never touched; copies: how many the
// runtime was asked for
static bool copy(pdp3::HostStage &hs, hipStream_t stream, size_t bytes, int *copies = nullptr) {
  std::string src(bytes, '\0');
  for (size_t j = 0; j < bytes; j++) src[j] = (char)(j * 2654435761u >> 13);
  void *dst = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  fakehip::copies = 0;
  g_no_memory = g_no_memory_in_copy.load();
  const hipError_t e = pdp3::copy_to_host(hs, stream->device, stream, dst, src.data(), bytes, true);
  g_no_memory = false;
  const bool same = std::memcmp(dst, src.data(), bytes) == 0;
  munmap(dst, bytes);
  if (copies) *copies = fakehip::copies;
  return e == hipSuccess && same;
}

int main(int argc, char **argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  fakehip::Object on0{0}, on1{1};
  const size_t kSizes[] = {200 << 10, 1 << 20, (5 << 20) + 12345};
  pdp3::HostStage hs;
  bool ok = true;
  int copies = 0;
  if (name == "same_device") {
    for (size_t n : kSizes) ok = ok && copy(hs, &on0, n, &copies) && copies == (int)((n + (512 << 10) - 1) / (512 << 10));
  } else if (name == "other_device_current") {
    // a context on device 1, its caller's current device is 0: staged as well,
    // and the caller's device stays
    for (size_t n : kSizes)
      ok = ok && copy(hs, &on1, n, &copies) && copies == (int)((n + (512 << 10) - 1) / (512 << 10)) && fakehip::current == 0;
    // and another current device at the next copy through the same slots
    fakehip::current = 1;
    for (size_t n : kSizes) ok = ok && copy(hs, &on1, n) && fakehip::current == 1;
  } else if (name == "record_fails") {
    for (int left : {0, 1, 3}) {
      fakehip::records_left = left;
      ok = ok && copy(hs, &on0, kSizes[2]);
    }
  } else if (name == "no_pinned_memory") {
    fakehip::no_pinned = true;
    ok = copy(hs, &on0, kSizes[2], &copies) && copies == 1;
  } else if (name == "no_threads") {
    g_no_threads = true;
    ok = copy(hs, &on0, kSizes[2]);
  } else if (name == "no_host_memory") {
    ok = copy(hs, &on0, kSizes[2]);  // the slots are there
    g_no_memory_in_copy = true;
    for (size_t n : kSizes) ok = ok && copy(hs, &on0, n);
    g_no_memory_in_copy = false;
  } else {
    std::fprintf(stderr, "no such case: %s\n", name.c_str());
    return 2;
  }
  hs.free_all();
  return ok && fakehip::live_events == 0 && fakehip::live_pinned == 0 ? 0 : 1;
}
