// The few runtime calls m2c_hostcopy.h makes, for its test without a GPU: one
// thread stands for the copy engine and carries out the copies of a stream in
// order; memory is "pinned" where hipHostMalloc or pin() made it so.  Copies
// are logged, and any call can be made to fail.
#pragma once
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
struct hipPointerAttribute_t { hipMemoryType type; };
struct FakeEvent { size_t at = 0; };
typedef FakeEvent* hipEvent_t;
typedef int hipStream_t;

struct FakeHip {
  struct Copy { void* dst; const void* src; size_t n; };
  std::mutex mu;
  std::condition_variable cv;
  std::deque<Copy> todo;
  std::vector<Copy> log;
  size_t given = 0, done = 0;
  size_t allocated = 0;  // calls of hipHostMalloc
  bool stop = false, no_pinned = false, unregistered_is_error = false;
  long fail_copy = -1;  // the copy with this number is refused
  std::map<const char*, size_t> pinned;
  std::thread engine;
  FakeHip() : engine([this] { run(); }) {}
  ~FakeHip() {
    { std::lock_guard<std::mutex> l(mu); stop = true; }
    cv.notify_all();
    engine.join();
  }
  void run() {
    std::unique_lock<std::mutex> l(mu);
    for (;;) {
      cv.wait(l, [this] { return stop || !todo.empty(); });
      if (todo.empty()) return;
      Copy c = todo.front();
      todo.pop_front();
      l.unlock();
      std::memcpy(c.dst, c.src, c.n);
      l.lock();
      done++;
      cv.notify_all();
    }
  }
  void pin(const void* p, size_t n) {
    std::lock_guard<std::mutex> l(mu);
    pinned[static_cast<const char*>(p)] = n;
  }
  bool is_pinned(const void* p) {
    std::lock_guard<std::mutex> l(mu);
    auto it = pinned.upper_bound(static_cast<const char*>(p));
    if (it == pinned.begin()) return false;
    --it;
    return static_cast<const char*>(p) < it->first + it->second;
  }
  void wait(size_t upto) {
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [&] { return done >= upto; });
  }
};
inline FakeHip& fake() { static FakeHip f; return f; }

inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (fake().no_pinned) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  { std::lock_guard<std::mutex> l(fake().mu); fake().allocated++; }
  fake().pin(*p, n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  { std::lock_guard<std::mutex> l(fake().mu); fake().pinned.erase(static_cast<char*>(p)); }
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new FakeEvent; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> l(fake().mu);
  e->at = fake().given;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  size_t at;
  { std::lock_guard<std::mutex> l(fake().mu); at = e->at; }
  fake().wait(at);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
  size_t g;
  { std::lock_guard<std::mutex> l(fake().mu); g = fake().given; }
  fake().wait(g);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  FakeHip& f = fake();
  std::lock_guard<std::mutex> l(f.mu);
  if ((long)f.log.size() == f.fail_copy) { f.fail_copy = -1; return hipErrorUnknown; }
  f.log.push_back({d, s, n});
  f.todo.push_back({d, s, n});
  f.given++;
  f.cv.notify_all();
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  const bool host = fake().is_pinned(p);
  a->type = host ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return !host && fake().unregistered_is_error ? hipErrorInvalidValue : hipSuccess;
}
