// Copies between device memory and the caller's (pageable) host arrays.
//
// A pageable copy of the runtime moves through one staging buffer on one
// thread, which also takes the page faults of a fresh destination: 256 MB take 63
// ms to a fresh array, 15 ms to one touched before and 9 ms from one, on a link
// that needs 4.7 ms to or from pinned memory.  Large copies here go
// through a ring of pinned chunks instead: the link fills (drains) the chunks
// in order while a few threads copy them to (from) the caller's array (11, 6.8
// and 6.6 ms).  The ring, 16 MB of pinned memory, belongs to one solver and is
// allocated at its first large copy; threads that wait give their time slice
// away but do not sleep, so that a process held to few CPUs by other means than
// its affinity mask (which sets their number) pays for the waiting.
// The fields of a 256^3 solver (0.75 GB) to fresh host arrays: 85 -> 30 ms.
// Memory that the link reaches itself (pinned or managed by the caller) is left
// to the runtime: 256 MB take 4.7 ms directly, 6.7 ms through the ring.
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace m2c {

class HostPipe {
 public:
  // 8 x 2 MB: 12 x 4 MB copies 0.69 GB 2% faster but its allocation adds 2 ms
  // to a solver's first copy; 1 MB chunks are 8% slower
  static constexpr size_t CHUNK = 2u << 20;
  static constexpr int RING = 8;
  static constexpr int MAX_THREADS = 8;
  // Smaller copies are left to the runtime.  Measured at 8 MB, ring and runtime:
  // to a fresh array 0.8 and 1.9 ms, to one touched before 0.33 and 0.51, from
  // one 0.30 and 0.30; at 6 MB from one 0.24 and 0.23.
  static constexpr size_t LEAST = 8u << 20;

  HostPipe() = default;
  HostPipe(const HostPipe&) = delete;
  HostPipe& operator=(const HostPipe&) = delete;
  ~HostPipe() { release(); }

  void release() {
    for (auto& e : ev_)
      if (e) hipEventDestroy(e);
    if (buf_) hipHostFree(buf_);
    for (auto& e : ev_) e = nullptr;
    buf_ = nullptr;
  }

  // both wait for the copy (and what `st` holds before it) to end
  hipError_t to_host(int device, void* host, const void* dev, size_t bytes, hipStream_t st) {
    return run(device, static_cast<char*>(host), const_cast<char*>(static_cast<const char*>(dev)), bytes, st, false);
  }
  hipError_t to_device(int device, void* dev, const void* host, size_t bytes, hipStream_t st) {
    return run(device, const_cast<char*>(static_cast<const char*>(host)), static_cast<char*>(dev), bytes, st, true);
  }

 private:
  char* buf_ = nullptr;
  hipEvent_t ev_[RING] = {};

  bool ready() {
    if (buf_) return true;
    if (hipHostMalloc(reinterpret_cast<void**>(&buf_), CHUNK * RING, hipHostMallocDefault) != hipSuccess) {
      buf_ = nullptr;
      (void)hipGetLastError();
      return false;
    }
    for (auto& e : ev_)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        release();
        return false;
      }
    return true;
  }

  static int thread_count(size_t chunks) {
    cpu_set_t set;
    CPU_ZERO(&set);
    const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    return (int)std::min<size_t>(chunks, (size_t)std::max(1, std::min(cpus, MAX_THREADS)));
  }

  // memory the runtime knows nothing of, which the link cannot reach itself
  static bool pageable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {  // how older runtimes say so
      (void)hipGetLastError();
      return true;
    }
    return a.type == hipMemoryTypeUnregistered;
  }

  static hipError_t plain(char* host, char* dev, size_t bytes, hipStream_t st, bool up) {
    hipError_t e = up ? hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st)
                      : hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipStreamSynchronize(st);
  }

  hipError_t run(int device, char* host, char* dev, size_t bytes, hipStream_t st, bool up) {
    if (bytes < LEAST || !pageable(host) || !pageable(host + bytes - 1) || !ready())
      return plain(host, dev, bytes, st, up);
    const size_t n = (bytes + CHUNK - 1) / CHUNK;
    // `host_done` counts per ring slot the chunks its threads have finished
    // with; `linked` is the number of chunks given to the link (to_host)
    std::atomic<size_t> next{0}, linked{0};
    std::atomic<size_t> host_done[RING];
    for (auto& d : host_done) d.store(0);
    std::atomic<bool> failed{false};
    auto span = [&](size_t c) { return std::min(CHUNK, bytes - c * CHUNK); };
    auto worker = [&]() {
      (void)hipSetDevice(device);
      for (size_t c; (c = next.fetch_add(1)) < n;) {
        const int s = (int)(c % RING);
        if (up) {
          // the slot is free once the link has taken the chunk before it
          while (linked.load(std::memory_order_acquire) + RING <= c && !failed.load()) std::this_thread::yield();
          if (failed.load()) return;
          if (c >= (size_t)RING && hipEventSynchronize(ev_[s]) != hipSuccess) failed.store(true);
          std::memcpy(buf_ + s * CHUNK, host + c * CHUNK, span(c));
        } else {
          while (linked.load(std::memory_order_acquire) <= c && !failed.load()) std::this_thread::yield();
          if (failed.load()) return;
          if (hipEventSynchronize(ev_[s]) != hipSuccess) failed.store(true);
          else std::memcpy(host + c * CHUNK, buf_ + s * CHUNK, span(c));
        }
        host_done[s].store(c / RING + 1, std::memory_order_release);
      }
    };
    std::vector<std::thread> pool;
    try {
      const int t = thread_count(n);
      pool.reserve(t);
      for (int q = 0; q < t; q++) pool.emplace_back(worker);
    } catch (...) {  // no (more) threads to be had: the ones there are do it
    }
    if (pool.empty()) return plain(host, dev, bytes, st, up);
    hipError_t err = hipSuccess;
    for (size_t c = 0; c < n && err == hipSuccess && !failed.load(); c++) {
      const int s = (int)(c % RING);
      const size_t need = up ? c / RING + 1 : c / RING;
      while (host_done[s].load(std::memory_order_acquire) < need && !failed.load()) std::this_thread::yield();
      if (failed.load()) break;
      err = up ? hipMemcpyAsync(dev + c * CHUNK, buf_ + s * CHUNK, span(c), hipMemcpyHostToDevice, st)
               : hipMemcpyAsync(buf_ + s * CHUNK, dev + c * CHUNK, span(c), hipMemcpyDeviceToHost, st);
      if (err == hipSuccess) err = hipEventRecord(ev_[s], st);
      if (err == hipSuccess) linked.store(c + 1, std::memory_order_release);
    }
    if (err != hipSuccess) failed.store(true);
    for (auto& t : pool) t.join();
    if (err == hipSuccess && failed.load()) err = hipErrorUnknown;
    const hipError_t e = hipStreamSynchronize(st);
    return err != hipSuccess ? err : e;
  }
};

}  // namespace m2c
