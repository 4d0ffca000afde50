// Copies between device memory and the caller's (pageable) host arrays.
//
// A pageable copy of the runtime moves through one staging buffer on one
// thread, which also takes the page faults of a fresh destination: 256 MB take 63
// ms to a fresh array, 15 ms to one touched before and 9 ms from one, on a link
// that needs 4.7 ms to or from pinned memory.  Large copies here go
// through a ring of pinned chunks instead: the link fills (drains) the chunks
// in order while a few threads copy them to (from) the caller's array (11, 6.8
// and 6.6 ms).  Threads that wait give their time slice away but do not sleep, so
// that a process held to few CPUs by other means than its affinity mask (which
// sets their number) pays for the waiting.
// The fields of a 256^3 solver (0.75 GB) to fresh host arrays: 85 -> 30 ms.
// Memory that the link reaches itself (pinned or managed by the caller) is left
// to the runtime: 256 MB take 4.7 ms directly, 6.7 ms through the ring.
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace m2c {

// 8 x 2 MB of pinned memory: 12 x 4 MB copies 0.69 GB 2% faster but its
// allocation adds 2 ms to a first copy; 1 MB chunks are 8% slower
struct HostRing {
  static constexpr size_t CHUNK = 2u << 20;
  static constexpr int RING = 8;
  char* buf = nullptr;
  hipEvent_t ev[RING] = {};

  bool create() {
    if (hipHostMalloc(reinterpret_cast<void**>(&buf), CHUNK * RING, hipHostMallocDefault) != hipSuccess) {
      buf = nullptr;
      (void)hipGetLastError();
      return false;
    }
    for (auto& e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
    return true;
  }
  ~HostRing() {
    for (auto& e : ev)
      if (e) hipEventDestroy(e);
    if (buf) hipHostFree(buf);
  }
};

// The rings of a device's solvers: a copy takes one for its duration, so that
// any number of threads copy at once, and at most KEEP idle ones wait for the
// next; the last solver of a device gives them back.  With a ring per solver 64
// of them held 1 GB pinned, each paid for its allocation (1 ms) and, in one
// process of three, creating solvers in turn with destroying others took 1.04
// instead of 0.64 ms every other time.
class HostRings {
 public:
  static HostRings& get() {
    static HostRings* all = new HostRings;  // outlives every solver
    return *all;
  }
  void join(int device) {
    std::lock_guard<std::mutex> lk(mu_);
    dev_[device].users++;
  }
  void leave(int device) {
    std::vector<HostRing*> out;
    {
      std::lock_guard<std::mutex> lk(mu_);
      Device& d = dev_[device];
      if (--d.users == 0) out.swap(d.idle);
    }
    for (HostRing* r : out) delete r;
  }
  HostRing* take(int device) {  // null: no pinned memory to be had
    {
      std::lock_guard<std::mutex> lk(mu_);
      Device& d = dev_[device];
      if (!d.idle.empty()) {
        HostRing* r = d.idle.back();
        d.idle.pop_back();
        return r;
      }
    }
    HostRing* r = new HostRing;
    if (r->create()) return r;
    delete r;
    return nullptr;
  }
  void give(int device, HostRing* r, bool sound) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      Device& d = dev_[device];
      if (sound && d.users > 0 && d.idle.size() < KEEP) {
        d.idle.push_back(r);
        return;
      }
    }
    delete r;
  }

 private:
  static constexpr size_t KEEP = 2;
  struct Device {
    int users = 0;
    std::vector<HostRing*> idle;
  };
  std::mutex mu_;
  std::map<int, Device> dev_;
};

// A solver's copies.
class HostPipe {
 public:
  static constexpr size_t CHUNK = HostRing::CHUNK;
  static constexpr int RING = HostRing::RING;
  static constexpr int MAX_THREADS = 8;
  // Smaller copies are left to the runtime.  Measured at 8 MB, ring and runtime:
  // to a fresh array 0.8 and 1.9 ms, to one touched before 0.33 and 0.51, from
  // one 0.30 and 0.30; at 6 MB from one 0.24 and 0.23.
  static constexpr size_t LEAST = 8u << 20;

  HostPipe() = default;
  HostPipe(const HostPipe&) = delete;
  HostPipe& operator=(const HostPipe&) = delete;
  ~HostPipe() {
    if (device_ >= 0) HostRings::get().leave(device_);
  }
  // the device whose rings the solver shares
  void attach(int device) {
    HostRings::get().join(device);
    device_ = device;
  }

  // both wait for the copy (and what `st` holds before it) to end
  hipError_t to_host(void* host, const void* dev, size_t bytes, hipStream_t st) const {
    return copy(static_cast<char*>(host), const_cast<char*>(static_cast<const char*>(dev)), bytes, st, false);
  }
  hipError_t to_device(void* dev, const void* host, size_t bytes, hipStream_t st) const {
    return copy(const_cast<char*>(static_cast<const char*>(host)), static_cast<char*>(dev), bytes, st, true);
  }

 private:
  int device_ = -1;

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

  hipError_t copy(char* host, char* dev, size_t bytes, hipStream_t st, bool up) const {
    HostRing* ring = nullptr;
    if (bytes >= LEAST && device_ >= 0 && pageable(host) && pageable(host + bytes - 1))
      ring = HostRings::get().take(device_);
    if (!ring) return plain(host, dev, bytes, st, up);
    const hipError_t e = through(*ring, host, dev, bytes, st, up);
    HostRings::get().give(device_, ring, e == hipSuccess);
    return e;
  }

  hipError_t through(HostRing& ring, char* host, char* dev, size_t bytes, hipStream_t st, bool up) const {
    char* const buf = ring.buf;
    hipEvent_t* const ev = ring.ev;
    const int device = device_;
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
          if (c >= (size_t)RING && hipEventSynchronize(ev[s]) != hipSuccess) failed.store(true);
          std::memcpy(buf + s * CHUNK, host + c * CHUNK, span(c));
        } else {
          while (linked.load(std::memory_order_acquire) <= c && !failed.load()) std::this_thread::yield();
          if (failed.load()) return;
          if (hipEventSynchronize(ev[s]) != hipSuccess) failed.store(true);
          else std::memcpy(host + c * CHUNK, buf + s * CHUNK, span(c));
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
      err = up ? hipMemcpyAsync(dev + c * CHUNK, buf + s * CHUNK, span(c), hipMemcpyHostToDevice, st)
               : hipMemcpyAsync(buf + s * CHUNK, dev + c * CHUNK, span(c), hipMemcpyDeviceToHost, st);
      if (err == hipSuccess) err = hipEventRecord(ev[s], st);
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
