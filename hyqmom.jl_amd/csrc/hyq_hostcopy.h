// Copies of large arrays between device and pageable host memory.
//
// The runtime moves pageable memory at 28 GB/s up and 18 GB/s down, and one thread faults in the
// pages of a fresh result (another 9 ms for a 242 MB state).  Pinned memory moves at 57 GB/s,
// and eight threads copy between it and pageable memory faster than that, page faults
// included.  So large copies go through a ring of pinned chunks, filled or emptied by threads
// beside the transfers.  Pinned and device pointers, small arrays, and an object's first copies
// below 24 MiB (early) are copied by the runtime as they are.  Down to fresh pages, in ms (runtime
// / ring, once it is pinned): 9 MB 0.52 / 0.46, 16 MB 0.89 / 0.66, 34 MB 3.3 / 1.15, 68 MB 6.4 /
// 1.9, 242 MB 22.6 / 5.6; up: 9 MB 0.26 / 0.36, 34 MB 1.04 / 0.97, 108 MB 3.7 / 2.6, 242 MB 8.3 / 5.4.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

namespace hyq {

class HostCopy {
 public:
  // Below these the threads' start costs what the ring saves.
  static constexpr size_t kMin = size_t(8) << 20, kMinUp = size_t(64) << 20;

  // An object for copies of up to `bytes`; its events belong to the current device.
  static HostCopy* create(size_t bytes) {
    HostCopy* h = new (std::nothrow) HostCopy();
    if (!h || bytes < kMin) return h;
    for (hipEvent_t& e : h->ev_)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        delete h;
        return nullptr;
      }
    h->max_ = bytes;
    return h;
  }
  ~HostCopy() {
    (void)hipHostFree(pin_);
    for (hipEvent_t e : ev_)
      if (e) (void)hipEventDestroy(e);
  }

  // Both return once the copy is complete.
  hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (!staged(dst, bytes, kMin) || early(bytes))
      return direct(dst, src, bytes, hipMemcpyDeviceToHost, s);
    std::lock_guard<std::mutex> lk(mu_);
    const Shape r = shape_of(bytes);
    const size_t chunk = r.chunk;
    Team t(static_cast<long>((bytes + chunk - 1) / chunk), r.slots);
    if (!pin() || !t.start([&](long k) {  // ready: its chunk has arrived
          std::memcpy((char*)dst + k * chunk, slot(k, r), std::min(chunk, bytes - k * chunk));
        }))
      return direct(dst, src, bytes, hipMemcpyDeviceToHost, s);
    long issued = 0;
    for (long k = 0; k < t.n; ++k) {
      // every transfer whose slot is empty, chunk k's in any case
      for (; issued < t.n && issued < k + r.slots; ++issued) {
        if (issued >= r.slots && !t.is_done(issued - r.slots)) {
          if (issued > k) break;
          t.wait_done(issued - r.slots);
        }
        const hipError_t e = move(slot(issued, r), (const char*)src + issued * chunk,
                                  std::min(chunk, bytes - issued * chunk), hipMemcpyDeviceToHost, s, issued % r.slots);
        if (e != hipSuccess) return stop(t, s, e);
      }
      const hipError_t e = hipEventSynchronize(ev_[k % r.slots]);
      if (e != hipSuccess) return stop(t, s, e);
      t.ready.store(k + 1, std::memory_order_release);
    }
    t.join();
    return hipSuccess;
  }
  hipError_t to_device(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (!staged(src, bytes, kMinUp)) return direct(dst, src, bytes, hipMemcpyHostToDevice, s);
    std::lock_guard<std::mutex> lk(mu_);
    const Shape r = shape_of(bytes);
    const size_t chunk = r.chunk;
    Team t(static_cast<long>((bytes + chunk - 1) / chunk), r.slots);
    if (!pin() || !t.start([&](long k) {  // ready: its slot is free
          std::memcpy(slot(k, r), (const char*)src + k * chunk, std::min(chunk, bytes - k * chunk));
        }))
      return direct(dst, src, bytes, hipMemcpyHostToDevice, s);
    t.ready.store(std::min<long>(r.slots, t.n), std::memory_order_release);
    for (long k = 0; k < t.n; ++k) {
      t.wait_done(k);
      hipError_t e = move((char*)dst + k * chunk, slot(k, r), std::min(chunk, bytes - k * chunk),
                          hipMemcpyHostToDevice, s, k % r.slots);
      // a slot is free again when its transfer is done: half a ring behind the newest
      const long f = k - r.slots / 2;
      if (e == hipSuccess && f >= 0 && f + r.slots < t.n) {
        e = hipEventSynchronize(ev_[f % r.slots]);
        t.ready.store(f + r.slots + 1, std::memory_order_release);
      }
      if (e != hipSuccess) return stop(t, s, e);
    }
    t.join();
    return hipStreamSynchronize(s);
  }

 private:
  static constexpr long kSlots = 10;  // at most
  static constexpr unsigned kThreads = 8;  // 4: a fresh 242 MB takes 5.2 ms, 8: 3.5, 12: 4.4

  // Threads that take chunks 0 .. n - 1 in turn, each as soon as `ready` passes it.
  struct Team {
    Team(long n_, long slots_) : n(n_), slots(slots_) {}
    ~Team() {
      quit.store(true);
      join();
    }
    // False if no thread could be started.
    template <typename F>
    bool start(F f) {
      const unsigned want = std::min<unsigned>(kThreads, std::thread::hardware_concurrency());
      if (want < 2) return false;
      try {
        for (; size < want; ++size)
          team[size] = std::thread([this, f] {
            for (long k; (k = next.fetch_add(1)) < n;) {
              while (ready.load(std::memory_order_acquire) <= k) {
                if (quit.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
              }
              f(k);
              last[k % slots].store(k + 1, std::memory_order_release);
            }
          });
      } catch (...) {  // fewer threads
      }
      return size > 0;
    }
    bool is_done(long k) const { return last[k % slots].load(std::memory_order_acquire) > k; }
    void wait_done(long k) const {
      while (!is_done(k)) std::this_thread::yield();
    }
    void join() {
      for (unsigned i = 0; i < size; ++i) team[i].join();
      size = 0;
    }
    const long n, slots;
    std::atomic<long> next{0}, ready{0};
    std::atomic<long> last[kSlots] = {};  // the latest chunk done in each slot, plus 1
    std::atomic<bool> quit{false};
    std::thread team[kThreads];
    unsigned size = 0;
  };

  HostCopy() = default;
  // Whether the copy goes through the ring: large, and the host pointer is pageable.
  bool staged(const void* host, size_t bytes, size_t least) const {
    if (bytes < least || bytes > max_) return false;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
  }
  // Whether an object's copy down comes too early for the ring: pinning it and giving it back
  // (in part paid by the next allocation) takes 0.3 to 1.3 ms at 12 MiB, by what pages the
  // system has at hand, and a copy saves 0.05 ms at 9 MB, 0.23 at 16, 1.0 at 31 and 2.1 at 34.
  // So below 24 MiB the ring is for objects that have copied about as often as it takes to
  // make up for that: 13 times at 9 MB, 4 at 16, twice at 24.  An object that copies once
  // (create, a state up, one down, destroy), ring at once / runtime, ms: 9 MB 1.4 to 2.4 / 1.0,
  // 16 MB 2.4 to 3.5 / 1.6, 34 MB 3.7 to 5.6 / 5.4, 56 MB 5.4 / 8.5, 68 MB 5.0 to 9.6 / 9.7.
  bool early(size_t bytes) {
    if (bytes >= (size_t(24) << 20)) return false;
    const double r = double(size_t(32) << 20) / bytes;
    const int n = early_.load();
    if (n >= std::max(1, (int)(r * r + 0.5))) return false;
    early_.store(n + 1);
    return true;
  }
  bool pin() {
    if (pin_) return true;
    if (hipHostMalloc((void**)&pin_, ring_of(max_), hipHostMallocPortable) == hipSuccess) return true;
    (void)hipGetLastError();
    pin_ = nullptr;
    return false;
  }
  struct Shape {
    size_t chunk;
    long slots;
  };
  // A chunk costs the issuing thread 34 us, the transfer of 2 MB.  Smaller copies take a smaller
  // ring, whose pinning they make up for: 34 MB with 2 MiB x 6 1.17 ms a copy, x 4 1.37, x 8
  // 1.12, 1 MiB x 8 1.32, 1.5 MiB x 6 1.22; 56 MB with 2 MiB x 6 2.2, x 8 1.9; 62 MB with 2 MiB
  // x 8 0.4 ms more than with 4 MiB x 10.
  static Shape shape_of(size_t bytes) {
    if (bytes >= (size_t(56) << 20)) return {size_t(4) << 20, kSlots};
    return {size_t(2) << 20, bytes < (size_t(48) << 20) ? 6 : 8};
  }
  static size_t ring_of(size_t bytes) { return shape_of(bytes).chunk * shape_of(bytes).slots; }
  char* slot(long k, const Shape& r) const { return pin_ + (size_t)(k % r.slots) * r.chunk; }
  hipError_t move(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s, long at) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
    return e != hipSuccess ? e : hipEventRecord(ev_[at], s);
  }
  static hipError_t direct(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
    return e != hipSuccess ? e : hipStreamSynchronize(s);
  }
  // After an error: the threads end, and nothing is in flight in the ring any more.
  static hipError_t stop(Team& t, hipStream_t s, hipError_t e) {
    t.quit.store(true);
    t.join();
    (void)hipStreamSynchronize(s);
    return e;
  }

  std::mutex mu_;
  std::atomic<int> early_{0};  // copies down that the ring left to the runtime
  char* pin_ = nullptr;
  hipEvent_t ev_[kSlots] = {};
  size_t max_ = 0;  // of a large object: the largest copy, for which the ring is pinned
};

}  // namespace hyq
