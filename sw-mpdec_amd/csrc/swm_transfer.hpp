// swm_transfer.hpp -- copies of states from the device to the caller's arrays.
//
// A copy to pageable memory goes through the runtime, one thread taking the page
// faults and moving the bytes.  Here a few threads move chunks between the array
// and a pinned ring, each chunk's transfer overlapping the others' host copies.
// Downloads by the runtime and by the ring, in us, with the layout kernel (fresh:
// into an array whose pages are not there yet):
//     bytes      fresh          used before    pinned
//     0.39 MB     39 / 45         38 / 45        29 / 45
//     0.96 MB    203 / 196        64 / 71        40 / 71
//     1.6 MB     365 / 278       106 / 99        51 / 104
//     6.3 MB     949 / 462       368 / 337      140 / 364
//     101 MB    9503 / 4610     5803 / 4570    1823 / 4679
// so the ring takes pageable arrays from 1.5 MB on, and the runtime pinned ones,
// smaller ones and all uploads (fresh arrays of 0.39 MB 34 / 37, 1.6 MB 94 / 116,
// 101 MB 3536 / 4798).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace swm {

class HostRing {
 public:
  // The ring of a device, shared by its engines (pinning its 8 MB takes longer
  // than most transfers) and given back with the last of them.
  static std::shared_ptr<HostRing> of_device(int device) {
    static std::mutex lock;
    static std::vector<std::weak_ptr<HostRing>> rings;
    std::lock_guard<std::mutex> g(lock);
    if (device < 0) return nullptr;
    if ((size_t)device >= rings.size()) rings.resize(device + 1);
    std::shared_ptr<HostRing> r = rings[device].lock();
    if (!r) {
      r.reset(new HostRing());
      r->device_ = device;
      rings[device] = r;
    }
    return r;
  }
  HostRing(const HostRing&) = delete;
  HostRing& operator=(const HostRing&) = delete;
  ~HostRing() {
    for (hipEvent_t e : done_)
      if (e) (void)hipEventDestroy(e);
    if (ring_) (void)hipHostFree(ring_);
  }

  // The device's bytes to host, complete on return.  A transfer that finds the
  // ring in use by another thread's leaves it to the runtime.
  hipError_t to_host(void* host, const void* dev, size_t bytes, hipStream_t s) {
    if (bytes >= kRingFrom && pageable(host) && use_.try_lock()) {
      std::lock_guard<std::mutex> g(use_, std::adopt_lock);
      if (prepare() == hipSuccess)
        return copy(static_cast<const char*>(dev), static_cast<char*>(host), bytes, s);
    }
    const hipError_t er = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
    return er == hipSuccess ? hipStreamSynchronize(s) : er;
  }

 private:
  HostRing() = default;
  static constexpr size_t kChunk = size_t(1) << 19;
  static constexpr size_t kRingFrom = 3 * kChunk;
  static constexpr int kThreads = 8;
  static constexpr int kSlots = 2 * kThreads;  // two per thread: one moves while one is copied

  // Memory the runtime does not know.
  static bool pageable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
  }

  hipError_t prepare() {
    hipError_t er = hipSuccess;
    for (int i = 0; i < kSlots && er == hipSuccess; ++i)
      if (!done_[i]) er = hipEventCreateWithFlags(&done_[i], hipEventDisableTiming);
    if (er == hipSuccess && !ring_) {
      er = hipHostMalloc((void**)&ring_, kSlots * kChunk, hipHostMallocDefault);
      if (er != hipSuccess) ring_ = nullptr;
    }
    return er;
  }

  // Two chunks of every thread are on their way at a time.  The first ones start
  // before the threads do.  All are awaited, so the next call finds every slot free.
  hipError_t copy(const char* dev, char* host, size_t bytes, hipStream_t s) {
    const size_t chunks = (bytes + kChunk - 1) / kChunk;
    // a thread costs about 20 us to start: one per 2 chunks
    const int nt = (int)std::min<size_t>(kThreads, (chunks + 1) / 2);
    hipError_t err[kThreads] = {};
    for (size_t c = 0; c < std::min<size_t>(chunks, 2 * nt) && err[0] == hipSuccess; ++c)
      err[0] = start(dev, bytes, c, nt, s);
    if (err[0] == hipSuccess) {
      auto work = [&](int w) {
        if (w > 0) (void)hipSetDevice(device_);
        err[w] = part(dev, host, bytes, chunks, nt, w, s);
      };
      std::thread threads[kThreads];
      for (int w = 1; w < nt; ++w) {
        try {
          threads[w] = std::thread(work, w);
        } catch (...) {  // no thread to be had: this one does its part
          work(w);
        }
      }
      work(0);
      for (int w = 1; w < nt; ++w)
        if (threads[w].joinable()) threads[w].join();
    }
    for (hipError_t e : err)
      if (e != hipSuccess) {
        (void)hipStreamSynchronize(s);
        return e;
      }
    return hipSuccess;
  }

  static size_t length(size_t bytes, size_t c) { return std::min(kChunk, bytes - c * kChunk); }

  // Chunk c is thread c % nt's, by turns in its two slots.
  static int slot(size_t c, int nt) { return 2 * (int)(c % nt) + (int)(c / nt % 2); }

  hipError_t start(const char* dev, size_t bytes, size_t c, int nt, hipStream_t s) {
    const int i = slot(c, nt);
    const hipError_t er = hipMemcpyAsync(ring_ + i * kChunk, dev + c * kChunk, length(bytes, c),
                                         hipMemcpyDeviceToHost, s);
    return er == hipSuccess ? hipEventRecord(done_[i], s) : er;
  }

  hipError_t part(const char* dev, char* host, size_t bytes, size_t chunks, int nt, int w,
                  hipStream_t s) {
    hipError_t er = hipSuccess;
    for (size_t c = w; c < chunks && er == hipSuccess; c += nt) {
      const int i = slot(c, nt);
      er = hipEventSynchronize(done_[i]);
      if (er != hipSuccess) break;
      std::memcpy(host + c * kChunk, ring_ + i * kChunk, length(bytes, c));
      if (c + 2 * nt < chunks) er = start(dev, bytes, c + 2 * nt, nt, s);
    }
    return er;
  }

  std::mutex use_;
  int device_ = 0;
  char* ring_ = nullptr;
  hipEvent_t done_[kSlots] = {};
};

}  // namespace swm
