// swm_transfer.hpp -- copies between the caller's pageable arrays and the
// device for the boundary's large arrays.
//
// A copy from or to pageable memory goes through the runtime: into fresh pages
// it brought 1 MB down in 0.62 ms, 25 MB in 6.0 and 100 MB in 23.9 ms, one
// thread taking the page faults and moving the bytes.  Here a few threads move
// chunks between the array and a pinned ring, each chunk's transfer overlapping
// the others' host copies: 0.24, 1.6 and 5 ms.  Upwards
// the runtime pins larger arrays in place at 27 GB/s, as fast as the ring;
// below that it takes 0.37 ms for 1 MB and 0.72 for 2, the ring 0.06 and 0.10.
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

  // host[0..bytes) to the device, ordered on the stream (the caller
  // synchronizes before host may change), and back, complete on return.  A
  // transfer that finds the ring in use by another thread's leaves it to the
  // runtime.
  hipError_t to_device(void* dev, const void* host, size_t bytes, hipStream_t s) {
    if (bytes <= kRingUp && use_.try_lock()) {
      std::lock_guard<std::mutex> g(use_, std::adopt_lock);
      if (prepare() == hipSuccess)
        return copy(static_cast<char*>(dev), const_cast<char*>(static_cast<const char*>(host)),
                    bytes, s, true);
    }
    return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
  }
  hipError_t to_host(void* host, const void* dev, size_t bytes, hipStream_t s) {
    if (use_.try_lock()) {
      std::lock_guard<std::mutex> g(use_, std::adopt_lock);
      if (prepare() == hipSuccess)
        return copy(const_cast<char*>(static_cast<const char*>(dev)), static_cast<char*>(host),
                    bytes, s, false);
    }
    const hipError_t er = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
    return er == hipSuccess ? hipStreamSynchronize(s) : er;
  }

 private:
  HostRing() = default;
  static constexpr size_t kChunk = size_t(1) << 19;
  static constexpr size_t kRingUp = size_t(4) << 20;
  static constexpr int kThreads = 8;
  static constexpr int kSlots = 2 * kThreads;  // two per thread: one moves while one is copied

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

  // Slot i once its last transfer, of this call or an earlier one, is done.
  hipError_t slot(int i, char*& p) {
    p = ring_ + (size_t)i * kChunk;
    return hipEventSynchronize(done_[i]);
  }

  hipError_t copy(char* dev, char* host, size_t bytes, hipStream_t s, bool up) {
    if (bytes == 0) return hipSuccess;
    const size_t chunks = (bytes + kChunk - 1) / kChunk;
    // a thread costs about 20 us to start: one per 2 chunks
    const int nt = (int)std::min<size_t>(kThreads, (chunks + 1) / 2);
    std::vector<hipError_t> err(nt, hipSuccess);
    auto work = [&](int w) {
      if (w > 0) (void)hipSetDevice(device_);
      err[w] = up ? up_part(dev, host, bytes, chunks, nt, w, s)
                  : down_part(dev, host, bytes, chunks, nt, w, s);
    };
    std::vector<std::thread> threads;
    for (int w = 1; w < nt; ++w) {
      try {
        threads.emplace_back(work, w);
      } catch (...) {  // no thread to be had: this one does its part
        work(w);
      }
    }
    work(0);
    for (std::thread& t : threads) t.join();
    for (hipError_t e : err)
      if (e != hipSuccess) return e;
    return hipSuccess;
  }

  static size_t length(size_t bytes, size_t c) { return std::min(kChunk, bytes - c * kChunk); }

  hipError_t up_part(char* dev, const char* host, size_t bytes, size_t chunks, int nt, int w,
                     hipStream_t s) {
    int turn = 0;
    for (size_t c = w; c < chunks; c += nt, turn ^= 1) {
      char* p;
      hipError_t er = slot(2 * w + turn, p);
      if (er != hipSuccess) return er;
      std::memcpy(p, host + c * kChunk, length(bytes, c));
      er = hipMemcpyAsync(dev + c * kChunk, p, length(bytes, c), hipMemcpyHostToDevice, s);
      if (er == hipSuccess) er = hipEventRecord(done_[2 * w + turn], s);
      if (er != hipSuccess) return er;
    }
    return hipSuccess;
  }

  hipError_t down_part(const char* dev, char* host, size_t bytes, size_t chunks, int nt, int w,
                       hipStream_t s) {
    auto start = [&](size_t c, int turn) {
      char* p;
      hipError_t er = slot(2 * w + turn, p);
      if (er == hipSuccess)
        er = hipMemcpyAsync(p, dev + c * kChunk, length(bytes, c), hipMemcpyDeviceToHost, s);
      return er == hipSuccess ? hipEventRecord(done_[2 * w + turn], s) : er;
    };
    int turn = 0;
    hipError_t er = (size_t)w < chunks ? start(w, 0) : hipSuccess;
    for (size_t c = w; c < chunks && er == hipSuccess; c += nt, turn ^= 1) {
      if (c + nt < chunks) er = start(c + nt, turn ^ 1);
      if (er != hipSuccess) break;
      er = hipEventSynchronize(done_[2 * w + turn]);
      if (er == hipSuccess)
        std::memcpy(host + c * kChunk, ring_ + (size_t)(2 * w + turn) * kChunk, length(bytes, c));
    }
    return er;
  }

  std::mutex use_;
  int device_ = 0;
  char* ring_ = nullptr;
  hipEvent_t done_[kSlots] = {};
};

}  // namespace swm
