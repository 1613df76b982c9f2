// swm_transfer.hpp -- copies of states between the caller's arrays and the device.
//
// A copy of pageable memory goes through the runtime, one thread taking the page
// faults and moving the bytes, by way of a buffer of 16 MB per stream.  Here a few
// threads move chunks between the array and a pinned ring of 8 MB, each chunk's way
// over the bus, by a small kernel, overlapping the others' host copies.  By the
// runtime and by the ring, in us, with the layout kernel; down: into an array whose
// pages are not there yet; (new): the first transfer of a new solver, the ring's
// pinning with it:
//     bytes      down            up             down (new), after a step   up (new)
//     3.8 MB      275 / 142      176 / 159        600 / 170                 180 / 160
//     6.3 MB      426 / 200      244 / 221        980 / 210                 240 / 220
//     25 MB      1525 / 618      754 / 692       3690 / 640          820-6100 / 700-1800
//     101 MB    10283 / 3307    4031 / 2508     15700 / 2980        3900-9000 / 2500-3900
// A first transfer of 2.2 MB takes 380 by the runtime and as much by the ring, which
// has 0.3 ms of pinning then; so the ring takes pageable arrays from 3 MB on, and the
// runtime smaller ones and pinned ones (6.3 MB down 140, 101 MB 1823).
//
// The chunks go by a kernel because the runtime's copies are not even: after a new
// solver's first step some hundred of them take 0.1 ms more each than later ones
// (25 MB down by chunks of 512 KB 5.4 ms, then 1.2), and the first pass over a new
// stream's buffer takes 0.3 ms a MB wherever its pages were not used before.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace swm {

// n doubles from device memory to the pinned ring or (up) back (swm_kernels.hip).
void launch_ring_copy(const double* from, double* to, size_t n, bool up, hipStream_t s);

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

  // The device's bytes (a multiple of 8) to host, complete on return, and back,
  // ordered on the stream (the caller synchronizes before host may change).  A
  // transfer that finds the ring in use by another thread's leaves it to the runtime.
  hipError_t to_host(void* host, const void* dev, size_t bytes, hipStream_t s) {
    char* d = const_cast<char*>(static_cast<const char*>(dev));
    return transfer(d, static_cast<char*>(host), bytes, s, false);
  }
  hipError_t to_device(void* dev, const void* host, size_t bytes, hipStream_t s) {
    char* h = const_cast<char*>(static_cast<const char*>(host));
    return transfer(static_cast<char*>(dev), h, bytes, s, true);
  }

 private:
  HostRing() = default;
  static constexpr size_t kChunk = size_t(1) << 20;
  static constexpr size_t kRingFrom = 3 * kChunk;
  static constexpr int kThreads = 4;
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
      er = hipHostMalloc((void**)&ring_, kSlots * kChunk, hipHostMallocCoherent);
      if (er != hipSuccess) ring_ = nullptr;
    }
    return er;
  }

  hipError_t transfer(char* dev, char* host, size_t bytes, hipStream_t s, bool up) {
    if (bytes >= kRingFrom && pageable(host) && use_.try_lock()) {
      std::lock_guard<std::mutex> g(use_, std::adopt_lock);
      if (prepare() == hipSuccess) return copy(dev, host, bytes, s, up);
    }
    if (up) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
    const hipError_t er = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
    return er == hipSuccess ? hipStreamSynchronize(s) : er;
  }

  // Two chunks of every thread are on their way at a time; the first ones down
  // start before the threads do.  All are awaited, so the next call finds every
  // slot free.
  hipError_t copy(char* dev, char* host, size_t bytes, hipStream_t s, bool up) {
    const size_t chunks = (bytes + kChunk - 1) / kChunk;
    // a thread costs about 20 us to start: one per 2 chunks
    const int nt = (int)std::min<size_t>(kThreads, (chunks + 1) / 2);
    hipError_t err[kThreads] = {};
    for (size_t c = 0; !up && c < std::min<size_t>(chunks, 2 * nt) && err[0] == hipSuccess; ++c)
      err[0] = start(dev, bytes, c, nt, s, false);
    if (err[0] == hipSuccess) {
      auto work = [&](int w) {
        if (w > 0) (void)hipSetDevice(device_);
        err[w] = up ? part_up(dev, host, bytes, chunks, nt, w, s)
                    : part_down(dev, host, bytes, chunks, nt, w, s);
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
    // on the way up the last kernels may still run, out of the ring
    return up ? hipStreamSynchronize(s) : hipSuccess;
  }

  static size_t length(size_t bytes, size_t c) { return std::min(kChunk, bytes - c * kChunk); }

  // Chunk c is thread c % nt's, by turns in its two slots.
  static int slot(size_t c, int nt) { return 2 * (int)(c % nt) + (int)(c / nt % 2); }

  hipError_t start(char* dev, size_t bytes, size_t c, int nt, hipStream_t s, bool up) {
    const int i = slot(c, nt);
    double* d = reinterpret_cast<double*>(dev + c * kChunk);
    double* r = reinterpret_cast<double*>(ring_ + i * kChunk);
    launch_ring_copy(up ? r : d, up ? d : r, length(bytes, c) / sizeof(double), up, s);
    const hipError_t er = hipGetLastError();
    return er == hipSuccess ? hipEventRecord(done_[i], s) : er;
  }

  hipError_t part_down(char* dev, char* host, size_t bytes, size_t chunks, int nt, int w,
                       hipStream_t s) {
    hipError_t er = hipSuccess;
    for (size_t c = w; c < chunks && er == hipSuccess; c += nt) {
      const int i = slot(c, nt);
      er = hipEventSynchronize(done_[i]);
      if (er != hipSuccess) break;
      std::memcpy(host + c * kChunk, ring_ + i * kChunk, length(bytes, c));
      if (c + 2 * nt < chunks) er = start(dev, bytes, c + 2 * nt, nt, s, false);
    }
    return er;
  }

  hipError_t part_up(char* dev, const char* host, size_t bytes, size_t chunks, int nt, int w,
                     hipStream_t s) {
    hipError_t er = hipSuccess;
    for (size_t c = w; c < chunks && er == hipSuccess; c += nt) {
      const int i = slot(c, nt);
      if (c >= (size_t)(2 * nt)) er = hipEventSynchronize(done_[i]);
      if (er != hipSuccess) break;
      std::memcpy(ring_ + i * kChunk, host + c * kChunk, length(bytes, c));
      er = start(dev, bytes, c, nt, s, true);
    }
    return er;
  }

  std::mutex use_;
  int device_ = 0;
  char* ring_ = nullptr;
  hipEvent_t done_[kSlots] = {};
};

}  // namespace swm
