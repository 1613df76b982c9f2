"""Which way a transfer goes (csrc/swm_transfer.hpp), on the CPU: the header is
compiled against a stand-in for the HIP runtime that copies at once and counts
the runtime's copies from and to the caller's array.  Pinned arrays of any size
and small pageable ones go by the runtime; large pageable ones through the
pinned ring, in chunks moved by kernels and none by the runtime; each brings
every byte."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "sw-mpdec_amd" / "csrc"

STAND_IN = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1 };
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2, hipEventDisableTiming = 2,
       hipHostMallocCoherent = 1 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t { hipMemoryType type; };
typedef int* hipStream_t;
typedef int* hipEvent_t;
struct Fake { char *pinned = nullptr, *user = nullptr; size_t n = 0; bool known = true;
              std::atomic<int> straight{0}, chunks{0}; };
inline Fake fake;
inline bool in_user(const void* p) {
  return (const char*)p >= fake.user && (const char*)p < fake.user + fake.n;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  if (in_user(d) || in_user(s))
    ++fake.straight;
  else
    fake.straight += 1000;  // the runtime moves no chunks
  std::memcpy(d, s, n);
  return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = p == fake.pinned ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return fake.known || p == fake.pinned ? hipSuccess : hipErrorInvalidValue;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = new int; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { *p = std::malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
"""

PROGRAM = r"""
#include "swm_transfer.hpp"
#include <cstdio>
void swm::launch_ring_copy(const double* a, double* b, size_t n, bool, hipStream_t) {
  ++fake.chunks;
  std::memcpy(b, a, n * sizeof(double));
}
int main() {
  auto ring = swm::HostRing::of_device(0);
  const size_t mb = size_t(1) << 20;
  for (size_t n : {size_t(24), mb, 3 * mb - 8, 3 * mb, 3 * mb + 8, 8 * mb, 9 * mb, 17 * mb + 24})
    for (int kind = 0; kind < 6; ++kind) {  // pageable; pinned; pageable, the runtime fails to
      // say; the same up
      std::vector<char> dev(n), host(n, 0);
      for (size_t i = 0; i < n; ++i) dev[i] = (char)(i * 7 + i / 251 + 1);
      fake.user = host.data();
      fake.n = n;
      fake.pinned = kind % 3 == 1 ? host.data() : nullptr;
      fake.known = kind % 3 != 2;
      fake.straight = fake.chunks = 0;
      if (kind > 2) std::swap(dev, host), fake.user = host.data();
      if (kind == 4) fake.pinned = host.data();
      const hipError_t er = kind < 3 ? ring->to_host(host.data(), dev.data(), n, nullptr)
                                     : ring->to_device(dev.data(), host.data(), n, nullptr);
      std::printf("%zu %d %d %d %d\n", n, kind, (int)fake.straight, (int)fake.chunks,
                  er == hipSuccess && host == dev);
    }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_routes(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STAND_IN)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{tmp_path}", f"-I{CSRC}",
                    str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")], check=True)
    out = subprocess.run([str(tmp_path / "main")], check=True, capture_output=True, text=True,
                         timeout=60).stdout
    rows = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert len(rows) == 48
    for n, kind, straight, chunks, right in rows:
        assert right, (n, kind)
        by_ring = kind % 3 != 1 and n >= 3 << 20
        assert straight == (0 if by_ring else 1), (n, kind)
        assert chunks == (-(-n // (1 << 20)) if by_ring else 0), (n, kind)
