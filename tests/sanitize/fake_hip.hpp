// The few HIP calls that the library's host-side memory code makes, over host
// memory: a device of `total` bytes, allocations counted against it.  For the
// CPU tests of that code (tests/sanitize/memory_driver.cpp); no GPU.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <mutex>
#include <string>

namespace fake {

struct Device {
  std::mutex mu;
  std::map<void*, size_t> blocks;
  size_t total = 1ull << 30, used = 0;
  bool capturing = false;            // hipDeviceSynchronize fails, as while a stream records a graph
  std::function<void()> on_failure;  // called once, without the lock, when an allocation fails
  size_t syncs = 0;
};
inline Device& device() {
  static Device* d = new Device;  // for as long as the process
  return *d;
}

}  // namespace fake

#define CHECK(c)                                                           \
  do {                                                                     \
    if (!(c)) {                                                            \
      std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
      std::_Exit(2);                                                       \
    }                                                                      \
  } while (0)

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  auto& d = fake::device();
  std::function<void()> f;
  {
    std::lock_guard<std::mutex> lk(d.mu);
    if (d.used + n <= d.total) {
      *p = std::malloc(64);
      d.blocks[*p] = n;
      d.used += n;
      return hipSuccess;
    }
    std::swap(f, d.on_failure);
  }
  if (f) f();
  return hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  auto& d = fake::device();
  std::lock_guard<std::mutex> lk(d.mu);
  if (!p) return hipSuccess;
  const auto it = d.blocks.find(p);
  CHECK(it != d.blocks.end());  // freed twice, or never allocated
  d.used -= it->second;
  d.blocks.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* fr, size_t* tot) {
  auto& d = fake::device();
  std::lock_guard<std::mutex> lk(d.mu);
  *fr = d.total - d.used;
  *tot = d.total;
  return hipSuccess;
}
hipError_t hipGetDevice(int* i) {
  *i = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() {
  auto& d = fake::device();
  std::lock_guard<std::mutex> lk(d.mu);
  ++d.syncs;
  return d.capturing ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
}
