// Device memory of graphs, index builds and trie levels, kept between uses.  A graph's
// index takes gigabytes, and the driver clears what one upload frees before
// the next may have it, at about 35 GB/s once the card's free memory has been
// handed out once: uploads of a few milliseconds of kernels then waited 40 to
// 85 ms for memory (R-MAT 18, 3.3 GB).  Freed blocks of at least kKeepMin
// bytes stay here, up to 1/32 of the device's memory, while a context of the
// device exists and until pool_trim frees them; an allocation takes one that
// is at most a quarter larger than asked.  They count as free memory
// (device_free_bytes), and every allocation of the library that fails gives
// them back and tries again.
#include <map>
#include <mutex>
#include <unordered_map>

#include "device.hpp"

namespace cuts {

namespace {

constexpr uint64_t kKeepMin = 1ull << 20;

struct Pool {
  std::mutex mu;
  std::multimap<uint64_t, void*> kept;          // by size
  std::unordered_map<void*, uint64_t> handed;   // sizes of the blocks in use
  uint64_t held = 0, limit = 0;
  int contexts = 0;
};

Pool& pool_of(int device) {
  // for as long as the process: a graph or a context of static lifetime may
  // end after everything that was constructed later than it
  static Pool* const pools = new Pool[64];
  if (device < 0 || device >= 64) throw Error(-1, "device index out of range");
  return pools[device];
}

// Frees every kept block (the caller holds the lock).
void release(Pool& p) {
  for (auto& b : p.kept) (void)hipFree(b.second);
  p.kept.clear();
  p.held = 0;
}

}  // namespace

hipError_t device_malloc(void** out, uint64_t bytes) {
  *out = nullptr;
  hipError_t e = hipMalloc(out, bytes);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return e;
  Pool& p = pool_of(device);
  {
    // nothing may be kept by now: another thread's failure has given it back,
    // and there is memory all the same
    std::lock_guard<std::mutex> lk(p.mu);
    release(p);
  }
  e = hipMalloc(out, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    *out = nullptr;
  }
  return e;
}

void* pool_take(int device, uint64_t bytes) {
  Pool& p = pool_of(device);
  if (bytes >= kKeepMin) {
    std::lock_guard<std::mutex> lk(p.mu);
    auto it = p.kept.lower_bound(bytes);
    if (it != p.kept.end() && it->first <= bytes + bytes / 4) {
      void* b = it->second;
      p.held -= it->first;
      p.handed[b] = it->first;
      p.kept.erase(it);
      return b;
    }
  }
  void* b = nullptr;
  if (device_malloc(&b, bytes) != hipSuccess) return nullptr;
  if (bytes >= kKeepMin) {
    std::lock_guard<std::mutex> lk(p.mu);
    p.handed[b] = bytes;
  }
  return b;
}

bool device_idle() {
  if (hipDeviceSynchronize() == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

void pool_give(int device, void* b, bool idle) {
  if (!b) return;
  Pool& p = pool_of(device);
  {
    std::lock_guard<std::mutex> lk(p.mu);
    const auto it = p.handed.find(b);
    if (it != p.handed.end()) {
      const uint64_t bytes = it->second;
      p.handed.erase(it);
      if (idle && p.contexts > 0 && p.held + bytes <= p.limit) {
        p.kept.emplace(bytes, b);
        p.held += bytes;
        return;
      }
    }
  }
  (void)hipFree(b);
}

void pool_context(int device, int change) {
  Pool& p = pool_of(device);
  std::lock_guard<std::mutex> lk(p.mu);
  p.contexts += change;
  if (p.contexts <= 0) {
    release(p);
  } else if (!p.limit) {
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) == hipSuccess) p.limit = tot / 32;
  }
}

uint64_t pool_trim(int device) {
  Pool& p = pool_of(device);
  std::lock_guard<std::mutex> lk(p.mu);
  const uint64_t held = p.held;
  release(p);
  return held;
}

uint64_t device_free_bytes(int device) {
  size_t fr = 0, tot = 0;
  HIPCHECK(hipMemGetInfo(&fr, &tot));
  Pool& p = pool_of(device);
  std::lock_guard<std::mutex> lk(p.mu);
  return fr + p.held;
}

}  // namespace cuts
