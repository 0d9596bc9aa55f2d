// Device arrays of the matcher: graphs' own, trie levels', and a scratch run's.
// Host code only, so that it can be checked without a GPU.
#pragma once
#include <algorithm>
#include <string>

#include "device.hpp"

namespace cuts {

// Back to the pool, once the device has finished with it, as hipFree waits.
// Where it cannot be waited for (a stream of the process is recording a
// graph), it is freed instead: the pool's next taker may be on any stream.
inline void dev_free(void* p) {
  if (!p) return;
  int device = 0;
  HIPCHECK(hipGetDevice(&device));
  pool_give(device, p, device_idle());
}

// An array on the current device, from the pool; the old one goes back.
template <typename T>
void dev_alloc(T*& p, uint64_t n) {
  T* const old = p;
  p = nullptr;
  dev_free(old);
  int device = 0;
  HIPCHECK(hipGetDevice(&device));
  p = (T*)pool_take(device, std::max<uint64_t>(n, 1) * sizeof(T));
  if (!p) throw Error(-5, "device allocation of " + std::to_string(n * sizeof(T)) + " bytes failed");
}

// An array of the device graph's own: of up to kSlabMost bytes from the graph's
// slab while that has room, else a block of its own.  Both come from the pool,
// which keeps slabs but not blocks that small: with an allocation for each of
// its 10 to 25 arrays a small graph's upload was mostly those.
constexpr uint64_t kSlab = 1ull << 20, kSlabMost = 128ull << 10;
template <typename T>
void graph_alloc(DeviceGraph& dg, T*& p, uint64_t n) {
  const uint64_t bytes = std::max<uint64_t>(n, 1) * sizeof(T);
  if (bytes <= kSlabMost) {
    if (!dg.slab) dg.slab = (char*)pool_take(dg.device, kSlab);
    const uint64_t at = (dg.slab_used + 255) & ~255ull;
    if (dg.slab && at + bytes <= kSlab) {
      p = (T*)(dg.slab + at);
      dg.slab_used = at + bytes;
      return;
    }
  }
  p = (T*)pool_take(dg.device, bytes);
  if (!p) throw Error(-5, "device allocation of " + std::to_string(bytes) + " bytes failed");
}
inline bool in_slab(const DeviceGraph& dg, const void* p) {
  return dg.slab && (const char*)p >= dg.slab && (const char*)p < dg.slab + kSlab;
}

// Device buffer of n elements: from the pool (the old one goes back to it), or
// carved from the arena when there is one (nothing given back; sizes are
// rounded up to a power of two so that regrowth wastes at most half of what
// was carved).
template <typename T>
void dev_alloc(ScratchArena* a, T*& p, uint64_t n) {
  if (!a) {
    dev_alloc(p, n);
    return;
  }
  uint64_t m = 1;
  while (m < std::max<uint64_t>(n, 1)) m <<= 1;
  p = (T*)a->carve(m * sizeof(T));
}

// The index builds' own memory beside what they build, of `free` bytes: the
// masks of one group of 64 rows are 8V bytes, those of as many groups are held
// at once as fit 512 MiB and a sixteenth of it (one at least; with fewer than
// all, the write pass builds them again).
inline uint32_t mask_groups(uint32_t groups, uint32_t V, uint64_t free) {
  const uint64_t bytes = std::min<uint64_t>(512ull << 20, free / 16);
  return (uint32_t)std::min<uint64_t>(groups, std::max<uint64_t>(1, bytes / (8ull * V)));
}
// The two-hop index is built on the device up to 2^17 vertices, where its
// counts per row and tile of 256 columns (V^2/64 bytes, 256 MiB at most) fit
// an eighth of the free memory; else on the host, which needs only the index.
inline bool two_hop_on_device(uint32_t V, uint64_t free) {
  return V <= (1u << 17) && (uint64_t)V * ((V + 255) / 256) * 4 <= free / 8;
}

// Makes sure level buffer `lv` can hold `rows` rows of `words` words plus
// the planning arrays for them.
inline void ensure_rows(ScratchArena* ar, LevelBuf& b, uint64_t rows, uint32_t words) {
  if (b.cap >= rows && b.rows) return;
  uint64_t cap = std::max<uint64_t>(rows, 1024);
  if (b.cap) cap = std::max<uint64_t>(cap, b.cap + b.cap / 2);
  b.cap = 0;  // until all arrays are there: an allocation may fail
  dev_alloc(ar, b.rows, cap * words);
  dev_alloc(ar, b.minlen, cap);
  dev_alloc(ar, b.minsel, cap);
  dev_alloc(ar, b.work_off, cap + 1);
  dev_alloc(ar, b.cbase, cap);
  b.cap = cap;
}
inline void ensure_rows_exact(ScratchArena* ar, LevelBuf& b, uint64_t rows, uint32_t words) {
  // like ensure_rows but never grows beyond `rows` (budget-bound levels)
  if (b.cap >= rows && b.rows) return;
  b.cap = 0;
  dev_alloc(ar, b.rows, std::max<uint64_t>(rows, 1) * words);
  dev_alloc(ar, b.minlen, std::max<uint64_t>(rows, 1));
  dev_alloc(ar, b.minsel, std::max<uint64_t>(rows, 1));
  dev_alloc(ar, b.work_off, std::max<uint64_t>(rows, 1) + 1);
  dev_alloc(ar, b.cbase, std::max<uint64_t>(rows, 1));
  b.cap = rows;
}
// The per-row arrays of the pair and chain levels, allocated only for the
// levels that use them (each grows to the level's row capacity).
template <typename T>
void ensure_aux(ScratchArena* ar, T*& p, uint64_t& cap, uint64_t rows) {
  if (cap >= rows && p) return;
  dev_alloc(ar, p, std::max<uint64_t>(rows, 1));
  cap = std::max<uint64_t>(rows, 1);
}

inline void ensure_bsum(ScratchArena* ar, LevelBuf& b, uint64_t nb) {
  if (b.bsum_cap >= nb + 1 && b.bsum) return;
  dev_alloc(ar, b.bsum, nb + 1);
  b.bsum_cap = nb + 1;
}
inline void ensure_tiles(ScratchArena* ar, LevelBuf& b, uint64_t nt) {
  if (b.tile_cap >= nt + 1 && b.tile_p) return;
  dev_alloc(ar, b.tile_p, nt + 1);
  b.tile_cap = nt + 1;
}

}  // namespace cuts
