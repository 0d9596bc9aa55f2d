// The network's buffers, and the live rows of its samples, packed for the copy
// to the GPU by all host threads at once (a sample of k query vertices has k of
// 16 rows; one thread's memcpy is slower than the copy itself).
#include <cstring>

#include <omp.h>

#include "mpnn.hpp"

namespace cuts {

void* mpnn_malloc(uint64_t bytes) {
  void* p = nullptr;
  if (device_malloc(&p, std::max<uint64_t>(bytes, 1)) != hipSuccess) throw Error(-5, "mpnn: device allocation failed");
  return p;
}

Mpnn::~Mpnn() {
  if (ctx) (void)hipSetDevice(ctx->device);
  for (void* q : {(void*)p, (void*)m, (void*)v, (void*)g, (void*)w, (void*)wt, (void*)part, (void*)loss,
                  (void*)x, (void*)row, (void*)adj, (void*)meta, (void*)t, (void*)y})
    if (q) (void)hipFree(q);
  if (stage) (void)hipHostFree(stage);
}

void mpnn_reserve(Mpnn& n, uint32_t cnt) {
  if (cnt <= n.cap) return;
  const uint32_t cap = std::max<uint32_t>(cnt, 1024);
  auto grow = [&](auto*& p, uint64_t each) {
    if (p) (void)hipFree(p);
    p = nullptr;
    p = (std::remove_reference_t<decltype(p)>)mpnn_malloc((uint64_t)cap * each * sizeof(*p));
  };
  n.cap = 0;  // until all are there: an allocation may fail
  grow(n.x, kMpnnNodes * kMpnnFeats);
  grow(n.row, 1);
  grow(n.adj, kMpnnNodes);
  grow(n.meta, 1);
  grow(n.t, 1);
  grow(n.y, 1);
  n.cap = cap;
}

void pack_rows(const float* x, const uint32_t* meta, const uint32_t* row, uint32_t first, uint32_t last, float* out) {
  const int threads = std::min(8, omp_get_max_threads());
#pragma omp parallel for schedule(static) num_threads(threads)
  for (int64_t s = first; s < (int64_t)last; ++s)
    std::memcpy(out + (uint64_t)(row[s] - row[first]) * kMpnnFeats, x + (uint64_t)s * kMpnnNodes * kMpnnFeats,
                (uint64_t)(meta[s] & 0xFF) * kMpnnFeats * 4);
}

}  // namespace cuts
