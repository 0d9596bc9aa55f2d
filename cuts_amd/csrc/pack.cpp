// Live rows of network samples, packed for the copy to the GPU by all host
// threads at once (a sample of k query vertices has k of 16 rows; one thread's
// memcpy is slower than the copy itself).
#include <cstring>

#include <omp.h>

#include "mpnn.hpp"

namespace cuts {

void pack_rows(const float* x, const uint32_t* meta, const uint32_t* row, uint32_t first, uint32_t last, float* out) {
  const int threads = std::min(8, omp_get_max_threads());
#pragma omp parallel for schedule(static) num_threads(threads)
  for (int64_t s = first; s < (int64_t)last; ++s)
    std::memcpy(out + (uint64_t)(row[s] - row[first]) * kMpnnFeats, x + (uint64_t)s * kMpnnNodes * kMpnnFeats,
                (uint64_t)(meta[s] & 0xFF) * kMpnnFeats * 4);
}

}  // namespace cuts
