// Common-neighbour rows of a symmetric data graph, built on the device at
// upload: |N(u) & N(v)| for a set of row vertices u and every v, as dense
// uint16 rows (hub rows) or as the two-hop index (ascending lists of the v
// with a nonzero count, plus dense rows for the longest lists).  No
// reference counterpart (cuTS intersects lists during the search,
// src/device_funcs.cu:57-100).
//
// The rows are taken 64 at a time: mask[x] has bit i set when row vertex i of
// the group is adjacent to x, so that row i's count of v is the number of
// x in N(v) whose mask has bit i.  A thread adds its masks as 64 one-bit
// numbers into bit-sliced counters (plane p holds bit p of all 64 counts): one
// 8-byte load and a few bitwise operations per list entry count 64 rows at
// once, where one atomic per wedge u-x-v went to L2 before (about 4e10 per
// second on the whole chip).  A block counts 256 consecutive v: lists of up to
// SHORT entries one per thread, longer ones a wave each (its lanes' counters
// added by a butterfly), and unpacks them into an LDS tile of 64 rows x 256 v,
// which goes out in row order.  Blocks of one group run on one XCD while there
// are groups for all eight, so that the group's masks stay in that XCD's L2.
// Bound by the gathers of the masks; R-MAT 18's 4,048 hub rows (2.1 GB):
// 88 -> 5.8 ms; both passes of the 36,692-vertex Chung-Lu graph's index
// (5.0e7 entries): 49 -> 5.9 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "batch.hpp"
#include "levels.hpp"

namespace cuts {

namespace {

constexpr int RB = 256;          // threads per block = vertices per tile
constexpr uint32_t SHORT = 64;   // longest list of one thread
constexpr int PT = 7;            // planes of a thread's counters (<= 64)
constexpr int PL = 11;           // planes of a lane's share of a long list (<= 1024: lists below 2^16)
constexpr int PW = 16;           // planes of a whole list's counters
constexpr int TS = RB + 2;       // row stride of the tile in LDS (odd number of words)
enum { HUB_ROWS = 0, H2_COUNT = 1, H2_WRITE = 2 };

struct RowArgs {
  const uint32_t *off, *adj;
  uint32_t V, ntiles;
  const uint2* mask;       // [groups][V]
  uint32_t groups, xcd;    // groups of this launch; 1: a group's blocks share an XCD
  const uint32_t* rowv;    // the rows' vertices, or null: r0 + row
  uint32_t r0, nrows;      // first row of the launch, rows in all
  uint16_t* out;           // HUB_ROWS: nrows x V
  uint32_t* tcnt;          // H2_COUNT: entries per (row, tile); H2_WRITE: the entries before the tile
  const uint64_t* h2_off;  // H2_WRITE
  uint32_t *hv, *hc;
  const int32_t* did;      // dense row of a vertex or -1, or null
  uint16_t* dense;
};

// One bit per row of the group: the row's vertex is adjacent to x.
__global__ __launch_bounds__(RB) void k_row_masks(const uint32_t* __restrict__ off, const uint32_t* __restrict__ adj,
                                                 uint32_t V, const uint32_t* __restrict__ rowv, uint32_t r0,
                                                 uint32_t n, unsigned long long* __restrict__ mask) {
  for (uint32_t r = blockIdx.x; r < n; r += gridDim.x) {
    const uint32_t u = rowv ? rowv[r0 + r] : r0 + r;
    unsigned long long* m = mask + (uint64_t)(r >> 6) * V;
    for (uint32_t i = off[u] + threadIdx.x; i < off[u + 1]; i += RB) atomicOr(&m[adj[i]], 1ull << (r & 63));
  }
}

// (carry, sum) of three one-bit numbers per bit position
__device__ __forceinline__ uint32_t add3(uint32_t& s, uint32_t a, uint32_t b) {
  const uint32_t c = (s & a) | (s & b) | (a & b);
  s = s ^ a ^ b;
  return c;
}

// Adds the carry c of plane Q - 1 to the planes Q.. of a counter.
template <int Q, int P>
__device__ __forceinline__ void ripple(uint32_t (&p)[P], uint32_t c) {
#pragma unroll
  for (int q = Q; q < P; ++q) {
    const uint32_t t = p[q] & c;
    p[q] ^= c;
    c = t;
  }
}

// Four masks: two pairs into plane 0, their carries into plane 1, one carry up.
template <int P>
__device__ __forceinline__ void add_four(uint32_t (&p)[P], uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  const uint32_t x = add3(p[0], a, b), y = add3(p[0], c, d);
  ripple<2>(p, add3(p[1], x, y));
}

// Adds the masks of adj[lo], adj[lo + step], .. below hi to the counters of
// the group's first (px) and last 32 rows (py); four at a time, so that the
// upper planes take one carry for every four masks.
template <int P>
__device__ __forceinline__ void count_masks(const uint32_t* __restrict__ adj, const uint2* __restrict__ mask, uint32_t lo,
                                            uint32_t hi, uint32_t step, uint32_t (&px)[P], uint32_t (&py)[P]) {
  uint32_t e = lo;
  for (; e < hi && hi - e > 3 * step; e += 4 * step) {
    uint32_t x[4];
    uint2 m[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = adj[e + i * step];
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = mask[x[i]];
    add_four(px, m[0].x, m[1].x, m[2].x, m[3].x);
    add_four(py, m[0].y, m[1].y, m[2].y, m[3].y);
  }
  for (; e < hi; e += step) {
    const uint2 m = mask[adj[e]];
    ripple<0>(px, m.x);
    ripple<0>(py, m.y);
  }
}

// Unpacks a thread's counters of 32 rows into its column of the tile.
__device__ __forceinline__ void unpack(const uint32_t (&p)[PT], uint16_t* col) {
  for (int b = 0; b < 32; ++b) {
    uint32_t c = 0;
#pragma unroll
    for (int q = 0; q < PT; ++q) c |= ((p[q] >> b) & 1u) << q;
    col[b * TS] = (uint16_t)c;
  }
}

template <int MODE>
__global__ __launch_bounds__(RB) void k_rows(RowArgs a) {
  __shared__ uint16_t s_tile[64 * TS];
  __shared__ uint32_t s_long[RB], s_nlong;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t grp, tile;
  if (a.xcd) {
    const uint32_t l = blockIdx.x >> 3;
    grp = (l / a.ntiles) * 8 + (blockIdx.x & 7u);
    tile = l % a.ntiles;
  } else {
    grp = blockIdx.x / a.ntiles;
    tile = blockIdx.x % a.ntiles;
  }
  if (grp >= a.groups) return;  // the whole block: the last eight groups may not be full
  const uint2* mask = a.mask + (uint64_t)grp * a.V;
  const uint32_t v0 = tile * RB;
  if (tid == 0) s_nlong = 0;
  __syncthreads();
  {
    const uint32_t v = v0 + tid;
    const uint32_t lo = v < a.V ? a.off[v] : 0u, hi = v < a.V ? a.off[v + 1] : 0u;
    if (hi - lo > SHORT) {
      s_long[atomicAdd(&s_nlong, 1u)] = tid;
    } else {
      uint32_t px[PT] = {}, py[PT] = {};
      count_masks<PT>(a.adj, mask, lo, hi, 1, px, py);
      unpack(px, s_tile + tid);
      unpack(py, s_tile + 32 * TS + tid);
    }
  }
  __syncthreads();
  for (uint32_t i = wave; i < s_nlong; i += RB / 64) {
    const uint32_t vl = s_long[i];
    const uint32_t lo = a.off[v0 + vl], hi = a.off[v0 + vl + 1];
    const int np = 32 - __builtin_clz(hi - lo);  // planes that the list's counts need, uniform
    uint32_t px[PW] = {}, py[PW] = {};
    {
      uint32_t lx[PL] = {}, ly[PL] = {};
      count_masks<PL>(a.adj, mask, lo + lane, hi, 64, lx, ly);
#pragma unroll
      for (int q = 0; q < PL; ++q) {
        px[q] = lx[q];
        py[q] = ly[q];
      }
    }
    for (int o = 1; o < 64; o <<= 1) {
      uint32_t cx = 0, cy = 0;
#pragma unroll
      for (int q = 0; q < PW; ++q)
        if (q < np) {
          cx = add3(px[q], __shfl_xor(px[q], o), cx);
          cy = add3(py[q], __shfl_xor(py[q], o), cy);
        }
    }
    uint32_t c = 0;
#pragma unroll
    for (int q = 0; q < PW; ++q)
      if (q < np) c |= (((lane < 32 ? px[q] : py[q]) >> (lane & 31)) & 1u) << q;
    s_tile[lane * TS + vl] = (uint16_t)c;
  }
  __syncthreads();
  // a wave per row, 64 vertices at a time
  for (uint32_t h = wave; h < 64; h += RB / 64) {
    const uint32_t r = a.r0 + grp * 64 + h;
    if (r >= a.nrows) break;
    const uint32_t u = a.rowv ? a.rowv[r] : r;
    uint32_t before = 0;
    if (MODE == H2_WRITE) before = a.tcnt[(uint64_t)r * a.ntiles + tile];
    const uint64_t base = MODE == H2_WRITE ? a.h2_off[u] : 0;
    const int32_t dr = MODE == H2_WRITE && a.did ? a.did[u] : -1;
#pragma unroll
    for (int k = 0; k < RB / 64; ++k) {
      const uint32_t vl = k * 64 + lane, v = v0 + vl;
      const uint32_t c = (v < a.V && v != u) ? s_tile[h * TS + vl] : 0u;
      if (MODE == HUB_ROWS) {
        if (v < a.V) a.out[(uint64_t)r * a.V + v] = (uint16_t)c;
        continue;
      }
      const uint64_t m = __ballot(c != 0);
      if (MODE == H2_WRITE) {
        if (dr >= 0 && v < a.V) a.dense[(uint64_t)dr * a.V + v] = (uint16_t)c;
        if (c) {
          const uint64_t at = base + before +
                              __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
          a.hv[at] = v;
          a.hc[at] = c;
        }
      }
      before += (uint32_t)__popcll(m);
    }
    if (MODE == H2_COUNT && lane == 0) a.tcnt[(uint64_t)r * a.ntiles + tile] = before;
  }
}

// Per row, the exclusive scan of its tiles' entries in place, and their sum;
// a wave per row.
__global__ __launch_bounds__(RB) void k_row_scan(uint32_t* __restrict__ tcnt, uint32_t rows, uint32_t ntiles,
                                                unsigned long long* __restrict__ total) {
  const uint32_t lane = threadIdx.x & 63;
  for (uint32_t r = blockIdx.x * (RB / 64) + (threadIdx.x >> 6); r < rows; r += gridDim.x * (RB / 64)) {
    uint32_t* t = tcnt + (uint64_t)r * ntiles;
    uint32_t carry = 0;
    for (uint32_t i0 = 0; i0 < ntiles; i0 += 64) {
      const uint32_t i = i0 + lane;
      const uint32_t c = i < ntiles ? t[i] : 0u;
      uint32_t s = c;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t q = __shfl_up(s, o);
        if (lane >= (uint32_t)o) s += q;
      }
      if (i < ntiles) t[i] = carry + s - c;
      carry += __shfl(s, 63);
    }
    if (lane == 0) total[r] = carry;
  }
}

// A device buffer of this build: a small one from the graph's slab, else from
// the pool; the stream has drained when it ends (each build synchronizes before
// it returns; an error may not have).
template <typename T>
struct Temp {
  Context& c;
  DeviceGraph& dg;
  T* p = nullptr;
  Temp(Context& ctx, DeviceGraph& g, uint64_t n) : c(ctx), dg(g) { graph_alloc(dg, p, n); }
  ~Temp() {
    if (in_slab(dg, p)) return;
    pool_give(c.device, p, hipStreamSynchronize(c.stream) == hipSuccess);
  }
  Temp(const Temp&) = delete;
  Temp& operator=(const Temp&) = delete;
};

// One launch of k_rows<MODE> per batch of groups.  fresh: build the masks
// (false: a single batch's are still there).
template <int MODE>
void row_passes(Context& c, RowArgs a, unsigned long long* mask, uint32_t at_once, bool fresh) {
  const uint32_t groups = (a.nrows + 63) / 64;
  for (uint32_t g0 = 0; g0 < groups; g0 += at_once) {
    a.r0 = g0 * 64;
    a.groups = std::min(at_once, groups - g0);
    const uint32_t n = std::min(a.groups * 64, a.nrows - a.r0);
    if (fresh) {
      HIPCHECK(hipMemsetAsync(mask, 0, (uint64_t)a.groups * a.V * 8, c.stream));
      hipLaunchKernelGGL(k_row_masks, dim3(std::min<uint32_t>(n, 65535)), dim3(RB), 0, c.stream, a.off, a.adj, a.V,
                         a.rowv, a.r0, n, mask);
      HIPCHECK(hipGetLastError());
    }
    a.mask = (const uint2*)mask;
    // with fewer than 32 groups some XCDs would run out of groups long before others
    a.xcd = a.groups >= 32;
    const uint64_t blocks = (uint64_t)(a.xcd ? (a.groups + 7) / 8 * 8 : a.groups) * a.ntiles;
    if (blocks >= (1ull << 31)) throw Error(-1, "index build: too many tiles for one launch");
    hipLaunchKernelGGL(k_rows<MODE>, dim3((uint32_t)blocks), dim3(RB), 0, c.stream, a);
    HIPCHECK(hipGetLastError());
  }
}

RowArgs row_args(const DeviceGraph& dg) {
  RowArgs a{};
  a.off = dg.off_out;
  a.adj = dg.adj_out;
  a.V = dg.V;
  a.ntiles = (dg.V + RB - 1) / RB;
  return a;
}

}  // namespace

void build_hub_rows(Context& c, DeviceGraph& dg, const std::vector<uint32_t>& hubs) {
  RowArgs a = row_args(dg);
  a.nrows = (uint32_t)hubs.size();
  a.out = dg.hr;
  const uint32_t at_once = mask_groups((a.nrows + 63) / 64, a.V, device_free_bytes(c.device));
  Temp<uint32_t> rowv(c, dg, hubs.size());
  Temp<unsigned long long> mask(c, dg, (uint64_t)at_once * a.V);
  HIPCHECK(hipMemcpy(rowv.p, hubs.data(), hubs.size() * 4, hipMemcpyHostToDevice));
  a.rowv = rowv.p;
  row_passes<HUB_ROWS>(c, a, mask.p, at_once, true);
  HIPCHECK(hipStreamSynchronize(c.stream));
}

void build_two_hop_device(Context& c, DeviceGraph& dg, std::vector<uint64_t>& off,
                          const std::function<std::vector<uint32_t>(const std::vector<uint64_t>&)>& dense_rows) {
  RowArgs a = row_args(dg);
  const uint32_t V = a.V, groups = (V + 63) / 64, at_once = mask_groups(groups, V, device_free_bytes(c.device));
  a.nrows = V;
  Temp<unsigned long long> mask(c, dg, (uint64_t)at_once * V), total(c, dg, V);
  Temp<uint32_t> tcnt(c, dg, (uint64_t)V * a.ntiles);
  a.tcnt = tcnt.p;
  row_passes<H2_COUNT>(c, a, mask.p, at_once, true);
  hipLaunchKernelGGL(k_row_scan, dim3(std::min<uint32_t>((V + 3) / 4, 65535)), dim3(RB), 0, c.stream, tcnt.p, V,
                     a.ntiles, total.p);
  HIPCHECK(hipGetLastError());
  std::vector<unsigned long long> t(V);
  HIPCHECK(hipMemcpyAsync(t.data(), total.p, (uint64_t)V * 8, hipMemcpyDeviceToHost, c.stream));
  HIPCHECK(hipStreamSynchronize(c.stream));
  for (uint32_t u = 0; u < V; ++u) off[u + 1] = off[u] + t[u];
  dg.h2_entries = off[V];
  const std::vector<uint32_t> cand = dense_rows(off);
  graph_alloc(dg, dg.h2_off, (uint64_t)V + 1);
  HIPCHECK(hipMemcpy(dg.h2_off, off.data(), ((uint64_t)V + 1) * 8, hipMemcpyHostToDevice));
  graph_alloc(dg, dg.h2_v, off[V]);
  graph_alloc(dg, dg.h2_c, off[V]);
  if (!cand.empty()) {
    std::vector<int32_t> did(V, -1);
    for (uint64_t r = 0; r < cand.size(); ++r) did[cand[r]] = (int32_t)r;
    graph_alloc(dg, dg.h2_did, V);
    HIPCHECK(hipMemcpy(dg.h2_did, did.data(), (uint64_t)V * 4, hipMemcpyHostToDevice));
    graph_alloc(dg, dg.h2_dense, cand.size() * V);
    dg.h2_dense_rows = (uint32_t)cand.size();
  }
  a.h2_off = dg.h2_off;
  a.hv = dg.h2_v;
  a.hc = dg.h2_c;
  a.did = dg.h2_did;
  a.dense = dg.h2_dense;
  row_passes<H2_WRITE>(c, a, mask.p, at_once, at_once < groups);
  HIPCHECK(hipStreamSynchronize(c.stream));
}

}  // namespace cuts
