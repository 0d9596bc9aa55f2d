// CPU driver of the library's device-memory code over a fake device
// (fake_hip.hpp), built with the sanitizers by tests/test_memory_host.py.  The
// first argument names the check.
#include "fake_hip.hpp"

#include <cstring>
#include <thread>
#include <vector>

#include "../../cuts_amd/csrc/levels.hpp"
#include "../../cuts_amd/csrc/mpnn.hpp"

namespace cuts {
void hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw Error(-4, what);
}
void* ScratchArena::carve(uint64_t) { return nullptr; }
}  // namespace cuts

using namespace cuts;
constexpr uint64_t MB = 1ull << 20;

// A graph of static lifetime: it ends after what was constructed later, the
// pool among it.
struct Late {
  void* block = nullptr;
  ~Late() {
    if (!block) return;
    pool_give(0, block);
    void* again = pool_take(0, 2 * MB);
    CHECK(again == block);
    pool_give(0, again);
    pool_context(0, -1);
    CHECK(fake::device().used == 0);
    std::printf("late ok\n");
    std::fflush(stdout);
  }
} late;

static void end_of_process() {
  pool_context(0, 1);
  late.block = pool_take(0, 2 * MB);
  CHECK(late.block);
}

// Another thread gives the kept blocks back between this one's failed
// allocation and its own look at them.
static void flushed_by_another() {
  auto& d = fake::device();
  d.total = 100 * MB;
  pool_context(0, 1);
  pool_give(0, pool_take(0, 3 * MB));  // kept (the limit is 1/32)
  CHECK(d.used == 3 * MB);
  void* big = nullptr;
  CHECK(device_malloc(&big, 96 * MB) == hipSuccess);
  d.on_failure = [] {
    void* p = nullptr;
    CHECK(device_malloc(&p, 4 * MB) == hipSuccess);  // gives the kept block back
    CHECK(hipFree(p) == hipSuccess);
  };
  void* p = nullptr;
  CHECK(device_malloc(&p, 4 * MB) == hipSuccess);
  CHECK(hipFree(p) == hipSuccess && hipFree(big) == hipSuccess);
  CHECK(device_malloc(&p, 200 * MB) == hipErrorOutOfMemory && p == nullptr);
  pool_context(0, -1);
  CHECK(d.used == 0);
}

// A block whose users cannot be waited for is not handed to another stream.
static void given_while_capturing() {
  auto& d = fake::device();
  pool_context(0, 1);
  uint32_t* p = nullptr;
  dev_alloc(p, MB);
  CHECK(d.used == 4 * MB);
  const size_t syncs = d.syncs;
  dev_free(p);
  CHECK(d.syncs == syncs + 1 && d.used == 4 * MB);  // waited for, and kept
  p = nullptr;
  dev_alloc(p, MB);
  d.capturing = true;
  dev_free(p);
  CHECK(d.used == 0);  // freed, as hipFree waits by itself
  d.capturing = false;
  p = nullptr;
  dev_alloc(p, MB / 2);
  uint32_t* const first = p;
  d.capturing = true;
  dev_alloc(p, MB);  // grown: the old block is freed too
  d.capturing = false;
  CHECK(p != first || d.used == 4 * MB);
  CHECK(d.used == 4 * MB);
  dev_free(p);
  pool_context(0, -1);
  CHECK(d.used == 0);
}

// Memory runs out while a level grows: the level holds what it says, and the
// next, smaller request gets all of its arrays.
static void growth_that_fails() {
  auto& d = fake::device();
  pool_context(0, 1);
  auto whole = [](const LevelBuf& b) { return b.rows && b.minlen && b.minsel && b.work_off && b.cbase; };
  for (int exact = 0; exact < 2; ++exact) {
    LevelBuf b;
    auto ensure = [&](uint64_t n) { exact ? ensure_rows_exact(nullptr, b, n, 4) : ensure_rows(nullptr, b, n, 4); };
    d.total = 1024 * MB;
    ensure(MB);
    CHECK(whole(b) && b.cap == MB);
    for (uint64_t room = 0; room < 64; room += 3) {  // out of memory at each array in turn
      d.total = d.used + room * MB;
      bool failed = false;
      try {
        ensure(2 * MB);
      } catch (const Error& e) {
        failed = e.code == -5;
      }
      CHECK(failed ? b.cap == 0 || whole(b) : whole(b) && b.cap >= 2 * MB);
      d.total = 1024 * MB;
      ensure(MB / 2);
      CHECK(whole(b) && b.cap >= MB / 2);
      if (!failed) break;
    }
    for (void* p : {(void*)b.rows, (void*)b.minlen, (void*)b.minsel, (void*)b.work_off, (void*)b.cbase}) dev_free(p);
  }
  pool_context(0, -1);
  CHECK(d.used == 0);
}

// Memory runs out while a network's buffers grow: a later call finds them
// whole, and no buffer is freed twice.
static void network_that_does_not_fit() {
  auto& d = fake::device();
  const uint64_t per = kMpnnNodes * (kMpnnFeats * 4 + 2) + 4 * 4;
  auto whole = [](const Mpnn& n) { return n.x && n.row && n.adj && n.meta && n.t && n.y; };
  for (uint64_t room = 0; room <= 10000 * per; room += 50 * 1024) {
    d.total = 1024 * MB;
    Mpnn n;
    mpnn_reserve(n, 5);
    CHECK(whole(n) && n.cap == 1024);
    const size_t first = d.used;
    d.total = d.used + room;
    bool failed = false;
    try {
      mpnn_reserve(n, 10000);
    } catch (const Error& e) {
      failed = e.code == -5;
    }
    CHECK(failed ? n.cap == 0 : whole(n) && n.cap == 10000);
    if (failed) {
      d.total = 1024 * MB;
      mpnn_reserve(n, 1024);
      CHECK(whole(n) && n.cap == 1024 && d.used >= first);
      mpnn_reserve(n, 2000);
      CHECK(whole(n) && n.cap == 2000);
    }
  }
  CHECK(d.used == 0);
}

// Eight threads take and give blocks, give the kept ones back and run out of
// memory now and then; nothing is kept beyond the limit or lost.
static void threads() {
  auto& d = fake::device();
  d.total = 256 * MB;
  pool_context(0, 1);
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([t] {
      unsigned seed = 7 + t;
      std::vector<void*> mine;
      for (int i = 0; i < 4000; ++i) {
        const uint64_t n = (1 + rand_r(&seed) % 8) * MB + rand_r(&seed) % 1000;
        if (void* p = pool_take(0, n)) mine.push_back(p);
        while (mine.size() > 6 || (!mine.empty() && rand_r(&seed) % 2)) {
          pool_give(0, mine.back(), rand_r(&seed) % 16 != 0);
          mine.pop_back();
        }
        if (i % 64 == 0) pool_trim(0);
        if (i % 97 == 0) {
          pool_context(0, 1);
          pool_context(0, -1);
        }
      }
      for (void* p : mine) pool_give(0, p);
    });
  for (auto& t : ts) t.join();
  CHECK(d.used <= d.total / 32);
  CHECK(device_free_bytes(0) == d.total);
  const uint64_t kept = d.used;
  CHECK(pool_trim(0) == kept && d.used == 0 && pool_trim(0) == 0);
  pool_give(0, pool_take(0, 2 * MB));
  CHECK(d.used == 2 * MB);
  pool_context(0, -1);
  CHECK(d.used == 0);
}

// What an index build takes for itself, on devices with little and much free
// memory: never more than the bounds that its comment gives, but one group.
static void index_builds() {
  for (uint64_t free : {0 * MB, 64 * MB, 600 * MB, 2048 * MB, 294912 * MB})
    for (uint32_t V : {2u, 255u, 257u, 36692u, 65536u, 131072u, 131073u, 1u << 20, 1u << 25}) {
      const uint32_t groups = (V + 63) / 64, at_once = mask_groups(groups, V, free);
      CHECK(at_once >= 1 && at_once <= groups);
      CHECK(at_once == 1 || 8ull * V * at_once <= std::min<uint64_t>(512 * MB, free / 16));
      CHECK(at_once == groups || 8ull * V * (at_once + 1) > std::min<uint64_t>(512 * MB, free / 16));
      const uint64_t counts = (uint64_t)V * ((V + 255) / 256) * 4;
      CHECK(two_hop_on_device(V, free) == (V <= 131072 && counts <= free / 8));
    }
  CHECK(mask_groups(2048, 131072, 288ull << 30) == 512 && two_hop_on_device(131072, 288ull << 30));
  CHECK(!two_hop_on_device(131072, 1024 * MB));
}

int main(int, char** argv) {
  const std::string what = argv[1];
  if (what == "end_of_process") end_of_process();
  else if (what == "flushed_by_another") flushed_by_another();
  else if (what == "given_while_capturing") given_while_capturing();
  else if (what == "growth_that_fails") growth_that_fails();
  else if (what == "network_that_does_not_fit") network_that_does_not_fit();
  else if (what == "threads") threads();
  else if (what == "index_builds") index_builds();
  else return 3;
  std::printf("%s ok\n", argv[1]);
  return 0;
}
