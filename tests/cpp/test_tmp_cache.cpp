// The cache of temporaries (morpheus_amd/csrc/tmp_cache.hpp) over a counting
// allocator in place of the device's: which blocks stay held, which are let
// go, and by whom.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>

#include "tmp_cache.hpp"

using namespace mph;

static std::atomic<int> allocations{0}, releases{0};
static std::mutex live_mutex;
static std::set<void*> live;  // blocks neither released nor held twice

#define CHECK(x)                                              \
  do {                                                        \
    if (!(x)) {                                               \
      std::printf("line %d: not so: %s\n", __LINE__, #x);     \
      std::exit(1);                                           \
    }                                                         \
  } while (0)

static void release(const TmpBlock& b) {
  releases++;
  std::lock_guard<std::mutex> lk(live_mutex);
  CHECK(live.erase(b.p) == 1);
}

static TmpBlock get(TmpCache& c, int device, size_t bytes) {
  TmpBlock b;
  bytes = TmpCache::rounded(bytes);
  if (c.take(device, bytes, &b)) return b;
  static std::atomic<uintptr_t> next{4096};
  allocations++;
  b = TmpBlock{reinterpret_cast<void*>(next.fetch_add(64)), bytes, device};
  std::lock_guard<std::mutex> lk(live_mutex);
  live.insert(b.p);
  return b;
}

// a call that holds blocks of these sizes, then gives them back
static int call(TmpCache& c, int device, const std::vector<size_t>& sizes) {
  const int before = allocations;
  std::vector<TmpBlock> held;
  for (size_t s : sizes) {
    const TmpBlock b = get(c, device, s);
    CHECK(b.bytes >= s && b.device == device);
    held.push_back(b);
  }
  for (const TmpBlock& b : held) c.give(b, release);
  return allocations - before;
}

int main() {
  const size_t MB = (size_t)1 << 20;
  {  // a large call fills the cache; a smaller one's blocks still get in
    TmpCache c;
    const std::vector<size_t> large(4, 500 * MB), small(5, 90 * MB);
    CHECK(call(c, 0, large) == 4);
    CHECK(call(c, 0, large) == 0);
    CHECK(call(c, 0, small) == 5);
    for (int i = 0; i < 3; i++) CHECK(call(c, 0, small) == 0);
    CHECK(c.held(0) <= kTmpKeepBytes);
    c.trim_all(release);
  }
  {  // more distinct sizes than blocks are held: the last ones stay
    TmpCache c;
    const auto size = [&](size_t i) { return (i + 1) * 5 * MB / 8; };
    for (size_t i = 0; i < 3 * kTmpKeepBlocks; i++) call(c, 0, {size(i % kTmpKeepBlocks)});
    for (size_t i = kTmpKeepBlocks; i < kTmpKeepBlocks + 20; i++) call(c, 0, {size(i)});
    for (size_t i = kTmpKeepBlocks; i < kTmpKeepBlocks + 20; i++) CHECK(call(c, 0, {size(i)}) == 0);
    c.trim_all(release);
  }
  {  // each device and the pinned memory have limits of their own
    TmpCache c;
    CHECK(call(c, 0, {1900 * MB}) == 1);
    CHECK(call(c, 1, {1900 * MB}) == 1);
    CHECK(call(c, kTmpHost, {1900 * MB, 4096}) == 2);
    for (int d : {0, 1}) CHECK(call(c, d, {1900 * MB}) == 0);
    CHECK(call(c, kTmpHost, {4096}) == 0);
    // memory that runs out on one is not asked of the others
    int tries = 0;
    CHECK(c.get_or_trim(1, [&]() { return ++tries == 2; }, release));
    CHECK(c.held(1) == 0 && c.held(0) > 0 && c.held(kTmpHost) > 0);
    CHECK(!c.get_or_trim(1, [&]() { return false; }, release));
    c.trim_all(release);
    CHECK(c.held(0) == 0 && c.held(kTmpHost) == 0);
  }
  {  // a block beyond the limit is released at once, and lets the others stay
    TmpCache c;
    call(c, 0, {100 * MB});
    call(c, 0, {4096 * MB});
    CHECK(c.held(0) < 200 * MB && c.held(0) >= 100 * MB);
    CHECK(call(c, 0, {100 * MB}) == 0);
    c.trim_all(release);
  }
  {  // threads: no block is with two calls, none is lost
    TmpCache c;
    std::mutex m;
    std::set<void*> used;
    std::vector<std::thread> ts;
    for (int t = 0; t < 8; t++)
      ts.emplace_back([&, t]() {
        for (int i = 0; i < 4000; i++) {
          const TmpBlock b = get(c, i % 2, ((size_t)(i * 7 + t) % 90 + 1) * MB);
          {
            std::lock_guard<std::mutex> lk(m);
            CHECK(used.insert(b.p).second);
          }
          {
            std::lock_guard<std::mutex> lk(m);
            used.erase(b.p);
          }
          c.give(b, release);
        }
      });
    for (auto& t : ts) t.join();
    c.trim_all(release);
  }
  CHECK(allocations == releases && live.empty());
  std::printf("ok\n");
  return 0;
}
