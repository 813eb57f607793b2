// Kept device memory (srbcrs_pool.h).
#include "srbcrs_pool.h"

#include <cstdint>
#include <map>
#include <mutex>
#include <set>
#include <tuple>
#include <unordered_map>
#include <vector>

namespace srbcrs {

namespace {

struct Block {
  void* p;
  size_t bytes;
  int device;
};

// Kept blocks by the time they were freed, and by (device, size, time): a
// process that has seen graphs of many sizes keeps thousands, and looking
// through them all took a small conversion from 90 to 320 us.
struct Pool {
  std::mutex mu;
  uint64_t now = 0;
  std::map<uint64_t, Block> kept;
  std::set<std::tuple<int, size_t, uint64_t>> by_size;
  size_t kept_bytes = 0;
  std::unordered_map<void*, Block> live;

  void keep(const Block& b) {
    kept.emplace(now, b);
    by_size.emplace(b.device, b.bytes, now++);
    kept_bytes += b.bytes;
  }
  Block take(std::map<uint64_t, Block>::iterator it) {
    const Block b = it->second;
    by_size.erase({b.device, b.bytes, it->first});
    kept.erase(it);
    kept_bytes -= b.bytes;
    return b;
  }
};

Pool& pool() {
  static Pool* p = new Pool;   // never destroyed: the runtime may be gone at exit
  return *p;
}

// 8 sizes per octave, so that arrays of similar graphs fit each other's
// blocks; 32 from 16 MB on, where an eighth of the size is much to leave
// unused; blocks that are not kept as they are.
size_t size_class(size_t n) {
  if (n <= 4096) return 4096;
  if (n > kPoolBytes) return n;
  const int o = 63 - __builtin_clzll((unsigned long long)n);
  const size_t step = size_t(1) << (o - (o < 24 ? 3 : 5));
  return (n + step - 1) / step * step;
}

void free_now(const Block& b) {
  int cur = 0;
  const bool known = hipGetDevice(&cur) == hipSuccess;
  if (known && cur != b.device) (void)hipSetDevice(b.device);
  (void)hipFree(b.p);
  if (known && cur != b.device) (void)hipSetDevice(cur);
}

}  // namespace

void* pool_alloc(size_t bytes, bool fresh, hipError_t* why) {
  Pool& P = pool();
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  auto refused = [&] {
    (void)hipGetLastError();
    if (why) *why = e;
    return nullptr;
  };
  if (e != hipSuccess) return refused();
  const size_t want = fresh ? bytes : size_class(bytes);
  if (!fresh) {
    std::lock_guard<std::mutex> lock(P.mu);
    const auto best = P.by_size.lower_bound({dev, want, 0});
    if (best != P.by_size.end() && std::get<0>(*best) == dev && std::get<1>(*best) - want <= want / 4) {
      const Block b = P.take(P.kept.find(std::get<2>(*best)));
      P.live.emplace(b.p, b);
      return b.p;
    }
  }
  Block b{nullptr, want, dev};
  e = hipMalloc(&b.p, want);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    pool_release(dev);
    e = hipMalloc(&b.p, want);
  }
  if (e != hipSuccess) return refused();
  std::lock_guard<std::mutex> lock(P.mu);
  P.live.emplace(b.p, b);
  return b.p;
}

void pool_free(void* p) {
  if (!p) return;
  Pool& P = pool();
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(P.mu);
    const auto it = P.live.find(p);
    if (it == P.live.end()) return;
    const Block b = it->second;
    P.live.erase(it);
    if (b.bytes > kPoolBytes) {
      out.push_back(b);
    } else {
      while (P.kept_bytes + b.bytes > kPoolBytes) out.push_back(P.take(P.kept.begin()));
      P.keep(b);
    }
  }
  for (const Block& b : out) free_now(b);
}

void pool_drop(void* p) {
  if (!p) return;
  Pool& P = pool();
  Block b{p, 0, 0};
  {
    std::lock_guard<std::mutex> lock(P.mu);
    const auto it = P.live.find(p);
    if (it == P.live.end()) return;
    b = it->second;
    P.live.erase(it);
  }
  free_now(b);
}

void pool_release(int device) {
  Pool& P = pool();
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(P.mu);
    for (auto it = P.kept.begin(); it != P.kept.end();) {
      const auto at = it++;
      if (device < 0 || at->second.device == device) out.push_back(P.take(at));
    }
  }
  for (const Block& b : out) free_now(b);
}

}  // namespace srbcrs
