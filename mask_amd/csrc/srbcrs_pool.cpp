// Kept device memory (srbcrs_pool.h).
#include "srbcrs_pool.h"

#include <cstdint>
#include <list>
#include <mutex>
#include <unordered_map>

namespace srbcrs {

namespace {

struct Block {
  void* p;
  size_t bytes;
  int device;
};

struct Pool {
  std::mutex mu;
  std::list<Block> kept;   // least recently freed first
  size_t kept_bytes = 0;
  std::unordered_map<void*, Block> live;
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

// Take kept blocks out of the list: all of a device, or the oldest until `room` bytes fit.
std::list<Block> take(Pool& P, int device, size_t room) {
  std::list<Block> out;
  for (auto it = P.kept.begin(); it != P.kept.end();) {
    auto next = std::next(it);
    if (room ? P.kept_bytes + room > kPoolBytes : device < 0 || it->device == device) {
      P.kept_bytes -= it->bytes;
      out.splice(out.end(), P.kept, it);
    }
    it = next;
  }
  return out;
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
    auto best = P.kept.end();
    for (auto it = P.kept.begin(); it != P.kept.end(); ++it)
      if (it->device == dev && it->bytes >= want && it->bytes - want <= want / 4 &&
          (best == P.kept.end() || it->bytes < best->bytes))
        best = it;
    if (best != P.kept.end()) {
      const Block b = *best;
      P.kept_bytes -= b.bytes;
      P.kept.erase(best);
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
  std::list<Block> out;
  {
    std::lock_guard<std::mutex> lock(P.mu);
    const auto it = P.live.find(p);
    if (it == P.live.end()) return;
    const Block b = it->second;
    P.live.erase(it);
    if (b.bytes > kPoolBytes) {
      out.push_back(b);
    } else {
      out = take(P, -1, b.bytes);
      P.kept.push_back(b);
      P.kept_bytes += b.bytes;
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
  std::list<Block> out;
  {
    std::lock_guard<std::mutex> lock(P.mu);
    out = take(P, device, 0);
  }
  for (const Block& b : out) free_now(b);
}

}  // namespace srbcrs
