// izh_memory.hip -- the library's device allocations.
//
// A lattice scan makes and ends a bunch per scan point.  Its about twenty
// buffers cost 0.3-0.7 ms to allocate and, above all, 1.2-4 ms to free (each
// hipFree waits for the device and unmaps): 1.2M particles on 64x64x128 spent
// 1.8 of 11.9 ms of a 64-step run on it.  So a released block is kept for the
// next allocation of about its size.
// - What is kept is bounded (kKeepBytes a device; the oldest blocks leave
//   first) and goes back when an allocation fails, when the last bunch or
//   field of the device ends and when the caller asks (izh_memory_trim).
// - A block serves requests down to 15/16 of its size, so a handle holds at
//   most that much more than it asked for.
// - A block is released by the owner's destroy or grow call, after it waited
//   for its stream, so the next owner may use it on any stream.
// - One lock guards the lists; hipMalloc and hipFree run outside of it.
#include <condition_variable>
#include <deque>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "izh_internal.hpp"

namespace izh {
namespace {

constexpr size_t kKeepBytes = (size_t)8 << 30;

struct Block {
  void *p;
  size_t bytes;
  int device;
};

struct Cache {
  std::mutex mu;
  std::unordered_map<void *, Block> used;
  std::unordered_map<int, size_t> used_bytes;
  std::unordered_map<int, std::deque<Block>> kept;  // by device, oldest first
  std::unordered_map<int, size_t> kept_bytes;
  std::unordered_map<int, int> handles;
  // blocks off the lists but not freed yet, and how often some have been
  std::condition_variable freed;
  int freeing = 0;
  uint64_t times_freed = 0;
};

// Never destroyed: at process exit the runtime may be gone before it.
Cache &cache() {
  static Cache *c = new Cache;
  return *c;
}

// Every kept block of the device, taken off the lists (the lock is held).
std::vector<Block> take_all(Cache &c, int device) {
  std::deque<Block> &q = c.kept[device];
  std::vector<Block> out(q.begin(), q.end());
  q.clear();
  c.kept_bytes[device] = 0;
  c.freeing += !out.empty();
  return out;
}

// Frees what was taken off the lists (counted in freeing when it was).
void give_back(Cache &c, const std::vector<Block> &blocks) {
  if (blocks.empty()) return;
  for (const Block &b : blocks) (void)hipFree(b.p);
  std::lock_guard<std::mutex> lock(c.mu);
  c.freeing--;
  c.times_freed++;
  c.freed.notify_all();
}

// A kept block for the request, if there is one (the lock is held).
void *take_kept(Cache &c, int device, size_t bytes) {
  std::deque<Block> &q = c.kept[device];
  auto best = q.end();
  for (auto it = q.begin(); it != q.end(); ++it)
    if (it->bytes >= bytes && it->bytes - it->bytes / 16 <= bytes &&
        (best == q.end() || it->bytes < best->bytes))
      best = it;
  if (best == q.end()) return nullptr;
  const Block b = *best;
  q.erase(best);
  c.kept_bytes[device] -= b.bytes;
  c.used[b.p] = b;
  c.used_bytes[device] += b.bytes;
  return b.p;
}

}  // namespace

// There is no memory only when the device has none with nothing kept and no
// other thread in the middle of giving some back: until then it tries again.
hipError_t dev_malloc(void **p, size_t bytes) {
  *p = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Cache &c = cache();
  for (;;) {
    uint64_t times;
    {
      std::lock_guard<std::mutex> lock(c.mu);
      if ((*p = take_kept(c, dev, bytes)) != nullptr) return hipSuccess;
      times = c.times_freed;
    }
    e = hipMalloc(p, bytes);
    std::unique_lock<std::mutex> lock(c.mu);
    if (e == hipSuccess) {
      c.used[*p] = Block{*p, bytes, dev};
      c.used_bytes[dev] += bytes;
      return hipSuccess;
    }
    (void)hipGetLastError();
    *p = nullptr;
    const std::vector<Block> all = take_all(c, dev);
    if (all.empty()) {
      c.freed.wait(lock, [&] { return c.freeing == 0 || c.times_freed != times; });
      if (c.times_freed == times) return e;
    }
    lock.unlock();
    give_back(c, all);
  }
}

void dev_release(void *p) {
  if (!p) return;
  Cache &c = cache();
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(c.mu);
    const auto it = c.used.find(p);
    if (it == c.used.end()) return;   // not a block of dev_malloc's
    const Block b = it->second;
    c.used.erase(it);
    c.used_bytes[b.device] -= b.bytes;
    if (b.bytes > kKeepBytes || c.handles[b.device] <= 0) {
      out.push_back(b);
    } else {
      std::deque<Block> &q = c.kept[b.device];
      size_t &held = c.kept_bytes[b.device];
      while (held + b.bytes > kKeepBytes) {
        out.push_back(q.front());
        held -= q.front().bytes;
        q.pop_front();
      }
      q.push_back(b);
      held += b.bytes;
    }
    c.freeing += !out.empty();
  }
  give_back(c, out);
}

void dev_free(void *p) {
  if (!p) return;
  Cache &c = cache();
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(c.mu);
    const auto it = c.used.find(p);
    if (it == c.used.end()) return;
    out.push_back(it->second);
    c.used_bytes[it->second.device] -= it->second.bytes;
    c.used.erase(it);
    c.freeing++;
  }
  give_back(c, out);
}

void dev_handles(int device, int change) {
  Cache &c = cache();
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(c.mu);
    int &h = c.handles[device];
    h += change;
    if (h <= 0) out = take_all(c, device);
  }
  give_back(c, out);
}

}  // namespace izh

using namespace izh;

extern "C" {

int izh_memory_info(int64_t *in_use, int64_t *kept) {
  int dev = 0;
  IZH_HIP(hipGetDevice(&dev));
  Cache &c = cache();
  std::lock_guard<std::mutex> lock(c.mu);
  if (in_use) *in_use = (int64_t)c.used_bytes[dev];
  if (kept) *kept = (int64_t)c.kept_bytes[dev];
  return IZH_OK;
}

int izh_memory_trim(void) {
  int dev = 0;
  IZH_HIP(hipGetDevice(&dev));
  Cache &c = cache();
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(c.mu);
    out = take_all(c, dev);
  }
  give_back(c, out);
  return IZH_OK;
}

}  // extern "C"
