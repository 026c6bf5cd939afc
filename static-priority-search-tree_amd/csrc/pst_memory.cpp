// Device memory of the library: hipMalloc with a bounded cache of freed
// blocks.
//
// Freeing device memory and taking it again is slow in ways a program that
// rebuilds its trees (a volume per time step) meets on every pass: hipMalloc
// and hipFree are driver calls (tens of microseconds each, a small tree with
// its search buffers makes about 20), and the driver clears freed memory in
// the background at about 65 GB/s, so a loop that frees faster than that
// waits for the clearing. Measured on MI355X: building 2^26 f32/u32 points
// and counting a batch takes 11 ms in a fresh process and 39 to 75 ms in a
// long loop; a 300,007-point tree 3.3 ms, or 22 ms while freed memory of
// earlier work is being cleared. Kernels take 10 and 1.0 ms of these.
//
// So a freed block is kept and handed to the next request of exactly its
// size (a rebuilt tree asks for the same sizes; nothing is split or rounded
// into a larger block, so a request never pins more than it asked for).
//   - Bounded: at most 1/32 of the device's memory is kept per device,
//     least recently freed blocks leave first, and larger blocks are never
//     kept. When less than 1/8 of the device is free nothing large is kept.
//   - Given back: every kept block of a device is freed when an allocation
//     on it fails, before that allocation is tried once more, and all of them
//     on request (dev_release_kept), for other allocators of the program.
//   - Only the library's own blocks: results go to callers, who free them by
//     pst_free or hipFree, so they come from hipMalloc and go by hipFree. (A
//     kept block that a caller could free behind the cache's back would be
//     handed out unmapped.) Up to 2 MB that pair takes 1.4 us, 64 MB 24 us.
//   - Safe over streams: a block enters the cache only when nothing on the
//     device can use it any more: dev_free waits for the device, by a hipFree,
//     and dev_free_idle is for callers that have waited themselves.
//   - Safe over threads: one mutex guards the tables; no HIP call that waits
//     is made under it.
// Blocks hold what their last user left; no caller may expect zeros.
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "pst_internal.hpp"

namespace pst {

namespace {

constexpr size_t kLargeBlock = size_t{32} << 20;
constexpr size_t kKeepShare = 32;  // of a device's memory at most one part in so many is kept

struct Block {
  void* p;
  size_t bytes;
  int dev;
};

struct Cache {
  std::mutex mu;
  std::unordered_map<void*, Block> live;
  // kept blocks in the order they were freed, and per (device, size) which
  std::map<unsigned long long, Block> kept;
  std::multimap<std::pair<int, size_t>, unsigned long long> by_size;
  std::map<int, size_t> kept_bytes, limit;
  unsigned long long tick = 0;

  void forget(std::map<unsigned long long, Block>::iterator it) {
    auto r = by_size.equal_range({it->second.dev, it->second.bytes});
    for (auto k = r.first; k != r.second; ++k)
      if (k->second == it->first) {
        by_size.erase(k);
        break;
      }
    kept_bytes[it->second.dev] -= it->second.bytes;
    kept.erase(it);
  }
};

// Never destroyed: blocks may be freed while the process ends.
Cache& cache() {
  static Cache* c = new Cache();
  return *c;
}

void free_all(const std::vector<void*>& ps) {
  for (void* p : ps) (void)hipFree(p);
}

// Takes every kept block of `dev` out of the cache.
std::vector<void*> take_kept(int dev) {
  Cache& c = cache();
  std::vector<void*> out;
  std::lock_guard<std::mutex> lk(c.mu);
  for (auto it = c.kept.begin(); it != c.kept.end();) {
    auto next = std::next(it);
    if (it->second.dev == dev) {
      out.push_back(it->second.p);
      c.forget(it);
    }
    it = next;
  }
  return out;
}

}  // namespace

// One pinned page per process, in slots of four words, taken by handles at
// their first blocking search. Reading a result from it after the stream's
// synchronisation replaces a device-to-host copy (13 us each for 8 bytes).
constexpr int kHostSlots = 128, kHostWords = 4;
struct HostPage {
  std::mutex mu;
  unsigned long long* page = nullptr;
  bool used[kHostSlots] = {};
};
HostPage& host_page() {
  static HostPage* h = new HostPage();
  return *h;
}

unsigned long long* host_words_take() {
  HostPage& h = host_page();
  std::lock_guard<std::mutex> lk(h.mu);
  if (!h.page) {
    void* p = nullptr;
    if (hipHostMalloc(&p, kHostSlots * kHostWords * 8, hipHostMallocPortable | hipHostMallocMapped) == hipSuccess)
      h.page = static_cast<unsigned long long*>(p);
    else  // refused for now (a capture in global mode, say): the caller copies its results
      (void)hipGetLastError();
  }
  if (!h.page) return nullptr;
  for (int k = 0; k < kHostSlots; k++)
    if (!h.used[k]) {
      h.used[k] = true;
      return h.page + k * kHostWords;
    }
  return nullptr;
}

void host_words_give(unsigned long long* p) {
  if (!p) return;
  HostPage& h = host_page();
  std::lock_guard<std::mutex> lk(h.mu);
  h.used[(p - h.page) / kHostWords] = false;
}

size_t dev_keep_limit() {
  size_t free_b = 0, total_b = 0;
  if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) total_b = size_t{288} << 30;
  return total_b / kKeepShare;
}

void dev_release_kept() {
  std::vector<int> devs;
  {
    Cache& c = cache();
    std::lock_guard<std::mutex> lk(c.mu);
    for (const auto& k : c.kept_bytes) devs.push_back(k.first);
  }
  for (int d : devs) free_all(take_kept(d));
}

namespace {
// hipMalloc on device `dev`, the current one, once more without the kept
// blocks where it finds too little.
hipError_t malloc_on(int dev, void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    const std::vector<void*> back = take_kept(dev);
    if (!back.empty()) {
      free_all(back);
      (void)hipGetLastError();  // the failed attempt's
      e = hipMalloc(p, bytes);
    }
  }
  if (e != hipSuccess) *p = nullptr;
  return e;
}
}  // namespace

hipError_t result_alloc_bytes(void** p, size_t bytes) {
  *p = nullptr;
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  return e == hipSuccess ? malloc_on(dev, p, bytes ? bytes : 1) : e;
}

hipError_t result_free(void* p) {
  if (!p) return hipSuccess;
  const hipError_t e = hipFree(p);
  if (e != hipSuccess) (void)hipGetLastError();  // the caller's mistake, not the next launch's
  return e;
}

hipError_t dev_alloc_bytes(void** p, size_t bytes) {
  *p = nullptr;
  if (bytes == 0) bytes = 1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Cache& c = cache();
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.by_size.find({dev, bytes});
    if (it != c.by_size.end()) {
      auto k = c.kept.find(it->second);
      const Block b = k->second;
      c.forget(k);
      c.live[b.p] = b;
      *p = b.p;
      return hipSuccess;
    }
  }
  e = malloc_on(dev, p, bytes);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(c.mu);
  c.live[*p] = Block{*p, bytes, dev};
  return hipSuccess;
}

hipError_t dev_free_idle(void* p) {
  if (!p) return hipSuccess;
  Cache& c = cache();
  Block b{};
  size_t limit = 0;
  bool known = false;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.live.find(p);
    if (it != c.live.end()) {
      b = it->second;
      c.live.erase(it);
      known = true;
      auto l = c.limit.find(b.dev);
      if (l != c.limit.end()) limit = l->second;
    }
  }
  if (!known) return hipFree(p);
  if (limit == 0 || b.bytes >= kLargeBlock) {
    int cur = 0;
    size_t free_b = 0, total_b = 0;
    bool ok = hipGetDevice(&cur) == hipSuccess;
    if (ok && cur != b.dev) ok = hipSetDevice(b.dev) == hipSuccess;
    if (ok) ok = hipMemGetInfo(&free_b, &total_b) == hipSuccess;
    if (cur != b.dev) (void)hipSetDevice(cur);
    if (!ok) return hipFree(p);
    limit = total_b / kKeepShare;
    if (b.bytes >= kLargeBlock && free_b < total_b / 8) return hipFree(p);
  }
  if (b.bytes > limit) return hipFree(p);
  std::vector<void*> out;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    c.limit[b.dev] = limit;
    for (auto it = c.kept.begin(); it != c.kept.end() && c.kept_bytes[b.dev] + b.bytes > limit;) {
      auto next = std::next(it);
      if (it->second.dev == b.dev) {
        out.push_back(it->second.p);
        c.forget(it);
      }
      it = next;
    }
    const unsigned long long t = c.tick++;
    c.kept[t] = b;
    c.by_size.insert({{b.dev, b.bytes}, t});
    c.kept_bytes[b.dev] += b.bytes;
  }
  free_all(out);
  return hipSuccess;
}

// The wait is a hipFree of eight bytes, which waits for every stream of the
// device and for running graphs. hipDeviceSynchronize would break a capture
// that any thread has running, also a relaxed one; a free does not (1.4 us on
// an idle device, with the allocation).
hipError_t dev_wait(const void* p) {
  Cache& c = cache();
  int dev = -1, cur = 0;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.live.find(const_cast<void*>(p));
    if (it != c.live.end()) dev = it->second.dev;
  }
  if (dev < 0) return hipSuccess;  // hipFree waits by itself
  hipError_t e = hipGetDevice(&cur);
  if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
  void* token = nullptr;
  if (e == hipSuccess) e = malloc_on(dev, &token, 8);
  if (e == hipSuccess) e = hipFree(token);
  if (cur != dev) (void)hipSetDevice(cur);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

hipError_t dev_free(void* p) {
  if (!p) return hipSuccess;
  if (dev_wait(p) == hipSuccess) return dev_free_idle(p);
  // no wait to be had: the block's own hipFree waits, or refuses, and then
  // the block stays the caller's
  Cache& c = cache();
  Block b{};
  bool known = false;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.live.find(p);
    known = it != c.live.end();
    if (known) {
      b = it->second;
      c.live.erase(it);
    }
  }
  const hipError_t e = hipFree(p);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    std::lock_guard<std::mutex> lk(c.mu);
    if (known) c.live[p] = b;
  }
  return e;
}

}  // namespace pst
