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
//   - Results go to callers, who may free them by pst_free, which keeps them,
//     or by hipFree, of which the cache learns nothing. So a result is known
//     by the runtime's ID of its allocation, and every use of a kept one
//     (handing it out, freeing it) first checks that the address still holds
//     that allocation; a second pst_free is refused. Results of up to 1 MB
//     come from hipMalloc and go by hipFree (1.4 us for both; 4 to 64 MB 24).
//   - Safe over streams: a block enters the cache only when nothing on the
//     device can use it any more: dev_free waits for the device, by a hipFree,
//     and dev_free_idle is for callers that have waited themselves.
//   - Safe over threads: one mutex guards the tables; no HIP call that waits
//     is made under it.
// Blocks hold what their last user left; no caller may expect zeros.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "pst_internal.hpp"

namespace pst {

namespace {

constexpr size_t kLargeBlock = size_t{32} << 20;
constexpr size_t kKeepShare = 32;  // of a device's memory at most one part in so many is kept
constexpr size_t kSmallResult = size_t{1} << 20;  // results up to here are not kept

struct Block {
  void* p;
  size_t bytes;
  int dev;
  unsigned long long id = 0;  // the runtime's ID of an allocation that was a result (0: never one)
};

// ID of the allocation that starts at p (0: none, or none to be had).
unsigned long long allocation_id(void* p) {
  unsigned long long id = 0;
  if (hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, p) == hipSuccess) return id;
  (void)hipGetLastError();
  return 0;
}
bool still_there(const Block& b) { return b.id == 0 || allocation_id(b.p) == b.id; }

struct Cache {
  std::mutex mu;
  std::unordered_map<void*, Block> live;
  // results that callers hold, and how many entries it takes to look for
  // those that were freed by hipFree
  std::unordered_map<void*, Block> results;
  size_t sweep_at = 256;
  // kept blocks in the order they were freed, and per (device, size) which
  std::map<unsigned long long, Block> kept;
  std::multimap<std::pair<int, size_t>, unsigned long long> by_size;
  std::unordered_map<void*, unsigned long long> kept_at;
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
    kept_at.erase(it->second.p);
    kept.erase(it);
  }
  // A kept block of exactly this size, out of the tables; blocks that are no
  // longer the library's are dropped on the way.
  bool take(int dev, size_t bytes, Block* out) {
    for (;;) {
      auto r = by_size.equal_range({dev, bytes});
      if (r.first == r.second) return false;
      auto k = kept.find(r.first->second);
      *out = k->second;
      forget(k);
      if (still_there(*out)) return true;
    }
  }
};

// Never destroyed: blocks may be freed while the process ends.
Cache& cache() {
  static Cache* c = new Cache();
  return *c;
}

void free_all(const std::vector<Block>& bs) {
  for (const Block& b : bs)
    if (still_there(b)) (void)hipFree(b.p);
}

// Takes every kept block of `dev` out of the cache.
std::vector<Block> take_kept(int dev) {
  Cache& c = cache();
  std::vector<Block> out;
  std::lock_guard<std::mutex> lk(c.mu);
  for (auto it = c.kept.begin(); it != c.kept.end();) {
    auto next = std::next(it);
    if (it->second.dev == dev) {
      out.push_back(it->second);
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
    const std::vector<Block> back = take_kept(dev);
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

namespace {
// Puts an idle block into the cache, within its bounds, or frees it.
hipError_t keep(const Block& b) {
  Cache& c = cache();
  size_t limit = 0;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto l = c.limit.find(b.dev);
    if (l != c.limit.end()) limit = l->second;
  }
  if (limit == 0 || b.bytes >= kLargeBlock) {
    int cur = 0;
    size_t free_b = 0, total_b = 0;
    bool ok = hipGetDevice(&cur) == hipSuccess;
    if (ok && cur != b.dev) ok = hipSetDevice(b.dev) == hipSuccess;
    if (ok) ok = hipMemGetInfo(&free_b, &total_b) == hipSuccess;
    if (cur != b.dev) (void)hipSetDevice(cur);
    if (!ok) return hipFree(b.p);
    limit = total_b / kKeepShare;
    if (b.bytes >= kLargeBlock && free_b < total_b / 8) return hipFree(b.p);
  }
  if (b.bytes > limit) return hipFree(b.p);
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    c.limit[b.dev] = limit;
    for (auto it = c.kept.begin(); it != c.kept.end() && c.kept_bytes[b.dev] + b.bytes > limit;) {
      auto next = std::next(it);
      if (it->second.dev == b.dev) {
        out.push_back(it->second);
        c.forget(it);
      }
      it = next;
    }
    // an entry of this address is of an allocation that a caller freed
    auto old = c.kept_at.find(b.p);
    if (old != c.kept_at.end()) c.forget(c.kept.find(old->second));
    const unsigned long long t = c.tick++;
    c.kept[t] = b;
    c.by_size.insert({{b.dev, b.bytes}, t});
    c.kept_at[b.p] = t;
    c.kept_bytes[b.dev] += b.bytes;
  }
  free_all(out);
  return hipSuccess;
}

// Waits for the work of device `dev` by a hipFree of eight bytes, which waits
// for every stream of the device and for running graphs. hipDeviceSynchronize
// would break a capture that any thread has running, also a relaxed one; a
// free does not (1.4 us on an idle device, with the allocation).
hipError_t wait_on(int dev) {
  int cur = 0;
  hipError_t e = hipGetDevice(&cur);
  if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
  void* token = nullptr;
  if (e == hipSuccess) e = malloc_on(dev, &token, 8);
  if (e == hipSuccess) e = hipFree(token);
  if (cur != dev) (void)hipSetDevice(cur);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}
}  // namespace

hipError_t plain_alloc_bytes(void** p, size_t bytes) {
  *p = nullptr;
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  return e == hipSuccess ? malloc_on(dev, p, bytes ? bytes : 1) : e;
}

hipError_t result_alloc_bytes(void** p, size_t bytes) {
  if (bytes <= kSmallResult) return plain_alloc_bytes(p, bytes);
  *p = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  Cache& c = cache();
  Block b{};
  {
    std::lock_guard<std::mutex> lk(c.mu);
    if (c.take(dev, bytes, &b)) *p = b.p;
  }
  if (!*p) {
    e = malloc_on(dev, p, bytes);
    if (e != hipSuccess) return e;
  }
  const unsigned long long id = b.id ? b.id : allocation_id(*p);
  if (id == 0) return hipSuccess;  // freed by hipFree
  std::lock_guard<std::mutex> lk(c.mu);
  c.results[*p] = Block{*p, bytes, dev, id};
  if (c.results.size() >= c.sweep_at) {
    for (auto it = c.results.begin(); it != c.results.end();) it = still_there(it->second) ? std::next(it) : c.results.erase(it);
    c.sweep_at = std::max<size_t>(256, 2 * c.results.size());
  }
  return hipSuccess;
}

hipError_t result_free(void* p) {
  if (!p) return hipSuccess;
  Cache& c = cache();
  Block b{};
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto k = c.kept_at.find(p);
    if ((k != c.kept_at.end() && still_there(c.kept[k->second])) || c.live.count(p)) return hipErrorInvalidValue;
    auto it = c.results.find(p);
    if (it != c.results.end()) {
      b = it->second;
      c.results.erase(it);
    }
  }
  if (b.p && still_there(b) && wait_on(b.dev) == hipSuccess) return keep(b);
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
    Block b{};
    if (c.take(dev, bytes, &b)) {
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
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.live.find(p);
    if (it != c.live.end()) {
      b = it->second;
      c.live.erase(it);
    }
  }
  return b.p ? keep(b) : hipFree(p);
}

hipError_t dev_wait(const void* p) {
  Cache& c = cache();
  int dev = -1;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.live.find(const_cast<void*>(p));
    if (it != c.live.end()) dev = it->second.dev;
  }
  return dev < 0 ? hipSuccess : wait_on(dev);  // hipFree waits by itself
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
