// Host check of the device memory tables (csrc/pst_memory.cpp) over a stub of
// the HIP runtime's memory calls: what is kept, handed out again and given
// back; results that callers free themselves; waits beside a stream capture.
// The stub refuses to free an address that is not allocated and gives freed
// addresses out again, as the runtime does.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "pst_capi.h"
#include "pst_internal.hpp"

namespace {
struct Dev {
  size_t total = size_t{1} << 30, used = 0;
};
Dev g_dev[2];
int g_cur = 0;
std::map<char*, std::pair<size_t, int>> g_mem;  // allocations: bytes, device
std::map<char*, unsigned long long> g_id;        // and the runtime's ID of each
unsigned long long g_ids = 0;
int g_mallocs = 0;
std::map<size_t, std::vector<char*>> g_free[2];  // freed addresses by size, reused last first
char* g_next = reinterpret_cast<char*>(size_t{1} << 40);
int g_waits = 0;          // hipFree calls that worked: each waits for the device
bool g_capturing = false;  // some stream is being captured (relaxed)
bool g_capture_broken = false;
bool g_refused = false;    // some stream is being captured in global mode: no call that may wait
int g_fail_host = 0;       // hipHostMalloc calls that fail
hipError_t g_last = hipSuccess;
std::mutex g_mu;
hipError_t set_last(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
bool allocated(void* p) { return g_mem.count(static_cast<char*>(p)) != 0; }
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { return *d = g_cur, hipSuccess; }
hipError_t hipSetDevice(int d) { return g_cur = d, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_refused) return set_last(hipErrorStreamCaptureUnsupported);
  Dev& d = g_dev[g_cur];
  if (n > d.total - d.used) return set_last(hipErrorOutOfMemory);
  auto& f = g_free[g_cur][n];
  char* a = g_next;
  if (!f.empty()) a = f.back(), f.pop_back();
  else g_next += n + 4096;
  g_mem[a] = {n, g_cur};
  g_id[a] = ++g_ids;
  g_mallocs++;
  d.used += n;
  *p = a;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (!p) return hipSuccess;
  if (g_refused) return set_last(hipErrorStreamCaptureUnsupported);
  auto it = g_mem.find(static_cast<char*>(p));
  if (it == g_mem.end()) return set_last(hipErrorInvalidValue);
  g_dev[it->second.second].used -= it->second.first;
  g_free[it->second.second][it->second.first].push_back(it->first);
  g_mem.erase(it);
  g_waits++;
  return hipSuccess;
}
hipError_t hipPointerGetAttribute(void* data, hipPointer_attribute what, hipDeviceptr_t p) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (what != HIP_POINTER_ATTRIBUTE_BUFFER_ID || !g_mem.count(static_cast<char*>(p))) return set_last(hipErrorInvalidValue);
  *static_cast<unsigned long long*>(data) = g_id[static_cast<char*>(p)];
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  if (g_capturing) return g_capture_broken = true, hipErrorStreamCaptureUnsupported;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = g_dev[g_cur].total - g_dev[g_cur].used;
  *t = g_dev[g_cur].total;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_fail_host > 0) return g_fail_host--, set_last(hipErrorOutOfMemory);
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
// the tree calls that a server makes when it is created
int pst_gpu_dtype(const pst_tree*) { return PST_F32; }
int pst_gpu_id_dtype(const pst_tree*) { return PST_U32; }
size_t pst_point_size(int, int) { return 12; }
const char* pst_last_error(void) { return ""; }
int pst_gpu_batch_count(pst_tree*, const void*, size_t, unsigned long long*, pst_stream_t) { return PST_OK; }
int pst_gpu_batch_write(pst_tree*, const void*, size_t, int, const unsigned long long*, const unsigned long long*, void*,
                        pst_stream_t) {
  return PST_OK;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
}

namespace {
int g_bad = 0;
void check(bool ok, const char* what, int line) {
  if (ok) return;
  g_bad++;
  std::printf("FAILED line %d: %s\n", line, what);
}
#define CHECK(x) check((x), #x, __LINE__)

void* take(size_t n) {
  void* p = nullptr;
  CHECK(pst::dev_alloc(&p, n) == hipSuccess);
  CHECK(allocated(p));
  return p;
}

// A result freed twice by pst_free, or by hipFree and then pst_free, is refused
// as hipFree refuses it; whatever a caller frees by hipFree, before or after,
// the memory handed out afterwards is allocated and nobody else's.
void results() {
  for (size_t n : {size_t{1} << 16, size_t{1} << 21}) {
    for (int how = 0; how < 4; how++) {
      void* r = nullptr;
      CHECK(pst::result_alloc(&r, n) == hipSuccess && allocated(r));
      const hipError_t first = how & 1 ? hipFree(r) : pst::result_free(r);
      const hipError_t second = how & 2 ? hipFree(r) : pst::result_free(r);
      CHECK(first == hipSuccess);
      CHECK((how & 2) || second != hipSuccess);
      CHECK((how & 2) || hipGetLastError() == hipSuccess);
      void* other = nullptr;  // may get the address that is free now
      CHECK(hipMalloc(&other, n) == hipSuccess);
      void* a = take(n);
      void* b = nullptr;
      CHECK(pst::result_alloc(&b, n) == hipSuccess && allocated(b));
      CHECK(a != b && a != other && b != other);
      CHECK(pst::dev_free(a) == hipSuccess && pst::result_free(b) == hipSuccess);
      CHECK(allocated(other));
      pst::dev_release_kept();
      CHECK(allocated(other));
      CHECK(hipFree(other) == hipSuccess);
      (void)hipGetLastError();
    }
  }
  constexpr size_t n = 1 << 20;
  // another owner's block of another size at a freed result's address
  void* r = nullptr;
  CHECK(pst::result_alloc(&r, 2 * n) == hipSuccess);
  CHECK(hipFree(r) == hipSuccess);
  g_free[0].clear();
  g_free[0][n / 2].push_back(static_cast<char*>(r));
  void* other = nullptr;
  CHECK(hipMalloc(&other, n / 2) == hipSuccess && other == r);
  CHECK(pst::result_free(other) == hipSuccess);
  CHECK(!allocated(other));
  void* big = take(2 * n);
  CHECK(g_mem[static_cast<char*>(big)].first == 2 * n);
  CHECK(pst::result_free(big) != hipSuccess && allocated(big));  // not the caller's
  CHECK(pst::dev_free(big) == hipSuccess);
  // a large result that pst_free took is used again, waits included; a block
  // that was a result stays one that callers may have kept the address of
  pst::dev_release_kept();
  CHECK(pst::result_alloc(&r, 2 * n) == hipSuccess);
  int w = g_waits, m = g_mallocs;
  CHECK(pst::result_free(r) == hipSuccess && allocated(r) && g_waits > w);
  m = g_mallocs;
  void* again = nullptr;
  CHECK(pst::result_alloc(&again, 2 * n) == hipSuccess && again == r && g_mallocs == m);
  CHECK(pst::result_free(again) == hipSuccess);
  void* own = take(2 * n);
  CHECK(own == r && pst::dev_free(own) == hipSuccess);
  CHECK(hipFree(r) == hipSuccess);  // by its old address
  void* fresh = take(2 * n);
  CHECK(allocated(fresh));
  CHECK(pst::dev_free(fresh) == hipSuccess);
  // results that callers free by hipFree do not pile up in the tables' way
  for (int k = 0; k < 2000; k++) {
    CHECK(pst::result_alloc(&r, 2 * n + 4096 * (k % 7)) == hipSuccess);
    CHECK(hipFree(r) == hipSuccess);
  }
  std::vector<void*> held(600);
  for (void*& h : held) CHECK(pst::result_alloc(&h, n + 16) == hipSuccess);
  for (void* h : held) CHECK(allocated(h) && pst::result_free(h) == hipSuccess);
  pst::dev_release_kept();
  for (void* h : held) CHECK(!allocated(h));
}

// Frees beside a capture neither break it nor lose the block; every block is
// waited for before it can be handed out again.
void captures() {
  constexpr size_t n = 3 << 20;
  void* a = take(n);
  g_capturing = true;
  const int before = g_waits;
  CHECK(pst::dev_free(a) == hipSuccess);
  CHECK(!g_capture_broken);
  CHECK(g_waits > before);
  void* b = take(n);
  CHECK(b == a);  // it was kept
  CHECK(pst::dev_wait(b) == hipSuccess);
  CHECK(pst::dev_free_idle(b) == hipSuccess);
  CHECK(!g_capture_broken);
  g_capturing = false;
  // refused outright: an error, the block stays the caller's and goes later
  void* c = take(2 * n);
  g_refused = true;
  CHECK(pst::dev_wait(c) != hipSuccess);
  CHECK(pst::dev_free(c) != hipSuccess);
  g_refused = false;
  CHECK(hipGetLastError() == hipSuccess);
  CHECK(allocated(c));
  void* d = take(2 * n);
  CHECK(d != c);
  CHECK(pst::dev_free(c) == hipSuccess && pst::dev_free(d) == hipSuccess);
  // a block of another device is waited for there
  g_cur = 1;
  void* e = take(n);
  g_cur = 0;
  CHECK(pst::dev_free(e) == hipSuccess);
  CHECK(g_cur == 0);
}

// The pinned words: a failed allocation (as beside a global capture) leaves no
// error for the next launch check and is tried again; slots are distinct,
// bounded and given back.
void host_words() {
  g_fail_host = 1;
  CHECK(pst::host_words_take() == nullptr);
  CHECK(hipGetLastError() == hipSuccess);
  std::set<unsigned long long*> got;
  while (unsigned long long* w = pst::host_words_take()) got.insert(w);
  CHECK(got.size() == 128);
  for (auto it = got.begin(); it != got.end() && std::next(it) != got.end(); ++it) CHECK(*std::next(it) - *it >= 4);
  pst::host_words_give(*got.begin());
  CHECK(pst::host_words_take() == *got.begin());
  for (unsigned long long* w : got) pst::host_words_give(w);
}

size_t used(int dev) { return g_dev[dev].used; }

// Kept blocks make room for a server's buffers where the device is full.
void server() {
  std::vector<void*> keep;
  for (int k = 0; k < 8; k++) keep.push_back(take(3 << 20));
  for (void* p : keep) CHECK(pst::dev_free(p) == hipSuccess);
  void* rest = nullptr;
  CHECK(hipMalloc(&rest, g_dev[0].total - used(0) - (4 << 20)) == hipSuccess);
  int dummy = 0;
  pst_tree* tree = reinterpret_cast<pst_tree*>(&dummy);
  pst_server* s = nullptr;
  CHECK(pst_server_create(&tree, 1, 10 << 20, 64, &s) == PST_OK);
  if (s) CHECK(pst_server_destroy(s) == PST_OK);
  CHECK(hipFree(rest) == hipSuccess);
  (void)hipGetLastError();
}

// The cache's bounds: at most 1/32 of the device, the least recently freed
// blocks leave first, larger blocks are never kept, nothing large on a nearly
// full device, each device its own; everything given back on request and where
// an allocation fails, which is then tried once more.
void bounds() {
  pst::dev_release_kept();
  const size_t base = used(0), base1 = used(1), limit = g_dev[0].total / 32;
  const size_t n = limit / 4 - 4096;  // four of them fit
  std::vector<void*> p;
  for (int k = 0; k < 6; k++) p.push_back(take(n + 16 * k));
  for (void* x : p) {
    CHECK(pst::dev_free(x) == hipSuccess);
    size_t held = used(0) - base;
    for (void* y : p) held -= allocated(y) && y > x ? g_mem[static_cast<char*>(y)].first : 0;
    CHECK(held <= limit);
  }
  CHECK(!allocated(p[0]) && !allocated(p[1]));
  for (int k = 2; k < 6; k++) CHECK(allocated(p[k]));
  CHECK(take(n + 16 * 3) == p[3]);  // exactly its size
  void* fresh = take(n + 16 * 3);
  CHECK(fresh != p[2] && fresh != p[4] && fresh != p[5]);
  CHECK(pst::dev_free(fresh) == hipSuccess && pst::dev_free(p[3]) == hipSuccess);
  void* big = take(limit + 1);
  CHECK(pst::dev_free(big) == hipSuccess);
  CHECK(!allocated(big));
  g_cur = 1;
  void* other = take(n);
  CHECK(pst::dev_free(other) == hipSuccess);
  CHECK(allocated(other) && used(1) == base1 + n);
  g_cur = 0;
  // an allocation that fails gives back this device's blocks alone
  void* rest = nullptr;
  CHECK(used(0) > base);
  CHECK(pst::dev_alloc(&rest, g_dev[0].total - base - 4096) == hipSuccess);
  CHECK(used(0) == g_dev[0].total - 4096 && used(1) == base1 + n);
  void* no = nullptr;
  CHECK(pst::dev_alloc(&no, 1 << 20) == hipErrorOutOfMemory && no == nullptr);
  CHECK(hipGetLastError() == hipErrorOutOfMemory);  // as hipMalloc leaves it
  CHECK(pst::dev_free(rest) == hipSuccess);
  CHECK(!allocated(rest));
  // on request: every device's
  void* a = take(n);
  CHECK(pst::dev_free(a) == hipSuccess && allocated(a));
  pst::dev_release_kept();
  CHECK(used(0) == base && used(1) == base1);
  // a block of 32 MB and more is not kept while less than 1/8 is free
  g_dev[0].total = size_t{4} << 30;
  void* fill = nullptr;
  CHECK(hipMalloc(&fill, (size_t{4} << 30) - (size_t{300} << 20)) == hipSuccess);
  g_dev[1].total = size_t{4} << 30;
  void* l = take(size_t{32} << 20);
  CHECK(pst::dev_free(l) == hipSuccess);
  CHECK(!allocated(l));
  CHECK(hipFree(fill) == hipSuccess);
  l = take(size_t{32} << 20);
  CHECK(pst::dev_free(l) == hipSuccess);
  CHECK(allocated(l));
  pst::dev_release_kept();
  CHECK(used(0) == base);
}

// Threads take and free blocks of the same sizes: no block is held twice, and
// all of them are given back.
void threads() {
  pst::dev_release_kept();
  const size_t base = used(0);
  std::mutex mu;
  std::set<void*> held;
  auto work = [&](unsigned seed) {
    for (int r = 0; r < 3000; r++) {
      seed = seed * 1664525u + 1013904223u;
      void* p = nullptr;
      const bool ok = pst::dev_alloc(&p, 4096u * (1 + (seed >> 28))) == hipSuccess;
      {
        std::lock_guard<std::mutex> lk(mu);
        CHECK(ok && held.insert(p).second);
      }
      std::lock_guard<std::mutex> lk(mu);
      held.erase(p);
      CHECK(pst::dev_free(p) == hipSuccess);
    }
  };
  std::vector<std::thread> ts;
  for (unsigned k = 0; k < 4; k++) ts.emplace_back(work, k + 1);
  for (auto& t : ts) t.join();
  pst::dev_release_kept();
  CHECK(used(0) == base);
}
}  // namespace

int main(int argc, char** argv) {
  const std::string only = argc > 1 ? argv[1] : "";
  if (only.empty() || only == "results") results();
  if (only.empty() || only == "captures") captures();
  if (only.empty() || only == "host_words") host_words();
  if (only.empty() || only == "server") server();
  if (only.empty() || only == "bounds") bounds();
  if (only.empty() || only == "threads") threads();
  std::printf(g_bad ? "%d checks failed\n" : "MEMORY OK\n", g_bad);
  return g_bad != 0;
}
