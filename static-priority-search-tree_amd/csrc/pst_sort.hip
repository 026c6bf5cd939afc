// Stable LSD radix sort of (unsigned key, 32-bit value) pairs for gfx950,
// used by tree construction, level index construction and query grouping.
//
// The reference sorts size_t index arrays with thrust::sort and an
// indirect comparator (pst/static-pst-gpu.tu:266-267, 317-318). Here the
// comparison keys are order-preserving unsigned integers (pst_common.hpp:
// ord_key), sorted 8 bits per pass, least significant digit first. Every
// pass is stable, which construction relies on for its index tie-breaks.
//
// A sort is one histogram pass over the keys and then one kernel per digit:
//   k_sort_hist     every digit's count for every pass, from one read of the
//                   keys (LDS counters, then one global atomic per counter
//                   and workgroup);
//   k_digit_starts  per pass, each digit's first output position;
//   k_sort_pass     per tile of 8192 keys (eight waves of 1024, lane l of
//                   round r holding key r * 64 + l of its wave):
//     1. takes the next tile number from a counter, so that tiles start in
//        tile order;
//     2. ranks every key stably within the tile: within a wave by ballot
//        matching of the 8 digit bits (lanes with the same digit in a
//        round), across rounds by per-wave digit counters in LDS, across
//        waves by their digit prefix;
//     3. publishes its digit counts, then adds up the counts of the tiles
//        before it by reading their published words backwards until one
//        carries an inclusive prefix (decoupled look-back), and publishes
//        its own inclusive prefix;
//     4. reorders the tile in LDS by (digit, rank) and writes the keys, then
//        the values through the same LDS buffer, so that each digit's keys
//        leave as one contiguous run.
// A tile waits only for tiles with smaller numbers, which took their
// numbers earlier and are therefore running, and every tile publishes its
// counts before it waits: every wait ends. The wait is still bounded; a
// tile that exceeds the bound sets the caller's failure word and goes on.
// Passes alternate between the output and a scratch buffer, ending in the
// output; the inputs are not modified. A pass in which all keys share the
// digit is left out (64-bit IDs and integers use few of their bytes).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "pst_internal.hpp"

namespace pst {

namespace {

constexpr int kDigitBits = 8;
constexpr int kDigits = 1 << kDigitBits;
constexpr int kPassBlock = 512;
constexpr int kPassWaves = kPassBlock / kWave;            // 8
// Keys per lane: tiles of 8192 keys, of 4096 where those are few (a pass then
// waits for its tile's rounds, and half the rounds run on twice the CUs).
// Building trees whose sorts take 8 and 4 instead of 16 keys per lane, MI355X:
// 20,000 f64 points 474, 442, 415 us; 300,007 615, 601, 625; 10^6 820, 828, 943.
constexpr int kPassPerFull = 16, kPassPerFew = 8;
constexpr uint32_t kFewKeys = 1u << 19;
constexpr uint32_t tile_keys(int per) { return kPassBlock * static_cast<uint32_t>(per); }
inline uint32_t tiles_of(size_t n) {
  const uint32_t t = tile_keys(n <= kFewKeys ? kPassPerFew : kPassPerFull);
  return static_cast<uint32_t>((n + t - 1) / t);
}
constexpr int kHistBlock = 512;
constexpr int kHistPer = 16;
constexpr uint32_t kHistChunk = kHistBlock * kHistPer;
constexpr unsigned kHistMaxBlocks = 1024;
constexpr uint32_t kLookbackSpins = 1u << 24;             // about a second
// Look-back words read at once. Where all tiles run at once none finds a
// prefix before the first tiles have finished, and each adds up every tile
// before it: such a sort reads more words per step.
constexpr uint32_t kLookAhead = 4, kLookAheadFew = 16;

template <typename K>
__device__ inline uint32_t digit_of(K k, uint32_t shift) {
  return static_cast<uint32_t>(k >> shift) & (kDigits - 1);
}

// LDS digit counters of the histogram are kept in kSub copies, lane l
// adding to copy l % kSub: lanes that share a digit (frequent in the high
// digits of clustered keys) collide on one counter kSub times less often.
constexpr int kSub = 4;

// Published per (tile, digit): the count in the low 32 bits, a tag in the
// high 32 bits: 0 nothing yet, 2 * pass + 2 the tile's own count, 2 * pass
// + 3 the inclusive prefix over tiles 0..tile. Tags differ between the
// passes of one sort, so the words are cleared once per sort.
__device__ inline uint32_t tag_count(uint32_t pass) { return 2 * pass + 2; }
__device__ inline uint32_t tag_prefix(uint32_t pass) { return 2 * pass + 3; }
__device__ inline unsigned long long pack_status(uint32_t tag, uint32_t v) {
  return (static_cast<unsigned long long>(tag) << 32) | v;
}

__global__ void k_fill_zero(uint32_t* __restrict__ p, size_t count) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < count) p[i] = 0u;
}

// hist[p * 256 + d] += keys of digit d at pass p.
template <typename K>
__global__ __launch_bounds__(kHistBlock) void k_sort_hist(const K* __restrict__ keys, uint32_t n,
                                                          uint32_t* __restrict__ hist) {
  constexpr int P = static_cast<int>(sizeof(K));
  __shared__ uint32_t h[kSub][P][kDigits];
  const uint32_t tid = threadIdx.x;
  for (uint32_t i = tid; i < kSub * P * kDigits; i += kHistBlock) (&h[0][0][0])[i] = 0u;
  __syncthreads();
  uint32_t(*mine)[kDigits] = h[tid % kSub];
  for (uint64_t b = static_cast<uint64_t>(blockIdx.x) * kHistChunk; b < n;
       b += static_cast<uint64_t>(gridDim.x) * kHistChunk) {
    K k[kHistPer];
#pragma unroll
    for (int e = 0; e < kHistPer; e++) {
      const uint64_t i = b + static_cast<uint64_t>(e) * kHistBlock + tid;
      k[e] = i < n ? keys[i] : K(0);
    }
#pragma unroll
    for (int e = 0; e < kHistPer; e++) {
      const bool ok = b + static_cast<uint64_t>(e) * kHistBlock + tid < n;
      if (ok) {
#pragma unroll
        for (int p = 0; p < P - 1; p++) atomicAdd(&mine[p][digit_of(k[e], p * kDigitBits)], 1u);
      }
      // the top digit, often shared by a whole wave of clustered keys: such
      // a wave adds once
      const uint32_t d = digit_of(k[e], (P - 1) * kDigitBits);
      const uint64_t act = __ballot(ok);
      const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
      if (act == ~0ull && __ballot(d != d0) == 0ull) {
        if (tid % kWave == 0) atomicAdd(&h[0][P - 1][d0], static_cast<uint32_t>(kWave));
      } else if (ok) {
        atomicAdd(&mine[P - 1][d], 1u);
      }
    }
  }
  __syncthreads();
  for (uint32_t i = tid; i < P * kDigits; i += kHistBlock) {
    uint32_t c = 0;
#pragma unroll
    for (int u = 0; u < kSub; u++) c += (&h[u][0][0])[i];
    if (c) atomicAdd(&hist[i], c);
  }
}

// Exclusive scan of each of `passes` rows of 256 digit totals, in place (one
// workgroup, four rows at a time), and the passes' order: a pass whose keys
// all share one digit would only copy and is left out. order[p]: passes that
// run before p, or kNoPass; order[kMaxPasses]: passes that run. With
// `keep_first` pass 0 always runs; some pass always does.
constexpr uint32_t kMaxPasses = 8;
constexpr uint32_t kNoPass = ~0u;
constexpr int kStartsBlock = 4 * kDigits;
__global__ __launch_bounds__(kStartsBlock) void k_digit_starts(uint32_t* __restrict__ hist, uint32_t passes, uint32_t n,
                                                               uint32_t keep_first, uint32_t* __restrict__ order) {
  __shared__ uint32_t wsum[kStartsBlock / kWave];
  __shared__ uint32_t one[kMaxPasses];
  const uint32_t d = threadIdx.x % kDigits, lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  if (threadIdx.x < kMaxPasses) one[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t p0 = 0; p0 < passes; p0 += kStartsBlock / kDigits) {
    const uint32_t p = p0 + threadIdx.x / kDigits;
    const uint32_t v = p < passes ? hist[p * kDigits + d] : 0u;
    uint32_t inc = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t o = __shfl_up(inc, off, kWave);
      if (static_cast<int>(lane) >= off) inc += o;
    }
    if (lane == kWave - 1) wsum[wave] = inc;
    if (p < passes && v == n) one[p] = 1;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = wave & ~3u; w < wave; w++) before += wsum[w];
    if (p < passes) hist[p * kDigits + d] = before + inc - v;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    uint32_t run = 0;
    for (uint32_t p = 0; p < passes; p++) {
      const bool skip = one[p] && !(keep_first && p == 0) && !(p + 1 == passes && run == 0);
      order[p] = skip ? kNoPass : run;
      run += skip ? 0u : 1u;
    }
    order[kMaxPasses] = run;
  }
}

template <typename K, typename V, int PER>
struct PassLds {
  static constexpr uint32_t kSortTile = tile_keys(PER);
  union {
    unsigned long long peer[kPassWaves][kDigits];  // while ranking: per-wave lane masks of a round's digits
    K sbuf[kSortTile];                             // then keys,
    V vbuf[kSortTile];                             // then values, in (digit, rank) order
  };
  uint32_t wcnt[kPassWaves][kDigits];   // per-wave digit counters, then their wave prefix
  uint32_t dcnt[kDigits];               // the tile's count of each digit
  uint32_t dstart[kDigits];             // first tile position of each digit
  uint32_t goff[kDigits];               // global position of each digit's first key of the tile
  uint32_t wtot[kDigits / kWave];
  uint32_t tile;
};

// Where a pass reads its pairs: key and value arrays, the value when the
// keys are ranked (value() is called again then).
template <typename K, typename V>
struct ArraySrc {
  const K* kin;
  const V* vin;
  __device__ void at(uint64_t base) {
    kin += base;
    vin += base;
  }
  __device__ K key(uint32_t i) const { return kin[i]; }
  __device__ V value(uint32_t i) const { return vin[i]; }
};

// Or the points themselves (the first pass of a point sort): the key is the
// dim1 key, the value (~dim2 key, ~ID key), ~index where there is no ID, so
// that of two values the smaller one belongs to the greater point in
// (dim2, ID) order.
template <typename T, typename I>
struct PointSrc {
  const Point<T, I>* pts;
  uint32_t first;
  __device__ void at(uint64_t base) {
    pts += base;
    first = static_cast<uint32_t>(base);
  }
  __device__ uint32_t key(uint32_t i) const { return ord_key(pts[i].dim1_val); }
  __device__ uint64_t value(uint32_t i) const {
    const Point<T, I> p = pts[i];
    uint32_t lo = first + i;
    if constexpr (has_id_v<I>) lo = ord_key(p.id);
    return (static_cast<uint64_t>(~ord_key(p.dim2_val)) << 32) | static_cast<uint32_t>(~lo);
  }
};

// One tile of a digit pass. FULL: the tile holds kSortTile keys, so no
// element needs a bounds check (and each lane's loads share one address).
template <typename K, typename V, bool FULL, uint32_t LOOK, int kPassPer, typename Src>
__device__ __forceinline__ void sort_tile(PassLds<K, V, kPassPer>& L, Src src,
                                          K* __restrict__ kout, V* __restrict__ vout, uint32_t tile,
                                          uint32_t valid, uint32_t pass, unsigned long long* __restrict__ status,
                                          const uint32_t* __restrict__ gstart, int* __restrict__ fail) {
  constexpr uint32_t kSortTile = tile_keys(kPassPer), kWaveKeys = kWave * kPassPer;
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  const uint32_t shift = pass * kDigitBits;
  const uint64_t base = static_cast<uint64_t>(tile) * kSortTile;
  const uint32_t wbase = wave * kWaveKeys;
  auto in_tile = [&](uint32_t i) { return FULL || i < valid; };
  src.at(base + wbase);
  K k[kPassPer];
#pragma unroll
  for (int r = 0; r < kPassPer; r++)
    if (in_tile(wbase + r * kWave + lane)) k[r] = src.key(r * kWave + lane);
  // stable rank within the wave: rounds in element order, lanes in order.
  // The lanes of a round that share a digit find each other through the
  // wave's peer word of that digit: each ORs in its lane bit, all read the
  // word back (one wave's LDS instructions complete in order), and the
  // lowest of them advances the digit's counter and clears the word.
  uint32_t rank[kPassPer];
  uint32_t* cnt = L.wcnt[wave];
  unsigned long long* pw = L.peer[wave];
  const uint64_t me = 1ull << lane;
  const uint64_t lt = me - 1ull;
#pragma unroll
  for (int r = 0; r < kPassPer; r++) {
    const bool ok = in_tile(wbase + r * kWave + lane);
    const uint32_t d = digit_of(k[r], shift);
    uint64_t peers = 0;
    if (ok) atomicOr(&pw[d], me);
    __builtin_amdgcn_wave_barrier();
    if (ok) peers = pw[d];
    const uint32_t below = static_cast<uint32_t>(__builtin_popcountll(peers & lt));
    uint32_t before = 0;
    if (ok) before = cnt[d];
    __builtin_amdgcn_wave_barrier();
    if (ok && below == 0) {
      cnt[d] = before + static_cast<uint32_t>(__builtin_popcountll(peers));
      pw[d] = 0ull;
    }
    __builtin_amdgcn_wave_barrier();
    rank[r] = before + below;
    // keep the rank computed here: sunk to its use, every round's peer
    // word would stay live until the reorder
    asm volatile("" : "+v"(rank[r]));
  }
  __syncthreads();
  // per digit (thread tid = digit): wave prefixes and the tile's count,
  // published at once, and the in-tile exclusive scan of the counts
  if (tid < kDigits) {
    uint32_t run = 0;
#pragma unroll
    for (int w = 0; w < kPassWaves; w++) {
      const uint32_t c = L.wcnt[w][tid];
      L.wcnt[w][tid] = run;
      run += c;
    }
    L.dcnt[tid] = run;
    __hip_atomic_store(&status[static_cast<size_t>(tile) * kDigits + tid],
                       pack_status(tile == 0 ? tag_prefix(pass) : tag_count(pass), run), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    uint32_t inc = run;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t o = __shfl_up(inc, off, kWave);
      if (static_cast<int>(lane) >= off) inc += o;
    }
    if (lane == kWave - 1) L.wtot[wave] = inc;
    L.dstart[tid] = inc - run;  // exclusive within the wave for now
  }
  __syncthreads();
  if (tid < kDigits) {
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; w++) before += L.wtot[w];
    L.dstart[tid] += before;
  }
  __syncthreads();
  // keys into LDS by (digit, rank); rank[] becomes the LDS position
#pragma unroll
  for (int r = 0; r < kPassPer; r++) {
    if (in_tile(wbase + r * kWave + lane)) {
      const uint32_t d = digit_of(k[r], shift);
      const uint32_t p = L.dstart[d] + L.wcnt[wave][d] + rank[r];
      L.sbuf[p] = k[r];
      rank[r] = p;
    }
  }
  V v[kPassPer];
#pragma unroll
  for (int r = 0; r < kPassPer; r++)
    if (in_tile(wbase + r * kWave + lane)) v[r] = src.value(r * kWave + lane);
  // look-back: the digit's count over the tiles before this one
  if (tid < kDigits) {
    const uint32_t run = L.dcnt[tid];
    uint32_t excl = 0;
    if (tile > 0) {
      const uint32_t ta = tag_count(pass), tp = tag_prefix(pass);
      uint32_t j = tile - 1;  // the next tile to read; tiles above j are summed
      uint32_t spins = 0;
      bool done = false;
      while (!done) {
        // LOOK words at a time (independent loads), then taken in
        // order: a prefix ends the walk, a count is added, a word not yet
        // published stops this step
        unsigned long long w[LOOK];
#pragma unroll
        for (uint32_t i = 0; i < LOOK; i++)
          w[i] = i <= j ? __hip_atomic_load(&status[static_cast<size_t>(j - i) * kDigits + tid], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT)
                        : 0ull;
        bool stalled = false;
#pragma unroll
        for (uint32_t i = 0; i < LOOK; i++) {
          if (done || stalled) continue;
          const uint32_t tag = static_cast<uint32_t>(w[i] >> 32);
          if (tag == tp) {
            excl += static_cast<uint32_t>(w[i]);
            done = true;
          } else if (tag == ta && j > 0) {  // tile 0 publishes a prefix
            excl += static_cast<uint32_t>(w[i]);
            j--;
          } else {
            stalled = true;
          }
        }
        if (done || !stalled) continue;
        if (++spins > kLookbackSpins) {
          *fail = 1;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      __hip_atomic_store(&status[static_cast<size_t>(tile) * kDigits + tid], pack_status(tp, excl + run),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    L.goff[tid] = gstart[tid] + excl;
  }
  __syncthreads();
  // write out: each digit's keys form a contiguous run of the output
  uint32_t g[kPassPer];
#pragma unroll
  for (int r = 0; r < kPassPer; r++) {
    const uint32_t i = r * kPassBlock + tid;
    if (in_tile(i)) {
      const K key = L.sbuf[i];
      const uint32_t d = digit_of(key, shift);
      g[r] = L.goff[d] + (i - L.dstart[d]);
      kout[g[r]] = key;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPassPer; r++)
    if (in_tile(wbase + r * kWave + lane)) L.vbuf[rank[r]] = v[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPassPer; r++) {
    const uint32_t i = r * kPassBlock + tid;
    if (in_tile(i)) vout[g[r]] = L.vbuf[i];
  }
}

// One digit pass: tiles in counter order, look-back over the published
// per-digit counts of earlier tiles, then a stable scatter.
// Six waves per SIMD: three workgroups per CU for 32-bit keys and values (LDS
// bounds 64-bit keys or values to two, four waves per SIMD).
// The first pass that runs reads `first`; the passes alternate between the
// scratch and the output so that the last one writes the output.
template <typename K, typename V, uint32_t LOOK, int PER, typename Src>
__global__ __launch_bounds__(kPassBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(V) == 8 ? 4 : 6))) void k_sort_pass(
    Src first, K* __restrict__ kout, V* __restrict__ vout, K* __restrict__ kx, V* __restrict__ vx, uint32_t n,
    uint32_t pass, const uint32_t* __restrict__ order, uint32_t* __restrict__ tile_ctr,
    unsigned long long* __restrict__ status, const uint32_t* __restrict__ gstart, int* __restrict__ fail) {
  const uint32_t c = __builtin_amdgcn_readfirstlane(
      __hip_atomic_load(&order[pass], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  if (c == kNoPass) return;
  const uint32_t runs = __builtin_amdgcn_readfirstlane(
      __hip_atomic_load(&order[kMaxPasses], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  const bool to_out = ((runs - c) & 1u) != 0;
  K* kdst = to_out ? kout : kx;
  V* vdst = to_out ? vout : vx;
  Src src = first;
  if constexpr (std::is_same<Src, ArraySrc<K, V>>::value) {
    if (c > 0) src = Src{to_out ? kx : kout, to_out ? vx : vout};
  }
  constexpr uint32_t kSortTile = tile_keys(PER);
  __shared__ PassLds<K, V, PER> L;
  const uint32_t tid = threadIdx.x;
  if (tid == 0) L.tile = atomicAdd(&tile_ctr[pass], 1u);
  for (uint32_t i = tid; i < kPassWaves * kDigits; i += kPassBlock) {
    (&L.wcnt[0][0])[i] = 0u;
    (&L.peer[0][0])[i] = 0ull;
  }
  __syncthreads();
  const uint32_t tile = L.tile;
  if (tile >= n / kSortTile + (n % kSortTile != 0 ? 1u : 0u)) return;  // one tile per workgroup
  // 32-bit arithmetic: tile * kSortTile < n < 2^32. (A 64-bit minimum here
  // was lowered to a select on a stale SCC, giving full tiles past n.)
  const uint32_t rem = n - tile * kSortTile;
  const uint32_t valid = rem < kSortTile ? rem : kSortTile;
  if (valid == kSortTile)
    sort_tile<K, V, true, LOOK, PER>(L, src, kdst, vdst, tile, valid, pass, status, gstart, fail);
  else
    sort_tile<K, V, false, LOOK, PER>(L, src, kdst, vdst, tile, valid, pass, status, gstart, fail);
}

// One pass over n pairs.
template <typename K, typename V, typename Src>
void launch_pass(Src first, K* kout, V* vout, K* kx, V* vx, uint32_t n, uint32_t pass, const uint32_t* order,
                 uint32_t* ctr, unsigned long long* status, const uint32_t* hist, int* fail, hipStream_t s) {
  const dim3 grid(tiles_of(n)), block(kPassBlock);
  if (n <= kFewKeys)
    hipLaunchKernelGGL((k_sort_pass<K, V, kLookAheadFew, kPassPerFew, Src>), grid, block, 0, s, first, kout, vout, kx, vx,
                       n, pass, order, ctr, status, hist + pass * kDigits, fail);
  else
    hipLaunchKernelGGL((k_sort_pass<K, V, kLookAhead, kPassPerFull, Src>), grid, block, 0, s, first, kout, vout, kx, vx,
                       n, pass, order, ctr, status, hist + pass * kDigits, fail);
}

constexpr uint32_t kOrderWord = 32;  // of the 64 counter words: tile counters, a failure word, then the order

inline size_t align256(size_t b) { return (b + 255) & ~size_t{255}; }

template <typename K>
hipError_t radix_sort(void* tmp, size_t& tmp_bytes, const K* kin, K* kout, const uint32_t* vin, uint32_t* vout,
                      size_t n, hipStream_t s, int* fail) {
  constexpr uint32_t passes = sizeof(K) * 8 / kDigitBits;
  const size_t ntiles = tiles_of(n);
  const size_t need_keys = align256(n * sizeof(K));
  const size_t need_vals = align256(n * 4);
  // cleared once per sort: the status words, the tile counters and the
  // failure word, the digit totals
  const size_t status_bytes = std::max<size_t>(ntiles, 1) * kDigits * 8;
  const size_t ctr_bytes = 256;
  const size_t hist_bytes = passes * kDigits * 4;
  const size_t need_clear = align256(status_bytes + ctr_bytes + hist_bytes);
  const size_t need = need_keys + need_vals + need_clear;
  if (!tmp) {
    tmp_bytes = std::max<size_t>(need, 256);
    return hipSuccess;
  }
  if (tmp_bytes < need) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  if (n >= (1ull << 32)) return hipErrorInvalidValue;
  unsigned char* p = static_cast<unsigned char*>(tmp);
  K* kt = reinterpret_cast<K*>(p);
  uint32_t* vt = reinterpret_cast<uint32_t*>(p + need_keys);
  unsigned char* clr = p + need_keys + need_vals;
  auto* status = reinterpret_cast<unsigned long long*>(clr);
  uint32_t* ctr = reinterpret_cast<uint32_t*>(clr + status_bytes);
  uint32_t* hist = reinterpret_cast<uint32_t*>(clr + status_bytes + ctr_bytes);
  if (!fail) fail = reinterpret_cast<int*>(ctr + passes);
  const uint32_t n32 = static_cast<uint32_t>(n);
  const size_t clear_words = (status_bytes + ctr_bytes + hist_bytes) / 4;
  hipLaunchKernelGGL(k_fill_zero, dim3(static_cast<unsigned>((clear_words + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<uint32_t*>(clr), clear_words);
  const unsigned hblocks =
      static_cast<unsigned>(std::min<size_t>((n + kHistChunk - 1) / kHistChunk, kHistMaxBlocks));
  hipLaunchKernelGGL((k_sort_hist<K>), dim3(hblocks), dim3(kHistBlock), 0, s, kin, n32, hist);
  uint32_t* order = ctr + kOrderWord;
  hipLaunchKernelGGL(k_digit_starts, dim3(1), dim3(kStartsBlock), 0, s, hist, passes, n32, 0u, order);
  for (uint32_t pass = 0; pass < passes; pass++)
    launch_pass(ArraySrc<K, uint32_t>{kin, vin}, kout, vout, kt, vt, n32, pass, order, ctr, status, hist, fail, s);
  return hipGetLastError();
}

// ---- points by dim1, with 64-bit values (pst_internal.hpp) ----
//
// The first pass reads the points themselves, so no key arrays are written
// beforehand. 2^26 f32/u32 points on MI355X: 0.20 ms for the digit totals,
// 0.45 ms for the first pass and 0.43 ms for each later one (24 B moved per
// point, 3.7 TB/s; LDS holds two workgroups per CU): 1.95 ms where the two
// sorts of 32-bit values with their key and rank-scatter kernels took 4.2.

constexpr uint32_t kPointPasses = 4;

// Digit totals of the points' dim1 keys, and what the points allow: flags[0]
// a NaN dim or ID, flags[1] a value that its key does not give back (-0) or
// IDs that do not rise strictly with the index.
template <typename T, typename I>
__global__ __launch_bounds__(kHistBlock) void k_point_hist(const Point<T, I>* __restrict__ pts, uint32_t n,
                                                           uint32_t* __restrict__ hist, int* __restrict__ flags) {
  constexpr int P = kPointPasses;
  __shared__ uint32_t h[kSub][P][kDigits];
  const uint32_t tid = threadIdx.x;
  for (uint32_t i = tid; i < kSub * P * kDigits; i += kHistBlock) (&h[0][0][0])[i] = 0u;
  __syncthreads();
  uint32_t(*mine)[kDigits] = h[tid % kSub];
  bool bad = false, plain = true;
  auto lossless = [](auto v) {
    if constexpr (std::is_floating_point<decltype(v)>::value) return __builtin_bit_cast(uint32_t, v) != 0x80000000u;
    else return true;
  };
  for (uint64_t b = static_cast<uint64_t>(blockIdx.x) * kHistChunk; b < n;
       b += static_cast<uint64_t>(gridDim.x) * kHistChunk) {
#pragma unroll 4
    for (int e = 0; e < kHistPer; e++) {
      const uint64_t i = b + static_cast<uint64_t>(e) * kHistBlock + tid;
      const bool ok = i < n;
      uint32_t k = 0;
      if (ok) {
        const Point<T, I> p = pts[i];
        bad |= is_nan(p.dim1_val) || is_nan(p.dim2_val);
        plain &= lossless(p.dim1_val) && lossless(p.dim2_val);
        if constexpr (has_id_v<I>) {
          bad |= is_nan(p.id);
          plain &= lossless(p.id);
          if (i + 1 < n) plain &= ord_key(p.id) < ord_key(pts[i + 1].id);
        }
        k = ord_key(p.dim1_val);
#pragma unroll
        for (int q = 0; q < P - 1; q++) atomicAdd(&mine[q][digit_of(k, q * kDigitBits)], 1u);
      }
      const uint32_t d = digit_of(k, (P - 1) * kDigitBits);
      const uint64_t act = __ballot(ok);
      const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
      if (act == ~0ull && __ballot(d != d0) == 0ull) {
        if (tid % kWave == 0) atomicAdd(&h[0][P - 1][d0], static_cast<uint32_t>(kWave));
      } else if (ok) {
        atomicAdd(&mine[P - 1][d], 1u);
      }
    }
  }
  if (bad) flags[0] = 1;
  if (!plain) flags[1] = 1;
  __syncthreads();
  for (uint32_t i = tid; i < P * kDigits; i += kHistBlock) {
    uint32_t c = 0;
#pragma unroll
    for (int u = 0; u < kSub; u++) c += (&h[u][0][0])[i];
    if (c) atomicAdd(&hist[i], c);
  }
}

struct PointSortTmp {
  unsigned long long* status;
  uint32_t* ctr;
  uint32_t* hist;
  size_t words;  // from status on, cleared once per sort
};
PointSortTmp point_sort_tmp(void* tmp, size_t n) {
  const size_t ntiles = tiles_of(n);
  const size_t status_bytes = std::max<size_t>(ntiles, 1) * kDigits * 8;
  PointSortTmp t{};
  auto* p = static_cast<unsigned char*>(tmp);
  t.status = reinterpret_cast<unsigned long long*>(p);
  t.ctr = reinterpret_cast<uint32_t*>(p + status_bytes);
  t.hist = reinterpret_cast<uint32_t*>(p + status_bytes + 256);
  t.words = (status_bytes + 256 + kPointPasses * kDigits * 4) / 4;
  return t;
}

template <typename F>
hipError_t with_point(int dtype, int id_dtype, F&& f) {
  auto ids = [&](auto t) {
    switch (id_dtype) {
      case NO_ID: return f(t, NoId{});
      case F32: return f(t, float{});
      case I32: return f(t, int32_t{});
      case U32: return f(t, uint32_t{});
    }
    return hipErrorInvalidValue;
  };
  switch (dtype) {
    case F32: return ids(float{});
    case I32: return ids(int32_t{});
  }
  return hipErrorInvalidValue;
}

}  // namespace

bool point_sort_takes(int dtype, int id_dtype) {
  return (dtype == F32 || dtype == I32) && (id_dtype == NO_ID || id_dtype == F32 || id_dtype == I32 || id_dtype == U32);
}

size_t point_sort_tmp_bytes(size_t n) { return align256(point_sort_tmp(nullptr, n).words * 4); }

hipError_t point_sort_count(int dtype, int id_dtype, const void* pts_d, size_t n, void* tmp, int* flags,
                            hipStream_t s) {
  const PointSortTmp t = point_sort_tmp(tmp, n);
  hipLaunchKernelGGL(k_fill_zero, dim3(static_cast<unsigned>((t.words + 255) / 256)), dim3(256), 0, s,
                     reinterpret_cast<uint32_t*>(t.status), t.words);
  const unsigned blocks = static_cast<unsigned>(std::min<size_t>((n + kHistChunk - 1) / kHistChunk, kHistMaxBlocks));
  return with_point(dtype, id_dtype, [&](auto tv, auto iv) {
    using Pt = Point<decltype(tv), decltype(iv)>;
    hipLaunchKernelGGL((k_point_hist<decltype(tv), decltype(iv)>), dim3(blocks), dim3(kHistBlock), 0, s,
                       static_cast<const Pt*>(pts_d), static_cast<uint32_t>(n), t.hist, flags);
    return hipGetLastError();
  });
}

hipError_t point_sort_passes(int dtype, int id_dtype, const void* pts_d, size_t n, void* tmp, uint32_t* key_x,
                             uint64_t* val_x, uint32_t* key_out, uint64_t* val_out, int* fail, hipStream_t s) {
  const PointSortTmp t = point_sort_tmp(tmp, n);
  const uint32_t n32 = static_cast<uint32_t>(n);
  uint32_t* order = t.ctr + kOrderWord;
  hipLaunchKernelGGL(k_digit_starts, dim3(1), dim3(kStartsBlock), 0, s, t.hist, kPointPasses, n32, 1u, order);
  const hipError_t e = with_point(dtype, id_dtype, [&](auto tv, auto iv) {
    using Src = PointSrc<decltype(tv), decltype(iv)>;
    using Pt = Point<decltype(tv), decltype(iv)>;
    launch_pass(Src{static_cast<const Pt*>(pts_d), 0u}, key_out, val_out, key_x, val_x, n32, 0u, order, t.ctr, t.status,
                t.hist, fail, s);
    return hipGetLastError();
  });
  for (uint32_t pass = 1; pass < kPointPasses && e == hipSuccess; pass++)
    launch_pass(ArraySrc<uint32_t, uint64_t>{nullptr, nullptr}, key_out, val_out, key_x, val_x, n32, pass, order, t.ctr,
                t.status, t.hist, fail, s);
  if (e == hipSuccess) return hipGetLastError();
  return e;
}

hipError_t radix_sort_u32(void* tmp, size_t& tmp_bytes, const uint32_t* kin, uint32_t* kout, const uint32_t* vin,
                          uint32_t* vout, size_t n, hipStream_t s, int* fail) {
  return radix_sort<uint32_t>(tmp, tmp_bytes, kin, kout, vin, vout, n, s, fail);
}

hipError_t radix_sort_u64(void* tmp, size_t& tmp_bytes, const uint64_t* kin, uint64_t* kout, const uint32_t* vin,
                          uint32_t* vout, size_t n, hipStream_t s, int* fail) {
  return radix_sort<uint64_t>(tmp, tmp_bytes, kin, kout, vin, vout, n, s, fail);
}

}  // namespace pst
