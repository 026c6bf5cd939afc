// Level index of one deep tree, and the batched searches that use it.
//
// For every depth t of the tree (t = 0 .. H-1, H = bit length of n) the
// index holds the points of all subtrees rooted at depth t, subtree by
// subtree in position order, each subtree's points sorted by dim2
// descending:
//   key[t * ns + k] = ~ord_key(dim2)   (ascending along a subtree's run)
//   id [t * ns + k] = the point's ID
// (level stride ns = n rounded up to 64, so every level starts aligned).
// The run of level-t position j starts at level_start(M, t, j) and holds
// level_size(M, t, j) points (M = n + 1, the closed-form tree shape).
//
// Why: a walk that reaches a subtree in REPORT_ABOVE state (both dim1
// bounds closed for it) reports exactly the subtree's points with
// dim2 >= min_dim2 (heap order: a node's dim2 is at least its
// descendants'), i.e. a prefix of the subtree's run, found by one binary
// search and copied as one contiguous range. What remains of the walk are
// the at most two paths on which a dim1 bound is still open, at most two
// nodes per level. A batch then costs a few dozen node visits and binary
// searches per query and one streaming copy of 4 bytes read + 4 bytes
// written per reported 4-byte ID, instead of a node visit per ID.
//
// Equal dim2 values keep breadth-first slot order inside a run, so a
// subtree root (the smallest slot of its subtree, with the largest dim2)
// is the first element of its run: a path node's own report is the
// one-element range at the front of its run.
//
// Construction: level 0 is one stable radix sort of all points by key (the
// input in slot order, last-level slots in bit-reversed position order);
// level t+1 is the stable partition of every level-t run into the runs of
// the root's left and right children (the root itself dropped), and level
// t+2 that of level t+1. One pass over level t writes both (the last level of
// an odd number takes a pass of its own). A point's destination is its child
// run's closed-form start plus its rank among the points of its run going the
// same way, from a global prefix count of the points of each way (per
// 4096-point tile, then scanned) less the closed-form count of same-way points
// in earlier runs.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pst_internal.hpp"

namespace pst {
namespace {

constexpr int kLvBlock = 256;
constexpr int kLvPer = 16;
constexpr uint32_t kLvTile = kLvBlock * kLvPer;  // points per partition tile
constexpr uint32_t kTaskCap = 128;               // ranges per query: <= 4 per level, <= 31 levels
constexpr uint32_t kFewQueries = 64;             // write plans of up to this many queries probe wider
// Copy chunks and workgroups. Copies spend their time moving between queries
// and ranges, where the hardware's own balancing of one chunk per workgroup
// hides each other's waits: 64 workgroups per CU and chunks of 8192 IDs. Small
// batches are cut into about eight chunks per CU, at least 1024 IDs each (one
// query of 1.5M IDs 33 us in chunks of 32768, which leave most CUs idle, now
// 11). us of write calls on MI355X with three workgroups per CU and chunks of
// 32768 / 64 and 8192 (2^26 points): 32768 queries of 8192 IDs 970 / 753, 2048
// of 65,636 299 / 231, 512 of 264,712 265 / 218, 256 of 1.0M 426 / 367, 1024
// mixed ones of 1.8M 2250 / 2140. 64 bytes of loads in flight per lane: with
// 256 the registers held the CU to half the waves (2785 instead of 2681 us on
// the last). The IDs are stored as streaming (2687 -> 2480 us there); loads
// stay ordinary, since queries share ranges (3154 us with both).
constexpr uint64_t kMinChunk = 1024, kMaxChunk = 8192;
constexpr uint64_t kChunkSpread = 2048;
constexpr uint64_t kChunkCap = 1u << 20;  // chunk table entries
// Up to 16 queries rarely fill more than eight workgroups per CU, and the idle
// ones of 64 cost 2 to 4 us: 8 / 64 per CU take 42 / 46 us for 8 queries of
// 335,000 IDs, 47 / 49 for 16, 48 / 48 for 24, 54 / 55 for 32, 73 / 67 for 64.
constexpr uint32_t kCopyPerCu = 64, kCopyPerCuFew = 8;
constexpr uint32_t kFewCopies = 16;
constexpr int kCopyBlock = 256;
constexpr int kCopyBytes = 64;  // bytes of loads in flight per lane in the copy
constexpr uint32_t kFlat = 4096;  // positions per flat pass of the copy (16 per lane)

template <typename T>
using key_of = decltype(ord_key(T{}));

// The kLvPer consecutive elements from a[base] (zeros past nt): aligned
// 16-byte loads when all are in range (base is a multiple of kLvPer and
// every level and slot array starts 256-byte aligned, level_stride).
template <typename V>
__device__ inline void load_run(const V* __restrict__ a, uint32_t base, uint32_t nt, V (&v)[kLvPer]) {
  if (base + kLvPer <= nt) {
    const uint4* q = reinterpret_cast<const uint4*>(a + base);
    constexpr int kVec = sizeof(V) * kLvPer / 16;
    constexpr int kPer = 16 / sizeof(V);
#pragma unroll
    for (int w = 0; w < kVec; w++) {
      const uint4 x = q[w];
      __builtin_memcpy(&v[w * kPer], &x, 16);
    }
  } else {
#pragma unroll
    for (int u = 0; u < kLvPer; u++) v[u] = base + u < nt ? a[base + u] : V{};
  }
}

// Points of level-(t+1) positions 2j'' + side, j'' < j: the same-way points
// of the level-t runs before run j.
__host__ __device__ inline uint64_t side_before(uint64_t M, uint32_t t, uint32_t j, uint32_t side) {
  const uint64_t base = (M >> (t + 1)) - 1;
  const uint64_t r1 = M & ((2ull << t) - 1ull);
  const uint64_t off = static_cast<uint64_t>(side) << t;
  const uint64_t r = r1 > off ? r1 - off : 0;
  return static_cast<uint64_t>(j) * base + brev_below(t, j, r);
}

// Slot of input element e of the level-0 sort: every slot above the last
// level in order, then the last level's occupied positions (those whose
// bit reversal is below the count) in bit-reversed order.
__host__ __device__ inline uint32_t input_slot(uint32_t e, uint32_t H) {
  const uint32_t F = (1u << (H - 1)) - 1u;
  return e < F ? e : F + brev_bits(e - F, H - 1);
}

template <typename T, typename IS>
__global__ __launch_bounds__(kLvBlock) void k_lv_keys(const Node<T, IS>* __restrict__ nodes, uint32_t n, uint32_t H,
                                                      key_of<T>* __restrict__ keys, uint32_t* __restrict__ slots) {
  const uint32_t e = blockIdx.x * kLvBlock + threadIdx.x;
  if (e >= n) return;
  const uint32_t s = input_slot(e, H);
  keys[e] = ~ord_key(nodes[s].dim2);
  slots[e] = s;
}

template <typename IS>
__global__ __launch_bounds__(kLvBlock) void k_lv_ids0(const IS* __restrict__ ids, const uint32_t* __restrict__ slots,
                                                      uint32_t n, IS* __restrict__ out) {
  const uint32_t e = blockIdx.x * kLvBlock + threadIdx.x;
  if (e >= n) return;
  out[e] = ids[slots[e]];
}

// Direction of the level-t point in slot s: 0 left, 1 right, 2 the root of
// its run (dropped).
__device__ inline uint32_t lv_side(uint32_t s, uint32_t t) {
  const uint32_t d = depth_of(s);
  if (d == t) return 2u;
  return ((s + 1u) >> (d - t - 1u)) & 1u;
}

// Per tile: left-going count (low 32 bits) and right-going count (high).
__global__ __launch_bounds__(kLvBlock) void k_lv_tile_counts(const uint32_t* __restrict__ slots, uint32_t nt,
                                                             uint32_t t, unsigned long long* __restrict__ agg) {
  __shared__ unsigned long long wsum[kLvBlock / kWave];
  const uint32_t base = blockIdx.x * kLvTile + threadIdx.x * kLvPer;
  uint32_t sl[kLvPer];
  load_run(slots, base, nt, sl);
  unsigned long long c = 0;
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    if (base + u < nt) {
      const uint32_t sd = lv_side(sl[u], t);
      c += sd == 0 ? 1ull : (sd == 1 ? (1ull << 32) : 0ull);
    }
  }
  for (int o = kWave / 2; o > 0; o >>= 1) c += __shfl_xor(c, o, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) wsum[threadIdx.x / kWave] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long s = 0;
    for (int w = 0; w < kLvBlock / kWave; w++) s += wsum[w];
    agg[blockIdx.x] = s;
  }
}

// Level t -> t+1: every point but its run's root moves to its child run.
// Phase 1 (a thread per 16 consecutive points): each point's destination,
// into LDS. Phase 2 (a thread per point, 256 consecutive points per pass):
// the moves, so that a wave's stores fall in at most a few contiguous
// stretches of the child runs and leave as whole lines.
constexpr uint32_t kDstPad = kLvPer + 1;  // LDS row of a thread's 16 destinations, padded against bank conflicts
template <typename K, typename IS>
__global__ __launch_bounds__(kLvBlock) void k_lv_scatter(const uint32_t* __restrict__ slots_in,
                                                         uint32_t* __restrict__ slots_out,
                                                         const K* __restrict__ key_in, K* __restrict__ key_out,
                                                         const IS* __restrict__ id_in, IS* __restrict__ id_out,
                                                         const unsigned long long* __restrict__ tile_pre,
                                                         uint32_t nt, uint32_t t, uint64_t M) {
  __shared__ unsigned long long wsum[kLvBlock / kWave];
  __shared__ uint32_t s_dst[kLvBlock * kDstPad];
  const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const uint32_t tile = blockIdx.x * kLvTile;
  const uint32_t base = tile + tid * kLvPer;
  uint32_t s[kLvPer];
  load_run(slots_in, base, nt, s);
  unsigned long long loc = 0;
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    if (base + u < nt) {
      const uint32_t sd = lv_side(s[u], t);
      loc += sd == 0 ? 1ull : (sd == 1 ? (1ull << 32) : 0ull);
    }
  }
  unsigned long long incl = loc;
  for (int o = 1; o < kWave; o <<= 1) {
    const unsigned long long y = __shfl_up(incl, o, kWave);
    if (static_cast<int>(lane) >= o) incl += y;
  }
  if (lane == kWave - 1) wsum[wave] = incl;
  __syncthreads();
  unsigned long long run = tile_pre[blockIdx.x] + incl - loc;
  for (uint32_t w = 0; w < wave; w++) run += wsum[w];
  // A thread's points lie in runs cj, cj + 1, ... (every level-t run
  // holds at least its root), so the closed-form counts of the first run
  // are advanced by the child run sizes from then on.
  uint32_t cj = 0;
  uint64_t cl = 0, cr = 0;
  bool have = false;
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    uint32_t dst = ~0u;  // the run's root (dropped) or past the level
    if (base + u < nt) {
      const uint32_t d = depth_of(s[u]);
      const uint32_t j = ((s[u] + 1u) >> (d - t)) - (1u << t);
      if (!have) {
        cj = j;
        cl = side_before(M, t, j, 0);
        cr = side_before(M, t, j, 1);
        have = true;
      }
      while (cj < j) {
        cl += static_cast<uint64_t>(level_size(M, t + 1, 2 * cj));
        cr += static_cast<uint64_t>(level_size(M, t + 1, 2 * cj + 1));
        cj++;
      }
      if (d != t) {
        const uint32_t sd = ((s[u] + 1u) >> (d - t - 1u)) & 1u;
        const uint64_t start = sd == 0 ? cl + cr : cl + cr + static_cast<uint64_t>(level_size(M, t + 1, 2 * cj));
        const uint64_t rank = sd == 0 ? (run & 0xffffffffull) - cl : (run >> 32) - cr;
        dst = static_cast<uint32_t>(start + rank);
        run += sd == 0 ? 1ull : (1ull << 32);
      }
    }
    s_dst[tid * kDstPad + u] = dst;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    const uint32_t r = u * kLvBlock + tid;  // point within the tile
    const uint32_t p = tile + r;
    const uint32_t dst = s_dst[(r / kLvPer) * kDstPad + r % kLvPer];
    if (p < nt && dst != ~0u) {
      key_out[dst] = key_in[p];
      id_out[dst] = id_in[p];
      slots_out[dst] = slots_in[p];
    }
  }
}

// ---------------------------------------------------------------------------
// Two levels at a time: level t's points go to level t + 1 (a child's run) and
// to level t + 2 (a grandchild's) from one read of their keys, IDs and slots;
// level t + 1 needs no slots of its own. A point's class is its two turns
// below level t (first turn high). In a run, the first point is the root, and
// among the points of one side the child's root comes first, so with the
// counts of the four classes before the point and before its run
//   level t + 2: run start + classes before its own + rank in its class,
//   level t + 1: run start + 1 + ranks in its side's two classes (0 for the
//                child's root itself).
// The runs before run j have dropped j roots by level t + 1 and 3j by level
// t + 2, so the starts there follow from the run's start at level t; that, and
// the class counts before it, are carried along the tile from root to root
// (closed form for the run that reaches into the tile from the left). For
// levels whose grandchild runs all exist or are empty: M >> (t + 2) >= 1.
//
// Bound by HBM: 36 B per point and two levels (56 with a pass per level). The
// moves hold keys and IDs in registers between the two levels, so that one
// LDS buffer of destinations serves both (with two, 12 waves per CU: 0.61
// ms). MI355X, 2^26 f32/u32 points: 0.52 ms per pair of levels after 0.08 ms of
// counts (4.2 TB/s), where single steps took 0.65 and 0.15.
// ---------------------------------------------------------------------------
__device__ inline uint32_t lv_class(uint32_t s, uint32_t t) {  // 4: the root or a child's root
  const uint32_t d = depth_of(s);
  return d < t + 2 ? 4u : ((s + 1u) >> (d - t - 2u)) & 3u;
}
// Class counts: classes 0 and 1 in the low and high half of a, 2 and 3 of b.
struct Counts4 {
  unsigned long long a, b;
  __device__ void add(uint32_t c) {
    const unsigned long long one = 1ull << (32 * (c & 1u));
    a += c < 2 ? one : 0ull;
    b += (c >> 1) == 1 ? one : 0ull;
  }
  __device__ uint32_t get(uint32_t c) const {
    const unsigned long long w = c < 2 ? a : b;
    return static_cast<uint32_t>((c & 1u) ? w >> 32 : w);
  }
};

// agg[tile], agg[stride + tile]: the tile's class counts.
__global__ __launch_bounds__(kLvBlock) void k_lv_tile_counts2(const uint32_t* __restrict__ slots, uint32_t nt,
                                                              uint32_t t, unsigned long long* __restrict__ agg,
                                                              uint32_t stride) {
  __shared__ Counts4 wsum[kLvBlock / kWave];
  const uint32_t base = blockIdx.x * kLvTile + threadIdx.x * kLvPer;
  uint32_t sl[kLvPer];
  load_run(slots, base, nt, sl);
  Counts4 c{0, 0};
#pragma unroll
  for (int u = 0; u < kLvPer; u++)
    if (base + u < nt) c.add(lv_class(sl[u], t));
  for (int o = kWave / 2; o > 0; o >>= 1) {
    c.a += __shfl_xor(c.a, o, kWave);
    c.b += __shfl_xor(c.b, o, kWave);
  }
  if ((threadIdx.x & (kWave - 1)) == 0) wsum[threadIdx.x / kWave] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    Counts4 s{0, 0};
    for (int w = 0; w < kLvBlock / kWave; w++) s.a += wsum[w].a, s.b += wsum[w].b;
    agg[blockIdx.x] = s.a;
    agg[stride + blockIdx.x] = s.b;
  }
}

template <typename K, typename IS>
__global__ __launch_bounds__(kLvBlock) void k_lv_scatter2(const uint32_t* __restrict__ slots_in,
                                                          uint32_t* __restrict__ slots_out,
                                                          const K* __restrict__ key_in, K* __restrict__ key1,
                                                          K* __restrict__ key2, const IS* __restrict__ id_in,
                                                          IS* __restrict__ id1, IS* __restrict__ id2,
                                                          const unsigned long long* __restrict__ tile_pre,
                                                          uint32_t stride, uint32_t nt, uint32_t t, uint64_t M) {
  constexpr int kWaves = kLvBlock / kWave;
  __shared__ Counts4 wsum[kWaves];
  __shared__ uint64_t wroots[kWaves];          // per wave: threads whose points hold a root
  __shared__ Counts4 s_at[kLvBlock + 1];       // the thread's last root: class counts before it,
  __shared__ uint32_t s_pos[kLvBlock + 1];     // its position (entry kLvBlock: the run that enters the tile)
  __shared__ uint32_t s_dst[kLvBlock * kDstPad];  // level t + 1, then t + 2
  const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const uint32_t tile = blockIdx.x * kLvTile;
  const uint32_t base = tile + tid * kLvPer;
  uint32_t s[kLvPer];
  load_run(slots_in, base, nt, s);
  Counts4 loc{0, 0};
#pragma unroll
  for (int u = 0; u < kLvPer; u++)
    if (base + u < nt) loc.add(lv_class(s[u], t));
  Counts4 inc = loc;
  for (int o = 1; o < kWave; o <<= 1) {
    const unsigned long long ya = __shfl_up(inc.a, o, kWave), yb = __shfl_up(inc.b, o, kWave);
    if (static_cast<int>(lane) >= o) inc.a += ya, inc.b += yb;
  }
  if (lane == kWave - 1) wsum[wave] = inc;
  if (tid == 0) {  // the run that holds the tile's first point
    const uint32_t d = depth_of(s[0]);
    const uint32_t j = ((s[0] + 1u) >> (d - t)) - (1u << t);
    s_pos[kLvBlock] = static_cast<uint32_t>(level_start(M, t, j));
    const uint64_t size = (M >> (t + 2)) - 1;
    const uint64_t r2 = M & ((4ull << t) - 1ull);
    uint32_t c[4];
    for (uint32_t k = 0; k < 4; k++) {
      // points of level-(t+2) positions 4j' + k, j' < j
      const uint64_t off = static_cast<uint64_t>(brev_bits(k, 2)) << t;
      c[k] = static_cast<uint32_t>(j * size + brev_below(t, j, r2 > off ? r2 - off : 0));
    }
    s_at[kLvBlock] = Counts4{c[0] | (static_cast<unsigned long long>(c[1]) << 32),
                             c[2] | (static_cast<unsigned long long>(c[3]) << 32)};
  }
  __syncthreads();
  Counts4 run{tile_pre[blockIdx.x] + inc.a - loc.a, tile_pre[stride + blockIdx.x] + inc.b - loc.b};
  for (uint32_t w = 0; w < wave; w++) run.a += wsum[w].a, run.b += wsum[w].b;
  // the thread's last root
  {
    Counts4 c = run;
    bool has = false;
#pragma unroll
    for (int u = 0; u < kLvPer; u++) {
      if (base + u < nt) {
        if (depth_of(s[u]) == t) {
          has = true;
          s_at[tid] = c;
          s_pos[tid] = base + u;
        }
        c.add(lv_class(s[u], t));
      }
    }
    const uint64_t b = __ballot(has);
    if (lane == 0) wroots[wave] = b;
  }
  __syncthreads();
  // the run the thread's first point lies in: the last root before it
  uint32_t from = kLvBlock;
  {
    uint64_t b = wroots[wave] & ((1ull << lane) - 1ull);
    uint32_t w = wave;
    while (!b && w > 0) b = wroots[--w];
    if (b) from = w * kWave + 63u - static_cast<uint32_t>(__clzll(static_cast<long long>(b)));
  }
  Counts4 at = s_at[from];
  uint32_t pos = s_pos[from];
  uint32_t cj = ~0u, s1 = 0, s2 = 0, left1 = 0, g[3] = {0, 0, 0};
  uint32_t dst2[kLvPer];
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    uint32_t d1 = ~0u, d2 = ~0u;
    if (base + u < nt) {
      const uint32_t d = depth_of(s[u]);
      const uint32_t j = ((s[u] + 1u) >> (d - t)) - (1u << t);
      if (d == t) {
        at = run;
        pos = base + u;
      }
      if (j != cj) {
        cj = j;
        s1 = pos - j;
        s2 = pos - 3 * j;
        left1 = static_cast<uint32_t>(level_size(M, t + 1, 2 * j));
        for (uint32_t k = 0; k < 3; k++) g[k] = static_cast<uint32_t>(level_size(M, t + 2, 4 * j + k));
      }
      if (d == t + 1) {
        d1 = s1 + (((s[u] + 1u) & 1u) ? left1 : 0u);
      } else if (d > t + 1) {
        const uint32_t c = ((s[u] + 1u) >> (d - t - 2u)) & 3u, side = c >> 1;
        const uint32_t r0 = run.get(2 * side) - at.get(2 * side), r1 = run.get(2 * side + 1) - at.get(2 * side + 1);
        d1 = s1 + (side ? left1 : 0u) + 1u + r0 + r1;
        d2 = s2 + (c > 0 ? g[0] : 0u) + (c > 1 ? g[1] : 0u) + (c > 2 ? g[2] : 0u) + ((c & 1u) ? r1 : r0);
        run.add(c);
      }
    }
    s_dst[tid * kDstPad + u] = d1;
    dst2[u] = d2;
  }
  // the moves, a thread per point, 256 consecutive points per pass
  K k[kLvPer];
  IS id[kLvPer];
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    const uint32_t p = tile + u * kLvBlock + tid;
    if (p < nt) {
      k[u] = key_in[p];
      id[u] = id_in[p];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    const uint32_t r = u * kLvBlock + tid;
    const uint32_t d = s_dst[(r / kLvPer) * kDstPad + r % kLvPer];
    if (tile + r < nt && d != ~0u) {
      key1[d] = k[u];
      id1[d] = id[u];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kLvPer; u++) s_dst[tid * kDstPad + u] = dst2[u];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kLvPer; u++) {
    const uint32_t r = u * kLvBlock + tid;
    const uint32_t d = s_dst[(r / kLvPer) * kDstPad + r % kLvPer];
    if (tile + r < nt && d != ~0u) {
      key2[d] = k[u];
      id2[d] = id[u];
      slots_out[d] = slots_in[tile + r];
    }
  }
}

// IDs per chunk of a batch that writes W IDs.
__host__ __device__ inline uint64_t chunk_len(uint64_t W) {
  uint64_t c = (W + kChunkCap - 1) / kChunkCap;
  c = (c + 255) & ~255ull;
  if (c >= kMaxChunk) return c;
  uint64_t f = (W / kChunkSpread + 255) & ~255ull;
  f = f < kMinChunk ? kMinChunk : (f > kMaxChunk ? kMaxChunk : f);
  return f > c ? f : c;
}

template <typename T, typename IS>
struct LvParams {
  const Node<T, IS>* nodes;
  const key_of<T>* key;
  const IS* id;
  uint64_t n;
  uint64_t ns;  // level stride
  uint32_t M, H;
  const Query<T>* queries;
  Query<T> single;
  uint32_t use_single;
  uint32_t keep;  // count mode: also keep the ranges (unclipped) for a later write from them
  uint32_t nq;
  unsigned long long* counts;  // count mode: per-query counts; write mode: per-query totals
  const unsigned long long* offsets;
  const unsigned long long* caps;
  unsigned long long cap_all;
  unsigned long long out_total;
  uint64_t* tsrc;   // per query, kTaskCap ranges: first index in the level arrays
  uint32_t* tpre;   // per query, kTaskCap: output position of each range (then the query's total)
  uint32_t* ntask;  // ranges per query
  unsigned long long* wq;  // IDs written per query
  unsigned long long* woff;  // one query (use_single, write mode): its work offsets, written by the plan
  uint32_t* chunk_task;      // and its chunk table
  unsigned long long* host;  // and its count, in pinned host memory (null: none)
};

// First index of the sorted run kk[0, len) whose key is above qk: a search
// with PROBES (3 or 7) loads in flight per step, which narrows the run 4 or 8
// times per memory round trip.
template <int PROBES, typename K>
__device__ inline uint32_t run_prefix(const K* __restrict__ kk, uint32_t len, K qk) {
  static_assert(PROBES == 3 || PROBES == 7, "quarters or eighths");
  constexpr uint32_t kParts = PROBES + 1;
  uint32_t lo = 0, hi = len;
  while (lo < hi) {
    const uint32_t w = hi - lo;
    uint32_t p[PROBES];
    K v[PROBES];
#pragma unroll
    for (int k = 0; k < PROBES; k++) {
      p[k] = lo + (w / kParts) * (k + 1) + ((w % kParts) * (k + 1)) / kParts;  // lo + floor(w (k + 1) / kParts) < hi
      v[k] = kk[p[k]];
    }
    uint32_t nlo = lo, nhi = hi;
#pragma unroll
    for (int k = 0; k < PROBES; k++)
      if (v[k] <= qk) nlo = p[k] + 1;
#pragma unroll
    for (int k = PROBES - 1; k >= 0; k--)
      if (!(v[k] <= qk)) nhi = p[k];
    lo = nlo;
    hi = nhi;
  }
  return lo;
}

// Chunks c0..c1-1 start in the lane's range: their table entries. All lanes
// take part in a range that starts many (one lane per range took 33 us for
// 56,000 chunks of 1024 queries on MI355X, this 3; in one query's plan 14).
__device__ inline void mark_chunks(uint32_t* __restrict__ chunk_task, uint32_t entry, uint32_t c0, uint32_t c1,
                                   uint32_t lane) {
  const bool many = c1 > c0 + 4;
  if (!many)
    for (uint32_t c = c0; c < c1; c++) chunk_task[c] = entry;
  uint64_t m = __ballot(many);
  while (m) {
    const int f = __builtin_ctzll(m);
    m &= m - 1;
    const uint32_t v = __shfl(entry, f, kWave), e = __shfl(c1, f, kWave);
    for (uint32_t c = __shfl(c0, f, kWave) + lane; c < e; c += kWave) chunk_task[c] = v;
  }
}

// One workgroup (one wave) per query: the open paths, then the REPORT_ABOVE
// subtrees' run searches, one lane per subtree.
//
// Bound by the chain of dependent loads, one per tree level and one per
// search step when taken singly. So the wave loads five levels of the (at
// most two) path nodes' subtrees at once, 31 nodes each on lanes 0-30 and
// 31-61, steps the paths down through the lanes' registers (a lane takes its
// state from its parent's lane), and starts again from the nodes reached;
// the closed-form starts of the ranges, a loop over the levels each, are left
// to the end, where every lane has a range of its own; and the searches keep
// several probes in flight. MI355X, 2^26 f32 points: one query 62 -> 20 us,
// 1024 queries 99 -> 27 us; 8192 queries on 2^25 i32 points 113 -> 41 us.
constexpr uint32_t kSpecLevels = 5;                      // levels loaded at once
constexpr uint32_t kSpecNodes = (1u << kSpecLevels) - 1;  // nodes per path
template <typename T, typename IS, bool W, int PROBES>
__global__ __launch_bounds__(kWave) void k_lv_plan(LvParams<T, IS> P) {
  using K = key_of<T>;
  __shared__ uint64_t s_src[kTaskCap];  // first: level << 33 | searched << 32 | position; then the source
  const uint32_t lane = threadIdx.x;
  const uint32_t q = blockIdx.x;
  const Query<T> Q = P.use_single ? P.single : P.queries[q];
  const Bounds<T> qb{Q.min_dim1, Q.max_dim1, Q.min_dim2};
  const BoundNum bn = bound_num<T, 1>(&qb);
  const uint64_t ns = P.ns;
  // the lane's place in its path's block
  const uint32_t blk = lane >= kSpecNodes ? 1u : 0u;
  const uint32_t r = lane - blk * kSpecNodes;
  const uint32_t rd = 31u - static_cast<uint32_t>(__builtin_clz(r + 1));  // depth in the block
  const bool in_block = lane < 2 * kSpecNodes;
  const int parent = static_cast<int>(blk * kSpecNodes + (r ? (r - 1) / 2 : 0));
  // path states: 4 valid, 2 upper bound open, 1 lower bound open
  uint32_t root[2] = {0, 0};
  uint32_t state[2] = {4u | lo_open(Q.kind) | (hi_open(Q.kind) << 1), 0u};
  uint32_t ntask = 0;
  for (uint32_t t = 0; t < P.H && (state[0] | state[1]); t += kSpecLevels) {
    const uint32_t rs = blk ? root[1] : root[0], rst = blk ? state[1] : state[0];
    const uint32_t depth = t + rd;
    const uint32_t slot = ((rs + 1) << rd) + r - (1u << rd);
    int32_t m = 0;
    if (in_block && rst && depth < P.H) m = subtree_size32(P.M, slot);
    const Node<T, IS> nd = P.nodes[m >= 1 ? slot : 0u];
    uint32_t st = r == 0 && m >= 1 ? rst : 0u;
    uint32_t kids = 0;  // open children: left state | right state << 3
#pragma unroll
    for (uint32_t d = 0; d < kSpecLevels; d++) {
      bool rep = false, ra = false;
      uint32_t side = 0;
      kids = 0;
      if (rd == d && st) {
        const StepOut o = node_step<T, 1>(nd.dim1, nd.dim2, nd.med, m, &qb, bn, 1u, st & 1u, (st >> 1) & 1u);
        rep = o.rep != 0;
        const uint32_t ol = o.ll | (o.hl << 1), orr = o.lr | (o.hr << 1);
        if (o.al) {
          if (ol) kids |= 4u | ol;
          else ra = true;
        }
        if (o.ar) {
          if (orr) kids |= (4u | orr) << 3;
          else {
            ra = true;
            side = 1;
          }
        }
      }
      // ranges in path order (left to right), a node's own point first
      const uint64_t b1 = __ballot(rep), b2 = __ballot(ra);
      uint32_t at = ntask + lanes_below(b1) + lanes_below(b2);
      const uint32_t j = slot + 1u - (1u << depth);
      if (rep) s_src[at++] = (static_cast<uint64_t>(depth) << 33) | j;
      if (ra) s_src[at] = (static_cast<uint64_t>(depth + 1) << 33) | (1ull << 32) | (2u * j + side);
      ntask += static_cast<uint32_t>(__popcll(b1) + __popcll(b2));
      if (d + 1 < kSpecLevels) {
        const uint32_t up = static_cast<uint32_t>(__shfl(static_cast<int>(kids), parent, kWave));
        if (rd == d + 1) st = m >= 1 ? ((r & 1u) ? up & 7u : up >> 3) : 0u;
      }
    }
    // the paths' nodes below the block, left to right (at most two)
    uint64_t bl = __ballot((kids & 7u) != 0), br = __ballot((kids >> 3) != 0);
    state[0] = state[1] = 0;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint64_t any = bl | br;
      if (any) {
        const int f = __builtin_ctzll(any);
        const uint64_t bit = 1ull << f;
        const bool left = (bl & bit) != 0;
        const uint32_t ps = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(slot), f));
        const uint32_t kd = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(kids), f));
        root[k] = 2 * ps + (left ? 1u : 2u);
        state[k] = left ? kd & 7u : kd >> 3;
        if (left) bl &= ~bit;
        else br &= ~bit;
      }
    }
  }
  __syncthreads();
  // each range's place in the level arrays and its length: one for a node's
  // own point, else the points of the subtree's run with key <= ~ord_key(min2)
  const K qk = ~ord_key(qb.min2);
  uint32_t cnt[2] = {0, 0};
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t i = lane + h * kWave;
    if (i < ntask) {
      const uint64_t e = s_src[i];
      const uint32_t t = static_cast<uint32_t>(e >> 33), j = static_cast<uint32_t>(e);
      const uint64_t src = static_cast<uint64_t>(t) * ns + static_cast<uint64_t>(level_start(P.M, t, j));
      s_src[i] = src;
      cnt[h] = (e >> 32) & 1u
                   ? run_prefix<PROBES>(P.key + src, static_cast<uint32_t>(level_size(P.M, t, j)), qk)
                   : 1u;
    }
  }
  // inclusive prefix over the ranges in order
  uint32_t inc0 = cnt[0], inc1 = cnt[1];
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t y0 = __shfl_up(inc0, o, kWave), y1 = __shfl_up(inc1, o, kWave);
    if (static_cast<int>(lane) >= o) {
      inc0 += y0;
      inc1 += y1;
    }
  }
  const uint32_t tot0 = __shfl(inc0, kWave - 1, kWave);
  inc1 += tot0;
  const uint32_t total = __shfl(inc1, kWave - 1, kWave);
  if (!W && !P.keep) {
    if (lane == 0) P.counts[q] = total;
  } else {
    unsigned long long clip = total;
    if constexpr (W) {
      const unsigned long long off = P.offsets ? P.offsets[q] : 0ull;
      const unsigned long long cap = P.caps ? P.caps[q] : P.cap_all;
      const unsigned long long room = off < P.out_total ? P.out_total - off : 0ull;
      if (cap < clip) clip = cap;
      if (room < clip) clip = room;
    }
    const uint32_t cw = static_cast<uint32_t>(clip);
    // keep the ranges that start before the clip point and hold IDs
    const uint32_t pre0 = inc0 - cnt[0], pre1 = inc1 - cnt[1];
    const bool k0 = lane < ntask && cnt[0] > 0 && pre0 < cw;
    const bool k1 = lane + kWave < ntask && cnt[1] > 0 && pre1 < cw;
    const uint64_t b0 = __ballot(k0), b1 = __ballot(k1);
    const uint32_t at0 = lanes_below(b0), at1 = static_cast<uint32_t>(__builtin_popcountll(b0)) + lanes_below(b1);
    const uint64_t qb0 = static_cast<uint64_t>(q) * kTaskCap;
    if (k0) {
      P.tsrc[qb0 + at0] = s_src[lane];
      P.tpre[qb0 + at0] = pre0;
    }
    if (k1) {
      P.tsrc[qb0 + at1] = s_src[lane + kWave];
      P.tpre[qb0 + at1] = pre1;
    }
    if (lane == 0) {
      const uint32_t nt = static_cast<uint32_t>(__builtin_popcountll(b0) + __builtin_popcountll(b1));
      P.tpre[qb0 + nt] = cw;
      P.ntask[q] = nt;
      if constexpr (W) P.wq[q] = clip;
      P.counts[q] = total;
    }
    if constexpr (W) {
      if (P.use_single) {
        // one query: its work offsets and chunk table directly (no scan or
        // marking launch); a kept range ends where the next one starts
        if (lane == 0) {
          P.woff[0] = 0;
          P.woff[1] = clip;
          if (P.host)
            __hip_atomic_store(P.host, static_cast<unsigned long long>(total), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        const uint32_t L = static_cast<uint32_t>(chunk_len(clip));
        auto mark = [&](bool keep, uint32_t at, uint32_t pre, uint32_t c) {
          const uint32_t end = keep ? (pre + c < cw ? pre + c : cw) : 0u;
          mark_chunks(P.chunk_task, at, keep ? (pre + L - 1) / L : 0u, (end + L - 1) / L, lane);
        };
        mark(k0, at0, pre0, cnt[0]);
        mark(k1, at1, pre1, cnt[1]);
      }
    }
  }
}

// Write step from ranges kept by a count pass: clip each query's ranges to
// its capacity and the output's size (a thread per query).
__global__ __launch_bounds__(kLvBlock) void k_lv_clip(uint32_t* __restrict__ tpre, uint32_t* __restrict__ ntask,
                                                      unsigned long long* __restrict__ wq,
                                                      unsigned long long* __restrict__ totals,
                                                      const unsigned long long* __restrict__ offsets,
                                                      const unsigned long long* __restrict__ caps,
                                                      unsigned long long cap_all, unsigned long long out_total,
                                                      uint32_t nq) {
  const uint32_t q = blockIdx.x * kLvBlock + threadIdx.x;
  if (q >= nq) return;
  const uint64_t qb = static_cast<uint64_t>(q) * kTaskCap;
  uint32_t nt = ntask[q];
  const uint32_t total = tpre[qb + nt];
  const unsigned long long off = offsets ? offsets[q] : 0ull;
  const unsigned long long cap = caps ? caps[q] : cap_all;
  const unsigned long long room = off < out_total ? out_total - off : 0ull;
  unsigned long long clip = total;
  if (cap < clip) clip = cap;
  if (room < clip) clip = room;
  if (clip < total) {
    while (nt > 0 && tpre[qb + nt - 1] >= clip) nt--;
    ntask[q] = nt;
    tpre[qb + nt] = static_cast<uint32_t>(clip);
  }
  wq[q] = clip;
  totals[q] = total;
}

// Chunk table: chunk c (IDs [c L, (c+1) L) of the batch's concatenated
// writes) starts in range i of query q: entry q << 7 | i.
__global__ __launch_bounds__(kLvBlock) void k_lv_mark(const unsigned long long* __restrict__ woff,
                                                      const uint32_t* __restrict__ tpre,
                                                      const uint32_t* __restrict__ ntask, uint32_t nq,
                                                      uint32_t* __restrict__ chunk_task) {
  // one wave per query, a lane per range
  const uint32_t q = blockIdx.x * (kLvBlock / kWave) + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (q >= nq) return;
  const uint32_t nt = ntask[q];
  const uint64_t L = chunk_len(woff[nq]);
  const uint64_t base = woff[q];
  const uint64_t qb = static_cast<uint64_t>(q) * kTaskCap;
  for (uint32_t i0 = 0; i0 < nt; i0 += kWave) {
    const uint32_t i = i0 + lane;
    uint32_t c0 = 0, c1 = 0;  // chunks that start in the lane's range (at most kChunkCap in all)
    if (i < nt) {
      c0 = static_cast<uint32_t>((base + tpre[qb + i] + L - 1) / L);
      c1 = static_cast<uint32_t>((base + tpre[qb + i + 1] + L - 1) / L);
    }
    mark_chunks(chunk_task, (q << 7) | i, c0, c1, lane);
  }
}

// All lanes of the workgroup copy len IDs, a multiple of the pass size,
// with kCopyBytes of loads in flight per lane (every load of a pass issued
// before its stores).
template <typename IS>
__device__ inline void copy_passes(const IS* __restrict__ src, IS* __restrict__ dst, uint64_t len, uint32_t tid) {
  constexpr int U = kCopyBytes / sizeof(IS);
  constexpr uint64_t kPass = static_cast<uint64_t>(kCopyBlock) * U;
  for (uint64_t k0 = 0; k0 < len; k0 += kPass) {
    IS v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = src[k0 + u * kCopyBlock + tid];
#pragma unroll
    for (int u = 0; u < U; u++) stream_store(&dst[k0 + u * kCopyBlock + tid], v[u]);
  }
}

// Streams the batch's ranges to the outputs, a chunk of IDs per workgroup
// pass. The current query's range table (output positions and sources) is
// staged in LDS. A range's whole passes are copied with all lanes on it;
// what is left of it, and the ranges after it in the same query and chunk,
// go in flat passes of kFlat positions where each lane finds its
// position's range in the table, so short ranges share a memory round
// trip.
template <typename IS>
__global__ __launch_bounds__(kCopyBlock) void k_lv_copy(const IS* __restrict__ ids, const uint64_t* __restrict__ tsrc,
                                                        const uint32_t* __restrict__ tpre,
                                                        const uint32_t* __restrict__ ntask,
                                                        const unsigned long long* __restrict__ woff,
                                                        const unsigned long long* __restrict__ offsets,
                                                        const uint32_t* __restrict__ chunk_task, uint32_t nq,
                                                        IS* __restrict__ out) {
  __shared__ uint32_t s_pre[kTaskCap + 1];
  __shared__ uint64_t s_src[kTaskCap];
  const uint64_t W = woff[nq];
  const uint64_t L = chunk_len(W);
  const uint64_t nch = (W + L - 1) / L;
  const uint32_t tid = threadIdx.x;
  for (uint64_t c = blockIdx.x; c < nch; c += gridDim.x) {
    const uint32_t e = chunk_task[c];
    uint32_t q = e >> 7, i = e & 127u;
    uint64_t x = c * L;
    const uint64_t x1 = x + L < W ? x + L : W;
    uint32_t staged = ~0u, nt = 0;
    uint64_t wbase = 0, obase = 0;
    while (x < x1) {
      if (q != staged) {
        __syncthreads();  // every lane is done with the previous table
        nt = ntask[q];
        wbase = woff[q];
        obase = offsets ? offsets[q] : 0ull;
        const uint64_t qb = static_cast<uint64_t>(q) * kTaskCap;
        if (tid <= nt) s_pre[tid] = tpre[qb + tid];
        if (tid < nt) s_src[tid] = tsrc[qb + tid];
        __syncthreads();
        staged = q;
      }
      if (i >= nt) {
        // the next query with IDs: the last q' with woff[q'] <= x
        uint32_t lo = q + 1, hi = nq - 1;
        while (lo < hi) {
          const uint32_t mid = (lo + hi + 1) >> 1;
          if (woff[mid] <= x) lo = mid;
          else hi = mid - 1;
        }
        if (lo > hi) break;
        q = lo;
        i = 0;
        continue;
      }
      const uint64_t a = wbase + s_pre[i], b = wbase + s_pre[i + 1];
      if (x < a || x >= b) break;  // not a range of this batch's plan
      const uint64_t hi = b < x1 ? b : x1;
      constexpr uint64_t kPass = static_cast<uint64_t>(kCopyBlock) * (kCopyBytes / sizeof(IS));
      const uint64_t bulk = ((hi - x) / kPass) * kPass;
      if (bulk) {
        copy_passes(ids + s_src[i] + (x - a), out + obase + (x - wbase), bulk, tid);
        x += bulk;
        if (x == b) i++;
        continue;
      }
      // a flat pass from x to the query's, the chunk's or the pass's end
      const uint64_t qend = wbase + s_pre[nt];
      uint64_t fend = x + kFlat;
      if (fend > qend) fend = qend;
      if (fend > x1) fend = x1;
      {
        constexpr int V = kFlat / kCopyBlock;
        IS v[V];
        uint32_t loc[V];
        uint32_t ii = i;
#pragma unroll
        for (int u = 0; u < V; u++) {
          const uint64_t pos = x + u * kCopyBlock + tid;
          loc[u] = static_cast<uint32_t>(pos - wbase);
          if (pos < fend) {
            while (s_pre[ii + 1] <= loc[u]) ii++;
            v[u] = ids[s_src[ii] + (loc[u] - s_pre[ii])];
          }
        }
#pragma unroll
        for (int u = 0; u < V; u++)
          if (x + u * kCopyBlock + tid < fend) stream_store(&out[obase + loc[u]], v[u]);
      }
      x = fend;
      while (i < nt && wbase + s_pre[i + 1] <= x) i++;
    }
  }
}

template <typename F>
Status lv_with_t(int dt, F&& f) {
  switch (dt) {
    case F32: return f(float{});
    case F64: return f(double{});
    case I32: return f(int32_t{});
    case I64: return f(int64_t{});
  }
  return Status{1, "Error: unsupported data type code " + std::to_string(dt)};
}
template <typename F>
Status lv_with_is(int idt, F&& f) {
  switch (idt) {
    case F32: case I32: case U32: return f(uint32_t{});
    case F64: case I64: case U64: return f(uint64_t{});
  }
  return Status{1, "Error: the level index needs a tree with IDs"};
}

uint32_t bit_length(uint64_t n) { return n ? 64u - static_cast<uint32_t>(__builtin_clzll(n)) : 0u; }

}  // namespace

size_t level_index_bytes(int dtype, int id_dtype, size_t n) {
  if (n == 0) return 0;
  const size_t per = dtype_size(dtype) + (id_dtype == F64 || id_dtype == I64 || id_dtype == U64 ? 8 : 4);
  return static_cast<size_t>(bit_length(n)) * level_stride(n) * per;
}

Status build_level_index(int dtype, int id_dtype, size_t n, const void* nodes_d, const void* ids_d, void* key_d,
                         void* id_d, hipStream_t s) {
  if (n == 0) return Status{};
  if (n >= (1ull << 31)) return Status{1, "Error: the level index holds trees of fewer than 2^31 points"};
  if (!ids_d) return Status{1, "Error: the level index needs a tree with IDs"};
  const uint32_t H = bit_length(n);
  const uint64_t M = n + 1;
  const size_t ns = level_stride(n);
  return lv_with_t(dtype, [&](auto tv) -> Status {
    using T = decltype(tv);
    using K = key_of<T>;
    return lv_with_is(id_dtype, [&](auto iv) -> Status {
      using IS = decltype(iv);
      K* key = static_cast<K*>(key_d);
      IS* id = static_cast<IS*>(id_d);
      const uint32_t n32 = static_cast<uint32_t>(n);
      const uint32_t ntiles = (n32 + kLvTile - 1) / kLvTile;
      K* kin = nullptr;
      uint32_t *sa = nullptr, *sb = nullptr;
      unsigned long long *agg = nullptr, *pre = nullptr;
      void* tmp = nullptr;
      size_t tmp_bytes = 0;
      hipError_t e = sizeof(K) == 4
                         ? radix_sort_u32(nullptr, tmp_bytes, nullptr, nullptr, nullptr, nullptr, n, s)
                         : radix_sort_u64(nullptr, tmp_bytes, nullptr, nullptr, nullptr, nullptr, n, s);
      // The slot arrays take the block that construction of a tree of this
      // size used and gave back. The sort of level 0 works in the key array's
      // deeper levels, which are written after it, where they hold it.
      const size_t slots = build_arena_bytes(dtype, id_dtype, n);
      const LevelSlots ls = level_slots(n);
      const bool inside = H >= 2 && ns * sizeof(K) * (H - 2) >= tmp_bytes && ls.bytes <= slots;
      uint32_t* slot_block = nullptr;
      void* sort_block = nullptr;
      if (e == hipSuccess) e = dev_alloc(&slot_block, std::max(slots, ls.bytes));
      if (e == hipSuccess) e = dev_alloc(&agg, 2 * (ntiles + 1) * 8ull);
      if (e == hipSuccess) e = dev_alloc(&pre, 2 * (ntiles + 2) * 8ull);
      const size_t kin_bytes = (n * sizeof(K) + 255) & ~size_t{255};
      if (e == hipSuccess && !inside) e = dev_alloc(&sort_block, kin_bytes + std::max<size_t>(tmp_bytes, 16));
      sa = slot_block;
      sb = slot_block + ls.second;
      kin = inside ? key + ns : static_cast<K*>(sort_block);
      tmp = inside ? static_cast<void*>(key + 2 * ns) : static_cast<unsigned char*>(sort_block) + kin_bytes;
      Status st = hip_status(e, "Error in allocating level index construction buffers");
      if (st.ok()) {
        const unsigned blocks = (n32 + kLvBlock - 1) / kLvBlock;
        const Node<T, IS>* nodes = static_cast<const Node<T, IS>*>(nodes_d);
        hipLaunchKernelGGL((k_lv_keys<T, IS>), dim3(blocks), dim3(kLvBlock), 0, s, nodes, n32, H, kin, sb);
        size_t tb = std::max<size_t>(tmp_bytes, 16);
        if constexpr (sizeof(K) == 4)
          e = radix_sort_u32(tmp, tb, kin, key, sb, sa, n, s);
        else
          e = radix_sort_u64(tmp, tb, kin, key, sb, sa, n, s);
        st = hip_status(e, "Error in sorting the level index");
      }
      if (st.ok()) {
        const unsigned blocks = (n32 + kLvBlock - 1) / kLvBlock;
        hipLaunchKernelGGL((k_lv_ids0<IS>), dim3(blocks), dim3(kLvBlock), 0, s, static_cast<const IS*>(ids_d), sa,
                           n32, id);
        for (uint32_t t = 0; t + 1 < H && st.ok(); t++) {
          const uint32_t nt = n32 - ((1u << t) - 1u);
          const uint32_t tiles = (nt + kLvTile - 1) / kLvTile;
          if ((M >> (t + 2)) >= 1 && t + 2 < H) {
            hipLaunchKernelGGL(k_lv_tile_counts2, dim3(tiles), dim3(kLvBlock), 0, s, sa, nt, t, agg, ntiles + 1);
            st = exclusive_scan(agg, pre, tiles, s, 2, ntiles + 1);
            if (!st.ok()) break;
            hipLaunchKernelGGL((k_lv_scatter2<K, IS>), dim3(tiles), dim3(kLvBlock), 0, s, sa, sb,
                               key + static_cast<size_t>(t) * ns, key + static_cast<size_t>(t + 1) * ns,
                               key + static_cast<size_t>(t + 2) * ns, id + static_cast<size_t>(t) * ns,
                               id + static_cast<size_t>(t + 1) * ns, id + static_cast<size_t>(t + 2) * ns, pre,
                               ntiles + 1, nt, t, M);
            std::swap(sa, sb);
            t++;
            continue;
          }
          hipLaunchKernelGGL(k_lv_tile_counts, dim3(tiles), dim3(kLvBlock), 0, s, sa, nt, t, agg);
          st = exclusive_scan(agg, pre, tiles, s);
          if (!st.ok()) break;
          hipLaunchKernelGGL((k_lv_scatter<K, IS>), dim3(tiles), dim3(kLvBlock), 0, s, sa, sb,
                             key + static_cast<size_t>(t) * ns, key + static_cast<size_t>(t + 1) * ns,
                             id + static_cast<size_t>(t) * ns, id + static_cast<size_t>(t + 1) * ns, pre, nt, t, M);
          std::swap(sa, sb);
        }
        if (st.ok()) st = hip_status(hipGetLastError(), "Error in launching level index construction");
        if (st.ok()) st = hip_status(hipStreamSynchronize(s), "Error in building the level index");
      }
      for (void* p : {static_cast<void*>(slot_block), sort_block, static_cast<void*>(agg), static_cast<void*>(pre)})
        (void)(st.ok() ? dev_free_idle(p) : dev_free(p));
      return st;
    });
  });
}

Status level_scratch_reserve(LevelScratch& sc, size_t nq) {
  if (sc.cap >= nq && sc.chunk_task) return Status{};
  if (sc.external) return Status{1, "Error: the batch holds more queries than the search buffers"};
  if (sc.pinned) return Status{1, kPinnedScratchMsg};
  level_scratch_release(sc);
  const size_t cap = std::max<size_t>(nq, 64);
  hipError_t e = dev_alloc(&sc.tsrc, cap * kTaskCap * 8);
  if (e == hipSuccess) e = dev_alloc(&sc.tpre, cap * kTaskCap * 4);
  if (e == hipSuccess) e = dev_alloc(&sc.ntask, cap * 4);
  if (e == hipSuccess) e = dev_alloc(&sc.wq, cap * 8);
  if (e == hipSuccess) e = dev_alloc(&sc.woff, (cap + 1) * 8);
  if (e == hipSuccess) e = dev_alloc(&sc.chunk_task, kChunkCap * 4);
  if (e != hipSuccess) {
    level_scratch_release(sc);
    return hip_status(e, "Error in allocating level search buffers");
  }
  sc.cap = cap;
  return Status{};
}

void level_scratch_release(LevelScratch& sc, bool idle) {
  if (sc.external) {
    sc = LevelScratch{};
    return;
  }
  for (void* p : {static_cast<void*>(sc.tsrc), static_cast<void*>(sc.tpre), static_cast<void*>(sc.ntask),
                  static_cast<void*>(sc.wq), static_cast<void*>(sc.woff), static_cast<void*>(sc.chunk_task)})
    (void)(idle ? dev_free_idle(p) : dev_free(p));
  sc = LevelScratch{};
}

Status level_search(const SearchArgs& a, const void* key_d, const void* id_d, LevelScratch& sc, hipStream_t s,
                    int plan) {
  if (a.nq == 0 || a.n == 0) return Status{};
  if (a.mode == 1 && a.ret_point) return Status{1, "Error: the level index returns IDs only"};
  if (plan == 2 && (a.mode != 1 || sc.cap < a.nq || !sc.tsrc))
    return Status{1, "Error: no kept ranges for this batch"};
  if (a.mode == 1 || plan == 1) {
    Status st = level_scratch_reserve(sc, a.nq);
    if (!st.ok()) return st;
  }
  return lv_with_t(a.dtype, [&](auto tv) -> Status {
    using T = decltype(tv);
    using K = key_of<T>;
    return lv_with_is(a.id_dtype, [&](auto iv) -> Status {
      using IS = decltype(iv);
      LvParams<T, IS> P{};
      P.nodes = static_cast<const Node<T, IS>*>(a.nodes);
      P.key = static_cast<const K*>(key_d);
      P.id = static_cast<const IS*>(id_d);
      P.n = a.n;
      P.ns = level_stride(a.n);
      P.M = static_cast<uint32_t>(a.n + 1);
      P.H = bit_length(a.n);
      P.queries = static_cast<const Query<T>*>(a.queries);
      if (a.single_query) {
        P.single = *static_cast<const Query<T>*>(a.single_query);
        P.use_single = 1;
        P.host = a.host;
      }
      P.nq = static_cast<uint32_t>(a.nq);
      P.counts = a.counts;
      P.offsets = a.offsets;
      P.caps = a.caps;
      P.cap_all = a.cap_all;
      P.out_total = a.out_total;
      P.tsrc = sc.tsrc;
      P.tpre = sc.tpre;
      P.ntask = sc.ntask;
      P.wq = sc.wq;
      P.woff = sc.woff;
      P.chunk_task = sc.chunk_task;
      if (a.mode == 0) {
        P.keep = plan == 1;
        hipLaunchKernelGGL((k_lv_plan<T, IS, false, 3>), dim3(P.nq), dim3(kWave), 0, s, P);
        return hip_status(hipGetLastError(), "Error in launching level search");
      }
      if (plan == 2) {
        hipLaunchKernelGGL(k_lv_clip, dim3((P.nq + kLvBlock - 1) / kLvBlock), dim3(kLvBlock), 0, s, sc.tpre, sc.ntask,
                           sc.wq, a.counts, a.offsets, a.caps, a.cap_all, P.out_total, P.nq);
      } else {
        // few queries leave the memory system idle: more probes per search step
        if (P.nq <= kFewQueries) hipLaunchKernelGGL((k_lv_plan<T, IS, true, 7>), dim3(P.nq), dim3(kWave), 0, s, P);
        else hipLaunchKernelGGL((k_lv_plan<T, IS, true, 3>), dim3(P.nq), dim3(kWave), 0, s, P);
      }
      if (!(P.use_single && plan != 2)) {  // a single query's plan wrote these itself
        Status st = exclusive_scan(sc.wq, sc.woff, a.nq, s);
        if (!st.ok()) return st;
        constexpr uint32_t kWaves = kLvBlock / kWave;
        hipLaunchKernelGGL(k_lv_mark, dim3((P.nq + kWaves - 1) / kWaves), dim3(kLvBlock), 0, s, sc.woff, sc.tpre, sc.ntask, P.nq, sc.chunk_task);
      }
      int dev = 0, cus = 0;
      hipGetDevice(&dev);
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
      const uint32_t per = P.nq <= kFewCopies ? kCopyPerCuFew : kCopyPerCu;
      hipLaunchKernelGGL((k_lv_copy<IS>), dim3(static_cast<unsigned>(cus) * per), dim3(kCopyBlock), 0, s, P.id, sc.tsrc,
                         sc.tpre, sc.ntask, sc.woff, a.offsets, sc.chunk_task, P.nq,
                         static_cast<IS*>(a.out));
      return hip_status(hipGetLastError(), "Error in launching level search");
    });
  });
}

}  // namespace pst
