// Tree construction for StaticPSTGPU on gfx950.
//
// Replaces the reference's construction (pst/static-pst-gpu.tu:19-437:
// index init, two thrust::sorts, then populateTree, a one-block kernel that
// builds nodes thread-per-node and relaunches itself through dynamic
// parallelism, pst/static-pst-gpu-populate-tree.tu:10-158) with rank arrays
// and level-synchronous passes:
//
//   1. The points are listed in key1 order as values that compare like
//      key2 (the smaller value is the greater point). Points with 32-bit
//      dims and 32-bit IDs that rise with the index sort once, by dim1,
//      carrying (dim2, ID) as a 64-bit value from which the node records are
//      formed: nothing is gathered (point_sort_*, pst_sort.hip). Others
//      first sort by key2 = (dim2, id, index), and the value is the 32-bit
//      key2 rank.
//   2. The levels above LDS size move no point: a static hierarchy of block
//      minima (64 values each) gives a segment's node as a range minimum,
//      taken around the at most `level` nodes already removed from the
//      segment; the median and the children's ranges follow by counting
//      those. Their sizes follow from n alone (pst_common.hpp).
//   3. Once every segment fits in LDS (<= kFinishTile points), one
//      workgroup finishes its whole subtree in LDS.
// The node chosen, the median rule and the child split are those of the
// reference's constructNode (pst/static-pst-gpu.tu:706-806 and
// pst/static-pst-cpu-iter.tpp:488-598); the tree is bit-identical to the
// reference's CPU iterative tree on the same input.
#include <algorithm>
#include <vector>

#include "pst_internal.hpp"

namespace pst {

namespace {

constexpr int kFinishBlock = 512;      // threads per LDS subtree of the deep tree
constexpr int kForestBlock = 256;       // threads per forest tree
// Levels of the forest trees that k_forest_reg builds (pst_forest_build.hip):
// trees of 31 to 511 points, a wave each (2.99 -> 0.174 ms for 16.7M points
// in trees of 127). Smaller trees leave most of a wave's lanes to tree ends;
// trees of 1023 points would need 16 points per lane, whose sort keys alone
// fill a lane's registers.
constexpr uint32_t kForestRegMin = 5, kForestRegMax = 9;

template <typename I>
struct IdStore {
  using type = typename std::conditional<sizeof(I) == 8, uint64_t, uint32_t>::type;
};
template <>
struct IdStore<NoId> {
  using type = NoId;
};

// ---------------------------------------------------------------------------
// Key kernels. Keys are order-preserving unsigned integers; for the
// descending key2 order the keys are complemented and the input visited
// back to front, so that a stable ascending sort also orders equal keys by
// descending index, as the reference's comparisonTiebreaker does for
// compareDim2(...) > 0.
// ---------------------------------------------------------------------------
// ORDER_CHECK: also sets flags[1] when some point's ID is above the next
// point's (IDs not in index order), and flags[0] for a NaN ID. With key1
// (32-bit keys only), the same read of point i also stores its ascending
// dim1 key at key1[i], the keys of the dim1 sort.
template <typename T, typename I, typename K, bool DIM2, bool DESC, bool WITH_ID, bool ORDER_CHECK = false>
__global__ void k_keys_single(const Point<T, I>* __restrict__ pts, uint32_t n, K* __restrict__ keys,
                              uint32_t* __restrict__ vals, const uint32_t* __restrict__ r2,
                              int* __restrict__ flags, uint32_t* __restrict__ key1 = nullptr) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const uint32_t i = DESC ? n - 1 - j : j;
  const Point<T, I> p = pts[i];
  const T d = DIM2 ? p.dim2_val : p.dim1_val;
  bool bad = is_nan(d);
  K k;
  if constexpr (WITH_ID) {
    bad |= is_nan(p.id);
    k = (static_cast<K>(ord_key(d)) << 32) | static_cast<K>(ord_key(p.id));
  } else {
    k = static_cast<K>(ord_key(d));
  }
  if constexpr (ORDER_CHECK) {
    bad |= is_nan(p.id);
    if (i + 1 < n && ord_key(p.id) > ord_key(pts[i + 1].id)) flags[1] = 1;
  }
  if constexpr (sizeof(K) == 4) {
    if (key1) {
      bad |= is_nan(p.dim1_val);
      key1[i] = static_cast<uint32_t>(ord_key(p.dim1_val));
    }
  }
  if (bad) flags[0] = 1;
  keys[j] = DESC ? ~k : k;
  vals[j] = r2 ? r2[i] : i;
}

// Keys of points whose IDs are not in index order: by ID first, then by dim
// over the points in that order (`perm`; backwards for a descending order, so
// that equal dims come by descending (id, index)).
template <typename T, typename I, typename K>
__global__ void k_keys_id(const Point<T, I>* __restrict__ pts, uint32_t n, K* __restrict__ keys,
                          uint32_t* __restrict__ vals, int* __restrict__ nan_flag) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const I id = pts[i].id;
  if (is_nan(id)) *nan_flag = 1;
  keys[i] = static_cast<K>(ord_key(id));
  vals[i] = i;
}

template <typename T, typename I, typename K, bool DIM2, bool DESC>
__global__ void k_keys_dim_perm(const Point<T, I>* __restrict__ pts, uint32_t n,
                                const uint32_t* __restrict__ perm, K* __restrict__ keys,
                                uint32_t* __restrict__ vals, const uint32_t* __restrict__ r2,
                                int* __restrict__ nan_flag) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const uint32_t i = perm[DESC ? n - 1 - j : j];
  const T d = DIM2 ? pts[i].dim2_val : pts[i].dim1_val;
  if (is_nan(d)) *nan_flag = 1;
  const K k = static_cast<K>(ord_key(d));
  keys[j] = DESC ? static_cast<K>(~k) : k;
  vals[j] = r2 ? r2[i] : i;
}

__global__ void k_scatter_rank(const uint32_t* __restrict__ perm2, uint32_t n, uint32_t* __restrict__ r2) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) r2[perm2[p]] = p;
}

// ---------------------------------------------------------------------------
// The levels above LDS size. V: uint32_t ranks or uint64_t values, all
// different; the smallest of a segment is its node. A segment of level t is
// the input range [b_j, b_(j+1)) of the key1-ordered array less the nodes of
// the levels above that lie in it (its holes, a sorted list of at most t
// positions; one per segment on average, since a node lies in one segment).
// ---------------------------------------------------------------------------
constexpr int kTopBlock = 256;

// mins1[k]: minimum of values [64 k, 64 k + 64); mins2 of 64 such, one
// workgroup per 4096 values.
template <typename V>
__global__ __launch_bounds__(kTopBlock) void k_block_min(const V* __restrict__ a, uint32_t n, V* __restrict__ mins1,
                                                         V* __restrict__ mins2) {
  constexpr int kPer = 16 / sizeof(V);            // values per 16-byte load
  constexpr int kLanes = kFan / kPer;             // lanes per block of 64
  constexpr int kRounds = 4096 / (kTopBlock * kPer);
  __shared__ V m1[kFan];
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * 4096;
  V x[kRounds][kPer];
  if (base + 4096 <= n) {
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
      const uint4 w = *reinterpret_cast<const uint4*>(a + base + (r * kTopBlock + threadIdx.x) * kPer);
      __builtin_memcpy(x[r], &w, 16);
    }
  } else {
#pragma unroll
    for (int r = 0; r < kRounds; r++)
#pragma unroll
      for (int k = 0; k < kPer; k++) {
        const uint64_t i = base + (r * kTopBlock + threadIdx.x) * kPer + k;
        x[r][k] = i < n ? a[i] : static_cast<V>(~V(0));
      }
  }
#pragma unroll
  for (int r = 0; r < kRounds; r++) {
    V m = x[r][0];
#pragma unroll
    for (int k = 1; k < kPer; k++) m = x[r][k] < m ? x[r][k] : m;
#pragma unroll
    for (int o = 1; o < kLanes; o <<= 1) {
      const V y = __shfl_xor(m, o, kWave);
      m = y < m ? y : m;
    }
    const uint32_t k = (r * kTopBlock + threadIdx.x) / kLanes;
    if (threadIdx.x % kLanes == 0) {
      m1[k] = m;
      if (base + k * kFan < n) mins1[base / kFan + k] = m;
    }
  }
  __syncthreads();
  if (threadIdx.x < kFan) {
    V m = m1[threadIdx.x];
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const V y = __shfl_xor(m, o, kWave);
      m = y < m ? y : m;
    }
    if (threadIdx.x == 0) mins2[blockIdx.x] = m;
  }
}

// mins3: minima of 64 values of mins2 (a wave each).
template <typename V>
__global__ __launch_bounds__(kTopBlock) void k_min_of_mins(const V* __restrict__ mins2, uint32_t n2,
                                                           V* __restrict__ mins3, uint32_t n3) {
  const uint32_t k = blockIdx.x * (kTopBlock / kWave) + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (k >= n3) return;
  const uint32_t i = k * kFan + lane;
  V m = i < n2 ? mins2[i] : static_cast<V>(~V(0));
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const V y = __shfl_xor(m, o, kWave);
    m = y < m ? y : m;
  }
  if (lane == 0) mins3[k] = m;
}

// Segments of one level: first positions, hole counts, hole lists.
struct Segs {
  uint32_t* b;
  uint32_t* cnt;
  uint32_t* holes;  // kMaxHoles per segment
};

__global__ void k_segs_root(Segs s) {
  s.b[0] = 0;
  s.cnt[0] = 0;
}

// A value of the dim's type from its key (not for -0, which shares +0's key).
template <typename T>
__device__ inline T from_key(uint32_t k) {
  if constexpr (std::is_same<T, float>::value) return __builtin_bit_cast(float, (k & 0x80000000u) ? k ^ 0x80000000u : ~k);
  else if constexpr (std::is_same<T, int32_t>::value) return static_cast<int32_t>(k ^ 0x80000000u);
  else return static_cast<T>(k);
}

// Where the records' fields come from. Ranked: V = uint32_t ranks into the
// key2 order, records gathered from the points. Direct: V = uint64_t values
// and the sorted dim1 keys; id_code says how IDs map to keys.
template <typename T, typename IS>
struct Ranked {
  using V = uint32_t;
  const uint32_t* perm2;
  const Point<T, IS>* pts;
  __device__ Point<T, IS> point(V v, uint32_t) const { return pts[perm2[v]]; }
};
template <typename T, typename IS>
struct Direct {
  using V = uint64_t;
  const uint32_t* key1;
  int id_code;
  __device__ Point<T, IS> make(V v, uint32_t k1) const {
    Point<T, IS> p;
    p.dim1_val = from_key<T>(k1);
    p.dim2_val = from_key<T>(~static_cast<uint32_t>(v >> 32));
    if constexpr (has_id_v<IS>) {
      const uint32_t k = ~static_cast<uint32_t>(v);
      p.id = id_code == F32 ? __builtin_bit_cast(uint32_t, from_key<float>(k))
                            : (id_code == I32 ? static_cast<uint32_t>(from_key<int32_t>(k)) : k);
    }
    return p;
  }
  __device__ Point<T, IS> point(V v, uint32_t pos) const { return make(v, key1[pos]); }
};

template <typename T, typename IS>
__device__ inline void write_node(Node<T, IS>* nodes, uint64_t slot, const Point<T, IS>& p, T med) {
  Node<T, IS> r;
  r.dim1 = p.dim1_val;
  r.dim2 = p.dim2_val;
  r.med = med;
  if constexpr (has_id_v<IS>) r.id = p.id;
  nodes[slot] = r;
}

// One level: a wave per segment finds the node, writes its record and hands
// the two halves of what remains to the next level. The minimum is taken
// over the stretches between the segment's holes; a stretch reads at most 126
// values at each end of each step of the hierarchy (and the middle of the
// top one), all at once, and the winner is traced down a step at a time.
// Bound by latency (about eight dependent loads). On MI355X the 15 levels of
// 2^26 points take 0.17 ms after 0.12 ms for the block minima, where moving
// the points level by level (8 B per point and level) took 1.78 ms.
template <typename T, typename IS, typename Src>
__global__ __launch_bounds__(kTopBlock) void k_top_level(Src src, const typename Src::V* __restrict__ a,
                                                         const typename Src::V* __restrict__ m1,
                                                         const typename Src::V* __restrict__ m2,
                                                         const typename Src::V* __restrict__ m3, uint32_t n, uint32_t t,
                                                         uint64_t M, Segs in, Segs out, Node<T, IS>* __restrict__ nodes) {
  using V = typename Src::V;
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t j = __builtin_amdgcn_readfirstlane(blockIdx.x * (kTopBlock / kWave) + threadIdx.x / kWave);
  const uint32_t nseg = 1u << t;
  if (j >= nseg) return;
  const uint32_t b = in.b[j], e = j + 1 < nseg ? in.b[j + 1] : n;
  const uint32_t cnt = in.cnt[j];
  uint32_t hole = lane < cnt ? in.holes[static_cast<size_t>(j) * kMaxHoles + lane] : ~0u;
  const uint32_t n1 = blocks_of(n), n2 = blocks_of(n1);
  // the lane's best candidate: its value, step of the hierarchy and index
  V best = static_cast<V>(~V(0));
  uint32_t step = 0, at = ~0u;
  auto take = [&](uint32_t st, uint32_t i) {
    const V v = (st == 0 ? a : (st == 1 ? m1 : (st == 2 ? m2 : m3)))[i];
    if (v < best || at == ~0u) {
      best = v;
      step = st;
      at = i;
    }
  };
  for (uint32_t r = 0; r <= cnt; r++) {
    const uint32_t lo = r == 0 ? b : __builtin_amdgcn_readlane(hole, r - 1) + 1;
    const uint32_t hi = r == cnt ? e : static_cast<uint32_t>(__builtin_amdgcn_readlane(hole, r));
    stretch_minima(lo, hi, lane, take);
  }
  V mn = best;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const V y = __shfl_xor(mn, o, kWave);
    mn = y < mn ? y : mn;
  }
  const uint64_t won = __ballot(best == mn && at != ~0u);
  if (won == 0) return;  // never: the segment holds points
  const int f = __builtin_ctzll(won);
  uint32_t q = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(at), f));
  int st = __builtin_amdgcn_readlane(static_cast<int>(step), f);
  for (; st > 0; st--) {
    const V* arr = st == 3 ? m2 : (st == 2 ? m1 : a);
    const uint32_t len = st == 3 ? n2 : (st == 2 ? n1 : n);
    const uint32_t i = q * kFan + lane;
    const uint64_t eq = __ballot(i < len && arr[i < len ? i : 0] == mn);
    q = q * kFan + static_cast<uint32_t>(eq ? __builtin_ctzll(eq) : 0);
  }
  // the node joins the holes (in position order)
  const uint32_t below = static_cast<uint32_t>(__popcll(__ballot(lane < cnt && hole < q)));
  const uint32_t prev = static_cast<uint32_t>(__shfl_up(static_cast<int>(hole), 1, kWave));
  hole = lane < below ? hole : (lane == below ? q : prev);
  const uint32_t nh = cnt + 1;
  // position of the last point of the left half: the (L - 1)-th that remains
  const uint32_t L = static_cast<uint32_t>(level_size(M, t, j)) >> 1;
  uint32_t last = b + L - 1;
  for (uint32_t i = 0; i < nh; i++) {
    const uint32_t h = static_cast<uint32_t>(__builtin_amdgcn_readlane(hole, i));
    last += h <= last ? 1u : 0u;
  }
  const uint32_t c = last + 1;
  const uint32_t nl = static_cast<uint32_t>(__popcll(__ballot(lane < nh && hole < c)));
  if (lane < nh) {
    if (lane < nl) out.holes[static_cast<size_t>(2 * j) * kMaxHoles + lane] = hole;
    else out.holes[static_cast<size_t>(2 * j + 1) * kMaxHoles + lane - nl] = hole;
  }
  if (lane == 0) {
    out.b[2 * j] = b;
    out.b[2 * j + 1] = c;
    out.cnt[2 * j] = nl;
    out.cnt[2 * j + 1] = nh - nl;
    write_node(nodes, nseg - 1ull + j, src.point(mn, q), src.point(a[last], last).dim1_val);
  }
}

// Subtree minima of dim2 and IDs of the levels above LDS size: levels
// [s, t0) by one workgroup per subtree of level s, then levels [0, s) by one
// workgroup (what k_submin_level computes, in two launches).
template <typename T, typename IS>
__global__ __launch_bounds__(kTopBlock) void k_top_submin(const Node<T, IS>* __restrict__ nodes, T* submin,
                                                          IS* __restrict__ ids, uint32_t s, uint32_t t0) {
  for (uint32_t u = t0; u-- > s;) {
    const uint32_t per = 1u << (u - s);
    for (uint32_t k = threadIdx.x; k < per; k += kTopBlock) {
      const uint32_t slot = (1u << u) - 1 + blockIdx.x * per + k;
      const Node<T, IS> nd = nodes[slot];
      if constexpr (has_id_v<IS>) {
        if (ids) ids[slot] = nd.id;
      }
      T v = nd.dim2;
      const T l = submin[2 * slot + 1], r = submin[2 * slot + 2];  // every such node has both children
      v = l < v ? l : v;
      v = r < v ? r : v;
      submin[slot] = v;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Whole subtree in LDS: A-segment of m <= kFinishTile points in bufA.
// ---------------------------------------------------------------------------
template <typename T, typename IS, typename PermF>
__device__ void lds_build(uint32_t* bufA, uint32_t* bufB, unsigned long long* sres,
                          unsigned long long* wred, uint32_t m, uint64_t root_slot,
                          const Point<T, IS>* __restrict__ pts, PermF perm, Node<T, IS>* __restrict__ nodes) {
  const uint32_t tid = threadIdx.x;
  const uint32_t nthr = blockDim.x;
  const uint64_t Mp = static_cast<uint64_t>(m) + 1;
  for (uint32_t u = 0; (Mp >> u) != 0; u++) {
    const uint32_t nsub = 1u << u;
    if (nsub <= nthr) {
      const uint32_t G = nthr / nsub;
      const uint32_t k = tid / G, g = tid % G;
      const int64_t sz = level_size(Mp, u, k);
      const uint32_t st = static_cast<uint32_t>(sz > 0 ? level_start(Mp, u, k) : 0);
      unsigned long long best = ~0ull;
      for (int64_t x = g; x < sz; x += G) {
        const unsigned long long key = (static_cast<unsigned long long>(bufA[st + x]) << 32) |
                                       static_cast<unsigned long long>(x);
        best = key < best ? key : best;
      }
      const uint32_t wg = G < kWave ? G : kWave;
      for (uint32_t off = wg >> 1; off >= 1; off >>= 1) {
        const unsigned long long o = __shfl_xor(best, off, kWave);
        best = o < best ? o : best;
      }
      if (G > kWave) {  // uniform across the block
        if ((tid & (kWave - 1)) == 0) wred[tid / kWave] = best;
        __syncthreads();
        if (g == 0) {
          const uint32_t w0 = tid / kWave, nw = G / kWave;
          for (uint32_t w = 0; w < nw; w++) best = wred[w0 + w] < best ? wred[w0 + w] : best;
        }
      }
      if (g == 0) sres[k] = best;
      __syncthreads();
      if (sz > 0) {
        const unsigned long long mn = sres[k];
        const uint32_t q = static_cast<uint32_t>(mn);
        const uint32_t L = static_cast<uint32_t>(sz) >> 1;
        if (g == 0) {
          const Point<T, IS> p = pts[perm(static_cast<uint32_t>(mn >> 32))];
          T med = p.dim1_val;
          if (L >= 1) med = pts[perm(bufA[st + (q < L ? L : L - 1)])].dim1_val;
          write_node(nodes, (root_slot + 1) * nsub - 1 + k, p, med);
        }
        const uint32_t dst0 = static_cast<uint32_t>(sz > 1 ? level_start(Mp, u + 1, 2 * k) : 0);
        for (int64_t x = g; x < sz; x += G) {
          if (static_cast<uint32_t>(x) == q) continue;
          bufB[dst0 + x - (static_cast<uint32_t>(x) > q ? 1 : 0)] = bufA[st + x];
        }
      }
    } else {
      for (uint32_t k = tid; k < nsub; k += nthr) {
        const int64_t sz = level_size(Mp, u, k);
        if (sz <= 0) continue;
        const uint32_t st = static_cast<uint32_t>(level_start(Mp, u, k));
        unsigned long long best = ~0ull;
        for (int64_t x = 0; x < sz; x++) {
          const unsigned long long key = (static_cast<unsigned long long>(bufA[st + x]) << 32) |
                                         static_cast<unsigned long long>(x);
          best = key < best ? key : best;
        }
        const uint32_t q = static_cast<uint32_t>(best);
        const uint32_t L = static_cast<uint32_t>(sz) >> 1;
        const Point<T, IS> p = pts[perm(static_cast<uint32_t>(best >> 32))];
        T med = p.dim1_val;
        if (L >= 1) med = pts[perm(bufA[st + (q < L ? L : L - 1)])].dim1_val;
        write_node(nodes, (root_slot + 1) * nsub - 1 + k, p, med);
        if (sz > 1) {
          const uint32_t dst0 = static_cast<uint32_t>(level_start(Mp, u + 1, 2 * k));
          for (int64_t x = 0; x < sz; x++) {
            if (static_cast<uint32_t>(x) == q) continue;
            bufB[dst0 + x - (static_cast<uint32_t>(x) > q ? 1 : 0)] = bufA[st + x];
          }
        }
      }
    }
    __syncthreads();
    uint32_t* tmp = bufA;
    bufA = bufB;
    bufB = tmp;
  }
}

// Orders a wave's LDS accesses around it (the compiler keeps them on their
// side; the wave's LDS instructions execute in order).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Threads of the subtree passes: from level kWaveLevel of a subtree on, the
// segment of position k and every segment below it belong to wave
// k >> (u - kWaveLevel), so those levels need no workgroup barrier.
constexpr uint32_t kFinishLog = 9;
static_assert((1u << kFinishLog) == kFinishBlock, "block size is a power of two");
constexpr uint16_t kNoPos = 0xffffu;
constexpr uint32_t kWaveLevel = kFinishLog - 6;
static_assert(kWave == 64, "64-lane waves");

// The subtree build of the deep tree's last levels. Every point's rank is
// read once up front, all reads in flight together; the levels then work
// on 16-bit local positions in LDS: the node of a
// segment is the position of least rank, and the level only notes, per
// point, the subtree slot it fills and its med point. The node records are
// read from the input and written after the last level, all reads in
// flight together, so that no level waits on global memory. The levels
// above kWaveLevel share segments between waves and end in a workgroup
// barrier; from it on each wave works on its own part of the subtree.
template <typename V>
__device__ void lds_build_local(uint16_t* bufA, uint16_t* bufB, const V* rank, uint16_t* slot_of, uint16_t* med_of,
                                uint16_t* sst, uint16_t* sres, V* wred, uint16_t* wredx, uint32_t m) {
  const uint32_t tid = threadIdx.x;
  constexpr uint32_t nthr = kFinishBlock;  // the launch's block size
  const uint64_t Mp = static_cast<uint64_t>(m) + 1;
  // node of segment k of level u: point bufA[st + q]; its subtree slot
  // h = 2^u - 1 + k; med: the point at position L or L - 1 (L = floor(sz /
  // 2)), or the node itself when L = 0. Segment starts are kept per slot
  // (sst[h], sst[0] = 0 set by the caller): with the node removed, the
  // children start at st and st + L of the next level's array. Children stay
  // within their parent's positions (the next array has gaps where nodes
  // left), so that a wave's part of both arrays never moves.
  auto note = [&](uint32_t u, uint32_t k, uint32_t st, uint32_t sz, uint32_t q) {
    const uint32_t L = sz >> 1;
    const uint16_t x = bufA[st + q];
    const uint32_t h = (1u << u) - 1 + k;
    slot_of[x] = static_cast<uint16_t>(h);
    med_of[x] = L >= 1 ? bufA[st + (q < L ? L : L - 1)] : x;
    if (sz > 1) {
      sst[2 * h + 1] = static_cast<uint16_t>(st);
      sst[2 * h + 2] = static_cast<uint16_t>(st + L);
    }
  };
  // level sync: a workgroup barrier while segments span waves, else the
  // wave's own
  auto level_sync = [&](uint32_t u) {
    if (u < kWaveLevel) __syncthreads();
    else wave_sync();
  };
  for (uint32_t u = 0; (Mp >> u) != 0; u++) {
    const uint32_t nsub = 1u << u;
    if (nsub <= nthr) {
      // segment k on threads [k G, (k + 1) G)
      const uint32_t G = nthr / nsub;
      const uint32_t k = tid / G, g = tid % G;
      const int64_t sz = level_size(Mp, u, k);
      const uint32_t st = sz > 0 ? sst[(1u << u) - 1 + k] : 0u;
      // the smallest value, then its position from the one thread that holds it
      V mine = static_cast<V>(~V(0));
      uint32_t bx = ~0u;
      for (int64_t x = g; x < sz; x += G) {
        const V v = rank[bufA[st + x]];
        if (v <= mine) {
          mine = v;
          bx = static_cast<uint32_t>(x);
        }
      }
      V best = mine;
      const uint32_t wg = G < kWave ? G : kWave;
      for (uint32_t off = wg >> 1; off >= 1; off >>= 1) {
        const V o = __shfl_xor(best, off, kWave);
        best = o < best ? o : best;
      }
      // the segment's result sits at its first thread's entry, which no
      // other wave uses at any level
      if (G > kWave) {  // uniform across the block
        if (bx != ~0u && mine == best) {
          wred[tid / kWave] = best;
          wredx[tid / kWave] = static_cast<uint16_t>(bx);
        }
        if (__ballot(bx != ~0u) == 0 && (tid & (kWave - 1)) == 0) {  // a wave without points
          wred[tid / kWave] = static_cast<V>(~V(0));
          wredx[tid / kWave] = kNoPos;
        }
        __syncthreads();
        if (g == 0) {
          const uint32_t w0 = tid / kWave, nw = G / kWave;
          V b2 = wred[w0];
          uint16_t x2 = wredx[w0];
          for (uint32_t w = 1; w < nw; w++) {
            if (wredx[w0 + w] != kNoPos && (x2 == kNoPos || wred[w0 + w] < b2)) {
              b2 = wred[w0 + w];
              x2 = wredx[w0 + w];
            }
          }
          sres[k * G] = x2;
        }
      } else if (bx != ~0u && mine == best) {
        sres[k * G] = static_cast<uint16_t>(bx);
      }
      level_sync(u);
      if (sz > 0) {
        const uint32_t q = sres[k * G];
        if (g == 0) note(u, k, st, static_cast<uint32_t>(sz), q);
        const uint32_t dst0 = st;
        for (int64_t x = g; x < sz; x += G) {
          if (static_cast<uint32_t>(x) == q) continue;
          bufB[dst0 + x - (static_cast<uint32_t>(x) > q ? 1 : 0)] = bufA[st + x];
        }
      }
    } else {
      // thread t takes the 2^(u - kFinishLog) segments below its segment of
      // level kFinishLog
      const uint32_t per = nsub >> kFinishLog;
      for (uint32_t k = tid * per; k < (tid + 1) * per; k++) {
        const int64_t sz = level_size(Mp, u, k);
        if (sz <= 0) continue;
        const uint32_t st = sst[(1u << u) - 1 + k];
        V best = rank[bufA[st]];
        uint32_t q = 0;
        for (int64_t x = 1; x < sz; x++) {
          const V v = rank[bufA[st + x]];
          if (v < best) {
            best = v;
            q = static_cast<uint32_t>(x);
          }
        }
        note(u, k, st, static_cast<uint32_t>(sz), q);
        if (sz > 1) {
          const uint32_t dst0 = st;
          for (int64_t x = 0; x < sz; x++) {
            if (static_cast<uint32_t>(x) == q) continue;
            bufB[dst0 + x - (static_cast<uint32_t>(x) > q ? 1 : 0)] = bufA[st + x];
          }
        }
      }
    }
    level_sync(u);
    uint16_t* tmp = bufA;
    bufA = bufB;
    bufB = tmp;
  }
  __syncthreads();
}

// Direct: 1.36 ms for 2^26 f32/u32 points on MI355X, bound by the LDS passes
// of the subtree build (12 B read and 24 B written per point are 0.5 ms at a
// large copy's rate). Ranked, with two 128-byte gathers per point: 2.75 ms.
// One workgroup per level-t0 segment: its whole subtree in LDS, then every
// node record; with `submin` also the subtree minima of dim2 and the IDs of
// the subtree's slots (the bottom levels of what k_submin_level computes).
template <typename T, typename IS, typename Src>
__global__ __launch_bounds__(kFinishBlock) void k_finish(
    Src src, const typename Src::V* __restrict__ A, uint32_t n, uint32_t t0, uint64_t M, Segs segs,
    Node<T, IS>* __restrict__ nodes, T* __restrict__ submin, IS* __restrict__ ids) {
  using V = typename Src::V;
  constexpr bool kDirect = sizeof(V) == 8;  // records from values and dim1 keys, else gathered
  union FinishLds {
    struct {
      uint16_t bufA[kFinishTile];
      uint16_t bufB[kFinishTile];
      uint16_t sst[2 * kFinishTile];  // segment start per subtree slot
    } b;
    T d2[2 * kFinishTile];  // after the build: dim2 per subtree slot, then its subtree minimum
  };
  __shared__ FinishLds U;
  union RankLds {
    V rank[kFinishTile];
    T d1[kFinishTile];  // gathered records, after the lookups: dim1 of every point, for the meds
  };
  __shared__ RankLds R;
  __shared__ uint32_t s_key1[kDirect ? kFinishTile : 1];
  V* rank = R.rank;
  __shared__ uint16_t slot_of[kFinishTile];  // the subtree slot (heap order) each point fills
  __shared__ uint16_t med_of[kFinishTile];   // and the point whose dim1 is its med
  __shared__ uint16_t sres[kFinishBlock];    // a segment's result, at its first thread's entry
  __shared__ V wred[kFinishBlock / kWave];
  __shared__ uint16_t wredx[kFinishBlock / kWave];
  __shared__ uint32_t s_hole[kMaxHoles];
  const uint32_t j = blockIdx.x;
  const int64_t m = level_size(M, t0, j);
  if (m <= 0) return;
  const uint32_t st = segs.b[j], len = (j + 1 < gridDim.x ? segs.b[j + 1] : n) - st;
  const uint32_t nh = segs.cnt[j];
  if (threadIdx.x < nh) s_hole[threadIdx.x] = segs.holes[static_cast<size_t>(j) * kMaxHoles + threadIdx.x] - st;
  const uint64_t root = (1ull << t0) - 1 + j;
  constexpr int kPer = kFinishTile / kFinishBlock;
  // the segment's values close up over its holes: point x is the x-th that
  // is left (a range of at most kFinishTile + kMaxHoles positions)
  V av[kPer + 1];
  uint32_t kv[kPer + 1];
#pragma unroll
  for (int e = 0; e < kPer + 1; e++) {
    const uint32_t p = threadIdx.x + e * kFinishBlock;
    if (p < len) {
      av[e] = A[st + p];
      if constexpr (kDirect) kv[e] = src.key1[st + p];
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kPer + 1; e++) {
    const uint32_t p = threadIdx.x + e * kFinishBlock;
    if (p < len) {
      uint32_t x = p;
      bool gone = false;
      for (uint32_t i = 0; i < nh; i++) {
        const uint32_t h = s_hole[i];
        x -= h < p ? 1u : 0u;
        gone |= h == p;
      }
      if (!gone && x < m) {
        rank[x] = av[e];
        if constexpr (kDirect) s_key1[x] = kv[e];
        U.b.bufA[x] = static_cast<uint16_t>(x);
      }
    }
  }
  if (threadIdx.x == 0) U.b.sst[0] = 0;
  __syncthreads();
  lds_build_local<V>(U.b.bufA, U.b.bufB, rank, slot_of, med_of, U.b.sst, sres, wred, wredx, static_cast<uint32_t>(m));
  // every point's node record: subtree slot h (level u, position k) is slot
  // ((root + 1) << u) - 1 + k of the tree. A med is the dim1 of a point of
  // the same subtree. Gathered records: rank -> input index -> record, all
  // loads in flight together.
  Point<T, IS> p[kPer];
  T med[kPer];
  if constexpr (kDirect) {
#pragma unroll
    for (int e = 0; e < kPer; e++) {
      const uint32_t x = threadIdx.x + e * kFinishBlock;
      if (x < m) {
        p[e] = src.make(rank[x], s_key1[x]);
        med[e] = from_key<T>(s_key1[med_of[x]]);
      }
    }
    __syncthreads();  // the build's LDS arrays are free from here
  } else {
    uint32_t ix[kPer];
#pragma unroll
    for (int e = 0; e < kPer; e++) {
      const uint32_t x = threadIdx.x + e * kFinishBlock;
      if (x < m) ix[e] = src.perm2[rank[x]];
    }
#pragma unroll
    for (int e = 0; e < kPer; e++) {
      const uint32_t x = threadIdx.x + e * kFinishBlock;
      if (x < m) p[e] = src.pts[ix[e]];
    }
    __syncthreads();  // the build's LDS arrays and the ranks are free from here
#pragma unroll
    for (int e = 0; e < kPer; e++) {
      const uint32_t x = threadIdx.x + e * kFinishBlock;
      if (x < m) R.d1[x] = p[e].dim1_val;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPer; e++) {
      const uint32_t x = threadIdx.x + e * kFinishBlock;
      if (x < m) med[e] = R.d1[med_of[x]];
    }
  }
  const uint32_t mdepth = 32u - static_cast<uint32_t>(__builtin_clz(static_cast<uint32_t>(m)));
#pragma unroll
  for (int e = 0; e < kPer; e++) {
    const uint32_t x = threadIdx.x + e * kFinishBlock;
    if (x < m) {
      const uint32_t h = slot_of[x] + 1u;
      if ((h >> mdepth) != 0) continue;  // never: the subtree has mdepth levels
      const uint32_t u = 31u - static_cast<uint32_t>(__builtin_clz(h));
      const uint64_t slot = ((root + 1) << u) - 1 + (h - (1u << u));
      write_node(nodes, slot, p[e], med[e]);
      if (submin) {
        U.d2[h - 1] = p[e].dim2_val;
        if constexpr (has_id_v<IS>) {
          if (ids) ids[slot] = p[e].id;
        }
      }
    }
  }
  if (!submin) return;
  // subtree minima, bottom level first: min(dim2(s), minima of the children
  // that exist); a slot of size ms has a left child if ms >= 2, a right one
  // if ms >= 3. Levels from kWaveLevel down: wave w takes the slots below
  // slot w of level kWaveLevel, with no workgroup barrier between levels;
  // the levels above them are one thread's.
  __syncthreads();
  const uint64_t Mp = static_cast<uint64_t>(m) + 1;
  const int depth = 32 - __builtin_clz(static_cast<uint32_t>(m));
  auto min_slot = [&](uint32_t u, uint32_t k) {
    const int64_t ms = level_size(Mp, u, k);
    if (ms < 1) return;
    const uint32_t sl = (1u << u) - 1 + k;
    T v = U.d2[sl];
    if (ms >= 2) {
      const T c = U.d2[2 * sl + 1];
      v = c < v ? c : v;
    }
    if (ms >= 3) {
      const T c = U.d2[2 * sl + 2];
      v = c < v ? c : v;
    }
    U.d2[sl] = v;
    submin[((root + 1) << u) - 1 + k] = v;
  };
  const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  for (int u = depth - 1; u >= static_cast<int>(kWaveLevel); u--) {
    const uint32_t per = 1u << (u - kWaveLevel);
    for (uint32_t i = lane; i < per; i += kWave) min_slot(static_cast<uint32_t>(u), wave * per + i);
    wave_sync();
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int top = depth - 1 < static_cast<int>(kWaveLevel) - 1 ? depth - 1 : static_cast<int>(kWaveLevel) - 1;
    for (int u = top; u >= 0; u--)
      for (uint32_t k = 0; k < (1u << u); k++) min_slot(static_cast<uint32_t>(u), k);
  }
}

// ---------------------------------------------------------------------------
// Subtree minimum of dim2, one level at a time from the bottom: submin(s) =
// min(dim2(s), submin(2s+1), submin(2s+2)) over the children that exist.
// A walk that meets a REPORT_ABOVE subtree with min_dim2 <= submin knows
// that every node in it is reported. Level t of every tree of a forest is
// done by one launch (ntrees x 2^t positions). The same pass copies each
// slot's ID into a dense ID array (null: none), which whole-subtree copies
// read instead of the full records.
// ---------------------------------------------------------------------------
template <typename T, typename IS>
__global__ void k_submin_level(const Node<T, IS>* __restrict__ nodes, T* __restrict__ submin, IS* __restrict__ ids,
                               uint32_t t, uint32_t shift, uint32_t ntrees, uint32_t full_M, uint32_t last_M) {
  const uint64_t k = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t per_tree = 1ull << t;
  if (k >= per_tree * ntrees) return;
  const uint32_t tree = static_cast<uint32_t>(k >> t);
  const uint32_t local = static_cast<uint32_t>((1ull << t) - 1 + (k & (per_tree - 1)));
  const uint32_t M = tree + 1 < ntrees ? full_M : last_M;
  const int32_t m = subtree_size32(M, local);
  if (m < 1) return;
  const uint64_t base = static_cast<uint64_t>(tree) << shift;
  const Node<T, IS> nd = nodes[base + local];
  if constexpr (has_id_v<IS>) {
    if (ids) ids[base + local] = nd.id;
  }
  T v = nd.dim2;
  if (m >= 2) {
    const T c = submin[base + 2 * local + 1];
    v = c < v ? c : v;
  }
  if (m >= 3) {
    const T c = submin[base + 2 * local + 2];
    v = c < v ? c : v;
  }
  submin[base + local] = v;
}

template <typename T, typename IS>
Status submin_typed(const void* nodes, void* submin, void* ids, uint32_t levels, uint32_t shift, uint32_t ntrees,
                    uint32_t full_M, uint32_t last_M, hipStream_t s) {
  for (int t = static_cast<int>(levels) - 1; t >= 0; t--) {
    const uint64_t work = (1ull << t) * ntrees;
    k_submin_level<T, IS><<<static_cast<unsigned>((work + 255) / 256), 256, 0, s>>>(
        static_cast<const Node<T, IS>*>(nodes), static_cast<T*>(submin), static_cast<IS*>(ids),
        static_cast<uint32_t>(t), shift, ntrees, full_M, last_M);
  }
  return hip_status(hipGetLastError(), "Error in launching subtree minima");
}

// ---------------------------------------------------------------------------
// Forest of shallow trees (StaticPSTGPUArr). Tree c holds the input points
// [c*St, min(n, (c+1)*St)), the reference's consecutive chunks
// (pst/static-pst-gpu-arr-populate-trees.tu:25-40, pst/static-pst-gpu-arr.tu:
// 1037-1060), and is the tree the deep construction would build for that
// chunk alone. One workgroup per tree: the chunk's key1 and key2 orders come
// from bitonic sorts in LDS, then lds_build fills the tree level by level.
// Tree c's records start at c << L, with St = 2^L - 1.
// ---------------------------------------------------------------------------
template <typename Before>
__device__ void bitonic_sort(uint16_t* idx, uint32_t N, Before before) {
  for (uint32_t k = 2; k <= N; k <<= 1) {
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      for (uint32_t t = threadIdx.x; t < N / 2; t += blockDim.x) {
        const uint32_t i = (t / j) * 2 * j + (t % j);
        const uint32_t l = i + j;
        const uint16_t a = idx[i], b = idx[l];
        const bool up = (i & k) == 0;
        if (up ? before(b, a) : before(a, b)) {
          idx[i] = b;
          idx[l] = a;
        }
      }
      __syncthreads();
    }
  }
}

struct LocalPerm {
  const uint16_t* ord2;
  uint64_t first;
  __device__ uint32_t operator()(uint32_t r) const { return static_cast<uint32_t>(first + ord2[r]); }
};

// Dynamic LDS for a tree of up to N (a power of two) points.
__host__ __device__ constexpr size_t forest_lds_bytes(uint32_t N) {
  return static_cast<size_t>(N) * (3 * 8 + 2 * 2 + 2 * 4) + kForestBlock * 8 + (kForestBlock / kWave) * 8;
}

template <typename T, typename I>
__global__ __launch_bounds__(kForestBlock) void k_forest_build(const Point<T, I>* __restrict__ pts, uint64_t n,
                                                               uint64_t tree0, uint32_t St, uint32_t L, uint32_t N,
                                                               Node<T, typename IdStore<I>::type>* nodes, T* submin,
                                                               typename IdStore<I>::type* ids, T* bounds,
                                                               int* __restrict__ nan_flag) {
  using IS = typename IdStore<I>::type;
  extern __shared__ __align__(16) unsigned char lds[];
  uint64_t* k1 = reinterpret_cast<uint64_t*>(lds);
  uint64_t* k2 = k1 + N;
  uint64_t* kid = k2 + N;
  unsigned long long* sres = reinterpret_cast<unsigned long long*>(kid + N);
  unsigned long long* wred = sres + kForestBlock;
  uint32_t* bufA = reinterpret_cast<uint32_t*>(wred + kForestBlock / kWave);
  uint32_t* bufB = bufA + N;
  uint16_t* o1 = reinterpret_cast<uint16_t*>(bufB + N);
  uint16_t* o2 = o1 + N;

  const uint64_t c = tree0 + blockIdx.x;
  const uint64_t first = c * St;
  const uint32_t m = static_cast<uint32_t>(n - first < St ? n - first : St);
  for (uint32_t x = threadIdx.x; x < N; x += blockDim.x) {
    o1[x] = static_cast<uint16_t>(x);
    o2[x] = static_cast<uint16_t>(x);
    if (x < m) {
      const Point<T, I> p = pts[first + x];
      bool bad = is_nan(p.dim1_val) || is_nan(p.dim2_val);
      k1[x] = static_cast<uint64_t>(ord_key(p.dim1_val));
      k2[x] = static_cast<uint64_t>(ord_key(p.dim2_val));
      if constexpr (has_id_v<I>) {
        bad |= is_nan(p.id);
        kid[x] = static_cast<uint64_t>(ord_key(p.id));
      } else {
        kid[x] = 0;
      }
      if (bad) *nan_flag = 1;
    }
  }
  __syncthreads();
  // key1 = (dim1, id, index) ascending; key2 = (dim2, id, index) descending
  // (rank 0 is the node point), the reference's compareDim1/compareDim2 with
  // comparisonTiebreaker (helpers/point-struct.h:54-92, 146-188)
  bitonic_sort(o1, N, [&](uint16_t a, uint16_t b) {
    if (a >= m) return false;
    if (b >= m) return true;
    if (k1[a] != k1[b]) return k1[a] < k1[b];
    if (kid[a] != kid[b]) return kid[a] < kid[b];
    return a < b;
  });
  bitonic_sort(o2, N, [&](uint16_t a, uint16_t b) {
    if (a >= m) return false;
    if (b >= m) return true;
    if (k2[a] != k2[b]) return k2[a] > k2[b];
    if (kid[a] != kid[b]) return kid[a] > kid[b];
    return a > b;
  });
  if (threadIdx.x == 0) {  // the tree's dim1 range
    bounds[2 * c] = pts[first + o1[0]].dim1_val;
    bounds[2 * c + 1] = pts[first + o1[m - 1]].dim1_val;
  }
  for (uint32_t r = threadIdx.x; r < m; r += blockDim.x) bufB[o2[r]] = r;
  __syncthreads();
  for (uint32_t x = threadIdx.x; x < m; x += blockDim.x) bufA[x] = bufB[o1[x]];
  __syncthreads();
  nodes += c << L;
  lds_build<T, IS>(bufA, bufB, sres, wred, m, 0, reinterpret_cast<const Point<T, IS>*>(pts), LocalPerm{o2, first},
                   nodes);
  // subtree minima of dim2 and the ID array, bottom level first (what
  // k_submin_level computes), from the records this workgroup wrote
  submin += c << L;
  const uint64_t Mp = static_cast<uint64_t>(m) + 1;
  for (int u = 31 - __clz(static_cast<int>(m)); u >= 0; u--) {
    for (uint32_t k = threadIdx.x; k < (1u << u); k += blockDim.x) {
      const int64_t ms = level_size(Mp, u, k);
      if (ms < 1) continue;
      const uint32_t s = (1u << u) - 1 + k;
      T v = nodes[s].dim2;
      if constexpr (has_id_v<I>) {
        if (ids) ids[(c << L) + s] = nodes[s].id;
      }
      if (ms >= 2) {
        const T b = submin[2 * s + 1];
        v = b < v ? b : v;
      }
      if (ms >= 3) {
        const T b = submin[2 * s + 2];
        v = b < v ? b : v;
      }
      submin[s] = v;
    }
    __syncthreads();
  }
}

// Forest export: per tree the reference's layout for its own slot count,
// trees concatenated (tree c at position c*St of every array).
template <typename T, typename IS>
__global__ void k_forest_export(const Node<T, IS>* __restrict__ nodes, uint64_t n, uint64_t St, uint32_t L,
                                uint64_t ntrees, uint64_t total, unsigned char* __restrict__ blob, size_t o1,
                                size_t o2, size_t om, size_t oi, size_t ob) {
  const uint64_t p = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= total) return;
  uint64_t c = p / St;
  if (c >= ntrees) c = ntrees - 1;
  const uint64_t s = p - c * St;
  const uint64_t mc = (c + 1 < ntrees) ? St : n - c * St;
  const int64_t m = subtree_size(mc + 1, s);
  T d1 = T(0), d2 = T(0), md = T(0);
  unsigned char bc = 0;
  const Node<T, IS>* nd = nodes + (c << L) + s;
  if (m >= 1) {
    d1 = nd->dim1;
    md = nd->med;
    d2 = nd->dim2;
    bc = static_cast<unsigned char>((m >= 2 ? 2 : 0) | (m >= 3 ? 1 : 0));
  }
  reinterpret_cast<T*>(blob + o1)[p] = d1;
  reinterpret_cast<T*>(blob + o2)[p] = d2;
  reinterpret_cast<T*>(blob + om)[p] = md;
  if constexpr (has_id_v<IS>) {
    IS id = 0;
    if (m >= 1) id = nd->id;
    reinterpret_cast<IS*>(blob + oi)[p] = id;
  }
  blob[ob + p] = bc;
}

// Reference-layout export: dim1[S] dim2[S] med[S] ids[S] bitcodes[S].
template <typename T, typename IS>
__global__ void k_export(const Node<T, IS>* __restrict__ nodes, uint64_t S,
                         uint64_t M, unsigned char* __restrict__ blob, size_t o1, size_t o2, size_t om,
                         size_t oi, size_t ob) {
  const uint64_t s = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= S) return;
  const int64_t m = subtree_size(M, s);
  T d1 = T(0), d2 = T(0), md = T(0);
  unsigned char bc = 0;
  if (m >= 1) {
    d1 = nodes[s].dim1;
    md = nodes[s].med;
    d2 = nodes[s].dim2;
    bc = static_cast<unsigned char>((m >= 2 ? 2 : 0) | (m >= 3 ? 1 : 0));
  }
  reinterpret_cast<T*>(blob + o1)[s] = d1;
  reinterpret_cast<T*>(blob + o2)[s] = d2;
  reinterpret_cast<T*>(blob + om)[s] = md;
  if constexpr (has_id_v<IS>) {
    IS id = 0;
    if (m >= 1) id = nodes[s].id;
    reinterpret_cast<IS*>(blob + oi)[s] = id;
  }
  blob[ob + s] = bc;
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
struct DevBuf {
  void* p = nullptr;
  ~DevBuf() { (void)dev_free(p); }  // early returns: queued kernels may still use it
  hipError_t alloc(size_t bytes) { return dev_alloc(&p, bytes); }
  void release_idle() {  // after the caller has waited for every use
    (void)dev_free_idle(p);
    p = nullptr;
  }
  template <typename U>
  U* as() const {
    return static_cast<U*>(p);
  }
};

inline unsigned grid_for(size_t n, unsigned block) { return static_cast<unsigned>((n + block - 1) / block); }

// Construction buffers of n points, carved from two blocks. Block A: keys and
// three 32-bit words per point; block B: keys, two words per point, sort
// scratch, minima and segment tables. Values that carry (dim2, ID) take two
// words per point in each block.
struct BuildLayout {
  size_t key0, v0, v2, flags;                       // in A
  size_t key1, v1, r2, tmp, mins, segs;             // in B
  size_t total_a, total_b, total;
  size_t tmp_bytes;
  uint32_t t0;
};

inline size_t al256(size_t b) { return (b + 255) & ~size_t{255}; }

// Block minima of n values: steps 1, 2 and 3 of the hierarchy.
inline size_t min_words(size_t n) {
  const size_t n1 = blocks_of(n), n2 = blocks_of(n1);
  return n1 + n2 + blocks_of(n2);
}
// One level's segment table, for levels up to t0.
inline size_t segs_bytes(uint32_t t0) { return (size_t{1} << t0) * (2 + kMaxHoles) * 4; }
inline Segs segs_at(unsigned char* p, uint32_t t0) {
  auto* w = reinterpret_cast<uint32_t*>(p);
  return Segs{w, w + (size_t{1} << t0), w + 2 * (size_t{1} << t0)};
}

template <typename K>
BuildLayout build_layout(size_t n) {
  BuildLayout L{};
  size_t tb = 0;
  if constexpr (sizeof(K) == 4) radix_sort_u32(nullptr, tb, nullptr, nullptr, nullptr, nullptr, n, nullptr);
  else radix_sort_u64(nullptr, tb, nullptr, nullptr, nullptr, nullptr, n, nullptr);
  if (point_sort_tmp_bytes(n) > tb) tb = point_sort_tmp_bytes(n);
  L.tmp_bytes = tb;
  L.t0 = finish_level(static_cast<uint64_t>(n) + 1);
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += al256(bytes ? bytes : 1);
    return at;
  };
  // part A: what the first key kernel writes
  L.key0 = take(n * sizeof(K));
  L.v0 = take(n * 4);
  L.v2 = take(n * 4);
  L.flags = take(16);
  L.total_a = o;
  // part B (offsets from its own start): the rest
  o = 0;
  L.key1 = take(n * sizeof(K));
  L.v1 = take(n * 4);
  L.r2 = take(n * 4);
  L.tmp = take(tb);
  L.mins = take(min_words(n) * 8);
  L.segs = take(2 * segs_bytes(L.t0));
  L.total_b = o;
  L.total = L.total_a + L.total_b;
  return L;
}

// Sort keys wide enough for a dim or an ID of the point type.
template <typename T, typename I>
using BuildKey = typename std::conditional<(sizeof(T) == 8 || (has_id_v<I> && sizeof(I) == 8)), uint64_t,
                                           uint32_t>::type;

// From the key1-ordered array on: the levels above LDS size, the LDS
// subtrees, and the subtree minima and IDs of the levels above them.
template <typename T, typename IS, typename Src>
Status build_levels(Src src, const typename Src::V* A, uint32_t n, uint32_t t0, unsigned char* mins, unsigned char* segs,
                    const BuildOut& out, hipStream_t s) {
  using V = typename Src::V;
  const uint64_t M = static_cast<uint64_t>(n) + 1;
  auto* nodes = static_cast<Node<T, IS>*>(out.nodes);
  Segs cur = segs_at(segs, t0), nxt = segs_at(segs + segs_bytes(t0), t0);
  k_segs_root<<<1, 1, 0, s>>>(cur);
  if (t0 > 0) {
    const uint32_t n1 = blocks_of(n), n2 = blocks_of(n1), n3 = blocks_of(n2);
    V* m1 = reinterpret_cast<V*>(mins);
    V* m2 = m1 + n1;
    V* m3 = m2 + n2;
    constexpr unsigned kWaves = kTopBlock / kWave;
    k_block_min<V><<<n2, kTopBlock, 0, s>>>(A, n, m1, m2);
    k_min_of_mins<V><<<grid_for(n3, kWaves), kTopBlock, 0, s>>>(m2, n2, m3, n3);
    for (uint32_t t = 0; t < t0; t++) {
      k_top_level<T, IS, Src><<<grid_for(size_t{1} << t, kWaves), kTopBlock, 0, s>>>(src, A, m1, m2, m3, n, t, M, cur, nxt,
                                                                                    nodes);
      std::swap(cur, nxt);
    }
  }
  k_finish<T, IS, Src><<<1u << t0, kFinishBlock, 0, s>>>(src, A, n, t0, M, cur, nodes, static_cast<T*>(out.submin),
                                                         static_cast<IS*>(out.ids));
  if (out.submin && t0 > 0) {
    const uint32_t split = t0 > 7 ? t0 - 7 : 0;
    k_top_submin<T, IS><<<1u << split, kTopBlock, 0, s>>>(nodes, static_cast<T*>(out.submin), static_cast<IS*>(out.ids),
                                                          split, t0);
    if (split)
      k_top_submin<T, IS><<<1, kTopBlock, 0, s>>>(nodes, static_cast<T*>(out.submin), static_cast<IS*>(out.ids), 0u,
                                                  split);
  }
  return hip_status(hipGetLastError(), "Error in launching construction kernels");
}

template <typename T, typename I>
Status build_typed(int dtype, int id_dtype, const void* pts_v, size_t n64, BuildOut& out, hipStream_t s,
                   BuildTimes* times) {
  using IS = typename IdStore<I>::type;
  using K = BuildKey<T, I>;
  Status st;
  if (n64 == 0) return st;
  if (n64 >= (1ull << 32) - 1) {
    st.code = 1;
    st.msg = "Error: StaticPSTGPU supports fewer than 2^32 - 1 points";
    return st;
  }
  const uint32_t n = static_cast<uint32_t>(n64);
  const auto* pts = static_cast<const Point<T, I>*>(pts_v);
  constexpr bool kHasId = has_id_v<I>;

  hipEvent_t ev[3] = {};
  if (times)
    for (auto& e : ev) hipEventCreate(&e);
  auto mark = [&](int k) {
    if (times) hipEventRecord(ev[k], s);
  };

  hipError_t e;
#define PST_TRY(expr, what)                         \
  do {                                              \
    e = (expr);                                     \
    if (e != hipSuccess) return hip_status(e, what); \
  } while (0)
  const BuildLayout BL = build_layout<K>(n64);
  DevBuf arena_a, arena_b;
  PST_TRY(arena_a.alloc(BL.total_a), "Error in allocating construction arrays");
  PST_TRY(arena_b.alloc(BL.total_b), "Error in allocating construction arrays");
  unsigned char* base_a = arena_a.as<unsigned char>();
  unsigned char* base_b = arena_b.as<unsigned char>();
  // flags[0]: NaN seen; flags[1]: IDs not in index order (a point sort: keys
  // and values do not stand for the points); flags[2]: a sort's wait ran out
  int* flags = reinterpret_cast<int*>(base_a + BL.flags);
  void* tmp = base_b + BL.tmp;
  auto read_flags = [&](int (&h)[3]) -> hipError_t {
    hipError_t r = hipMemcpyAsync(h, flags, sizeof(h), hipMemcpyDeviceToHost, s);
    return r == hipSuccess ? hipStreamSynchronize(s) : r;
  };
  int hflag[3] = {0, 0, 0};
  mark(0);
  PST_TRY(hipMemsetAsync(flags, 0, 3 * sizeof(int), s), "Error in clearing construction flags");
  // the output arrays: the caller's hook allocates them while the first pass runs
  auto out_arrays = [&]() -> Status {
    if (!out.alloc || out.nodes) return Status{};
    Status sa = out.alloc(out);
    if (!sa.ok()) (void)hipStreamSynchronize(s);  // the queued passes still use the scratch
    return sa;
  };
  bool direct = false;
  if constexpr (sizeof(T) == 4 && sizeof(K) == 4) {
    if (point_sort_takes(dtype, id_dtype)) {
      PST_TRY(point_sort_count(dtype, id_dtype, pts_v, n64, tmp, flags, s), "Error in counting construction keys");
      st = out_arrays();
      if (!st.ok()) return st;
      PST_TRY(read_flags(hflag), "Error in reading construction flags");
      direct = hflag[1] == 0 && hflag[0] == 0;
      if (direct) {
        uint32_t* key_x = reinterpret_cast<uint32_t*>(base_a + BL.key0);
        uint64_t* val_x = reinterpret_cast<uint64_t*>(base_a + BL.v0);  // v0 and v2
        uint32_t* key1 = reinterpret_cast<uint32_t*>(base_b + BL.key1);
        uint64_t* val = reinterpret_cast<uint64_t*>(base_b + BL.v1);    // v1 and r2
        PST_TRY(point_sort_passes(dtype, id_dtype, pts_v, n64, tmp, key_x, val_x, key1, val, flags + 2, s),
                "Error in sorting by dimension 1");
        mark(1);
        st = build_levels<T, IS>(Direct<T, IS>{key1, id_dtype}, val, n, BL.t0, base_b + BL.mins, base_b + BL.segs, out, s);
        if (!st.ok()) return st;
      }
    }
  }
  if (!direct) {
    PST_TRY(hipMemsetAsync(flags, 0, 3 * sizeof(int), s), "Error in clearing construction flags");
    K* key0 = reinterpret_cast<K*>(base_a + BL.key0);
    uint32_t* v0 = reinterpret_cast<uint32_t*>(base_a + BL.v0);
    uint32_t* v2 = reinterpret_cast<uint32_t*>(base_a + BL.v2);
    K* key1 = reinterpret_cast<K*>(base_b + BL.key1);
    uint32_t* v1 = reinterpret_cast<uint32_t*>(base_b + BL.v1);
    uint32_t* r2 = reinterpret_cast<uint32_t*>(base_b + BL.r2);
    const unsigned B = 256;
    const unsigned G = grid_for(n, B);
    int* nan_flag = flags;
    // ---- key2 descending -> perm2 (v1), r2. One sort by dim2 when the IDs
    // are in index order (the sort's index tie-break is then the (id, index)
    // tie-break), else a sort by ID and then a stable one by dim2.
    // 32-bit keys: the dim1 keys are stored by the same kernel, into v2
    constexpr bool kKey1First = sizeof(K) == 4;
    k_keys_single<T, I, K, true, true, false, kHasId>
        <<<G, B, 0, s>>>(pts, n, key0, v0, nullptr, flags, kKey1First ? v2 : nullptr);
    // stable radix sort of (key, value) pairs: kin/vin to kout/vout
    auto sortK = [&](const K* kin, K* kout, const uint32_t* vin, uint32_t* vout) -> hipError_t {
      size_t tb = BL.tmp_bytes;
      if constexpr (sizeof(K) == 4) return radix_sort_u32(tmp, tb, kin, kout, vin, vout, n, s, flags + 2);
      else return radix_sort_u64(tmp, tb, kin, kout, vin, vout, n, s, flags + 2);
    };
    st = out_arrays();
    if (!st.ok()) return st;
    bool ordered = true;
    if constexpr (kHasId) {
      PST_TRY(read_flags(hflag), "Error in reading construction flags");
      ordered = hflag[1] == 0;
    }
    if (ordered) {
      PST_TRY(sortK(key0, key1, v0, v1), "Error in sorting by dimension 2");
    } else {
      if constexpr (kHasId) {
        // v2: the points in (id, index) order, read backwards for key2
        k_keys_id<T, I, K><<<G, B, 0, s>>>(pts, n, key0, v0, nan_flag);
        PST_TRY(sortK(key0, key1, v0, v2), "Error in sorting by ID");
        k_keys_dim_perm<T, I, K, true, true><<<G, B, 0, s>>>(pts, n, v2, key0, v0, nullptr, nan_flag);
        PST_TRY(sortK(key0, key1, v0, v1), "Error in sorting by dimension 2");
      }
    }
    const uint32_t* perm2 = v1;
    k_scatter_rank<<<G, B, 0, s>>>(perm2, n, r2);
    // ---- key1 ascending, carrying r2 -> A (v2; v0 when the dim1 keys came
    // with the dim2 keys, whose sort reads them from v2 and r2 in place)
    const uint32_t* A = v2;
    if (ordered && kKey1First) {
      PST_TRY(sortK(reinterpret_cast<const K*>(v2), key0, r2, v0), "Error in sorting by dimension 1");
      A = v0;
    } else if (ordered) {
      k_keys_single<T, I, K, false, false, false><<<G, B, 0, s>>>(pts, n, key0, v0, r2, flags);
      PST_TRY(sortK(key0, key1, v0, v2), "Error in sorting by dimension 1");
    } else {
      if constexpr (kHasId) {
        k_keys_dim_perm<T, I, K, false, false><<<G, B, 0, s>>>(pts, n, v2, key0, v0, r2, nan_flag);
        PST_TRY(sortK(key0, key1, v0, v2), "Error in sorting by dimension 1");
      }
    }
    mark(1);
    st = build_levels<T, IS>(Ranked<T, IS>{perm2, static_cast<const Point<T, IS>*>(pts_v)}, A, n, BL.t0,
                             base_b + BL.mins, base_b + BL.segs, out, s);
    if (!st.ok()) return st;
  }
  mark(2);
  PST_TRY(read_flags(hflag), "Error in synchronising after construction");
  arena_b.release_idle();
  arena_a.release_idle();
  if (times) {
    hipEventElapsedTime(&times->sort_ms, ev[0], ev[1]);
    hipEventElapsedTime(&times->levels_ms, ev[1], ev[2]);
    for (auto& x : ev) hipEventDestroy(x);
  }
  if (hflag[2]) {
    st.code = 5;
    st.msg = "Error: a construction sort pass waited too long for earlier tiles";
  } else if (hflag[0]) {
    st.code = 3;
    st.msg = "Error: input contains NaN values, which have no order";
  }
#undef PST_TRY
  return st;
}

template <typename T, typename IS>
Status export_typed(size_t n, const void* nodes, void* blob, size_t o1, size_t o2, size_t om,
                    size_t oi, size_t ob, hipStream_t s) {
  if (n == 0) return Status{};
  uint64_t S = 1;
  while (S <= n) S <<= 1;
  S -= 1;
  k_export<T, IS><<<grid_for(S, 256), 256, 0, s>>>(static_cast<const Node<T, IS>*>(nodes), S, n + 1,
                                                    static_cast<unsigned char*>(blob), o1, o2, om, oi, ob);
  return hip_status(hipGetLastError(), "Error in launching tree export");
}

template <typename T, typename I>
Status forest_build_typed(int dtype, int id_dtype, const void* pts_v, size_t n, size_t St, void* nodes_v,
                          void* submin_v, void* ids_v, void* bounds_v, hipStream_t s) {
  using IS = typename IdStore<I>::type;
  if (n == 0) return Status{};
  uint32_t L = 0;
  while ((1ull << L) < St + 1) L++;
  if ((1ull << L) != St + 1 || St > kFinishTile - 1)
    return Status{1, "Error: forest trees hold 2^k - 1 <= 2047 points"};
  const uint64_t ntrees = (n + St - 1) / St;
  const uint32_t N = static_cast<uint32_t>(St + 1);
  const size_t lds = forest_lds_bytes(N);
  auto kern = k_forest_build<T, I>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
  if (e != hipSuccess) return hip_status(e, "Error in sizing forest construction LDS");
  DevBuf flag;
  e = flag.alloc(sizeof(int));
  if (e == hipSuccess) e = hipMemsetAsync(flag.p, 0, sizeof(int), s);
  if (e != hipSuccess) return hip_status(e, "Error in allocating construction flag");
  // full trees of kForestRegMin..kForestRegMax levels a wave each, in
  // registers; a partial last tree and other sizes a workgroup each
  size_t done = 0;
  if (L >= kForestRegMin && L <= kForestRegMax && n >= St) {
    done = n / St;
    Status st = build_forest_full(dtype, id_dtype, L, pts_v, done, nodes_v, submin_v, ids_v, bounds_v, flag.as<int>(), s);
    if (!st.ok()) return st;
  }
  if (done < ntrees)
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(ntrees - done)), dim3(kForestBlock), lds, s,
                       static_cast<const Point<T, I>*>(pts_v), static_cast<uint64_t>(n), static_cast<uint64_t>(done),
                       static_cast<uint32_t>(St), L, N, static_cast<Node<T, IS>*>(nodes_v), static_cast<T*>(submin_v),
                       static_cast<IS*>(ids_v), static_cast<T*>(bounds_v), flag.as<int>());
  e = hipGetLastError();
  if (e != hipSuccess) return hip_status(e, "Error in launching forest construction");
  int hflag = 0;
  e = hipMemcpyAsync(&hflag, flag.p, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return hip_status(e, "Error in synchronising after forest construction");
  flag.release_idle();
  if (hflag) return Status{3, "Error: input contains NaN values, which have no order"};
  return Status{};
}

template <typename T, typename IS>
Status forest_export_typed(size_t n, size_t St, const void* nodes, void* blob, size_t total, size_t o1, size_t o2,
                           size_t om, size_t oi, size_t ob, hipStream_t s) {
  if (n == 0) return Status{};
  uint32_t L = 0;
  while ((1ull << L) < St + 1) L++;
  const uint64_t ntrees = (n + St - 1) / St;
  k_forest_export<T, IS><<<grid_for(total, 256), 256, 0, s>>>(static_cast<const Node<T, IS>*>(nodes), n, St, L,
                                                              ntrees, total, static_cast<unsigned char*>(blob), o1,
                                                              o2, om, oi, ob);
  return hip_status(hipGetLastError(), "Error in launching forest export");
}

template <typename F>
Status with_t(int dt, F&& f) {
  switch (dt) {
    case F32: return f(float{});
    case F64: return f(double{});
    case I32: return f(int32_t{});
    case I64: return f(int64_t{});
  }
  return Status{1, "Error: unsupported data type code " + std::to_string(dt)};
}
template <typename F>
Status with_id(int idt, F&& f) {
  switch (idt) {
    case NO_ID: return f(NoId{});
    case F32: return f(float{});
    case F64: return f(double{});
    case I32: return f(int32_t{});
    case I64: return f(int64_t{});
    case U32: return f(uint32_t{});
    case U64: return f(uint64_t{});
  }
  return Status{1, "Error: unsupported ID type code " + std::to_string(idt)};
}

}  // namespace

Status build_tree(int dtype, int id_dtype, const void* pts_d, size_t n, BuildOut& out, hipStream_t stream,
                  BuildTimes* times) {
  return with_t(dtype, [&](auto t) {
    return with_id(id_dtype, [&](auto i) { return build_typed<decltype(t), decltype(i)>(dtype, id_dtype, pts_d, n, out, stream, times); });
  });
}

Status build_tree(int dtype, int id_dtype, const void* pts_d, size_t n, void* nodes_d, hipStream_t stream,
                  BuildTimes* times, void* submin_d, void* ids_d) {
  BuildOut out;
  out.nodes = nodes_d;
  out.submin = submin_d;
  out.ids = ids_d;
  return build_tree(dtype, id_dtype, pts_d, n, out, stream, times);
}

namespace {
BuildLayout layout_of(int dtype, int id_dtype, size_t n) {
  BuildLayout L{};
  (void)with_t(dtype, [&](auto t) {
    return with_id(id_dtype, [&](auto i) {
      L = build_layout<BuildKey<decltype(t), decltype(i)>>(n);
      return Status{};
    });
  });
  return L;
}
}  // namespace

size_t build_scratch_bytes(int dtype, int id_dtype, size_t n) { return layout_of(dtype, id_dtype, n).total; }
size_t build_arena_bytes(int dtype, int id_dtype, size_t n) { return layout_of(dtype, id_dtype, n).total_a; }

Status export_tree(int dtype, int id_dtype, size_t n, const void* nodes_d, void* blob_d,
                   size_t o1, size_t o2, size_t om, size_t oi, size_t ob, hipStream_t stream) {
  return with_t(dtype, [&](auto t) {
    return with_id(id_dtype, [&](auto i) {
      using IS = typename IdStore<decltype(i)>::type;
      return export_typed<decltype(t), IS>(n, nodes_d, blob_d, o1, o2, om, oi, ob, stream);
    });
  });
}

}  // namespace pst

namespace pst {

Status build_forest(int dtype, int id_dtype, const void* pts_d, size_t n, size_t slots_per_tree, void* nodes_d,
                    void* submin_d, void* ids_d, void* bounds_d, hipStream_t stream) {
  return with_t(dtype, [&](auto t) {
    return with_id(id_dtype, [&](auto i) {
      return forest_build_typed<decltype(t), decltype(i)>(dtype, id_dtype, pts_d, n, slots_per_tree, nodes_d, submin_d,
                                                          ids_d, bounds_d, stream);
    });
  });
}

Status export_forest(int dtype, int id_dtype, size_t n, size_t slots_per_tree, const void* nodes_d, void* blob_d,
                     size_t total_slots, size_t o1, size_t o2, size_t om, size_t oi, size_t ob,
                     hipStream_t stream) {
  return with_t(dtype, [&](auto t) {
    return with_id(id_dtype, [&](auto i) {
      using IS = typename IdStore<decltype(i)>::type;
      return forest_export_typed<decltype(t), IS>(n, slots_per_tree, nodes_d, blob_d, total_slots, o1, o2, om, oi,
                                                  ob, stream);
    });
  });
}

}  // namespace pst

namespace pst {

Status build_submin(int dtype, int id_dtype, size_t n, size_t slots_per_tree, const void* nodes_d, void* submin_d,
                    void* ids_d, hipStream_t stream) {
  if (n == 0) return Status{};
  uint32_t shift, ntrees, full_M, last_M, levels = 0;
  if (slots_per_tree == 0) {
    shift = 31;
    ntrees = 1;
    full_M = last_M = static_cast<uint32_t>(n + 1);
    while ((1ull << levels) <= n) levels++;
  } else {
    shift = 0;
    while ((1ull << shift) < slots_per_tree + 1) shift++;
    ntrees = static_cast<uint32_t>((n + slots_per_tree - 1) / slots_per_tree);
    full_M = static_cast<uint32_t>(slots_per_tree + 1);
    last_M = static_cast<uint32_t>(n - (ntrees - 1ull) * slots_per_tree + 1);
    levels = shift;
  }
  return with_t(dtype, [&](auto t) {
    return with_id(id_dtype, [&](auto i) {
      using IS = typename IdStore<decltype(i)>::type;
      return submin_typed<decltype(t), IS>(nodes_d, submin_d, ids_d, levels, shift, ntrees, full_M, last_M, stream);
    });
  });
}

}  // namespace pst
