// Construction of the full trees of a forest (StaticPSTGPUArr) whose trees
// hold 2^LOGN - 1 points, LOGN = 5..9: one wave per tree (two trees of 31
// points share a wave), every point in a register, no workgroup barrier.
//
// The tree is the one k_forest_build (pst_build.hip) gives for the chunk:
// node = max key2, med = dim1 of the floor(m/2)-th remaining point in key1
// order, key1 = (dim1, id, index), key2 = (dim2, id, index). Here both
// orders come from bitonic sorts over registers and lane exchanges, and the
// levels use what a full tree's sizes allow: with N = 2^LOGN positions (the
// last one a hole), the segment of level u, position k sits at the aligned
// block [k g, (k + 1) g), g = N >> u, its last position a hole. Taking the
// node at position q out and splitting the rest into halves of L = g/2 - 1
// points then moves no point by more than one position:
//   q < mid (= block + L): positions q..mid-1 take their right neighbour;
//   q > mid:               positions mid+1..q take their left neighbour;
//   position mid becomes the hole after the left half.
// So a level is one segmented minimum and one shift by a lane. The med is
// the last point of the new left half (position mid - 1).
//
// The kernel also writes what searches need beside the records: each slot's
// subtree minimum of dim2, the ID array and the tree's dim1 range.
//
// Bound by instruction issue and memory together: 16.7M f32/u32 points in
// trees of 127 points (2^24 metacells) on MI355X take 0.174 ms, 3.4 TB/s of
// the 0.6 GB read and written. One 256-thread workgroup per tree with sorts
// in LDS took 2.99 ms, plus 0.15 ms of subtree-minimum passes and 0.05 ms for
// the ranges, which this kernel gives on the way.
#include "pst_internal.hpp"

namespace pst {

namespace {

// Waves per workgroup: four, two where four trees of 511 points with 64-bit
// dims would pass the 64 KB of static LDS.
constexpr int reg_waves(int log_n) { return log_n >= 9 ? 2 : 4; }

// Orders a wave's LDS accesses around it.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value of lane ^ MASK: DPP where a pattern exists, else the LDS crossbar.
template <int MASK>
__device__ inline uint32_t lane_xor(uint32_t v) {
  const int x = static_cast<int>(v);
  if constexpr (MASK == 1) return __builtin_amdgcn_mov_dpp(x, 0xB1, 0xf, 0xf, true);        // quad_perm 1,0,3,2
  else if constexpr (MASK == 2) return __builtin_amdgcn_mov_dpp(x, 0x4E, 0xf, 0xf, true);   // quad_perm 2,3,0,1
  else if constexpr (MASK == 4)  // half-row mirror (lane ^ 7), then quad_perm 3,2,1,0 (lane ^ 3)
    return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(x, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
  else if constexpr (MASK == 8) return __builtin_amdgcn_mov_dpp(x, 0x128, 0xf, 0xf, true);  // row_ror:8
  else if constexpr (MASK == 16) return __builtin_amdgcn_ds_swizzle(x, 0x401F);             // xor 16
  else return static_cast<uint32_t>(__shfl_xor(x, MASK, kWave));
}
template <int MASK>
__device__ inline uint64_t lane_xor(uint64_t v) {
  return (static_cast<uint64_t>(lane_xor<MASK>(static_cast<uint32_t>(v >> 32))) << 32) |
         lane_xor<MASK>(static_cast<uint32_t>(v));
}

// A key with its tie-break word (tie << 16 | index): one 64-bit integer for
// 32-bit keys.
template <typename K>
struct El;
template <>
struct El<uint32_t> {
  uint64_t v;
  __device__ static El make(uint32_t k, uint32_t w) { return {(static_cast<uint64_t>(k) << 32) | w}; }
  __device__ uint32_t word() const { return static_cast<uint32_t>(v); }
  __device__ bool before(const El& o) const { return v < o.v; }
  template <int MASK>
  __device__ El xored() const {
    return {lane_xor<MASK>(v)};
  }
};
template <>
struct El<uint64_t> {
  uint64_t k;
  uint32_t w;
  __device__ static El make(uint64_t k, uint32_t w) { return {k, w}; }
  __device__ uint32_t word() const { return w; }
  __device__ bool before(const El& o) const { return k < o.k || (k == o.k && w < o.w); }
  template <int MASK>
  __device__ El xored() const {
    return {lane_xor<MASK>(k), lane_xor<MASK>(w)};
  }
};

// Bitonic sort of the N positions p0 + e (E consecutive ones per lane),
// ascending; for N < 64 each aligned group of N lanes sorts its own.
template <int N, int E, int K, int J, typename X>
__device__ inline void bitonic_steps(X (&x)[E], uint32_t p0) {
  if constexpr (J < E) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int f = e ^ J;
      if (f > e) {
        const bool up = ((p0 + e) & K) == 0;
        const bool swap = x[f].before(x[e]) == up;
        const X a = x[e], b = x[f];
        x[e] = swap ? b : a;
        x[f] = swap ? a : b;
      }
    }
  } else {
    // keep the smaller where bit J of the position agrees with the direction
    const bool small = ((p0 & J) == 0) == ((p0 & K) == 0);
#pragma unroll
    for (int e = 0; e < E; e++) {
      const X o = x[e].template xored<J / E>();
      if (o.before(x[e]) == small) x[e] = o;
    }
  }
  if constexpr (J > 1) bitonic_steps<N, E, K, J / 2>(x, p0);
  else if constexpr (K < N) bitonic_steps<N, E, K * 2, K>(x, p0);
}

// Minimum over aligned groups of LANES lanes, in every lane (inputs of the
// mirrored steps are already equal within the mirrored halves).
template <int LANES>
__device__ inline uint32_t group_min(uint32_t v) {
  auto mn = [](uint32_t a, uint32_t b) { return a < b ? a : b; };
  if constexpr (LANES >= 2) v = mn(v, lane_xor<1>(v));
  if constexpr (LANES >= 4) v = mn(v, lane_xor<2>(v));
  if constexpr (LANES >= 8)
    v = mn(v, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x141, 0xf, 0xf, true)));
  if constexpr (LANES >= 16)
    v = mn(v, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x140, 0xf, 0xf, true)));
  if constexpr (LANES >= 32) v = mn(v, lane_xor<16>(v));
  if constexpr (LANES >= 64) v = mn(v, lane_xor<32>(v));
  return v;
}

// Order key of a stored ID of the given code (a float ID is stored as its bits).
template <typename IS>
__device__ inline IS id_key(IS id, int code) {
  if constexpr (sizeof(IS) == 4) {
    if (code == F32) return ord_key(__builtin_bit_cast(float, id));
    if (code == I32) return ord_key(static_cast<int32_t>(id));
  } else {
    if (code == F64) return ord_key(__builtin_bit_cast(double, id));
    if (code == I64) return ord_key(static_cast<int64_t>(id));
  }
  return id;
}
template <typename IS>
__device__ inline bool id_nan(IS id, int code) {
  if constexpr (sizeof(IS) == 4) return code == F32 && is_nan(__builtin_bit_cast(float, id));
  else return code == F64 && is_nan(__builtin_bit_cast(double, id));
}

template <typename T>
struct Range1 {
  T lo, hi;
};

constexpr uint32_t kHole = 0xffffu;  // position without a point

// One level: v[e] is the key2 rank of the point at position p0 + e (kHole:
// none). Notes each segment's node and med (as ranks) at their slots and
// moves the points to the next level's positions.
template <int LOGN, int E, int U>
__device__ inline void level_steps(uint32_t (&v)[E], uint32_t p0, uint16_t* node_r, uint16_t* med_r) {
  constexpr int N = 1 << LOGN;
  constexpr int g = N >> U;  // positions per segment
  uint32_t m[E];
  if constexpr (g > E) {
    uint32_t best = ~0u;
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t k = (v[e] << 16) | (p0 + e);
      best = k < best ? k : best;
    }
    best = group_min<g / E>(best);
#pragma unroll
    for (int e = 0; e < E; e++) m[e] = best;
  } else {
#pragma unroll
    for (int b = 0; b < E; b += g) {
      uint32_t best = ~0u;
#pragma unroll
      for (int e = b; e < b + g; e++) {
        const uint32_t k = (v[e] << 16) | (p0 + e);
        best = k < best ? k : best;
      }
#pragma unroll
      for (int e = b; e < b + g; e++) m[e] = best;
    }
  }
  // neighbours across lanes (wave_shl / wave_shr by one)
  const uint32_t after = __builtin_amdgcn_update_dpp(static_cast<int>(kHole), static_cast<int>(v[0]), 0x130, 0xf, 0xf, false);
  const uint32_t prior = __builtin_amdgcn_update_dpp(static_cast<int>(kHole), static_cast<int>(v[E - 1]), 0x138, 0xf, 0xf, false);
  uint32_t nv[E];
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t p = p0 + e;
    const uint32_t q = m[e] & 0xffffu;
    const uint32_t mid = (p & ~static_cast<uint32_t>(g - 1)) + g / 2 - 1;
    const uint32_t next = e + 1 < E ? v[e + 1 < E ? e + 1 : e] : after;
    const uint32_t prev = e > 0 ? v[e > 0 ? e - 1 : 0] : prior;
    uint32_t x = v[e];
    if (p >= q && p < mid) x = next;
    if (p > mid && p <= q) x = prev;
    if (p == mid) x = kHole;
    nv[e] = x;
    const uint32_t h = (1u << U) - 1 + (p >> (LOGN - U));
    if (p == q) {
      node_r[h] = static_cast<uint16_t>(m[e] >> 16);
      if constexpr (g == 2) med_r[h] = static_cast<uint16_t>(m[e] >> 16);
    }
    if constexpr (g > 2) {
      if (p + 1 == mid) med_r[h] = static_cast<uint16_t>(x);
    }
  }
#pragma unroll
  for (int e = 0; e < E; e++) v[e] = nv[e];
  if constexpr (U + 1 < LOGN) level_steps<LOGN, E, U + 1>(v, p0, node_r, med_r);
}

template <typename T, typename IS, int LOGN>
__global__ __launch_bounds__(reg_waves(LOGN) * kWave) void k_forest_reg(const Point<T, IS>* __restrict__ pts, uint32_t ntrees,
                                                          int id_code, Node<T, IS>* __restrict__ nodes,
                                                          T* __restrict__ submin, IS* __restrict__ ids,
                                                          Range1<T>* __restrict__ bounds, int* __restrict__ nan_flag) {
  constexpr int kRegWaves = reg_waves(LOGN);
  constexpr int N = 1 << LOGN;
  constexpr int E = N > kWave ? N / kWave : 1;   // points per lane
  constexpr int TPW = N < kWave ? kWave / N : 1;  // trees per wave
  constexpr int W = N * TPW;                      // positions per wave
  constexpr bool kHasId = has_id_v<IS>;
  using K = decltype(ord_key(T{}));
  __shared__ T s_d1[kRegWaves][W];
  __shared__ T s_d2[kRegWaves][W];
  __shared__ T s_sub[kRegWaves][W];
  using IdSlot = typename std::conditional<kHasId, IS, uint8_t>::type;
  __shared__ IdSlot s_id[kRegWaves][kHasId ? W : 1];
  __shared__ uint16_t s_r2[kRegWaves][W];    // point -> key2 rank (before that: point -> ID order)
  __shared__ uint16_t s_ord2[kRegWaves][W];  // key2 rank -> point
  __shared__ uint16_t s_node[kRegWaves][W];  // slot -> rank of its node
  __shared__ uint16_t s_med[kRegWaves][W];   // slot -> rank of its med point
  const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const uint32_t sub = TPW > 1 ? lane / N : 0;  // tree within the wave
  const uint32_t tree = (blockIdx.x * kRegWaves + wave) * TPW + sub;
  const bool active = tree < ntrees;
  const uint32_t p0 = TPW > 1 ? lane % N : lane * E;
  T* d1 = s_d1[wave] + sub * N;
  T* d2 = s_d2[wave] + sub * N;
  T* smin = s_sub[wave] + sub * N;
  IdSlot* idv = s_id[wave] + (kHasId ? sub * N : 0);
  uint16_t* r2 = s_r2[wave] + sub * N;
  uint16_t* ord2 = s_ord2[wave] + sub * N;
  uint16_t* node_r = s_node[wave] + sub * N;
  uint16_t* med_r = s_med[wave] + sub * N;

  const Point<T, IS>* tp = pts + static_cast<uint64_t>(active ? tree : 0) * (N - 1);
  K k1[E], k2[E];
  uint32_t tie[E];
  bool bad = false;
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t p = p0 + e;
    k1[e] = k2[e] = 0;
    tie[e] = p;
    if (active && p < N - 1) {
      const Point<T, IS> r = tp[p];
      bad |= is_nan(r.dim1_val) || is_nan(r.dim2_val);
      d1[p] = r.dim1_val;
      d2[p] = r.dim2_val;
      k1[e] = ord_key(r.dim1_val);
      k2[e] = ord_key(r.dim2_val);
      if constexpr (kHasId) {
        bad |= id_nan(r.id, id_code);
        idv[p] = r.id;
      }
    }
  }
  if (bad) *nan_flag = 1;
  wave_sync();
  if constexpr (kHasId) {
    // ties are broken by (id, index): the index alone where IDs ascend with
    // it, else the position in (id, index) order
    bool unordered = false;
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t p = p0 + e;
      if (active && p + 2 < N) unordered |= id_key(idv[p], id_code) > id_key(idv[p + 1], id_code);
    }
    if (__ballot(unordered)) {
      El<IS> x[E];
#pragma unroll
      for (int e = 0; e < E; e++) {
        const uint32_t p = p0 + e;
        const bool real = active && p < N - 1;
        x[e] = El<IS>::make(real ? id_key(idv[p], id_code) : static_cast<IS>(~IS(0)), p);
      }
      bitonic_steps<N, E, 2, 1>(x, p0);
#pragma unroll
      for (int e = 0; e < E; e++) r2[x[e].word() & (N - 1)] = static_cast<uint16_t>(p0 + e);
      wave_sync();
#pragma unroll
      for (int e = 0; e < E; e++) tie[e] = r2[p0 + e];
      wave_sync();
    }
  }
  El<K> x[E];
  // key2 descending: rank 0 is the node point; holes last
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t p = p0 + e;
    x[e] = active && p < N - 1 ? El<K>::make(static_cast<K>(~k2[e]), ((0xffffu - tie[e]) << 16) | p)
                               : El<K>::make(static_cast<K>(~K(0)), ~0u);
  }
  bitonic_steps<N, E, 2, 1>(x, p0);
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t i = x[e].word() & (N - 1);
    ord2[p0 + e] = static_cast<uint16_t>(i);
    r2[i] = static_cast<uint16_t>(p0 + e);
  }
  // key1 ascending
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t p = p0 + e;
    x[e] = active && p < N - 1 ? El<K>::make(k1[e], (tie[e] << 16) | p) : El<K>::make(static_cast<K>(~K(0)), ~0u);
  }
  bitonic_steps<N, E, 2, 1>(x, p0);
  wave_sync();
  uint32_t v[E];
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t p = p0 + e;
    const uint32_t i = x[e].word() & (N - 1);
    v[e] = p < N - 1 ? r2[i] : kHole;
    if (active && p == 0) bounds[tree].lo = d1[i];
    if (active && p == N - 2) bounds[tree].hi = d1[i];
  }
  level_steps<LOGN, E, 0>(v, p0, node_r, med_r);
  wave_sync();
  // node records, IDs and subtree minima, slot by slot
  const uint64_t base = static_cast<uint64_t>(tree) << LOGN;
  const uint32_t h0 = TPW > 1 ? lane % N : lane;
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t h = h0 + e * kWave;
    if (h < N - 1) {
      const uint32_t i = ord2[node_r[h] & (N - 1)];
      const uint32_t im = ord2[med_r[h] & (N - 1)];
      smin[h] = d2[i];
      if (active) {
        Node<T, IS> r;
        r.dim1 = d1[i];
        r.dim2 = d2[i];
        r.med = d1[im];
        if constexpr (kHasId) {
          r.id = idv[i];
          if (ids) ids[base + h] = r.id;
        }
        nodes[base + h] = r;
      }
    }
  }
  wave_sync();
#pragma unroll
  for (int u = LOGN - 2; u >= 0; u--) {
    for (uint32_t k = h0; k < (1u << u); k += kWave) {
      const uint32_t s = (1u << u) - 1 + k;
      T b = smin[s];
      const T l = smin[2 * s + 1], r = smin[2 * s + 2];
      b = l < b ? l : b;
      b = r < b ? r : b;
      smin[s] = b;
    }
    wave_sync();
  }
  if (active) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t h = h0 + e * kWave;
      if (h < N - 1) submin[base + h] = smin[h];
    }
  }
}

template <typename T, typename IS, int LOGN>
Status launch(const void* pts, uint32_t ntrees, int id_code, void* nodes, void* submin, void* ids, void* bounds,
              int* nan_flag, hipStream_t s) {
  constexpr uint32_t per = reg_waves(LOGN) * ((1 << LOGN) < kWave ? kWave >> LOGN : 1);
  k_forest_reg<T, IS, LOGN><<<(ntrees + per - 1) / per, reg_waves(LOGN) * kWave, 0, s>>>(
      static_cast<const Point<T, IS>*>(pts), ntrees, id_code, static_cast<Node<T, IS>*>(nodes),
      static_cast<T*>(submin), static_cast<IS*>(ids), static_cast<Range1<T>*>(bounds), nan_flag);
  return hip_status(hipGetLastError(), "Error in launching forest construction");
}

template <typename T, typename IS>
Status launch_n(uint32_t log_n, const void* pts, uint32_t ntrees, int id_code, void* nodes, void* submin, void* ids,
                void* bounds, int* nan_flag, hipStream_t s) {
  switch (log_n) {
    case 5: return launch<T, IS, 5>(pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
    case 6: return launch<T, IS, 6>(pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
    case 7: return launch<T, IS, 7>(pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
    case 8: return launch<T, IS, 8>(pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
    case 9: return launch<T, IS, 9>(pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
  }
  return Status{1, "Error: forest trees of this size are built by workgroups"};
}

template <typename T>
Status launch_id(int id_code, uint32_t log_n, const void* pts, uint32_t ntrees, void* nodes, void* submin, void* ids,
                 void* bounds, int* nan_flag, hipStream_t s) {
  switch (id_code) {
    case NO_ID: return launch_n<T, NoId>(log_n, pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
    case F32: case I32: case U32:
      return launch_n<T, uint32_t>(log_n, pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
    case F64: case I64: case U64:
      return launch_n<T, uint64_t>(log_n, pts, ntrees, id_code, nodes, submin, ids, bounds, nan_flag, s);
  }
  return Status{1, "Error: unsupported ID type code " + std::to_string(id_code)};
}

}  // namespace

Status build_forest_full(int dtype, int id_dtype, uint32_t log_n, const void* pts_d, size_t ntrees, void* nodes_d,
                         void* submin_d, void* ids_d, void* bounds_d, int* nan_flag_d, hipStream_t s) {
  const uint32_t nt = static_cast<uint32_t>(ntrees);
  switch (dtype) {
    case F32: return launch_id<float>(id_dtype, log_n, pts_d, nt, nodes_d, submin_d, ids_d, bounds_d, nan_flag_d, s);
    case F64: return launch_id<double>(id_dtype, log_n, pts_d, nt, nodes_d, submin_d, ids_d, bounds_d, nan_flag_d, s);
    case I32: return launch_id<int32_t>(id_dtype, log_n, pts_d, nt, nodes_d, submin_d, ids_d, bounds_d, nan_flag_d, s);
    case I64: return launch_id<int64_t>(id_dtype, log_n, pts_d, nt, nodes_d, submin_d, ids_d, bounds_d, nan_flag_d, s);
  }
  return Status{1, "Error: unsupported data type code " + std::to_string(dtype)};
}

}  // namespace pst
