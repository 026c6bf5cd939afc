// Isosurface extraction over active metacells: the consumer of the metacell
// IDs an isovalue search returns. The reference stops at those IDs and
// copies them back "for on-device marching cubes"
// (testers/pst-tester-functions.tu:230-252).
//
// Method: marching tetrahedra. Each voxel (cube of 8 grid vertices, corner k
// at offset (k & 1, k >> 1 & 1, k >> 2)) is cut into the 6 tetrahedra
// {0, e_a, e_a + e_b, 7} of the axis orders (a, b, c) (Freudenthal / Kuhn);
// neighbouring voxels cut their shared faces along the same diagonal, so the
// surface has no cracks. A tetrahedron with one vertex on the other side of
// the isovalue q from the rest gives one triangle, with two on each side a
// quad (two triangles). A vertex is "below" when its value is < q. A surface
// vertex on grid edge (u, v) is u + (q - f(u)) / (f(v) - f(u)) (v - u) with u
// the endpoint of lower linear vertex index, so every voxel sharing the edge
// computes the same bits. Triangles are wound so that their normal points
// from below to above q.
//
// Metacell (a, b, c) of size (mx, my, mz) holds the voxels with base vertex
// x in [a mx, min((a + 1) mx, px - 1)) (likewise in y and z); its ID is
// a + (b + c gy) gx, as formMetacellTags numbers them. Count pass: one wave
// per metacell, a lane per voxel, the wave's total per metacell. Write pass:
// the same walk; for each tetrahedron index the lanes' triangles are staged
// in LDS and stored as one contiguous run after the metacell's offset
// (order: 64-voxel chunk, tetrahedron, voxel). Positions are grid
// coordinates (x, y, z) as float, 9 floats per triangle.
#include <cstring>

#include "pst_internal.hpp"

namespace pst {

namespace {

constexpr int kIsoWave = 64;
constexpr int kIsoWavesPerCu = 24;  // measured on 1.6M metacells: 24 beats 16 and 32

// interpolation precision: float for float volumes, double otherwise
template <typename T>
using Acc = typename std::conditional<std::is_same<T, float>::value, float, double>::type;

// The six tetrahedra of a voxel as corner indices (corner k: x = k & 1,
// y = k >> 1 & 1, z = k >> 2): 0 -> e_a -> e_a + e_b -> 7.
__constant__ uint8_t kTets[6][4] = {{0, 1, 3, 7}, {0, 1, 5, 7}, {0, 2, 3, 7},
                                    {0, 2, 6, 7}, {0, 4, 5, 7}, {0, 4, 6, 7}};

struct Voxel {
  uint32_t x, y, z;
};

// Triangles of one tetrahedron: 0, 1 or 2.
__device__ inline int tet_tris(uint32_t below_mask) {
  const int nb = __popc(below_mask);
  return (nb == 0 || nb == 4) ? 0 : (nb == 2 ? 2 : 1);
}

template <typename T>
__device__ inline int voxel_count(const T f[8], T q) {
  int n = 0;
#pragma unroll
  for (int t = 0; t < 6; t++) {
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) m |= (f[kTets[t][k]] < q ? 1u : 0u) << k;
    n += tet_tris(m);
  }
  return n;
}

template <typename T>
__device__ inline void load_corners(const T* __restrict__ vol, uint32_t px, uint32_t py, const Voxel& v, T f[8]) {
  const size_t base = v.x + (static_cast<size_t>(v.y) + static_cast<size_t>(v.z) * py) * px;
#pragma unroll
  for (int k = 0; k < 8; k++)
    f[k] = vol[base + (k & 1) + (static_cast<size_t>((k >> 1) & 1) + static_cast<size_t>(k >> 2) * py) * px];
}

// Surface point on the edge between corners i and j of voxel v.
template <typename T>
__device__ inline float3 edge_point(const Voxel& v, const T f[8], int i, int j, T q) {
  // corner index order is linear vertex index order: interpolate from the lower one
  const int u = i < j ? i : j, w = i < j ? j : i;
  using A = Acc<T>;
  const A t = (static_cast<A>(q) - static_cast<A>(f[u])) / (static_cast<A>(f[w]) - static_cast<A>(f[u]));
  const float ux = static_cast<float>(v.x + (u & 1)), uy = static_cast<float>(v.y + ((u >> 1) & 1)),
              uz = static_cast<float>(v.z + (u >> 2));
  const float tf = static_cast<float>(t);
  return make_float3(ux + tf * static_cast<float>((w & 1) - (u & 1)),
                     uy + tf * static_cast<float>(((w >> 1) & 1) - ((u >> 1) & 1)),
                     uz + tf * static_cast<float>((w >> 2) - (u >> 2)));
}

__device__ inline float3 corner_pos(const Voxel& v, int k) {
  return make_float3(static_cast<float>(v.x + (k & 1)), static_cast<float>(v.y + ((k >> 1) & 1)),
                     static_cast<float>(v.z + (k >> 2)));
}

// Whether the normal of triangle (a, b, c) points against `up`.
__device__ inline bool faces_away(float3 a, float3 b, float3 c, float3 up) {
  const float3 e1 = make_float3(b.x - a.x, b.y - a.y, b.z - a.z), e2 = make_float3(c.x - a.x, c.y - a.y, c.z - a.z);
  const float3 n = make_float3(e1.y * e2.z - e1.z * e2.y, e1.z * e2.x - e1.x * e2.z, e1.x * e2.y - e1.y * e2.x);
  return n.x * up.x + n.y * up.y + n.z * up.z < 0.0f;
}

// Writes triangle (a, b, c), wound so that its normal points along `up`.
__device__ inline void put_tri(float* __restrict__ out, float3 a, float3 b, float3 c, float3 up) {
  if (faces_away(a, b, c, up)) {
    const float3 s = b;
    b = c;
    c = s;
  }
  out[0] = a.x, out[1] = a.y, out[2] = a.z;
  out[3] = b.x, out[4] = b.y, out[5] = b.z;
  out[6] = c.x, out[7] = c.y, out[8] = c.z;
}

// Triangles of tetrahedron t of voxel v (0, 1 or 2), written at `out`.
template <typename T>
__device__ inline void tet_write(const Voxel& v, const T f[8], T q, int t, float* out) {
  int below[4], above[4], nb = 0, na = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int c = kTets[t][k];
    if (f[c] < q) below[nb++] = c;
    else above[na++] = c;
  }
  if (nb == 0 || na == 0) return;
  // a direction from below to above q across this tetrahedron
  const float3 pb = corner_pos(v, below[0]), pa = corner_pos(v, above[0]);
  const float3 up = make_float3(pa.x - pb.x, pa.y - pb.y, pa.z - pb.z);
  if (nb == 1 || na == 1) {
    const int s = nb == 1 ? below[0] : above[0];
    const int* o = nb == 1 ? above : below;
    put_tri(out, edge_point(v, f, s, o[0], q), edge_point(v, f, s, o[1], q), edge_point(v, f, s, o[2], q), up);
  } else {
    const float3 p0 = edge_point(v, f, below[0], above[0], q), p1 = edge_point(v, f, below[0], above[1], q);
    const float3 p2 = edge_point(v, f, below[1], above[1], q), p3 = edge_point(v, f, below[1], above[0], q);
    put_tri(out, p0, p1, p2, up);
    put_tri(out + 9, p0, p2, p3, up);
  }
}

template <typename T>
__device__ inline int tet_count(const T f[8], T q, int t) {
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) m |= (f[kTets[t][k]] < q ? 1u : 0u) << k;
  return tet_tris(m);
}

struct IsoGrid {
  uint32_t px, py, pz;  // vertices per axis
  uint32_t mx, my, mz;  // voxels per metacell edge
  uint32_t gx, gy, gz;  // metacells per axis
};

// Voxel j of metacell `id` (false when past the metacell's voxels).
__device__ inline bool metacell_voxel(const IsoGrid& g, uint64_t id, uint32_t j, Voxel& v, uint32_t& nvox) {
  const uint32_t a = static_cast<uint32_t>(id % g.gx);
  const uint64_t r = id / g.gx;
  const uint32_t b = static_cast<uint32_t>(r % g.gy), c = static_cast<uint32_t>(r / g.gy);
  const uint32_t x0 = a * g.mx, y0 = b * g.my, z0 = c * g.mz;
  const uint32_t nx = min(g.mx, g.px - 1 - x0), ny = min(g.my, g.py - 1 - y0), nz = min(g.mz, g.pz - 1 - z0);
  nvox = nx * ny * nz;
  if (j >= nvox) return false;
  v.x = x0 + j % nx;
  v.y = y0 + (j / nx) % ny;
  v.z = z0 + j / (nx * ny);
  return true;
}

template <typename T, typename I>
__global__ __launch_bounds__(kIsoWave) void k_iso_count(const T* __restrict__ vol, IsoGrid g,
                                                         const I* __restrict__ ids, uint64_t nids, T q,
                                                         unsigned long long* __restrict__ counts,
                                                         unsigned long long* __restrict__ err) {
  const uint32_t lane = threadIdx.x;
  const uint64_t ncells = static_cast<uint64_t>(g.gx) * g.gy * g.gz;
  for (uint64_t i = blockIdx.x; i < nids; i += gridDim.x) {
    const uint64_t id = static_cast<uint64_t>(ids[i]);
    unsigned long long n = 0;
    if (id >= ncells) {
      if (lane == 0) atomicOr(err, 1ull);
    } else {
      uint32_t nvox = 1;
      for (uint32_t j0 = 0; j0 < nvox; j0 += kIsoWave) {
        Voxel v;
        if (metacell_voxel(g, id, j0 + lane, v, nvox)) {
          T f[8];
          load_corners(vol, g.px, g.py, v, f);
          n += voxel_count(f, q);
        }
      }
    }
    for (int o = kIsoWave / 2; o > 0; o >>= 1) n += __shfl_xor(n, o, kIsoWave);
    if (lane == 0) counts[i] = n;
  }
}

// One wave per metacell; per chunk of 64 voxels and per tetrahedron index,
// the lanes' triangles (at most 128) are staged in LDS at their prefix
// positions and written out as one contiguous run of floats, so the stores
// are coalesced. Order within a metacell: voxel chunk, tetrahedron, voxel.
template <typename T, typename I>
__global__ __launch_bounds__(kIsoWave) void k_iso_write(const T* __restrict__ vol, IsoGrid g,
                                                         const I* __restrict__ ids, uint64_t nids, T q,
                                                         const unsigned long long* __restrict__ offsets,
                                                         unsigned long long capacity, float* __restrict__ out) {
  __shared__ float stage[2 * kIsoWave * 9];
  const uint32_t lane = threadIdx.x;
  const uint64_t ncells = static_cast<uint64_t>(g.gx) * g.gy * g.gz;
  for (uint64_t i = blockIdx.x; i < nids; i += gridDim.x) {
    const uint64_t id = static_cast<uint64_t>(ids[i]);
    if (id >= ncells) continue;
    unsigned long long base = offsets[i];  // triangles written so far, as an output index
    uint32_t nvox = 1;
    for (uint32_t j0 = 0; j0 < nvox; j0 += kIsoWave) {
      Voxel v;
      T f[8];
      const bool have = metacell_voxel(g, id, j0 + lane, v, nvox);
      if (have) load_corners(vol, g.px, g.py, v, f);
      for (int t = 0; t < 6; t++) {
        const uint32_t n = have ? static_cast<uint32_t>(tet_count(f, q, t)) : 0u;
        uint32_t incl = n;
        for (int o = 1; o < kIsoWave; o <<= 1) {
          const uint32_t u = __shfl_up(incl, o, kIsoWave);
          if (static_cast<int>(lane) >= o) incl += u;
        }
        const uint32_t total = __shfl(incl, kIsoWave - 1, kIsoWave);
        if (total == 0) continue;
        if (n) tet_write(v, f, q, t, stage + 9 * (incl - n));
        __syncthreads();
        for (uint32_t k = lane; k < 9 * total; k += kIsoWave) {
          const unsigned long long tri = base + k / 9;
          if (tri < capacity) out[9 * base + k] = stage[k];
        }
        __syncthreads();
        base += total;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Marching cubes: one surface patch per voxel from a 256-case table over the
// 8 corner signs (corner k below when f < q). The table is generated at
// compile time from one rule, so no case list is transcribed:
//  - on each face of the cube, walked counter-clockwise as seen from outside,
//    every maximal run of below corners is cut off by one segment, from the
//    edge where the walk leaves the run to the edge where it entered it; a
//    face with two diagonal below corners thus gets two segments, each
//    cutting off one corner (the below corners stay apart), and the choice
//    depends on the face's corner signs alone, so the two voxels that share
//    a face cut it the same way and the surface has no cracks;
//  - every crossing edge starts one segment and ends one (the two faces of
//    an edge walk it in opposite directions), so the segments form closed
//    loops; each loop becomes a triangle fan, wound so that the normal
//    points from below to above q.
// Edges are numbered by axis: x edges 0-3 (corner pairs 0-1, 2-3, 4-5,
// 6-7), y edges 4-7 (0-2, 1-3, 4-6, 5-7), z edges 8-11 (0-4, 1-5, 2-6, 3-7).
// Surface vertices interpolate from the edge endpoint of lower linear
// index, as for the tetrahedra, so shared edges give identical vertices.
// ---------------------------------------------------------------------------
constexpr int kMcMaxTri = 5;
struct McCase {
  uint8_t ntri;
  uint8_t e[3 * kMcMaxTri];  // edge triples of the triangles
};
struct McTable {
  McCase c[256];
  int maxtri;
};
constexpr uint8_t kMcEdgeLo[12] = {0, 2, 4, 6, 0, 1, 4, 5, 0, 1, 2, 3};
constexpr uint8_t kMcEdgeHi[12] = {1, 3, 5, 7, 2, 3, 6, 7, 4, 5, 6, 7};

constexpr int mc_edge_of(int a, int b) {
  for (int e = 0; e < 12; e++)
    if ((kMcEdgeLo[e] == a && kMcEdgeHi[e] == b) || (kMcEdgeLo[e] == b && kMcEdgeHi[e] == a)) return e;
  return -1;
}

constexpr McTable make_mc_table() {
  McTable T{};
  // faces: axis bit, side, and corner offsets u, v with u x v along the
  // outward normal (x = 1, y = 2, z = 4)
  const int ax[6] = {1, 1, 2, 2, 4, 4};
  const int side[6] = {0, 1, 0, 1, 0, 1};
  const int uu[6] = {4, 2, 1, 4, 2, 1};
  const int vv[6] = {2, 4, 4, 1, 1, 2};
  for (int cfg = 0; cfg < 256; cfg++) {
    int next[12] = {-1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1};
    for (int f = 0; f < 6; f++) {
      const int b = side[f] ? ax[f] : 0;
      const int c[4] = {b, b | uu[f], b | uu[f] | vv[f], b | vv[f]};
      bool in[4] = {};
      for (int i = 0; i < 4; i++) in[i] = (cfg >> c[i]) & 1;
      for (int i = 0; i < 4; i++) {
        if (!in[i] || in[(i + 1) % 4]) continue;  // the walk leaves a run at corner i
        int j = i;
        while (in[(j + 3) % 4]) j = (j + 3) % 4;  // back to the run's first corner
        next[mc_edge_of(c[i], c[(i + 1) % 4])] = mc_edge_of(c[(j + 3) % 4], c[j]);
      }
    }
    bool seen[12] = {};
    int nt = 0;
    for (int e0 = 0; e0 < 12; e0++) {
      if (next[e0] < 0 || seen[e0]) continue;
      int cyc[12] = {};
      int len = 0;
      for (int e = e0; !seen[e]; e = next[e]) {
        seen[e] = true;
        cyc[len++] = e;
      }
      for (int k = 1; k + 1 < len; k++) {
        if (nt < kMcMaxTri) {
          T.c[cfg].e[3 * nt] = static_cast<uint8_t>(cyc[0]);
          T.c[cfg].e[3 * nt + 1] = static_cast<uint8_t>(cyc[k + 1]);
          T.c[cfg].e[3 * nt + 2] = static_cast<uint8_t>(cyc[k]);
        }
        nt++;
      }
    }
    T.c[cfg].ntri = static_cast<uint8_t>(nt);
    if (nt > T.maxtri) T.maxtri = nt;
  }
  return T;
}

constexpr McTable kMcHost = make_mc_table();
static_assert(kMcHost.maxtri == kMcMaxTri, "marching cubes table capacity");
__constant__ McTable kMc = make_mc_table();

template <typename T>
__device__ inline uint32_t mc_config(const T f[8], T q) {
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) m |= (f[k] < q ? 1u : 0u) << k;
  return m;
}

template <typename T, typename I>
__global__ __launch_bounds__(kIsoWave) void k_mc_count(const T* __restrict__ vol, IsoGrid g,
                                                        const I* __restrict__ ids, uint64_t nids, T q,
                                                        unsigned long long* __restrict__ counts,
                                                        unsigned long long* __restrict__ err) {
  const uint32_t lane = threadIdx.x;
  const uint64_t ncells = static_cast<uint64_t>(g.gx) * g.gy * g.gz;
  for (uint64_t i = blockIdx.x; i < nids; i += gridDim.x) {
    const uint64_t id = static_cast<uint64_t>(ids[i]);
    unsigned long long n = 0;
    if (id >= ncells) {
      if (lane == 0) atomicOr(err, 1ull);
    } else {
      uint32_t nvox = 1;
      for (uint32_t j0 = 0; j0 < nvox; j0 += kIsoWave) {
        Voxel v;
        if (metacell_voxel(g, id, j0 + lane, v, nvox)) {
          T f[8];
          load_corners(vol, g.px, g.py, v, f);
          n += kMc.c[mc_config(f, q)].ntri;
        }
      }
    }
    for (int o = kIsoWave / 2; o > 0; o >>= 1) n += __shfl_xor(n, o, kIsoWave);
    if (lane == 0) counts[i] = n;
  }
}

// One wave per metacell; per chunk of 64 voxels the lanes' triangles are
// staged in LDS at their prefix positions (voxel order) and written out as
// one contiguous run. Order within a metacell: voxel, then the voxel's
// table order.
template <typename T, typename I>
__global__ __launch_bounds__(kIsoWave) void k_mc_write(const T* __restrict__ vol, IsoGrid g,
                                                        const I* __restrict__ ids, uint64_t nids, T q,
                                                        const unsigned long long* __restrict__ offsets,
                                                        unsigned long long capacity, float* __restrict__ out) {
  __shared__ float stage[kIsoWave * kMcMaxTri * 9];
  const uint32_t lane = threadIdx.x;
  const uint64_t ncells = static_cast<uint64_t>(g.gx) * g.gy * g.gz;
  for (uint64_t i = blockIdx.x; i < nids; i += gridDim.x) {
    const uint64_t id = static_cast<uint64_t>(ids[i]);
    if (id >= ncells) continue;
    unsigned long long base = offsets[i];
    uint32_t nvox = 1;
    for (uint32_t j0 = 0; j0 < nvox; j0 += kIsoWave) {
      Voxel v;
      T f[8];
      const bool have = metacell_voxel(g, id, j0 + lane, v, nvox);
      uint32_t cfg = 0, n = 0;
      if (have) {
        load_corners(vol, g.px, g.py, v, f);
        cfg = mc_config(f, q);
        n = kMc.c[cfg].ntri;
      }
      uint32_t incl = n;
      for (int o = 1; o < kIsoWave; o <<= 1) {
        const uint32_t u = __shfl_up(incl, o, kIsoWave);
        if (static_cast<int>(lane) >= o) incl += u;
      }
      const uint32_t total = __shfl(incl, kIsoWave - 1, kIsoWave);
      if (total == 0) continue;
      float* my = stage + 9 * (incl - n);
      for (uint32_t t = 0; t < n; t++) {
        const uint8_t* e = kMc.c[cfg].e + 3 * t;
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const float3 p = edge_point(v, f, kMcEdgeLo[e[k]], kMcEdgeHi[e[k]], q);
          my[9 * t + 3 * k] = p.x;
          my[9 * t + 3 * k + 1] = p.y;
          my[9 * t + 3 * k + 2] = p.z;
        }
      }
      __syncthreads();
      for (uint32_t k = lane; k < 9 * total; k += kIsoWave) {
        const unsigned long long tri = base + k / 9;
        if (tri < capacity) out[9 * base + k] = stage[k];
      }
      __syncthreads();
      base += total;
    }
  }
}

// ---------------------------------------------------------------------------
// Marching cubes for metacells of at most 4 x 4 x 4 voxels. A wave holds the
// metacell's 5 x 5 x 5 vertices, two per lane (vertex u = x + 5 y + 25 z at
// lanes u and u - 64), as registers and as a 125-bit mask of the vertices
// below q; lane j is voxel (j & 3, j >> 2 & 3, j >> 4), which is also the
// voxel order of partial metacells (lanes past the grid are skipped). A
// voxel's case is eight bits of the mask's 32-bit window at its base vertex.
//
// The write computes each crossing edge's parameter once per metacell (the
// voxels around an edge share it: a quarter of the divisions), lists the
// triangles' vertices as edge numbers in LDS at their output positions, and
// then takes lanes over the output's vertices, whose 12-byte stores are
// contiguous across the wave. A wave takes a contiguous run of the ID list,
// so that neighbouring metacells share the cache lines of their vertex rows,
// and loads the next metacell's vertices while it works on one.
//
// Measured on 670,647 active metacells of a 1024^3 volume (49.1M triangles,
// 1.77 GB) on MI355X, against the general kernels above: count 0.309 -> 0.207
// ms (4.3 TB/s of 128-byte row requests), write 1.68 -> 0.63 ms (1.23 GB read
// and 1.79 GB written, 4.8 TB/s; 0.75 before the triangles were stored as
// streaming, which leaves the L2 to the vertices that metacells share).
// ---------------------------------------------------------------------------
constexpr int kMc4Waves = 4;               // waves per workgroup (one LDS case table)
constexpr int kMc4BlocksPerCu = 20;
constexpr uint32_t kVerts = 125;           // vertices of a 4 x 4 x 4 metacell
constexpr uint32_t kMc4List = 3 * kMcMaxTri * kIsoWave;

__device__ inline void iso_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The lane's two vertices of a 5 x 5 x 5 block, with their byte offsets from
// the metacell's base vertex.
struct LaneVerts {
  uint32_t x[2], y[2], z[2], off[2];
  bool in[2];
};
template <typename T>
__device__ inline LaneVerts lane_verts(const IsoGrid& g, uint32_t lane) {
  LaneVerts v;
#pragma unroll
  for (uint32_t h = 0; h < 2; h++) {
    const uint32_t u = lane + h * kIsoWave;
    v.x[h] = u % 5, v.y[h] = (u / 5) % 5, v.z[h] = u / 25;
    v.in[h] = u < kVerts;
    v.off[h] = (v.x[h] + (v.y[h] + v.z[h] * g.py) * g.px) * static_cast<uint32_t>(sizeof(T));
  }
  return v;
}

// 64 list entries at a time: lane k holds entry base + k's base vertex and
// voxels per axis (n: nx | ny << 8 | nz << 16; 0: past the list or no such ID).
struct CellLane {
  uint32_t x0, y0, z0, n;
};
template <typename I>
__device__ inline CellLane cell_lane(const IsoGrid& g, const I* __restrict__ ids, uint64_t i, uint64_t i1) {
  CellLane c{0, 0, 0, 0};
  if (i >= i1) return c;
  const uint64_t id = static_cast<uint64_t>(ids[i]);
  if (id >= static_cast<uint64_t>(g.gx) * g.gy * g.gz) return c;
  const uint64_t r = id / g.gx;
  c.x0 = static_cast<uint32_t>(id - r * g.gx) * g.mx;
  const uint32_t d = static_cast<uint32_t>(r / g.gy);
  c.y0 = static_cast<uint32_t>(r - static_cast<uint64_t>(d) * g.gy) * g.my;
  c.z0 = d * g.mz;
  c.n = min(g.mx, g.px - 1 - c.x0) | (min(g.my, g.py - 1 - c.y0) << 8) | (min(g.mz, g.pz - 1 - c.z0) << 16);
  return c;
}
// Entry k of the 64, in scalar registers.
struct Cell {
  uint32_t x0, y0, z0, nx, ny, nz;
};
__device__ inline Cell cell_at(const CellLane& c, int k) {
  const uint32_t n = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(c.n), k));
  return Cell{static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(c.x0), k)),
              static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(c.y0), k)),
              static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(c.z0), k)),
              n & 0xff, (n >> 8) & 0xff, n >> 16};
}

template <typename T>
__device__ inline void load_verts(const T* __restrict__ vol, const IsoGrid& g, const Cell& c, const LaneVerts& lv,
                                  T (&f)[2], bool (&ok)[2]) {
  const char* p = reinterpret_cast<const char*>(vol + c.x0 + (c.y0 + static_cast<size_t>(c.z0) * g.py) * g.px);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    ok[h] = lv.in[h] && c.nx && lv.x[h] <= c.nx && lv.y[h] <= c.ny && lv.z[h] <= c.nz;
    f[h] = T(0);
    if (ok[h]) f[h] = *reinterpret_cast<const T*>(p + lv.off[h]);
  }
}

// The lane's voxel's case from the vertices' below mask (lo: vertices 0-63).
__device__ inline uint32_t voxel_case(uint64_t lo, uint64_t hi, uint32_t b) {
  const uint64_t w64 = b < 64 ? (lo >> b) | (b ? hi << (64 - b) : 0ull) : hi >> (b - 64);
  const uint32_t w = static_cast<uint32_t>(w64);
  return (w & 3u) | (((w >> 5) & 3u) << 2) | (((w >> 25) & 3u) << 4) | ((w >> 30) << 6);
}

// The list range of a wave: contiguous, balanced to one ID.
__device__ inline void wave_range(uint64_t nids, uint64_t wave, uint64_t waves, uint64_t& i0, uint64_t& i1) {
  const uint64_t per = nids / waves, rest = nids % waves;
  i0 = wave * per + (wave < rest ? wave : rest);
  i1 = i0 + per + (wave < rest ? 1 : 0);
}

template <typename T, typename I>
__global__ __launch_bounds__(kMc4Waves * kIsoWave) void k_mc_count4(const T* __restrict__ vol, IsoGrid g,
                                                                    const I* __restrict__ ids, uint64_t nids, T q,
                                                                    unsigned long long* __restrict__ counts,
                                                                    unsigned long long* __restrict__ err) {
  __shared__ uint8_t s_ntri[256];
  if (threadIdx.x < 256) s_ntri[threadIdx.x] = kMc.c[threadIdx.x].ntri;
  __syncthreads();
  const uint32_t lane = threadIdx.x % kIsoWave;
  const LaneVerts lv = lane_verts<T>(g, lane);
  const uint32_t vx = lane & 3, vy = (lane >> 2) & 3, vz = lane >> 4;
  const uint32_t vb = vx + 5 * vy + 25 * vz;
  uint64_t i0, i1;
  wave_range(nids, blockIdx.x * kMc4Waves + __builtin_amdgcn_readfirstlane(threadIdx.x / kIsoWave),
             static_cast<uint64_t>(gridDim.x) * kMc4Waves, i0, i1);
  for (uint64_t ib = i0; ib < i1; ib += kIsoWave) {
    const int m = static_cast<int>(i1 - ib < kIsoWave ? i1 - ib : kIsoWave);
    const CellLane cl = cell_lane(g, ids, ib + lane, i1);
    T f[2], fn[2];
    bool ok[2], okn[2];
    Cell c = cell_at(cl, 0), cn = c;
    load_verts(vol, g, c, lv, f, ok);
    uint32_t mine = 0;  // entry ib + lane's triangles
    for (int k = 0; k < m; k++) {
      if (k + 1 < m) {
        cn = cell_at(cl, k + 1);
        load_verts(vol, g, cn, lv, fn, okn);
      }
      const uint64_t lo = __ballot(ok[0] && f[0] < q), hi = __ballot(ok[1] && f[1] < q);
      const bool have = vx < c.nx && vy < c.ny && vz < c.nz;
      const uint32_t n = have ? s_ntri[voxel_case(lo, hi, vb)] : 0u;
      const uint32_t total = __popcll(__ballot(n & 1)) + 2 * __popcll(__ballot(n & 2)) + 4 * __popcll(__ballot(n & 4));
      mine = static_cast<int>(lane) == k ? total : mine;
      c = cn;
#pragma unroll
      for (int h = 0; h < 2; h++) f[h] = fn[h], ok[h] = okn[h];
    }
    if (static_cast<int>(lane) < m) {
      counts[ib + lane] = mine;
      if (cl.n == 0) atomicOr(err, 1ull);
    }
  }
}

// Bound by HBM: its reads and stores move at 84% of a large copy's rate.
template <typename T, typename I>
__global__ __launch_bounds__(kMc4Waves * kIsoWave) void k_mc_write4(const T* __restrict__ vol, IsoGrid g,
                                                                    const I* __restrict__ ids, uint64_t nids, T q,
                                                                    const unsigned long long* __restrict__ offsets,
                                                                    unsigned long long capacity,
                                                                    float* __restrict__ out) {
  using A = Acc<T>;
  // per case: triangle count, then edge numbers (axis * 125 + vertex) relative to the voxel's base vertex
  __shared__ __align__(16) uint16_t s_case[256][16];
  // edge number -> its base vertex's place (bytes x, y, z), its direction (bytes)
  __shared__ uint2 s_place[3 * kVerts];
  __shared__ A s_val[kMc4Waves][kVerts];
  __shared__ float s_t[kMc4Waves][3 * kVerts];
  __shared__ uint16_t s_list[kMc4Waves][kMc4List];
  for (uint32_t i = threadIdx.x; i < 256 * 16; i += kMc4Waves * kIsoWave) {
    const uint32_t cfg = i >> 4, k = i & 15;
    uint32_t v = kMc.c[cfg].ntri;
    if (k > 0) {
      const uint32_t e = kMc.c[cfg].e[k - 1], lo = kMcEdgeLo[e];
      v = (e >> 2) * kVerts + (lo & 1) + 5 * ((lo >> 1) & 1) + 25 * (lo >> 2);
    }
    s_case[cfg][k] = static_cast<uint16_t>(v);
  }
  for (uint32_t i = threadIdx.x; i < 3 * kVerts; i += kMc4Waves * kIsoWave) {
    const uint32_t u = i % kVerts;
    s_place[i] = make_uint2((u % 5) | (((u / 5) % 5) << 8) | ((u / 25) << 16), 1u << (8 * (i / kVerts)));
  }
  __syncthreads();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kIsoWave), lane = threadIdx.x % kIsoWave;
  A* val = s_val[wave];
  float* tpar = s_t[wave];
  uint16_t* list = s_list[wave];
  const LaneVerts lv = lane_verts<T>(g, lane);
  const uint32_t vx = lane & 3, vy = (lane >> 2) & 3, vz = lane >> 4;
  const uint32_t vb = vx + 5 * vy + 25 * vz;
  uint64_t i0, i1;
  wave_range(nids, blockIdx.x * kMc4Waves + wave, static_cast<uint64_t>(gridDim.x) * kMc4Waves, i0, i1);
  for (uint64_t ib = i0; ib < i1; ib += kIsoWave) {
    const int m = static_cast<int>(i1 - ib < kIsoWave ? i1 - ib : kIsoWave);
    const CellLane cl = cell_lane(g, ids, ib + lane, i1);
    const unsigned long long base_lane = ib + lane < i1 ? offsets[ib + lane] : 0;
    T f[2], fn[2];
    bool ok[2], okn[2];
    Cell c = cell_at(cl, 0), cn = c;
    load_verts(vol, g, c, lv, f, ok);
    for (int k = 0; k < m; k++) {
      if (k + 1 < m) {
        cn = cell_at(cl, k + 1);
        load_verts(vol, g, cn, lv, fn, okn);
      }
      const unsigned long long base =
          (static_cast<unsigned long long>(static_cast<uint32_t>(
               __builtin_amdgcn_readlane(static_cast<int>(base_lane >> 32), k))) << 32) |
          static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(base_lane), k));
      const uint64_t lo = __ballot(ok[0] && f[0] < q), hi = __ballot(ok[1] && f[1] < q);
      const bool have = vx < c.nx && vy < c.ny && vz < c.nz;
      const uint32_t cfg = have ? voxel_case(lo, hi, vb) : 0u;
      // 16 entries of the case: its count and at most 15 edges
      const uint4 ca = *reinterpret_cast<const uint4*>(&s_case[cfg][0]),
                  cb = *reinterpret_cast<const uint4*>(&s_case[cfg][8]);
      const uint32_t w[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
      const uint32_t n = w[0] & 0xffffu;
      const uint64_t b0 = __ballot(n & 1), b1 = __ballot(n & 2), b2 = __ballot(n & 4);
      const uint32_t total = __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2);
      if (total && base < capacity) {
        const uint32_t pre = lanes_below(b0) + 2 * lanes_below(b1) + 4 * lanes_below(b2);
#pragma unroll
        for (int h = 0; h < 2; h++)
          if (lv.in[h]) val[lane + h * kIsoWave] = static_cast<A>(f[h]);
        iso_wave_sync();
        // crossing edges from the lane's vertices u to u + 1, u + 5, u + 25
        // (both ends in the metacell), as lane masks from the below mask
#pragma unroll
        for (int a = 0; a < 3; a++) {
          constexpr uint32_t kStep[3] = {1, 5, 25};
          const uint32_t step = kStep[a];
          const uint64_t olo = (lo >> step) | (hi << (64 - step)), ohi = hi >> step;
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const bool end = a == 0 ? lv.x[h] < c.nx : (a == 1 ? lv.y[h] < c.ny : lv.z[h] < c.nz);
            if (__builtin_amdgcn_inverse_ballot_w64(h ? hi ^ ohi : lo ^ olo) && ok[h] && end) {
              const uint32_t u = lane + h * kIsoWave;
              const A fu = static_cast<A>(f[h]);
              const A t = (static_cast<A>(q) - fu) / (val[u + step] - fu);
              tpar[a * kVerts + u] = static_cast<float>(t);
            }
          }
        }
        // the voxel's triangles as edge numbers, at their output positions
        uint16_t* my = list + 3 * pre;
#pragma unroll
        for (int t = 0; t < kMcMaxTri; t++) {
          if (t < static_cast<int>(n)) {
#pragma unroll
            for (int j = 0; j < 3; j++) {
              const int at = 1 + 3 * t + j;
              my[3 * t + j] = static_cast<uint16_t>(((w[at >> 1] >> (16 * (at & 1))) & 0xffffu) + vb);
            }
          }
        }
        iso_wave_sync();
        const unsigned long long room = capacity - base;
        const uint32_t nv = 3 * (room < total ? static_cast<uint32_t>(room) : total);
        float* o = out + 9 * base;
        const float fx = static_cast<float>(c.x0), fy = static_cast<float>(c.y0), fz = static_cast<float>(c.z0);
        for (uint32_t j = lane; j < nv; j += kIsoWave) {
          const uint32_t e = list[j];
          const float t = tpar[e];
          const uint2 pl = s_place[e];
          float3 p;
          p.x = fx + static_cast<float>(pl.x & 0xff) + t * static_cast<float>(pl.y & 0xff);
          p.y = fy + static_cast<float>((pl.x >> 8) & 0xff) + t * static_cast<float>((pl.y >> 8) & 0xff);
          p.z = fz + static_cast<float>((pl.x >> 16) & 0xff) + t * static_cast<float>((pl.y >> 16) & 0xff);
          stream_store(reinterpret_cast<float3*>(o + 3 * j), p);
        }
        iso_wave_sync();
      }
      c = cn;
#pragma unroll
      for (int h = 0; h < 2; h++) f[h] = fn[h], ok[h] = okn[h];
    }
  }
}

// ---------------------------------------------------------------------------
// Marching tetrahedra for the same metacells, in the same manner: edges run
// from a vertex in the seven directions of the Kuhn subdivision (dir = bits
// of the corner difference), edge number (dir - 1) * 128 + vertex. Triangles
// come tetrahedron by tetrahedron, voxel order within; lanes over triangles
// settle each winding (put_tri's test on the same positions) before lanes
// take the output's vertices.
//
// Measured on the same 670,647 metacells on MI355X against the general
// kernels above: count 0.316 -> 0.229 ms, write 4.14 -> 1.56 ms (bound by
// instruction issue: seven divisions per vertex pair and two passes over the
// triangles).
// ---------------------------------------------------------------------------
constexpr uint32_t kTet4List = 3 * 12 * kIsoWave;  // at most 12 triangles per voxel

// Case of tetrahedron t with below mask m: triangles, their edges as local
// corner pairs (lo, hi), and the corners the winding points between.
struct TetCase {
  uint8_t ntri;
  uint8_t lo[6], hi[6];  // corners of the cube
  uint8_t below, above;
};
constexpr uint8_t kTetCorner[6][4] = {{0, 1, 3, 7}, {0, 1, 5, 7}, {0, 2, 3, 7}, {0, 2, 6, 7}, {0, 4, 5, 7}, {0, 4, 6, 7}};
constexpr TetCase tet_case(int t, int m) {
  TetCase c{};
  uint8_t below[4] = {}, above[4] = {};
  int nb = 0, na = 0;
  for (int k = 0; k < 4; k++) {
    if (m >> k & 1) below[nb++] = kTetCorner[t][k];
    else above[na++] = kTetCorner[t][k];
  }
  if (nb == 0 || na == 0) return c;
  c.below = below[0];
  c.above = above[0];
  uint8_t p[6][2] = {};
  if (nb == 1 || na == 1) {
    c.ntri = 1;
    const uint8_t s = nb == 1 ? below[0] : above[0];
    for (int k = 0; k < 3; k++) p[k][0] = s, p[k][1] = nb == 1 ? above[k] : below[k];
  } else {
    c.ntri = 2;
    const int b[6] = {0, 0, 1, 0, 1, 1}, a[6] = {0, 1, 1, 0, 1, 0};
    for (int k = 0; k < 6; k++) p[k][0] = below[b[k]], p[k][1] = above[a[k]];
  }
  for (int k = 0; k < 6; k++) {
    c.lo[k] = p[k][0] < p[k][1] ? p[k][0] : p[k][1];
    c.hi[k] = p[k][0] < p[k][1] ? p[k][1] : p[k][0];
  }
  return c;
}
struct TetTable {
  TetCase c[6 * 16];
};
constexpr TetTable make_tet_table() {
  TetTable T{};
  for (int t = 0; t < 6; t++)
    for (int m = 0; m < 16; m++) T.c[t * 16 + m] = tet_case(t, m);
  return T;
}
__constant__ TetTable kTet = make_tet_table();

// Below mask of tetrahedron t's corners from a voxel's case.
__device__ inline uint32_t tet_mask(uint32_t cfg, int t) {
  return ((cfg >> kTetCorner[t][0]) & 1u) | (((cfg >> kTetCorner[t][1]) & 1u) << 1) |
         (((cfg >> kTetCorner[t][2]) & 1u) << 2) | (((cfg >> kTetCorner[t][3]) & 1u) << 3);
}

template <typename T, typename I>
__global__ __launch_bounds__(kMc4Waves * kIsoWave) void k_iso_count4(const T* __restrict__ vol, IsoGrid g,
                                                                     const I* __restrict__ ids, uint64_t nids, T q,
                                                                     unsigned long long* __restrict__ counts,
                                                                     unsigned long long* __restrict__ err) {
  __shared__ uint8_t s_ntri[256];  // triangles of a voxel's six tetrahedra
  {
    uint32_t n = 0;
#pragma unroll
    for (int t = 0; t < 6; t++) n += static_cast<uint32_t>(tet_tris(tet_mask(threadIdx.x, t)));
    s_ntri[threadIdx.x] = static_cast<uint8_t>(n);
  }
  static_assert(kMc4Waves * kIsoWave == 256, "a thread per case");
  __syncthreads();
  const uint32_t lane = threadIdx.x % kIsoWave;
  const LaneVerts lv = lane_verts<T>(g, lane);
  const uint32_t vx = lane & 3, vy = (lane >> 2) & 3, vz = lane >> 4;
  const uint32_t vb = vx + 5 * vy + 25 * vz;
  uint64_t i0, i1;
  wave_range(nids, blockIdx.x * kMc4Waves + __builtin_amdgcn_readfirstlane(threadIdx.x / kIsoWave),
             static_cast<uint64_t>(gridDim.x) * kMc4Waves, i0, i1);
  for (uint64_t ib = i0; ib < i1; ib += kIsoWave) {
    const int m = static_cast<int>(i1 - ib < kIsoWave ? i1 - ib : kIsoWave);
    const CellLane cl = cell_lane(g, ids, ib + lane, i1);
    T f[2], fn[2];
    bool ok[2], okn[2];
    Cell c = cell_at(cl, 0), cn = c;
    load_verts(vol, g, c, lv, f, ok);
    uint32_t mine = 0;
    for (int k = 0; k < m; k++) {
      if (k + 1 < m) {
        cn = cell_at(cl, k + 1);
        load_verts(vol, g, cn, lv, fn, okn);
      }
      const uint64_t lo = __ballot(ok[0] && f[0] < q), hi = __ballot(ok[1] && f[1] < q);
      const bool have = vx < c.nx && vy < c.ny && vz < c.nz;
      const uint32_t n = have ? s_ntri[voxel_case(lo, hi, vb)] : 0u;  // at most 12
      const uint32_t total = __popcll(__ballot(n & 1)) + 2 * __popcll(__ballot(n & 2)) +
                             4 * __popcll(__ballot(n & 4)) + 8 * __popcll(__ballot(n & 8));
      mine = static_cast<int>(lane) == k ? total : mine;
      c = cn;
#pragma unroll
      for (int h = 0; h < 2; h++) f[h] = fn[h], ok[h] = okn[h];
    }
    if (static_cast<int>(lane) < m) {
      counts[ib + lane] = mine;
      if (cl.n == 0) atomicOr(err, 1ull);
    }
  }
}

template <typename T, typename I>
__global__ __launch_bounds__(kMc4Waves * kIsoWave) void k_iso_write4(const T* __restrict__ vol, IsoGrid g,
                                                                     const I* __restrict__ ids, uint64_t nids, T q,
                                                                     const unsigned long long* __restrict__ offsets,
                                                                     unsigned long long capacity,
                                                                     float* __restrict__ out) {
  using A = Acc<T>;
  // per tetrahedron and mask: triangle count, 6 edge numbers relative to the
  // voxel's base vertex, and the winding's direction (2 bits per axis, + 1)
  __shared__ __align__(16) uint16_t s_case[6 * 16][8];
  __shared__ uint32_t s_place[128];  // vertex -> bytes x, y, z
  __shared__ A s_val[kMc4Waves][kVerts];
  __shared__ float s_t[kMc4Waves][7 * 128];
  __shared__ uint16_t s_list[kMc4Waves][kTet4List];
  __shared__ uint8_t s_dir[kMc4Waves][kTet4List / 3];
  if (threadIdx.x < 6 * 16) {
    const TetCase tc = kTet.c[threadIdx.x];
    s_case[threadIdx.x][0] = tc.ntri;
    for (int k = 0; k < 6; k++) {
      const uint32_t lo = tc.lo[k], dir = lo ^ tc.hi[k];
      s_case[threadIdx.x][1 + k] =
          static_cast<uint16_t>((dir ? dir - 1 : 0) * 128 + (lo & 1) + 5 * ((lo >> 1) & 1) + 25 * (lo >> 2));
    }
    uint32_t up = 0;
    for (int a = 0; a < 3; a++) up |= (1 + ((tc.above >> a) & 1) - ((tc.below >> a) & 1)) << (2 * a);
    s_case[threadIdx.x][7] = static_cast<uint16_t>(up);
  }
  if (threadIdx.x < 128) {
    const uint32_t u = threadIdx.x;
    s_place[u] = (u % 5) | (((u / 5) % 5) << 8) | ((u / 25) << 16);
  }
  __syncthreads();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kIsoWave), lane = threadIdx.x % kIsoWave;
  A* val = s_val[wave];
  float* tpar = s_t[wave];
  uint16_t* list = s_list[wave];
  uint8_t* dirs = s_dir[wave];
  const LaneVerts lv = lane_verts<T>(g, lane);
  const uint32_t vx = lane & 3, vy = (lane >> 2) & 3, vz = lane >> 4;
  const uint32_t vb = vx + 5 * vy + 25 * vz;
  uint64_t i0, i1;
  wave_range(nids, blockIdx.x * kMc4Waves + wave, static_cast<uint64_t>(gridDim.x) * kMc4Waves, i0, i1);
  for (uint64_t ib = i0; ib < i1; ib += kIsoWave) {
    const int m = static_cast<int>(i1 - ib < kIsoWave ? i1 - ib : kIsoWave);
    const CellLane cl = cell_lane(g, ids, ib + lane, i1);
    const unsigned long long base_lane = ib + lane < i1 ? offsets[ib + lane] : 0;
    T f[2], fn[2];
    bool ok[2], okn[2];
    Cell c = cell_at(cl, 0), cn = c;
    load_verts(vol, g, c, lv, f, ok);
    for (int k = 0; k < m; k++) {
      if (k + 1 < m) {
        cn = cell_at(cl, k + 1);
        load_verts(vol, g, cn, lv, fn, okn);
      }
      const unsigned long long base =
          (static_cast<unsigned long long>(static_cast<uint32_t>(
               __builtin_amdgcn_readlane(static_cast<int>(base_lane >> 32), k))) << 32) |
          static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(base_lane), k));
      const uint64_t lo = __ballot(ok[0] && f[0] < q), hi = __ballot(ok[1] && f[1] < q);
      const bool have = vx < c.nx && vy < c.ny && vz < c.nz;
      const uint32_t cfg = have ? voxel_case(lo, hi, vb) : 0u;
      if (base < capacity && __ballot(cfg != 0 && cfg != 255)) {
#pragma unroll
        for (int h = 0; h < 2; h++)
          if (lv.in[h]) val[lane + h * kIsoWave] = static_cast<A>(f[h]);
        iso_wave_sync();
#pragma unroll
        for (int d = 1; d < 8; d++) {
          const uint32_t step = (d & 1) + 5 * ((d >> 1) & 1) + 25 * (d >> 2);
          const uint64_t olo = (lo >> step) | (hi << (64 - step)), ohi = hi >> step;
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const bool end = (!(d & 1) || lv.x[h] < c.nx) && (!(d & 2) || lv.y[h] < c.ny) && (!(d & 4) || lv.z[h] < c.nz);
            if (__builtin_amdgcn_inverse_ballot_w64(h ? hi ^ ohi : lo ^ olo) && ok[h] && end) {
              const uint32_t u = lane + h * kIsoWave;
              const A fu = static_cast<A>(f[h]);
              const A t = (static_cast<A>(q) - fu) / (val[u + step] - fu);
              tpar[(d - 1) * 128 + u] = static_cast<float>(t);
            }
          }
        }
        // the triangles as edge numbers at their output positions
        uint32_t total = 0;
#pragma unroll
        for (int t = 0; t < 6; t++) {
          const uint32_t tm = t * 16 + tet_mask(cfg, t);
          const uint4 ca = *reinterpret_cast<const uint4*>(&s_case[tm][0]);
          const uint32_t w[4] = {ca.x, ca.y, ca.z, ca.w};
          const uint32_t n = w[0] & 0xffffu;
          const uint64_t b0 = __ballot(n & 1), b1 = __ballot(n & 2);
          const uint32_t at = total + lanes_below(b0) + 2 * lanes_below(b1);
          total += __popcll(b0) + 2 * __popcll(b1);
#pragma unroll
          for (int r = 0; r < 2; r++) {
            if (r < static_cast<int>(n)) {
#pragma unroll
              for (int j = 0; j < 3; j++) {
                const int e = 1 + 3 * r + j;
                list[3 * (at + r) + j] = static_cast<uint16_t>(((w[e >> 1] >> (16 * (e & 1))) & 0xffffu) + vb);
              }
              dirs[at + r] = static_cast<uint8_t>(w[3] >> 16);
            }
          }
        }
        iso_wave_sync();
        const unsigned long long room = capacity - base;
        const uint32_t nt = room < total ? static_cast<uint32_t>(room) : total;
        const float fx = static_cast<float>(c.x0), fy = static_cast<float>(c.y0), fz = static_cast<float>(c.z0);
        auto point = [&](uint32_t e) {
          const float t = tpar[e];
          const uint32_t pl = s_place[e & 127], d = (e >> 7) + 1;
          return make_float3(fx + static_cast<float>(pl & 0xff) + t * static_cast<float>(d & 1),
                             fy + static_cast<float>((pl >> 8) & 0xff) + t * static_cast<float>((d >> 1) & 1),
                             fz + static_cast<float>((pl >> 16) & 0xff) + t * static_cast<float>(d >> 2));
        };
        // windings
        for (uint32_t j = lane; j < nt; j += kIsoWave) {
          const uint16_t eb = list[3 * j + 1], ec = list[3 * j + 2];
          const float3 a = point(list[3 * j]), b = point(eb), p = point(ec);
          const uint32_t d = dirs[j];
          const float3 up = make_float3(static_cast<float>(static_cast<int>(d & 3) - 1),
                                        static_cast<float>(static_cast<int>((d >> 2) & 3) - 1),
                                        static_cast<float>(static_cast<int>((d >> 4) & 3) - 1));
          if (faces_away(a, b, p, up)) {
            list[3 * j + 1] = ec;
            list[3 * j + 2] = eb;
          }
        }
        iso_wave_sync();
        float* o = out + 9 * base;
        for (uint32_t j = lane; j < 3 * nt; j += kIsoWave) stream_store(reinterpret_cast<float3*>(o + 3 * j), point(list[j]));
        iso_wave_sync();
      }
      c = cn;
#pragma unroll
      for (int h = 0; h < 2; h++) f[h] = fn[h], ok[h] = okn[h];
    }
  }
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
Status with_idx(int idt, F&& f) {
  switch (idt) {
    case F32: case I32: case U32: return f(uint32_t{});
    case F64: case I64: case U64: return f(uint64_t{});
  }
  return Status{1, "Error: metacell IDs must be of an ID type with 4 or 8 bytes"};
}

Status iso_grid(const uint32_t pt_dims[3], const uint32_t mc_dims[3], IsoGrid& g) {
  for (int d = 0; d < 3; d++)
    if (pt_dims[d] < 2 || mc_dims[d] == 0)
      return Status{1, "Error: need at least 2 vertices and metacells of >= 1 voxel per axis"};
  g.px = pt_dims[0], g.py = pt_dims[1], g.pz = pt_dims[2];
  g.mx = mc_dims[0], g.my = mc_dims[1], g.mz = mc_dims[2];
  g.gx = (g.px - 1 + g.mx - 1) / g.mx;
  g.gy = (g.py - 1 + g.my - 1) / g.my;
  g.gz = (g.pz - 1 + g.mz - 1) / g.mz;
  return Status{};
}

unsigned iso_grid_blocks(size_t nids) {
  int dev = 0, cus = 0;
  hipGetDevice(&dev);
  hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const size_t cap = static_cast<size_t>(cus > 0 ? cus : 1) * kIsoWavesPerCu;
  return static_cast<unsigned>(std::max<size_t>(1, std::min(nids, cap)));
}

// Metacells that a wave can hold vertex by vertex (5 x 5 x 5 of them), on
// grids whose coordinates are exact as floats (a position is the sum of the
// metacell's and the vertex's) and whose vertex offsets within a metacell
// fit 32 bits.
bool small_cells(const IsoGrid& g) {
  return g.mx <= 4 && g.my <= 4 && g.mz <= 4 && g.px <= (1u << 24) && g.py <= (1u << 24) && g.pz <= (1u << 24) &&
         static_cast<uint64_t>(g.px) * (g.py + 2ull) < (1ull << 26);
}

// Workgroups for a list: about 8 metacells per wave, so that the case table's
// set-up (some microseconds) is shared, but two workgroups per CU before that
// and at most kMc4BlocksPerCu (5 to 40 per CU measured within 2% on 670,647
// metacells).
unsigned mc4_blocks(size_t nids) {
  int dev = 0, cus = 0;
  hipGetDevice(&dev);
  hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const size_t c = static_cast<size_t>(cus > 0 ? cus : 1);
  const size_t want = std::min(std::max(nids / (8 * kMc4Waves), 2 * c), c * kMc4BlocksPerCu);
  return static_cast<unsigned>(std::max<size_t>(1, std::min((nids + kMc4Waves - 1) / kMc4Waves, want)));
}

}  // namespace

Status mc_count(int dtype, int id_dtype, const void* vertices_d, const uint32_t pt_dims[3],
                const uint32_t mc_dims[3], const void* ids_d, size_t nids, const void* isovalue,
                unsigned long long* counts_d, unsigned long long* err_d, hipStream_t stream) {
  IsoGrid g;
  Status st = iso_grid(pt_dims, mc_dims, g);
  if (!st.ok() || nids == 0) return st;
  return with_t(dtype, [&](auto t) {
    return with_idx(id_dtype, [&](auto i) {
      using T = decltype(t);
      using I = decltype(i);
      T q;
      std::memcpy(&q, isovalue, sizeof(T));
      if (small_cells(g))
        k_mc_count4<T, I><<<mc4_blocks(nids), kMc4Waves * kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, counts_d, err_d);
      else
        k_mc_count<T, I><<<iso_grid_blocks(nids), kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, counts_d, err_d);
      return hip_status(hipGetLastError(), "Error in launching the marching cubes count");
    });
  });
}

Status mc_write(int dtype, int id_dtype, const void* vertices_d, const uint32_t pt_dims[3],
                const uint32_t mc_dims[3], const void* ids_d, size_t nids, const void* isovalue,
                const unsigned long long* offsets_d, size_t capacity, float* tri_d, hipStream_t stream) {
  IsoGrid g;
  Status st = iso_grid(pt_dims, mc_dims, g);
  if (!st.ok() || nids == 0) return st;
  return with_t(dtype, [&](auto t) {
    return with_idx(id_dtype, [&](auto i) {
      using T = decltype(t);
      using I = decltype(i);
      T q;
      std::memcpy(&q, isovalue, sizeof(T));
      if (small_cells(g))
        k_mc_write4<T, I><<<mc4_blocks(nids), kMc4Waves * kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, offsets_d, capacity, tri_d);
      else
        k_mc_write<T, I><<<iso_grid_blocks(nids), kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, offsets_d, capacity, tri_d);
      return hip_status(hipGetLastError(), "Error in launching the marching cubes write");
    });
  });
}

Status iso_count(int dtype, int id_dtype, const void* vertices_d, const uint32_t pt_dims[3],
                 const uint32_t mc_dims[3], const void* ids_d, size_t nids, const void* isovalue,
                 unsigned long long* counts_d, unsigned long long* err_d, hipStream_t stream) {
  IsoGrid g;
  Status st = iso_grid(pt_dims, mc_dims, g);
  if (!st.ok() || nids == 0) return st;
  return with_t(dtype, [&](auto t) {
    return with_idx(id_dtype, [&](auto i) {
      using T = decltype(t);
      using I = decltype(i);
      T q;
      std::memcpy(&q, isovalue, sizeof(T));
      if (small_cells(g))
        k_iso_count4<T, I><<<mc4_blocks(nids), kMc4Waves * kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, counts_d, err_d);
      else
        k_iso_count<T, I><<<iso_grid_blocks(nids), kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, counts_d, err_d);
      return hip_status(hipGetLastError(), "Error in launching the isosurface count");
    });
  });
}

Status iso_write(int dtype, int id_dtype, const void* vertices_d, const uint32_t pt_dims[3],
                 const uint32_t mc_dims[3], const void* ids_d, size_t nids, const void* isovalue,
                 const unsigned long long* offsets_d, size_t capacity, float* tri_d, hipStream_t stream) {
  IsoGrid g;
  Status st = iso_grid(pt_dims, mc_dims, g);
  if (!st.ok() || nids == 0) return st;
  return with_t(dtype, [&](auto t) {
    return with_idx(id_dtype, [&](auto i) {
      using T = decltype(t);
      using I = decltype(i);
      T q;
      std::memcpy(&q, isovalue, sizeof(T));
      if (small_cells(g))
        k_iso_write4<T, I><<<mc4_blocks(nids), kMc4Waves * kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, offsets_d, capacity, tri_d);
      else
        k_iso_write<T, I><<<iso_grid_blocks(nids), kIsoWave, 0, stream>>>(
            static_cast<const T*>(vertices_d), g, static_cast<const I*>(ids_d), nids, q, offsets_d, capacity, tri_d);
      return hip_status(hipGetLastError(), "Error in launching the isosurface write");
    });
  });
}

}  // namespace pst
