// surface.hip -- iso-surface extraction from particle positions.
//
// SurfaceSPH::extract (SurfaceSPH.cpp:29-190) lays a node grid over the
// particles' bounds plus a margin, evaluates the field of evaluateIso_Kernel
// (UniformGridKernel.cu:98-138) at every node, and polygonises it with
// marching cubes (MarchingCube_Kernel.cu:14-158).  Here, on the device:
//
//   k_bounds     min / max of the particle positions (order-independent)
//   k_sorted     particles in the order of a uniform grid of cell r
//   k_iso        field at each node, f = sum_j (r^2 - d_j^2)^3 / r^6 over
//                the particles within r = h / scale (27 cells), in sorted
//                order; one wave per 4 x 4 x 4 nodes, which takes its
//                candidates together where nodes are close (kBoxCells)
//   k_edges      crossed grid edges (one end <= iso, the other not), three
//                per node (+x, +y, +z); exclusive scan -> vertex numbers
//   k_vertices   one vertex per crossed edge, vertexInterpolate_MarchingCube
//                (MarchingCube_Kernel.cu:145-155), and its normal: the
//                direction of -grad f; waves and candidates as for k_iso
//   k_cubes      case index and triangle count per cube; exclusive scan
//   k_emit       triangles as vertex-index triples, cube by cube (x fastest)
//
// Vertices are shared through their grid edge, so the mesh is indexed
// without the host-side float-equality merge of SurfaceSPH.cpp:118-150.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "mc_cases.h"
#include "psb_internal.h"

namespace psb {

__constant__ McCases c_mc;
// cube edge -> (node offset x, y, z, axis of the grid edge from that node)
// for the corner numbering of polygonize_MarchingCube_Kernel
__constant__ int8_t c_edge_node[12][4] = {{0, 0, 0, 0}, {1, 0, 0, 2}, {0, 0, 1, 0}, {0, 0, 0, 2},
                                          {0, 1, 0, 0}, {1, 1, 0, 2}, {0, 1, 1, 0}, {0, 1, 0, 2},
                                          {0, 0, 0, 1}, {1, 0, 0, 1}, {1, 0, 1, 1}, {0, 0, 1, 1}};

// float -> unsigned key with the same order (for atomicMin / atomicMax)
__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
static float key_float(uint32_t k) {
  const uint32_t u = (k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

__device__ __forceinline__ bool kept(const uint32_t* ids, uint32_t limit, uint32_t p) {
  return !ids || ids[p] < limit;
}

__global__ __launch_bounds__(256) void k_bounds_init(uint32_t* out) {
  if (threadIdx.x < 6) out[threadIdx.x] = threadIdx.x < 3 ? 0xFFFFFFFFu : 0u;
}

// At most kBoundsBlocks workgroups, each with one atomic per bound: all
// atomics fall on one cache line, and one set per wave (4,096 waves at 262,144
// particles) took 281 us against 10.
constexpr uint32_t kBoundsBlocks = 128;
__global__ __launch_bounds__(256) void k_bounds(uint32_t n, const float4* __restrict__ pos,
                                                const uint32_t* __restrict__ ids, uint32_t limit,
                                                uint32_t* __restrict__ out) {
  __shared__ uint32_t red[4][6];
  uint32_t lo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, hi[3] = {0u, 0u, 0u};
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    if (!kept(ids, limit, p)) continue;
    const float4 x = pos[p];
    const float c[3] = {x.x, x.y, x.z};
    for (int a = 0; a < 3; ++a) {
      const uint32_t k = order_key(c[a]);
      lo[a] = min(lo[a], k);
      hi[a] = max(hi[a], k);
    }
  }
  for (int a = 0; a < 3; ++a) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo[a] = min(lo[a], (uint32_t)__shfl_xor((int)lo[a], o, 64));
      hi[a] = max(hi[a], (uint32_t)__shfl_xor((int)hi[a], o, 64));
    }
    if ((threadIdx.x & 63u) == 0) {
      red[threadIdx.x >> 6][a] = lo[a];
      red[threadIdx.x >> 6][3 + a] = hi[a];
    }
  }
  __syncthreads();
  const uint32_t a = threadIdx.x;
  if (a < 3) {
    const uint32_t v = min(min(red[0][a], red[1][a]), min(red[2][a], red[3][a]));
    if (v != 0xFFFFFFFFu) atomicMin(out + a, v);
  } else if (a < 6) {
    const uint32_t v = max(max(red[0][a], red[1][a]), max(red[2][a], red[3][a]));
    if (v != 0u) atomicMax(out + a, v);
  }
}

struct NodeGrid {
  int nx, ny, nz;
  float ox, oy, oz, cell;
  float iso, r2, inv_r6;
};

constexpr int kMaxNodes = 4096;   // per axis
// A wave takes its block's candidates together up to this node spacing over
// r; above, each lane walks its own 27 cells.  The box a wave has to look
// through grows with the cube of (3 spacings + 2 r), a lane's cells do not.
// Us per extraction, box / cells (particles; r in particle spacings):
//                    0.25         0.4        0.5        1          4
//   262,144; 3.1   336 / 443   275 / 298  308 / 246  850 / 253  10,450 / 219
//   32,768; 3.1    200 / 208   264 / 218  275 / 208  777 / 230   5,860 / 214
//   262,144; 2     340 / 423   220 / 274  208 / 195  321 / 156   2,400 / 141
//   32,768; 5                  607 / 522  780 / 500  2,265 / 520
constexpr float kBoxCells = 0.4f;

__device__ __forceinline__ void node_pos(const NodeGrid& G, int i, int j, int k, float& x, float& y,
                                         float& z) {
  x = G.ox + (float)i * G.cell;
  y = G.oy + (float)j * G.cell;
  z = G.oz + (float)k * G.cell;
}

// Positions in the grid's sorted order; a particle that is left out goes far
// away (finite, so that its zero weight makes no NaN).
constexpr float kFar = 1e18f;
__global__ __launch_bounds__(256) void k_sorted(uint32_t n, const uint32_t* __restrict__ perm,
                                                const float4* __restrict__ pos,
                                                const uint32_t* __restrict__ ids, uint32_t limit,
                                                float4* __restrict__ xs) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t p = perm[k];
  const float4 q = pos[p];
  xs[k] = kept(ids, limit, p) ? make_float4(q.x, q.y, q.z, 0.f) : make_float4(kFar, kFar, kFar, 0.f);
}

// A wave's block of kNodeBlock^3 nodes and the box [lo, hi] around the points
// its lanes evaluate.
constexpr int kNodeBlock = 4;
struct WaveBox {
  float lo[3], hi[3];
  int c0[3], c1[3];     // grid cells of the box's corners
};

__device__ __forceinline__ void box_cells(const GridDev& g, WaveBox& w) {
  uint32_t bad = 0;
  const float mn[3] = {g.minx, g.miny, g.minz};
  const int nc[3] = {g.nx, g.ny, g.nz};
  for (int a = 0; a < 3; ++a) {
    w.c0[a] = max(cell_coord(w.lo[a], mn[a], g.cell, nc[a], bad) - 1, 0);
    w.c1[a] = min(cell_coord(w.hi[a], mn[a], g.cell, nc[a], bad) + 1, nc[a] - 1);
  }
}

// Visit, in sorted order, the particles near a wave's box: rows of cells in
// ascending (z, y), 64 candidates at a time, one per lane; those within reach
// of the box go to LDS in order, and every lane then sees each of them (an
// LDS broadcast).  The field and normal sums of a lane's own 27 cells are
// ~780 candidates at r = 3 spacings of which ~120 lie within r; per wave ~620
// are near a block of 4^3 nodes a third of r apart, and one load serves 64 nodes
// instead of a gather (through the permutation) per candidate and node.  262,144
// particles, 440,000 nodes: k_iso 617 -> 106 us, k_vertices 245 -> 57 us; what
// is left is the ~13 VALU instructions per wave and survivor.
template <class F>
__device__ __forceinline__ void for_near_box(const GridDev& g, const uint32_t* __restrict__ start,
                                             const float4* __restrict__ xs, const WaveBox& w,
                                             float r2, float4* lds, F&& f) {
  const uint32_t lane = threadIdx.x & 63u;
  const float reach2 = r2 * 1.001f;   // the box test is conservative, the sums decide
  for (int zz = w.c0[2]; zz <= w.c1[2]; ++zz)
    for (int yy = w.c0[1]; yy <= w.c1[1]; ++yy) {
      const uint64_t base = (uint64_t)g.nx * ((uint64_t)yy + (uint64_t)g.ny * (uint64_t)zz);
      const uint32_t q1 = start[base + w.c1[0] + 1];
      for (uint32_t q0 = start[base + w.c0[0]]; q0 < q1; q0 += 64u) {
        const uint32_t q = q0 + lane;
        float4 x = make_float4(kFar, kFar, kFar, 0.f);
        if (q < q1) x = xs[q];
        const float dx = fmaxf(fmaxf(w.lo[0] - x.x, x.x - w.hi[0]), 0.f);
        const float dy = fmaxf(fmaxf(w.lo[1] - x.y, x.y - w.hi[1]), 0.f);
        const float dz = fmaxf(fmaxf(w.lo[2] - x.z, x.z - w.hi[2]), 0.f);
        const bool in = dot3(dx, dy, dz, dx, dy, dz) <= reach2;
        const uint64_t m = __ballot(in);
        const uint32_t ns = (uint32_t)__popcll(m);
        if (!ns) continue;
        if (in) lds[__popcll(m & ((1ull << lane) - 1ull))] = x;
        if (lane < 4u) lds[ns + lane] = make_float4(kFar, kFar, kFar, 0.f);   // pad to fours
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (uint32_t k = 0; k < ns; k += 4u) {
          float4 c[4];
#pragma unroll
          for (uint32_t u = 0; u < 4u; ++u) c[u] = lds[k + u];
#pragma unroll
          for (uint32_t u = 0; u < 4u; ++u) f(c[u]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
}

// Whether particle x lies in the 27 cells around the point whose cell is c.  A
// particle outside them is more than a cell (r) away but for rounding at the
// cell borders: only a distance this close to r needs the test.  An index
// (x - min) / r carries two roundings, so it is off by at most 2^-23 of itself:
// of two points in a grid of N cells along an axis the one more than a cell away
// is no nearer than (1 - 2^-22 N) r.  Where nodes are close enough for the block
// kernels N is at most 1,640; from 16,000 on the rounding does pass 0.999 of r^2.
constexpr float kNearEdge = 0.999f;
static_assert((kBoxCells * kMaxNodes + 2) / (1 << 21) + 1.f / (1 << 18) < 1.f - kNearEdge, "kNearEdge");
__device__ __forceinline__ bool in_cells(const GridDev& g, const int (&c)[3], const float4& x) {
  uint32_t bad = 0;
  const int kx = cell_coord(x.x, g.minx, g.cell, g.nx, bad);
  const int ky = cell_coord(x.y, g.miny, g.cell, g.ny, bad);
  const int kz = cell_coord(x.z, g.minz, g.cell, g.nz, bad);
  return abs(kx - c[0]) <= 1 && abs(ky - c[1]) <= 1 && abs(kz - c[2]) <= 1;
}
__device__ __forceinline__ void cells_of(const GridDev& g, float x, float y, float z, int (&c)[3]) {
  uint32_t bad = 0;
  c[0] = cell_coord(x, g.minx, g.cell, g.nx, bad);
  c[1] = cell_coord(y, g.miny, g.cell, g.ny, bad);
  c[2] = cell_coord(z, g.minz, g.cell, g.nz, bad);
}

// The same for each lane by itself: the particles of the 27 cells around c in
// sorted order, four loads in flight.
template <class F>
__device__ __forceinline__ void for_near_cells(const GridDev& g, const uint32_t* __restrict__ start,
                                               const float4* __restrict__ xs, const int (&c)[3],
                                               F&& f) {
  const int x0 = max(c[0] - 1, 0), x1 = min(c[0] + 1, g.nx - 1);
  for (int zz = max(c[2] - 1, 0); zz <= min(c[2] + 1, g.nz - 1); ++zz)
    for (int yy = max(c[1] - 1, 0); yy <= min(c[1] + 1, g.ny - 1); ++yy) {
      const uint64_t base = (uint64_t)g.nx * ((uint64_t)yy + (uint64_t)g.ny * (uint64_t)zz);
      const uint32_t q1 = start[base + x1 + 1];
      for (uint32_t q = start[base + x0]; q < q1; q += 4u) {
        float4 x[4];
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) x[u] = xs[min(q + u, q1 - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) f(x[u], q + u < q1);
      }
    }
}

// first node of wave `w`'s block (blocks x fastest), false past the last block
__device__ __forceinline__ bool block_origin(const NodeGrid& G, uint32_t w, int (&o)[3]) {
  const uint32_t bx = (G.nx + kNodeBlock - 1) / kNodeBlock, by = (G.ny + kNodeBlock - 1) / kNodeBlock,
                 bz = (G.nz + kNodeBlock - 1) / kNodeBlock;
  o[0] = (int)(w % bx) * kNodeBlock;
  o[1] = (int)(w / bx % by) * kNodeBlock;
  o[2] = (int)(w / (bx * by)) * kNodeBlock;
  return w / (bx * by) < bz;
}

constexpr uint32_t kIsoWaves = 4;   // waves per workgroup, one node block each
template <bool BOX>
__global__ __launch_bounds__(64 * kIsoWaves) void k_iso(NodeGrid G, GridDev g,
                                                        const uint32_t* __restrict__ start,
                                                        const float4* __restrict__ xs,
                                                        float* __restrict__ iso) {
  __shared__ float4 lds[BOX ? kIsoWaves : 1][BOX ? 64 + 4 : 1];
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int o[3];
  if (!block_origin(G, blockIdx.x * kIsoWaves + wv, o)) return;
  const int i = o[0] + (int)(lane & 3u), j = o[1] + (int)(lane >> 2 & 3u), k = o[2] + (int)(lane >> 4);
  const bool mine = i < G.nx && j < G.ny && k < G.nz;
  float x, y, z;
  node_pos(G, i, j, k, x, y, z);
  int c[3];
  cells_of(g, x, y, z, c);
  float acc = 0.f;
  if constexpr (!BOX) {
    if (!mine) return;
    // (the weight in a function of its own: written into the walk it came out
    // with a branch per candidate, 284 against 252 us an extraction at a
    // spacing of r)
    auto add = [&](float d2, bool in) {
      const float v = in ? G.r2 - d2 : 0.f;
      acc = __builtin_fmaf(v * v, v, acc);   // v = 0 leaves acc (never -0) unchanged
    };
    for_near_cells(g, start, xs, c, [&](const float4& q, bool in) {
      const float dx = x - q.x, dy = y - q.y, dz = z - q.z;
      const float d2 = dot3(dx, dy, dz, dx, dy, dz);
      add(d2, in && d2 <= G.r2);
    });
    iso[(uint64_t)i + (uint64_t)G.nx * ((uint64_t)j + (uint64_t)G.ny * (uint64_t)k)] = acc * G.inv_r6;
    return;
  }
  const int e[3] = {min(o[0] + kNodeBlock, G.nx) - 1, min(o[1] + kNodeBlock, G.ny) - 1,
                    min(o[2] + kNodeBlock, G.nz) - 1};
  WaveBox w;
  node_pos(G, o[0], o[1], o[2], w.lo[0], w.lo[1], w.lo[2]);
  node_pos(G, e[0], e[1], e[2], w.hi[0], w.hi[1], w.hi[2]);
  box_cells(g, w);
  const float edge2 = G.r2 * kNearEdge;
  for_near_box(g, start, xs, w, G.r2, lds[wv], [&](const float4& q) {
    const float dx = x - q.x, dy = y - q.y, dz = z - q.z;
    const float d2 = dot3(dx, dy, dz, dx, dy, dz);
    bool in = d2 <= G.r2;
    if (__any(in && d2 > edge2)) in = in && (d2 <= edge2 || in_cells(g, c, q));
    const float v = in ? G.r2 - d2 : 0.f;
    acc = __builtin_fmaf(v * v, v, acc);
  });
  if (mine)
    iso[(uint64_t)i + (uint64_t)G.nx * ((uint64_t)j + (uint64_t)G.ny * (uint64_t)k)] = acc * G.inv_r6;
}

__global__ __launch_bounds__(256) void k_edges(NodeGrid G, const float* __restrict__ iso,
                                               uint8_t* __restrict__ eflags,
                                               uint32_t* __restrict__ vcount) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nn = (uint64_t)G.nx * G.ny * G.nz;
  if (t >= nn) return;
  const int i = (int)(t % G.nx), j = (int)((t / G.nx) % G.ny), k = (int)(t / ((uint64_t)G.nx * G.ny));
  const bool b0 = iso[t] <= G.iso;
  uint32_t f = 0;
  if (i + 1 < G.nx && (iso[t + 1] <= G.iso) != b0) f |= 1u;
  if (j + 1 < G.ny && (iso[t + G.nx] <= G.iso) != b0) f |= 2u;
  if (k + 1 < G.nz && (iso[t + (uint64_t)G.nx * G.ny] <= G.iso) != b0) f |= 4u;
  eflags[t] = (uint8_t)f;
  vcount[t] = __builtin_popcount(f);
}

// One wave per node block: the block's crossed edges are dealt to the lanes
// (a wave of consecutive nodes had ~1 lane in 10 at work), 64 at a time.
template <bool BOX>
__global__ __launch_bounds__(64 * kIsoWaves) void k_vertices(
    NodeGrid G, GridDev g, const uint32_t* __restrict__ start, const float4* __restrict__ xs,
    const float* __restrict__ iso, const uint8_t* __restrict__ eflags,
    const uint32_t* __restrict__ vbase, float* __restrict__ verts, float* __restrict__ norms) {
  __shared__ float4 lds[BOX ? kIsoWaves : 1][BOX ? 64 + 4 : 1];
  __shared__ uint8_t edge[kIsoWaves][192];   // node of the block (6 bits), axis (2 bits)
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int o[3];
  if (!block_origin(G, blockIdx.x * kIsoWaves + wv, o)) return;
  const int i = o[0] + (int)(lane & 3u), j = o[1] + (int)(lane >> 2 & 3u), k = o[2] + (int)(lane >> 4);
  const uint64_t sy = (uint64_t)G.nx, sz = (uint64_t)G.nx * G.ny;
  const uint64_t t0 = (uint64_t)o[0] + sy * (uint64_t)o[1] + sz * (uint64_t)o[2];
  const uint32_t f = (i < G.nx && j < G.ny && k < G.nz)
                         ? eflags[(uint64_t)i + sy * (uint64_t)j + sz * (uint64_t)k] : 0u;
  uint32_t total = 0;
#pragma unroll
  for (uint32_t axis = 0; axis < 3u; ++axis) {
    const uint64_t m = __ballot(f >> axis & 1u);
    if (f >> axis & 1u)
      edge[wv][total + __popcll(m & ((1ull << lane) - 1ull))] = (uint8_t)(lane << 2 | axis);
    total += (uint32_t)__popcll(m);
  }
  if (!total) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  WaveBox w;
  if constexpr (BOX) {
    node_pos(G, o[0], o[1], o[2], w.lo[0], w.lo[1], w.lo[2]);
    node_pos(G, o[0] + kNodeBlock, o[1] + kNodeBlock, o[2] + kNodeBlock, w.hi[0], w.hi[1], w.hi[2]);
    box_cells(g, w);
  }
  const float edge2 = G.r2 * kNearEdge;
  for (uint32_t v0 = 0; v0 < total; v0 += 64u) {
    const bool on = v0 + lane < total;
    const uint32_t ed = edge[wv][on ? v0 + lane : v0];
    const int axis = (int)(ed & 3u);
    const int ni = o[0] + (int)(ed >> 2 & 3u), nj = o[1] + (int)(ed >> 4 & 3u), nk = o[2] + (int)(ed >> 6);
    const uint64_t t = t0 + (ed >> 2 & 3u) + sy * (ed >> 4 & 3u) + sz * (ed >> 6);
    float ax, ay, az, bx, by, bz;
    node_pos(G, ni, nj, nk, ax, ay, az);
    node_pos(G, ni + (axis == 0), nj + (axis == 1), nk + (axis == 2), bx, by, bz);
    const float va = iso[t], vb = iso[t + (axis == 0 ? 1 : axis == 1 ? sy : sz)];
    const uint32_t v = vbase[t] + __builtin_popcount(eflags[t] & ((1u << axis) - 1u));
    float px, py, pz;
    // vertexInterpolate_MarchingCube (MarchingCube_Kernel.cu:145-155)
    if (fabsf(G.iso - va) < 0.000001f) { px = ax; py = ay; pz = az; }
    else if (fabsf(G.iso - vb) < 0.000001f) { px = bx; py = by; pz = bz; }
    else if (fabsf(va - vb) < 0.000001f) { px = ax; py = ay; pz = az; }
    else {
      const float mu = (G.iso - va) / (vb - va);
      px = ax + mu * (bx - ax); py = ay + mu * (by - ay); pz = az + mu * (bz - az);
    }
    // normal: -grad f ~ sum_j (x - x_j)(r^2 - d_j^2)^2, normalised
    int c[3];
    cells_of(g, px, py, pz, c);
    float gx = 0.f, gy = 0.f, gz = 0.f;
    if constexpr (BOX) {
      for_near_box(g, start, xs, w, G.r2, lds[wv], [&](const float4& q) {
        const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
        const float d2 = dot3(dx, dy, dz, dx, dy, dz);
        bool in = d2 < G.r2;
        if (__any(in && d2 > edge2)) in = in && (d2 <= edge2 || in_cells(g, c, q));
        const float u = in ? G.r2 - d2 : 0.f;
        const float u2 = u * u;   // 0: adds a zero of either sign to sums that are never -0
        gx = __builtin_fmaf(dx, u2, gx);
        gy = __builtin_fmaf(dy, u2, gy);
        gz = __builtin_fmaf(dz, u2, gz);
      });
    } else if (on) {
      for_near_cells(g, start, xs, c, [&](const float4& q, bool in) {
        const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
        const float d2 = dot3(dx, dy, dz, dx, dy, dz);
        const float u = in && d2 < G.r2 ? G.r2 - d2 : 0.f;
        const float u2 = u * u;
        gx = __builtin_fmaf(dx, u2, gx);
        gy = __builtin_fmaf(dy, u2, gy);
        gz = __builtin_fmaf(dz, u2, gz);
      });
    }
    if (!on) continue;
    const float gl = sqrtf(dot3(gx, gy, gz, gx, gy, gz));
    if (gl > 0.f) { gx = gx / gl; gy = gy / gl; gz = gz / gl; }
    verts[3 * (size_t)v] = px; verts[3 * (size_t)v + 1] = py; verts[3 * (size_t)v + 2] = pz;
    norms[3 * (size_t)v] = gx; norms[3 * (size_t)v + 1] = gy; norms[3 * (size_t)v + 2] = gz;
  }
}

__device__ __forceinline__ uint32_t cube_case(const NodeGrid& G, const float* __restrict__ iso,
                                              uint64_t t) {
  const uint64_t sx = 1, sy = (uint64_t)G.nx, sz = (uint64_t)G.nx * G.ny;
  // corner order of polygonize_MarchingCube_Kernel (MarchingCube_Kernel.cu:45-53)
  const uint64_t c[8] = {t, t + sx, t + sx + sz, t + sz, t + sy, t + sx + sy, t + sx + sy + sz, t + sy + sz};
  uint32_t cs = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (iso[c[q]] <= G.iso) cs |= 1u << q;
  return cs;
}

__device__ __forceinline__ void cube_of(const NodeGrid& G, uint64_t u, int& i, int& j, int& k) {
  const uint64_t cx = G.nx - 1, cy = G.ny - 1;
  i = (int)(u % cx); j = (int)((u / cx) % cy); k = (int)(u / (cx * cy));
}

__global__ __launch_bounds__(256) void k_cubes(NodeGrid G, const float* __restrict__ iso,
                                               uint32_t* __restrict__ tcount) {
  const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nc = (uint64_t)(G.nx - 1) * (G.ny - 1) * (G.nz - 1);
  if (u >= nc) return;
  int i, j, k;
  cube_of(G, u, i, j, k);
  const uint64_t t = (uint64_t)i + (uint64_t)G.nx * ((uint64_t)j + (uint64_t)G.ny * k);
  tcount[u] = c_mc.ntri[cube_case(G, iso, t)];
}

__global__ __launch_bounds__(256) void k_emit(NodeGrid G, const float* __restrict__ iso,
                                              const uint8_t* __restrict__ eflags,
                                              const uint32_t* __restrict__ vbase,
                                              const uint32_t* __restrict__ tbase,
                                              uint32_t* __restrict__ tris) {
  const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nc = (uint64_t)(G.nx - 1) * (G.ny - 1) * (G.nz - 1);
  if (u >= nc) return;
  const uint32_t b = tbase[u], e = tbase[u + 1];
  if (b == e) return;
  int i, j, k;
  cube_of(G, u, i, j, k);
  const uint64_t t = (uint64_t)i + (uint64_t)G.nx * ((uint64_t)j + (uint64_t)G.ny * k);
  const uint32_t cs = cube_case(G, iso, t);
  for (uint32_t q = 0; q < 3 * (e - b); ++q) {
    const int ed = c_mc.tri[cs][q];
    const uint64_t nd = t + (uint64_t)c_edge_node[ed][0] +
                        (uint64_t)G.nx * ((uint64_t)c_edge_node[ed][1] + (uint64_t)G.ny * c_edge_node[ed][2]);
    const uint32_t below = eflags[nd] & ((1u << c_edge_node[ed][3]) - 1u);
    tris[3 * (size_t)b + q] = vbase[nd] + __builtin_popcount(below);
  }
}

psb_status scan_exclusive(uint32_t* count, uint64_t n, uint32_t* bsum, uint32_t* start,
                          hipStream_t s);

}  // namespace psb

using namespace psb;

struct psb_surface_s {
  psb_context ctx = nullptr;
  psb_grid grid = nullptr;
  psb_grid_desc gdesc{};
  uint32_t grid_cap = 0;
  NodeGrid G{};
  uint64_t nodes = 0, cubes = 0;
  // element capacities of the device arrays below
  size_t cap_iso = 0, cap_ef = 0, cap_vc = 0, cap_vb = 0, cap_tc = 0, cap_tb = 0, cap_bs = 0;
  size_t cap_v = 0, cap_n = 0, cap_t = 0, cap_xs = 0;
  float4* xs = nullptr;            // positions in the grid's sorted order
  float* iso = nullptr;
  uint8_t* eflags = nullptr;
  uint32_t *vcount = nullptr, *vbase = nullptr, *tcount = nullptr, *tbase = nullptr;
  uint32_t* bsum = nullptr;
  uint32_t* bounds = nullptr;
  uint32_t* h_counts = nullptr;   // pinned
  float *verts = nullptr, *norms = nullptr;
  uint32_t* tris = nullptr;
  uint32_t nv = 0, nt = 0;
};

namespace {
std::vector<bool> g_table_loaded;   // per device

psb_status load_table(int dev) {
  if ((int)g_table_loaded.size() <= dev) g_table_loaded.resize(dev + 1, false);
  if (g_table_loaded[dev]) return PSB_OK;
  static const McCases tab = mc_generate();
  PSB_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_mc), &tab, sizeof(tab)));
  g_table_loaded[dev] = true;
  return PSB_OK;
}

template <class T> psb_status grow(T*& p, size_t& cap, size_t want) {
  if (want <= cap && p) return PSB_OK;
  if (p) PSB_HIP(hipFree(p));
  p = nullptr;
  const size_t c = std::max<size_t>(want, 1);
  PSB_HIP(hipMalloc((void**)&p, sizeof(T) * c));
  cap = c;
  return PSB_OK;
}
}  // namespace

extern "C" {

psb_status psb_surface_default_params(psb_surface_params* p) {
  PSB_ARG(p, "null argument");
  p->cell_size = 0.03f;   // SurfaceSPH.cpp:31
  p->scale = 0.65f;       // SurfaceSPH.cpp:32
  p->iso_level = 0.5f;
  p->margin = 2.0f;       // SurfaceSPH.cpp:43: 2 h / scale
  return PSB_OK;
}

psb_status psb_surface_case_table(uint8_t* triangle_counts, int8_t* triangle_edges) {
  McCases t;
  try {
    t = mc_generate();
  } catch (const std::exception& e) {
    set_error(e.what());
    return PSB_ERR_STATE;
  }
  if (triangle_counts) std::memcpy(triangle_counts, t.ntri, sizeof(t.ntri));
  if (triangle_edges)
    for (int c = 0; c < 256; ++c)
      for (int k = 0; k < 16; ++k) triangle_edges[16 * c + k] = k < 3 * kMcMaxTri ? t.tri[c][k] : -1;
  return PSB_OK;
}

psb_status psb_surface_create(psb_context ctx, psb_surface* out) {
  PSB_ARG(ctx && out, "null argument");
  PSB_HIP(hipSetDevice(ctx->device));
  auto* s = new psb_surface_s;
  s->ctx = ctx;
  psb_status r = PSB_OK;
  if (hipMalloc((void**)&s->bounds, 64) != hipSuccess ||
      hipHostMalloc((void**)&s->h_counts, 64, hipHostMallocDefault) != hipSuccess) {
    set_error("surface allocation failed");
    r = PSB_ERR_OUT_OF_MEMORY;
  }
  if (r == PSB_OK) r = load_table(ctx->device);
  if (r != PSB_OK) { psb_surface_destroy(s); return r; }
  *out = s;
  return PSB_OK;
}

psb_status psb_surface_destroy(psb_surface s) {
  if (!s) return PSB_OK;
  (void)hipSetDevice(s->ctx->device);
  (void)hipStreamSynchronize(s->ctx->stream);
  if (s->grid) psb_finalize_grid(s->grid);
  for (void* p : {(void*)s->iso, (void*)s->eflags, (void*)s->vcount, (void*)s->vbase,
                  (void*)s->tcount, (void*)s->tbase, (void*)s->bsum, (void*)s->bounds,
                  (void*)s->verts, (void*)s->norms, (void*)s->tris, (void*)s->xs})
    if (p) (void)hipFree(p);
  if (s->h_counts) (void)hipHostFree(s->h_counts);
  delete s;
  return PSB_OK;
}

psb_status psb_surface_extract_points(psb_surface s, const float* pos4, const uint32_t* ids,
                                      uint32_t n, uint32_t id_limit, float support_radius,
                                      const psb_surface_params* prm, uint32_t* num_vertices,
                                      uint32_t* num_triangles) {
  PSB_ARG(s && prm && (n == 0 || pos4), "null argument");
  PSB_ARG(std::isfinite(support_radius) && support_radius > 0.f, "support radius must be > 0");
  PSB_ARG(std::isfinite(prm->scale) && prm->scale > 0.f && std::isfinite(prm->cell_size) &&
              prm->cell_size > 0.f && std::isfinite(prm->margin) && prm->margin >= 0.f &&
              std::isfinite(prm->iso_level),
          "surface parameters: scale, cell_size > 0, margin >= 0, finite iso_level");
  PSB_HIP(hipSetDevice(s->ctx->device));
  hipStream_t st = s->ctx->stream;
  const float4* P = reinterpret_cast<const float4*>(pos4);
  s->nv = s->nt = 0;
  s->nodes = s->cubes = 0;
  if (num_vertices) *num_vertices = 0;
  if (num_triangles) *num_triangles = 0;
  if (!n) return PSB_OK;
  // bounds of the kept particles
  hipLaunchKernelGGL(k_bounds_init, dim3(1), dim3(64), 0, st, s->bounds);
  hipLaunchKernelGGL(k_bounds, dim3(std::min(blocks_for(n), kBoundsBlocks)), dim3(kBlock), 0, st, n,
                     P, ids, id_limit, s->bounds);
  PSB_HIP(hipGetLastError());
  PSB_HIP(hipMemcpyAsync(s->h_counts, s->bounds, 24, hipMemcpyDeviceToHost, st));
  PSB_HIP(hipStreamSynchronize(st));
  if (s->h_counts[0] == 0xFFFFFFFFu) return PSB_OK;   // no particle kept
  float lo[3], hi[3];
  for (int a = 0; a < 3; ++a) { lo[a] = key_float(s->h_counts[a]); hi[a] = key_float(s->h_counts[3 + a]); }
  for (int a = 0; a < 3; ++a)
    PSB_ARG(std::isfinite(lo[a]) && std::isfinite(hi[a]), "non-finite particle positions");
  // node grid as SurfaceSPH::extract lays it (SurfaceSPH.cpp:38-60), in double
  const float r = support_radius / prm->scale;
  const double margin = (double)prm->margin * (double)r;
  double mn[3], mx[3];
  uint32_t dims[3];
  float org[3];
  for (int a = 0; a < 3; ++a) {
    mn[a] = (double)lo[a] - margin;
    mx[a] = (double)hi[a] + margin;
    const double len = std::fabs(mx[a] - mn[a]);
    const double nd = std::ceil(len / (double)prm->cell_size);
    PSB_ARG(nd >= 2 && nd <= kMaxNodes, "surface node grid must have 2..4096 nodes per axis");
    dims[a] = (uint32_t)nd;
    const double center = (mn[a] + mx[a]) / 2;
    org[a] = (float)(center - len / 2 + (double)prm->cell_size / 2);
  }
  NodeGrid& G = s->G;
  G.nx = (int)dims[0]; G.ny = (int)dims[1]; G.nz = (int)dims[2];
  G.ox = org[0]; G.oy = org[1]; G.oz = org[2];
  G.cell = prm->cell_size;
  G.iso = prm->iso_level;
  G.r2 = r * r;
  G.inv_r6 = 1.0f / (G.r2 * G.r2 * G.r2);
  s->nodes = (uint64_t)dims[0] * dims[1] * dims[2];
  s->cubes = (uint64_t)(dims[0] - 1) * (dims[1] - 1) * (dims[2] - 1);
  // particle grid of cell r over the margin-extended bounds
  psb_grid_desc gd{};
  for (int a = 0; a < 3; ++a) {
    gd.min[a] = (float)mn[a];
    gd.dims[a] = (int32_t)std::ceil((mx[a] - mn[a]) / (double)r) + 1;
  }
  gd.cell_size = r;
  PSB_ARG((uint64_t)gd.dims[0] * gd.dims[1] * gd.dims[2] <= (1ull << 31),
          "particle grid too fine for the surface radius");
  if (!s->grid || std::memcmp(&gd, &s->gdesc, sizeof gd) != 0 || n > s->grid_cap) {
    if (s->grid) { psb_finalize_grid(s->grid); s->grid = nullptr; }
    PSB_TRY(psb_create_grid_desc(s->ctx, &gd, n, &s->grid));
    s->gdesc = gd;
    s->grid_cap = n;
  }
  PSB_TRY(grid_build(s->grid, P, n, nullptr, st));
  const GridDev g = grid_dev(gd, r);
  PSB_TRY(grow(s->iso, s->cap_iso, s->nodes));
  PSB_TRY(grow(s->eflags, s->cap_ef, s->nodes));
  PSB_TRY(grow(s->vcount, s->cap_vc, s->nodes));
  PSB_TRY(grow(s->vbase, s->cap_vb, s->nodes + 1));
  PSB_TRY(grow(s->tcount, s->cap_tc, s->cubes));
  PSB_TRY(grow(s->tbase, s->cap_tb, s->cubes + 1));
  const uint64_t scan_tiles = (std::max(s->nodes, s->cubes) + kScanTile - 1) / kScanTile;
  PSB_TRY(grow(s->bsum, s->cap_bs, scan_tiles + 1));
  PSB_TRY(grow(s->xs, s->cap_xs, n));
  const uint32_t nbn = blocks_for(s->nodes), nbc = blocks_for(s->cubes);
  uint32_t nbb = 1;   // node blocks, kIsoWaves to a workgroup
  for (int a = 0; a < 3; ++a) nbb *= (dims[a] + kNodeBlock - 1) / kNodeBlock;
  nbb = blocks_for(nbb, kIsoWaves);
  hipLaunchKernelGGL(k_sorted, dim3(blocks_for(n)), dim3(kBlock), 0, st, n, s->grid->perm, P, ids,
                     id_limit, s->xs);
  const bool box = prm->cell_size < kBoxCells * r;
  if (box)
    hipLaunchKernelGGL(k_iso<true>, dim3(nbb), dim3(64 * kIsoWaves), 0, st, G, g, s->grid->start,
                       s->xs, s->iso);
  else
    hipLaunchKernelGGL(k_iso<false>, dim3(nbb), dim3(64 * kIsoWaves), 0, st, G, g, s->grid->start,
                       s->xs, s->iso);
  hipLaunchKernelGGL(k_edges, dim3(nbn), dim3(kBlock), 0, st, G, s->iso, s->eflags, s->vcount);
  PSB_HIP(hipGetLastError());
  PSB_TRY(scan_exclusive(s->vcount, s->nodes, s->bsum, s->vbase, st));
  if (s->cubes) {
    hipLaunchKernelGGL(k_cubes, dim3(nbc), dim3(kBlock), 0, st, G, s->iso, s->tcount);
    PSB_HIP(hipGetLastError());
  }
  PSB_TRY(scan_exclusive(s->tcount, s->cubes, s->bsum, s->tbase, st));
  PSB_HIP(hipMemcpyAsync(s->h_counts, s->vbase + s->nodes, 4, hipMemcpyDeviceToHost, st));
  PSB_HIP(hipMemcpyAsync(s->h_counts + 1, s->tbase + s->cubes, 4, hipMemcpyDeviceToHost, st));
  PSB_HIP(hipStreamSynchronize(st));
  s->nv = s->h_counts[0];
  s->nt = s->h_counts[1];
  PSB_TRY(grow(s->verts, s->cap_v, 3 * (size_t)s->nv));
  PSB_TRY(grow(s->norms, s->cap_n, 3 * (size_t)s->nv));
  PSB_TRY(grow(s->tris, s->cap_t, 3 * (size_t)s->nt));
  if (box)
    hipLaunchKernelGGL(k_vertices<true>, dim3(nbb), dim3(64 * kIsoWaves), 0, st, G, g,
                       s->grid->start, s->xs, s->iso, s->eflags, s->vbase, s->verts, s->norms);
  else
    hipLaunchKernelGGL(k_vertices<false>, dim3(nbb), dim3(64 * kIsoWaves), 0, st, G, g,
                       s->grid->start, s->xs, s->iso, s->eflags, s->vbase, s->verts, s->norms);
  if (s->cubes)
    hipLaunchKernelGGL(k_emit, dim3(nbc), dim3(kBlock), 0, st, G, s->iso, s->eflags, s->vbase,
                       s->tbase, s->tris);
  PSB_HIP(hipGetLastError());
  PSB_HIP(hipStreamSynchronize(st));
  if (num_vertices) *num_vertices = s->nv;
  if (num_triangles) *num_triangles = s->nt;
  return PSB_OK;
}

psb_status psb_surface_get_mesh(psb_surface s, float* vertices3, float* normals3,
                                uint32_t* triangles3) {
  PSB_ARG(s, "null surface");
  PSB_HIP(hipSetDevice(s->ctx->device));
  hipStream_t st = s->ctx->stream;
  if (vertices3 && s->nv)
    PSB_HIP(hipMemcpyAsync(vertices3, s->verts, 12 * (size_t)s->nv, hipMemcpyDeviceToHost, st));
  if (normals3 && s->nv)
    PSB_HIP(hipMemcpyAsync(normals3, s->norms, 12 * (size_t)s->nv, hipMemcpyDeviceToHost, st));
  if (triangles3 && s->nt)
    PSB_HIP(hipMemcpyAsync(triangles3, s->tris, 12 * (size_t)s->nt, hipMemcpyDeviceToHost, st));
  PSB_HIP(hipStreamSynchronize(st));
  return PSB_OK;
}

psb_status psb_surface_get_field(psb_surface s, float* field, uint32_t dims[3], float origin[3],
                                 float* cell) {
  PSB_ARG(s, "null surface");
  if (dims) { dims[0] = s->nodes ? s->G.nx : 0; dims[1] = s->nodes ? s->G.ny : 0; dims[2] = s->nodes ? s->G.nz : 0; }
  if (origin) { origin[0] = s->G.ox; origin[1] = s->G.oy; origin[2] = s->G.oz; }
  if (cell) *cell = s->G.cell;
  if (field && s->nodes) {
    PSB_HIP(hipSetDevice(s->ctx->device));
    PSB_HIP(hipMemcpyAsync(field, s->iso, 4 * s->nodes, hipMemcpyDeviceToHost, s->ctx->stream));
    PSB_HIP(hipStreamSynchronize(s->ctx->stream));
  }
  return PSB_OK;
}

}  // extern "C"
