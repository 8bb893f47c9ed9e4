// grid.hip -- uniform grid: cell hash, stable counting sort, cell ranges,
// reorder and neighbour search for gfx950.
//
// Replaces createGrid / reinitCells / storeParticles / searchNeighbooring
// (UniformGrid.cu:17-99, UniformGridKernel.cu:12-95).  The reference inserts
// particles into 64-slot cell buckets with atomicAdd (order depends on the
// race, no overflow check) and writes a 200-wide neighbour list with a global
// read-modify-write per hit.  Here:
//
//   1. k_hash_count   hash[i] = cell of x_i;  slot[i] = atomicAdd(count[c])
//   2. k_scan_*       start = exclusive prefix sum of count over all cells
//                     (start[c] = #particles with hash < c, start[ncells] = n);
//                     the per-tile sums come from step 1 (tsum), so the scan
//                     reads count once, and only where particles are; k_rank_reorder re-zeroes the occupied
//                     cells' counts for the next build
//   3. k_scatter      tmp[start[c] + slot[i]] = i      (order within a cell
//                     still depends on the atomics)
//   4. k_rank_reorder rank of i among its cell's tmp entries by index ->
//                     dst = start[c] + rank: the stable (hash, index) order;
//                     perm[dst] = i and the particle state is gathered here
//
// The dense lower-bound table start[] makes every stencil row of cells one
// contiguous particle range [start[c0], start[c1 + 1]) because the hash is
// x-fastest, so the neighbour kernel does two table loads per row.
#include "psb_internal.h"
#include "pcisph.h"

namespace psb {

constexpr int kTileSlots = 16;   // copies of the per-tile count table (atomic spreading)

// Bound by its atomics: one per run of lanes in the same cell and, where the
// scan's tiles fit in LDS, one per workgroup and tile (43,993 particles in
// random order 10.9 -> 6.0 us, where a wave went through up to 64 tiles in
// turn; 262,144 in cells of eight 27.3 -> 7.8).  Larger tables are counted by
// wave: a workgroup would pay more to clear and send the table.
constexpr uint32_t kLdsTiles = 512;   // scan tiles counted in LDS

// M: SingleMap or BatchMap (a batch hashes into its scene's cell range).
template <class M>
__global__ __launch_bounds__(M::kMaxThreads) void k_hash_count(M map, const float4* __restrict__ pos,
                                                               uint32_t n, GridDev g0,
                                                               uint32_t* __restrict__ hash,
                                                               uint32_t* __restrict__ slot,
                                                               uint32_t* __restrict__ count,
                                                               uint32_t* __restrict__ flags,
                                                               uint32_t* __restrict__ tsum,
                                                               uint32_t nscan, StepReset rs) {
  if (rs.st && blockIdx.x < rs.scenes) pci_reset_scene(rs.st, blockIdx.x, rs.done, rs.es);
  __shared__ uint32_t tiles[kLdsTiles];
  if (nscan <= kLdsTiles) {
    for (uint32_t t = threadIdx.x; t < nscan; t += blockDim.x) tiles[t] = 0u;
    __syncthreads();
  }
  uint32_t i = 0, sc = 0, off = 0, c = 0xFFFFFFFFu, bad = 0, f = 0;
  bool lead;
  const bool valid = map.locate(n, i, sc, lead);
  if (valid) {
    const GridDev g = map.grid(g0, sc, off);
    const float4 p = pos[i];
    const int cx = cell_coord(p.x, g.minx, g.cell, g.nx, bad);
    const int cy = cell_coord(p.y, g.miny, g.cell, g.ny, bad);
    const int cz = cell_coord(p.z, g.minz, g.cell, g.nz, bad);
    c = off + (uint32_t)cx + (uint32_t)g.nx * ((uint32_t)cy + (uint32_t)g.ny * (uint32_t)cz);
    hash[i] = c;
    if (bad) f |= PSB_FLAG_OUT_OF_GRID;
    if (!(isfinite(p.x) && isfinite(p.y) && isfinite(p.z))) f |= PSB_FLAG_NONFINITE;
    if (f) atomicOr(flags, f);
  }
  // one atomic per run of lanes in the same cell (a cell's slots are given out
  // in any order; atomics on one cell's word serialise)
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t prev = (uint32_t)__shfl_up((int)c, 1, 64);
  const uint64_t heads = __ballot(lane == 0u || c != prev);
  const uint32_t head = 63u - (uint32_t)__builtin_clzll(heads & (~0ull >> (63u - lane)));
  const uint64_t later = lane == 63u ? 0ull : heads >> (lane + 1u);
  const uint32_t run = later ? (uint32_t)__builtin_ctzll(later) + 1u : 64u - lane;
  uint32_t first = 0;
  if (valid && head == lane) first = atomicAdd(&count[c], run);
  first = (uint32_t)__shfl((int)first, (int)head, 64);
  if (valid) slot[i] = first + lane - head;
  // per-scan-tile particle counts (the scan's first pass), spread over
  // kTileSlots copies of the table by workgroup: counted in LDS where the
  // table fits, else one atomic per distinct tile of the wave (the particles
  // arrive in last step's sorted order, so a wave's cells mostly share a tile)
  const uint32_t t = c / kScanTile;
  uint32_t* __restrict__ ts = tsum + (size_t)(blockIdx.x % kTileSlots) * nscan;
  if (nscan <= kLdsTiles) {
    if (valid && head == lane) atomicAdd(&tiles[t], run);
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < nscan; k += blockDim.x)
      if (tiles[k]) atomicAdd(&ts[k], tiles[k]);
    return;
  }
  uint64_t todo = __ballot(valid);
  while (todo) {
    const int leader = __ffsll((unsigned long long)todo) - 1;
    const uint32_t tl = (uint32_t)__shfl((int)t, leader, 64);
    const uint64_t same = __ballot(t == tl) & todo;
    if ((int)(threadIdx.x & 63u) == leader) atomicAdd(&ts[tl], (uint32_t)__popcll(same));
    todo &= ~same;
  }
}

// exclusive scan of one value per thread over a workgroup of W waves
template <uint32_t W = 4>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* lds, uint32_t& total) {
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = (uint32_t)__shfl_up((int)x, o, 64);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 63) lds[wid] = x;
  __syncthreads();
  uint32_t woff = 0, tot = 0;
#pragma unroll
  for (uint32_t w = 0; w < W; ++w) {
    uint32_t t = lds[w];
    if (w < wid) woff += t;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return woff + x - v;
}

// per-tile sums of count
__global__ __launch_bounds__(256) void k_scan_reduce(const uint32_t* __restrict__ count,
                                                     uint64_t ncells, uint32_t* __restrict__ bsum) {
  __shared__ uint32_t lds[4];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
  uint32_t s = 0;
  if (base + kScanTile <= ncells) {
    const uint4* c4 = reinterpret_cast<const uint4*>(count + base);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint4 v = c4[threadIdx.x + 256 * j];
      s += v.x + v.y + v.z + v.w;
    }
  } else {
    for (uint64_t k = base + threadIdx.x; k < ncells; k += 256) s += count[k];
  }
  uint32_t tot;
  block_excl_scan(s, lds, tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// exclusive scan of the tile sums: dst[k] = sum of src[<k]; start[ncells] =
// total.  PARTS: src holds kTileSlots tables of nb partial sums (added here),
// dst is another array, and a workgroup takes kTilesPer tiles, adding up all
// earlier ones itself: 37 -> 10.9 us at 8,192 tiles, where one workgroup of
// 256 went through them a round trip to memory at a time.  Its reads grow with
// the square of the tiles, yet stay below that walk's time up to the largest
// table (8,000 particles: 65,536 tiles 302 -> 44 us, 262,144 1,244 -> 198,
// 1,000,000 4,813 -> 3,843 beside 3,037 for the table itself).  Otherwise one
// workgroup, and dst may be src.
constexpr uint32_t kTilesPer = 1024;
template <bool PARTS>
__global__ __launch_bounds__(kTilesPer) void k_scan_tiles(const uint32_t* src, uint32_t* dst,
                                                          uint32_t nb,
                                                          uint32_t* __restrict__ start,
                                                          uint64_t ncells) {
  constexpr uint32_t W = kTilesPer / 64;
  __shared__ uint32_t lds[W];
  auto tile = [&](uint32_t k) {
    if (!PARTS) return src[k];
    uint32_t v = 0u;
#pragma unroll
    for (int j = 0; j < kTileSlots; ++j) v += src[(size_t)j * nb + k];
    return v;
  };
  const uint32_t b1 = PARTS ? min((blockIdx.x + 1u) * kTilesPer, nb) : nb;
  uint32_t b0 = 0, carry = 0, tot;
  if (PARTS && blockIdx.x) {
    b0 = blockIdx.x * kTilesPer;
    uint32_t v = 0;
#pragma unroll 2
    for (uint32_t k = threadIdx.x; k < b0; k += kTilesPer) v += tile(k);
    block_excl_scan<W>(v, lds, carry);
  }
  for (; b0 < b1; b0 += kTilesPer) {
    const uint32_t k = b0 + threadIdx.x;
    const uint32_t ex = block_excl_scan<W>(k < nb ? tile(k) : 0u, lds, tot);
    if (k < nb) dst[k] = carry + ex;
    carry += tot;
  }
  if (b1 == nb && threadIdx.x == 0) start[ncells] = carry;
}

// start[c] = tile offset + in-tile exclusive prefix; ZERO: count[c] = 0;
// parts: the tile's kTileSlots partial sums zeroed for the next build.  Bound
// by the table's bytes: the counts of a tile without particles are not read,
// and every access of a wave is one contiguous kilobyte (33.5 million cells,
// a twentieth of their tiles occupied: 55 -> 34 us).
template <bool ZERO>
__global__ __launch_bounds__(256) void k_scan_apply(uint32_t* __restrict__ count, uint64_t ncells,
                                                    const uint32_t* __restrict__ bsum,
                                                    uint32_t* __restrict__ start,
                                                    uint32_t* __restrict__ parts) {
  constexpr int kSegs = 4;   // segments of 1,024 cells, four per thread
  __shared__ uint32_t lds[kSegs][4];
  const uint32_t nb = gridDim.x;
  const uint32_t toff = bsum[blockIdx.x];   // loaded with the counts, not after the block scan
  const uint32_t tend = blockIdx.x + 1u < nb ? bsum[blockIdx.x + 1u] : start[ncells];
  if (parts && threadIdx.x < (uint32_t)kTileSlots) parts[(size_t)threadIdx.x * nb + blockIdx.x] = 0u;
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * 4u;
  const bool full = (uint64_t)(blockIdx.x + 1) * kScanTile <= ncells;
  uint4 v[kSegs] = {};
  if (tend != toff) {   // the same for the whole workgroup
    if (full) {
#pragma unroll
      for (int j = 0; j < kSegs; ++j) v[j] = *reinterpret_cast<const uint4*>(count + base + 1024u * j);
    } else {
#pragma unroll
      for (int j = 0; j < kSegs; ++j) {
        const uint64_t c = base + 1024u * j;
        if (c < ncells) v[j].x = count[c];
        if (c + 1 < ncells) v[j].y = count[c + 1];
        if (c + 2 < ncells) v[j].z = count[c + 2];
        if (c + 3 < ncells) v[j].w = count[c + 3];
      }
    }
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    uint32_t x[kSegs];   // inclusive sums over the wave
#pragma unroll
    for (int j = 0; j < kSegs; ++j) x[j] = v[j].x + v[j].y + v[j].z + v[j].w;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
      for (int j = 0; j < kSegs; ++j) {
        const uint32_t y = (uint32_t)__shfl_up((int)x[j], o, 64);
        if (lane >= (uint32_t)o) x[j] += y;
      }
    if (lane == 63u)
#pragma unroll
      for (int j = 0; j < kSegs; ++j) lds[j][wid] = x[j];
    __syncthreads();
    uint32_t before = toff;
#pragma unroll
    for (int j = 0; j < kSegs; ++j) {
      uint32_t mine = before;
#pragma unroll
      for (uint32_t w = 0; w < 4u; ++w) {
        if (w < wid) mine += lds[j][w];
        before += lds[j][w];
      }
      const uint4 t = v[j];
      v[j].x = mine + x[j] - (t.x + t.y + t.z + t.w);
      v[j].y = v[j].x + t.x;
      v[j].z = v[j].y + t.y;
      v[j].w = v[j].z + t.z;
    }
  } else {
#pragma unroll
    for (int j = 0; j < kSegs; ++j) v[j] = make_uint4(toff, toff, toff, toff);
  }
#pragma unroll
  for (int j = 0; j < kSegs; ++j) {
    const uint64_t c = base + 1024u * j;
    if (full) {
      *reinterpret_cast<uint4*>(start + c) = v[j];
      if (ZERO && tend != toff) *reinterpret_cast<uint4*>(count + c) = make_uint4(0u, 0u, 0u, 0u);
    } else {
      const uint32_t e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (c + u < ncells) {
          start[c + u] = e[u];
          if (ZERO) count[c + u] = 0u;
        }
    }
  }
}

__global__ __launch_bounds__(256) void k_scatter(const uint32_t* __restrict__ hash,
                                                 const uint32_t* __restrict__ slot, uint32_t n,
                                                 const uint32_t* __restrict__ start,
                                                 uint32_t* __restrict__ tmp) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  tmp[start[hash[i]] + slot[i]] = i;
}

// Stable rank within the cell + gather of the particle state.
// The cell's first particle re-zeroes its count for the next build.
template <bool STATE>
__global__ __launch_bounds__(256) void k_rank_reorder(const uint32_t* __restrict__ hash, uint32_t n,
                                                      const uint32_t* __restrict__ start,
                                                      const uint32_t* __restrict__ tmp,
                                                      uint32_t* __restrict__ perm, ReorderArrays ra,
                                                      uint32_t* __restrict__ count) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t c = hash[i];
  const uint32_t s = start[c], e = start[c + 1];
  uint32_t rank = 0;
  if (e - s > 1)
    for (uint32_t q = s; q < e; ++q) rank += (tmp[q] < i) ? 1u : 0u;
  const uint32_t dst = s + rank;
  perm[dst] = i;
  if (rank == 0) count[c] = 0u;
  if (STATE) {
    ra.dx[dst] = ra.sx[i];
    ra.dv[dst] = ra.sv[i];
    ra.dvh[dst] = ra.svh[i];
    ra.did[dst] = ra.sid[i];
    ra.dp[dst] = ra.sp[i];
  }
}

// (in a wide scene every wave comes here: most find the word set)
__device__ __forceinline__ void report_wide(uint32_t* word) {
  if (!__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(word, 1u);
}

// End of a particle's search: count, density (with the epilogue fused), flags.
// (x.w written by the epilogue is not read by the search: it tests positions
// only.)
template <bool DENS, class M>
__device__ __forceinline__ void search_finish(const M& map, uint32_t p, uint32_t sc, uint32_t n,
                                              uint32_t cnt, uint32_t cap, bool wide, float S,
                                              uint32_t* __restrict__ ncount,
                                              float* __restrict__ rho, float mc,
                                              uint32_t* __restrict__ flags, const Compact16& c16,
                                              const EpiArgs& ep) {
  ncount[p] = cnt < cap ? cnt : cap;
  if (DENS) {
    if (ep.on) {
      Consts cc = ep.c;
      map.patch(cc, sc);
      density_epilogue_one(cc, ep, p, S * mc, rho);
    } else {
      rho[p] = S * mc;
    }
  }
  if (cnt > cap) atomicOr(flags, PSB_FLAG_NEIGHBOR_OVERFLOW);
  if (wide) report_wide(c16.wide + (size_t)sc * c16.wide_stride);
}

// Workgroup maximum of the neighbour counts, then one atomic per workgroup on
// a spread slot (every thread of the workgroup calls it).
template <class M>
__device__ __forceinline__ void report_max_count(const M& map, uint32_t cnt,
                                                 uint32_t* __restrict__ maxcnt, ErrSlots es) {
  if (!maxcnt && !es.base) return;
  __shared__ uint32_t red[8];
  const uint32_t m = wave_max_u(cnt);
  if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t b = 0;
    for (uint32_t w = 0; w < (blockDim.x >> 6); ++w) b = max(b, red[w]);
    if (b) {
      uint32_t* dst = es.base ? es.base + (size_t)(blockIdx.x % kErrSlots) * es.stride +
                                    (size_t)map.scene_of_block() * kMaxIterSlots + kCountEntry
                              : maxcnt;
      // most workgroups find a maximum no smaller than theirs already there
      if (b > __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(dst, b);
    }
  }
}

// searchNeighbooring (UniformGridKernel.cu:58-95) on sorted positions; the
// density sum of the same pairs rides along (SphKernel.cu:9-27).
// RT > 0: the stencil half-width is a compile-time constant; the (2RT+1)^2
// row ranges are loaded first (independent table loads) and the candidates of
// a row are gathered kRowSlots at a time before being tested in order.  RT =
// 0: any stencil width, rows visited one after the other.  With ep.on the
// density epilogue (density_epilogue_one) runs on the particle's sum.
constexpr int kRowSlots = 8;   // candidate loads in flight per stencil row

template <bool DENS, int RT, class M>
__global__ __launch_bounds__(M::kMaxThreads) void k_neighbors(M map, const float4* xs, uint32_t n,
                                                              GridDev g0,
                                                              const uint32_t* __restrict__ start0,
                                                              float r2, uint32_t cap,
                                                              uint32_t* __restrict__ ncount,
                                                              uint32_t* __restrict__ nlist,
                                                              float* __restrict__ rho, float mc,
                                                              uint32_t* __restrict__ flags,
                                                              uint32_t* __restrict__ maxcnt,
                                                              Compact16 c16, ErrSlots es,
                                                              const HaloTile* __restrict__ tiles,
                                                              EpiArgs ep) {
  uint32_t p, sc;
  bool lead;
  const bool valid = map.locate(n, p, sc, lead);
  uint32_t cnt = 0;
  if (valid) {
    uint32_t off;
    const GridDev g = map.grid(g0, sc, off);
    const uint32_t* __restrict__ start = start0 + off;
    const float4 xi = xs[p];
    uint32_t bad = 0;
    const int cx = cell_coord(xi.x, g.minx, g.cell, g.nx, bad);
    const int cy = cell_coord(xi.y, g.miny, g.cell, g.ny, bad);
    const int cz = cell_coord(xi.z, g.minz, g.cell, g.nz, bad);
    const int R = RT > 0 ? RT : g.R;
    const int x0 = max(cx - R, 0), x1 = min(cx + R, g.nx - 1);
    float S = 0.f;
    bool wide = false;
    // grouped 32-bit list of a system whose compact offsets have overflowed
    // (then in place of the compact list, which its readers no longer take)
    uint32_t* const l32g =
        (!tiles && c16.list32g && c16.want32 && *c16.want32) ? c16.list32g : nullptr;
    // staged tiles: the compact entry is the LDS slot q + sb of the row
    const HaloTile* T = tiles ? tiles + p / kHaloTile : nullptr;
    const bool hok = T && T->ok;
    int32_t sb = 0;
    auto visit = [&](uint32_t q, const float4& xj) {
      const float dx = xi.x - xj.x, dy_ = xi.y - xj.y, dz_ = xi.z - xj.z;
      const float d2 = dot3(dx, dy_, dz_, dx, dy_, dz_);
      const bool acc = d2 <= r2;
      if (DENS) {
        // a rejected candidate adds +0, which leaves S (never -0) unchanged
        const float w = acc ? r2 - d2 : 0.f;
        S = __builtin_fmaf(w * w, w, S);
      }
      if (acc && cnt < cap) {
        nlist[(uint64_t)cnt * n + p] = q;
        if (l32g) l32g[l32g_at(cnt, p, n)] = q;
        else if (c16.list16) {
          const int d = (int)(q - p);
          const bool fits = d >= -kCompactReach && d <= kCompactReach;
          const uint16_t e = hok ? (uint16_t)((int32_t)q + sb) : (uint16_t)(d + 32768);
          if (hok || fits) c16.list16[l16_at(cnt, p, n)] = e;
          wide = wide || (!hok && !fits);
        }
      }
      cnt += acc ? 1u : 0u;
    };
    // a row's candidates 8 at a time: one round of loads covers a typical
    // row (slots past the row's end load nothing and are not visited)
    auto row = [&](uint32_t q0, uint32_t q1) {
      for (uint32_t q = q0; q < q1; q += kRowSlots) {
        float4 xq[kRowSlots];
#pragma unroll
        for (int u = 0; u < kRowSlots; ++u)
          if (q + u < q1) xq[u] = xs[q + u];
#pragma unroll
        for (int u = 0; u < kRowSlots; ++u)
          if (q + u < q1) visit(q + u, xq[u]);
      }
    };
    if (RT > 0) {
      constexpr int W = 2 * RT + 1;
      uint32_t q0s[W * W], q1s[W * W];
#pragma unroll
      for (int r = 0; r < W * W; ++r) {
        const int z = cz + r / W - RT, y = cy + r % W - RT;
        const bool ok = z >= 0 && z < g.nz && y >= 0 && y < g.ny;
        const uint64_t base = ok ? (uint64_t)g.nx * ((uint64_t)y + (uint64_t)g.ny * (uint64_t)z) : 0;
        q0s[r] = ok ? start[base + x0] : 0u;
        q1s[r] = ok ? start[base + x1 + 1] : 0u;
      }
      for (int r = 0; r < W * W; ++r) {
        if (hok && q1s[r] > q0s[r]) sb = halo_slot_base(*T, cy + r % W - RT, cz + r / W - RT);
        row(q0s[r], q1s[r]);
      }
    } else {
      for (int dz = -R; dz <= R; ++dz) {
        const int z = cz + dz;
        if (z < 0 || z >= g.nz) continue;
        for (int dy = -R; dy <= R; ++dy) {
          const int y = cy + dy;
          if (y < 0 || y >= g.ny) continue;
          const uint64_t base = (uint64_t)g.nx * ((uint64_t)y + (uint64_t)g.ny * (uint64_t)z);
          if (hok) sb = halo_slot_base(*T, y, z);
          row(start[base + x0], start[base + x1 + 1]);
        }
      }
    }
    search_finish<DENS>(map, p, sc, n, cnt, cap, wide, S, ncount, rho, mc, flags, c16, ep);
  }
  report_max_count(map, cnt, maxcnt, es);
}

// The same search for few particles: a workgroup of kSplit waves serves 64
// particles, each lane a contiguous kPer of the (2 RT + 1)^2 stencil rows of
// one particle.  With a lane per particle the search is a serial chain of
// ~6,000 instructions however few the particles are; here a particle's tests
// run side by side, and what is left in sequence is the density sum over its
// neighbours' weights.
//
// Every lane keeps its accepted candidates in LDS, as 16-bit distances from the
// first candidate of its run of rows.  The rows of a run lie in one layer of
// cells, so the distance spans a few rows of particles and not the layers
// between (180 x 100 x 4 particles, whose layers are 18,000 apart: with the
// distance from the particle itself no buffer held its candidates, and the
// search with the density sum took 57 us against 29 for a lane per particle;
// now 22).  The counts of a particle's runs, in row order, place the entries in
// the list.  The waves take eight of a particle's entries each, write them
// (whole words of the compact list, rows of 64 in the plain one) and leave their
// weights in LDS, which the first wave adds in list order, 40 at a time: list
// and sum are the plain search's.  40 KB a workgroup, so that four fit a compute
// unit.
// Where a lane accepts more than its buffer holds, the particle's lanes write
// their own entries, that lane walking its rows again, and the weights are
// taken from the list written (32,768 particles with 185 neighbours 161 us when
// the first wave walked all rows by itself, now 69; a lane per particle 122).
// Bound by latency at 1,000 particles (with the density sum 9.0 us, a lane
// per particle 30), by instruction issue at 100,000 (27 us against 35).
constexpr int kSplit = 5;             // lanes per particle
constexpr uint32_t kSplitHits = 44;   // accepted candidates kept per lane
constexpr uint32_t kSplitSum = 8 * kSplit;   // weights kept per particle
// Candidate loads in flight per stencil row (an earlier form: 6 13.7 us at
// 32,768 particles, 8 14.5, 6 without those past the row's end 14.3).
constexpr int kSplitSlots = 6;
template <int RT> struct SplitShape {
  static constexpr int kWidth = 2 * RT + 1;
  static constexpr int kRows = kWidth * kWidth;
  static constexpr int kPer = (kRows + kSplit - 1) / kSplit;   // rows per lane
  // Runs of rows in one layer: one per lane, but that at RT = 1 the second
  // lane's two rows end a layer and begin the next.
  static constexpr bool kTwo = RT == 1;
  static constexpr uint32_t kRuns = kTwo ? kSplit + 1 : kSplit;
  static constexpr uint32_t lane_of(uint32_t run) { return kTwo && run >= 2u ? run - 1u : run; }
  static __device__ uint32_t run_of(uint32_t lane) { return kTwo && lane >= 2u ? lane + 1u : lane; }
};

template <bool DENS, int RT>
__global__ __launch_bounds__(64 * kSplit) void k_neighbors_split(
    const float4* xs, uint32_t n, GridDev g, const uint32_t* __restrict__ start, float r2,
    uint32_t cap, uint32_t* __restrict__ ncount, uint32_t* __restrict__ nlist,
    float* __restrict__ rho, float mc, uint32_t* __restrict__ flags, uint32_t* __restrict__ maxcnt,
    Compact16 c16, ErrSlots es, EpiArgs ep) {
  using Sh = SplitShape<RT>;
  constexpr int W = Sh::kWidth, kPer = Sh::kPer;
  constexpr uint32_t kRuns = Sh::kRuns;
  constexpr uint32_t kPitch = kSplitHits + 1;   // one more takes what does not fit
  __shared__ uint16_t rel[kSplit * kPitch * 64];
  __shared__ float weight[DENS ? kSplitSum * 64 : 1];
  // of a run: accepted candidates (6 bits) and first candidate; kOver candidates
  // where the lane's buffer does not hold them all (it then holds their number,
  // as 16-bit halves)
  __shared__ uint32_t info[kRuns][64];
  constexpr uint32_t kOver = 63u;
  static_assert(kSplitHits < kOver && kSplitHits >= 4u && (kSplit - 1) * kPitch < 256u, "packing");
  const uint32_t i = threadIdx.x & 63u;
  const uint32_t slice = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const bool two = Sh::kTwo && slice == 1u;   // this lane's last row is a run of its own
  const uint32_t p = xcd_block(blockIdx.x, gridDim.x) * 64u + i;
  const bool valid = p < n;
  uint32_t q0[kPer] = {}, q1[kPer] = {}, c = 0, c0 = 0;
  uint32_t from = 0, from2 = 0;   // first candidate of the run (of the second one)
  float4 xi = make_float4(0.f, 0.f, 0.f, 0.f);
  int cx = 0, cy = 0, cz = 0;
  bool over = false;
  auto range = [&](int r, uint32_t& lo, uint32_t& hi) {
    const int z = cz + r / W - RT, y = cy + r % W - RT;
    const bool in = r < Sh::kRows && z >= 0 && z < g.nz && y >= 0 && y < g.ny;
    const uint64_t base = in ? (uint64_t)g.nx * ((uint64_t)y + (uint64_t)g.ny * (uint64_t)z) : 0;
    lo = start[base + max(cx - RT, 0)];
    hi = start[base + min(cx + RT, g.nx - 1) + 1];
    if (!in) hi = lo;
  };
  auto weight_of = [&](const float4& xj, bool& acc) {
    const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
    const float d2 = dot3(dx, dy, dz, dx, dy, dz);
    acc = d2 <= r2;
    return r2 - d2;
  };
  // one round of kSplitSlots candidates (loads past the row's end stay inside
  // the array and are not accepted)
  auto load = [&](uint32_t q, float4 (&xq)[kSplitSlots]) {
#pragma unroll
    for (int u = 0; u < kSplitSlots; ++u) xq[u] = gather4(xs, min(q + u, n - 1u));
  };
  const uint32_t mine = slice * kPitch * 64u + i;
  if (valid) {
    xi = xs[p];
    uint32_t bad = 0;
    cx = cell_coord(xi.x, g.minx, g.cell, g.nx, bad);
    cy = cell_coord(xi.y, g.miny, g.cell, g.ny, bad);
    cz = cell_coord(xi.z, g.minz, g.cell, g.nz, bad);
#pragma unroll
    for (int r = 0; r < kPer; ++r) range((int)slice * kPer + r, q0[r], q1[r]);
    from = from2 = q0[kPer - 1];
#pragma unroll
    for (int r = kPer - 2; r >= 0; --r) from = two || q0[r] < q1[r] ? q0[r] : from;
    // candidates from q on, the row's last `left`
    auto test = [&](uint32_t q, uint32_t left, uint32_t first, const float4 (&xq)[kSplitSlots]) {
      const uint32_t d = q - first;
      over = over || d > 0xFFFFu - kSplitSlots;
#pragma unroll
      for (int u = 0; u < kSplitSlots; ++u) {
        bool acc;
        weight_of(xq[u], acc);
        rel[mine + 64u * min(c, kSplitHits)] = (uint16_t)(d + u);
        c += acc && (uint32_t)u < left ? 1u : 0u;
      }
    };
    // the next row's first round loaded before this row's tests
    float4 x0[2][kSplitSlots];
    load(q0[0], x0[0]);
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      if (r + 1 < kPer) load(q0[r + 1], x0[(r + 1) & 1]);
      if (Sh::kTwo && r == kPer - 1) c0 = c;
      if (q0[r] == q1[r]) continue;
      const uint32_t first = Sh::kTwo && r == kPer - 1 && two ? from2 : from;
      test(q0[r], q1[r] - q0[r], first, x0[r & 1]);
      for (uint32_t q = q0[r] + kSplitSlots; q < q1[r]; q += kSplitSlots) {
        float4 xq[kSplitSlots];
        load(q, xq);
        test(q, q1[r] - q, first, xq);
      }
    }
    over = over || c > kSplitHits;
    const uint32_t run = Sh::run_of(slice), m = two ? c0 : c;
    info[run][i] = from << 6 | (over ? kOver : m);
    if (two) info[run + 1u][i] = from2 << 6 | (over ? kOver : c - c0);
    if (over) {
      rel[mine] = (uint16_t)m;
      rel[mine + 64u] = (uint16_t)(m >> 16);
      if (two) {
        rel[mine + 128u] = (uint16_t)(c - c0);
        rel[mine + 192u] = (uint16_t)((c - c0) >> 16);
      }
    }
  }
  __syncthreads();
  bool wide = false, listed = true;   // listed: every buffer of the particle holds all
  // of a run: last entry + 1; first candidate (24 bits) and how much further an
  // entry lies in rel than in the list (at most 4 kPitch)
  uint32_t end[kRuns] = {}, where[kRuns] = {}, all = 0;
  if (valid) {
    uint32_t longest = 0;
#pragma unroll
    for (uint32_t s = 0; s < kRuns; ++s) {
      const uint32_t m = info[s][i], have = m & 63u;
      longest = max(longest, have);
      where[s] = (m & ~63u) << 2 |
                 (Sh::lane_of(s) * kPitch + (Sh::kTwo && s == 2u ? end[1] - end[0] : 0u) - all);
      all += have;
      end[s] = all;
    }
    listed = longest < kOver;
  }
  // entry k of the particle's list
  auto entry = [&](uint32_t k) {
    uint32_t w = where[0];
#pragma unroll
    for (uint32_t s = 1; s < kRuns; ++s) {
      const uint32_t next = where[s];   // (a choice between the two array elements goes through scratch)
      w = k >= end[s - 1] ? next : w;
    }
    return (w >> 8) + rel[(k + (w & 255u)) * 64u + i];
  };
  uint32_t* const l32g = (c16.list32g && c16.want32 && *c16.want32) ? c16.list32g : nullptr;
  // the same for every wave of the workgroup, as all that follows from info is
  if (__any(!listed)) {
    if (!listed) {
      uint32_t at = all = 0u;   // entries before this lane's, entries
#pragma unroll
      for (uint32_t s = 0; s < kRuns; ++s) {
        const uint32_t m = info[s][i] & 63u;
        const uint32_t b = (Sh::lane_of(s) * kPitch + (Sh::kTwo && s == 2u ? 2u : 0u)) * 64u + i;
        at = s == Sh::run_of(slice) ? all : at;
        all += m < kOver ? m : rel[b] | (uint32_t)rel[b + 64u] << 16;
      }
      auto put = [&](uint32_t k, uint32_t q) {
        if (k >= cap) return;
        nlist[(uint64_t)k * n + p] = q;
        if (l32g) l32g[l32g_at(k, p, n)] = q;
        else if (c16.list16) {
          const uint32_t e = q - p + 32768u;
          c16.list16[l16_at(k, p, n)] = (uint16_t)e;
          wide = wide || e - 1u >= 2u * kCompactReach + 1u;
        }
      };
      if (!over) {
        for (uint32_t k = 0; k < c; ++k)
          put(at + k, (two && k >= c0 ? from2 : from) + rel[mine + 64u * k]);
      } else {
#pragma unroll
        for (int r = 0; r < kPer; ++r)
          for (uint32_t q = q0[r]; q < q1[r]; q += kSplitSlots) {
            float4 xq[kSplitSlots];
            load(q, xq);
#pragma unroll
            for (int u = 0; u < kSplitSlots; ++u) {
              bool acc;
              weight_of(xq[u], acc);
              if (acc && q + u < q1[r]) put(at++, q + u);
            }
          }
      }
    }
    if (DENS) __syncthreads();   // the list just written is read below
  }
  const uint32_t kept = min(all, cap);
  // a list cut short holds no entry for the rest of the sum: rows again
  const bool rows = DENS && !listed && all > cap;
  float S = 0.f;
  const uint32_t todo = DENS ? (rows ? 0u : all) : (listed ? kept : 0u);
  for (uint32_t b0 = 0; DENS ? __any(b0 < todo) : b0 + 8u * slice < todo; b0 += kSplitSum) {
    const uint32_t k0 = b0 + 8u * slice;
    if (k0 < todo) {
      uint32_t q[8];
      if (!DENS || listed) {
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) q[u] = entry(min(k0 + u, all - 1u));
      } else {
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) q[u] = nlist[(uint64_t)min(k0 + u, all - 1u) * n + p];
      }
      if (DENS) {
        float4 xq[8];
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) xq[u] = gather4(xs, q[u]);
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) {
          bool acc;
          weight[(8u * slice + u) * 64u + i] = weight_of(xq[u], acc);
        }
      }
      if (listed && k0 < kept) {
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u)
          if (k0 + u < kept) nlist[(uint64_t)(k0 + u) * n + p] = q[u];
        if (l32g) {
          uint4* const dst = reinterpret_cast<uint4*>(l32g + l32g_at(k0, p, n));
          dst[0] = make_uint4(q[0], q[1], q[2], q[3]);
          dst[n] = make_uint4(q[4], q[5], q[6], q[7]);
        } else if (c16.list16) {
          uint32_t e[8], far = 0;
#pragma unroll
          for (uint32_t u = 0; u < 8u; ++u) {
            e[u] = q[u] - p + 32768u;
            far = max(far, e[u] - 1u);
          }
          // (past the list's end the last entry stands in; one cut off counts)
          wide = wide || far >= 2u * kCompactReach + 1u;
          *reinterpret_cast<uint4*>(c16.list16 + l16_at(k0, p, n)) =
              make_uint4((e[0] & 0xFFFFu) | e[1] << 16, (e[2] & 0xFFFFu) | e[3] << 16,
                         (e[4] & 0xFFFFu) | e[5] << 16, (e[6] & 0xFFFFu) | e[7] << 16);
        }
      }
    }
    if (DENS) {
      __syncthreads();
      if (slice == 0u)
        for (uint32_t k = b0; k < min(todo, b0 + kSplitSum); k += 8u) {
          float w[8];
#pragma unroll
          for (uint32_t u = 0; u < 8u; ++u) w[u] = weight[(k - b0 + u) * 64u + i];
#pragma unroll
          for (uint32_t u = 0; u < 8u; ++u)
            if (k + u < all) S = __builtin_fmaf(w[u] * w[u], w[u], S);
        }
      if (__any(b0 + kSplitSum < todo)) __syncthreads();
    }
  }
  if (wide && slice != 0u) report_wide(c16.wide);
  if (slice == 0u && rows)
    for (int r = 0; r < Sh::kRows; ++r) {
      uint32_t lo, hi;
      range(r, lo, hi);
      for (uint32_t q = lo; q < hi; q += kSplitSlots) {
        float4 xq[kSplitSlots];
        load(q, xq);
#pragma unroll
        for (int u = 0; u < kSplitSlots; ++u) {
          bool acc;
          const float w = weight_of(xq[u], acc);
          if (acc && q + u < hi) S = __builtin_fmaf(w * w, w, S);
        }
      }
    }
  if (valid && slice == 0u)
    search_finish<DENS>(SingleMap{}, p, 0u, n, all, cap, wide, S, ncount, rho, mc, flags, c16, ep);
  report_max_count(SingleMap{}, slice == 0u ? all : 0u, maxcnt, es);
}

template <int W>
__global__ __launch_bounds__(256) void k_gather(const float* __restrict__ src, float* __restrict__ dst,
                                                const uint32_t* __restrict__ perm, uint32_t n) {
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  if (W == 4) reinterpret_cast<float4*>(dst)[k] = reinterpret_cast<const float4*>(src)[perm[k]];
  else dst[k] = src[perm[k]];
}

// counting sort of the hashed particles + cell ranges + reorder
static psb_status grid_sort(psb_grid g, uint32_t n, const ReorderArrays* ra, hipStream_t s) {
  // the tile sums came with the hashes (tsum); the scan's second pass
  // leaves count alone, the reorder re-zeroes the occupied cells
  const uint32_t nb = blocks_for(n);
  hipLaunchKernelGGL(k_scan_tiles<true>, dim3(blocks_for(g->nscan, kTilesPer)), dim3(kTilesPer), 0,
                     s, g->tsum, g->bsum, g->nscan, g->start, g->ncells);
  hipLaunchKernelGGL(k_scan_apply<false>, dim3(g->nscan), dim3(kBlock), 0, s, g->count, g->ncells,
                     g->bsum, g->start, g->tsum);
  if (n) {
    hipLaunchKernelGGL(k_scatter, dim3(nb), dim3(kBlock), 0, s, g->hash, g->slot, n, g->start, g->tmp);
    if (ra) {
      hipLaunchKernelGGL(k_rank_reorder<true>, dim3(nb), dim3(kBlock), 0, s, g->hash, n, g->start,
                         g->tmp, g->perm, *ra, g->count);
    } else {
      ReorderArrays none{};
      hipLaunchKernelGGL(k_rank_reorder<false>, dim3(nb), dim3(kBlock), 0, s, g->hash, n, g->start,
                         g->tmp, g->perm, none, g->count);
    }
  }
  PSB_HIP(hipGetLastError());
  g->n = n;
  return PSB_OK;
}

// One workgroup per tile of kHaloTile sorted particles: the tile's halo rows
// (HaloTile) and, per LDS slot, the sorted index staged there.
__global__ __launch_bounds__(kHaloTile) void k_halo(const float4* __restrict__ xs, uint32_t n,
                                                    GridDev g, const uint32_t* __restrict__ start,
                                                    HaloTile* __restrict__ tiles,
                                                    uint32_t* __restrict__ src) {
  __shared__ int s_x0, s_x1, s_z0, s_z1, s_ok, s_nrows, s_total;
  __shared__ int s_ylo[kHaloMaxZ], s_yhi[kHaloMaxZ], s_rowbase[kHaloMaxZ + 1];
  __shared__ uint32_t s_gs[kHaloMaxRows], s_lb[kHaloMaxRows + 1];
  const uint32_t t = blockIdx.x;
  const uint32_t p = t * kHaloTile + threadIdx.x;
  const int R = g.R;
  if (threadIdx.x == 0) { s_x0 = 0x7FFFFFFF; s_x1 = -1; s_z0 = 0x7FFFFFFF; s_z1 = -1; }
  if (threadIdx.x < kHaloMaxZ) { s_ylo[threadIdx.x] = 0x7FFFFFFF; s_yhi[threadIdx.x] = -1; }
  if (threadIdx.x < kHaloMaxZ + 1) s_rowbase[threadIdx.x] = 0;
  __syncthreads();
  int cx = 0, cy = 0, cz = 0;
  const bool v = p < n;
  if (v) {
    uint32_t bad = 0;
    const float4 x = xs[p];
    cx = cell_coord(x.x, g.minx, g.cell, g.nx, bad);
    cy = cell_coord(x.y, g.miny, g.cell, g.ny, bad);
    cz = cell_coord(x.z, g.minz, g.cell, g.nz, bad);
    atomicMin(&s_x0, cx); atomicMax(&s_x1, cx);
    atomicMin(&s_z0, cz); atomicMax(&s_z1, cz);
  }
  __syncthreads();
  const int zlo = max(s_z0 - R, 0), zhi = min(s_z1 + R, g.nz - 1);
  const bool zok = s_z1 >= 0 && zhi - zlo + 1 <= kHaloMaxZ;
  if (v && zok)
    for (int z = max(cz - R, zlo); z <= min(cz + R, zhi); ++z) {
      atomicMin(&s_ylo[z - zlo], max(cy - R, 0));
      atomicMax(&s_yhi[z - zlo], min(cy + R, g.ny - 1));
    }
  __syncthreads();
  if (threadIdx.x == 0) {
    int ok = zok ? 1 : 0, rows = 0;
    const int nzr = zok ? zhi - zlo + 1 : 0;
    for (int i = 0; i < nzr; ++i) {
      s_rowbase[i] = rows;
      if (s_yhi[i] >= s_ylo[i]) rows += s_yhi[i] - s_ylo[i] + 1;
      else s_ylo[i] = 0;   // no row in this layer
    }
    s_rowbase[nzr] = rows;
    if (rows > kHaloMaxRows) ok = 0;
    s_ok = ok;
    s_nrows = ok ? rows : 0;
  }
  __syncthreads();
  const int x0 = max(s_x0 - R, 0), x1 = min(s_x1 + R, g.nx - 1);
  const int nrows = s_nrows;
  for (int r = threadIdx.x; r < nrows; r += blockDim.x) {
    int i = 0;
    while (s_rowbase[i + 1] <= r) ++i;
    const int y = s_ylo[i] + (r - s_rowbase[i]), z = zlo + i;
    const uint64_t base = (uint64_t)g.nx * ((uint64_t)y + (uint64_t)g.ny * (uint64_t)z);
    const uint32_t gs = start[base + x0];
    s_gs[r] = gs;
    s_lb[r] = start[base + x1 + 1] - gs;   // count, scanned below
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
    for (int r = 0; r < nrows; ++r) { const uint32_t c = s_lb[r]; s_lb[r] = tot; tot += c; }
    s_lb[nrows] = tot;
    if (tot > (uint32_t)kHaloCap) s_ok = 0;
    s_total = (int)tot;
  }
  __syncthreads();
  HaloTile& T = tiles[t];
  const int ok = s_ok;
  if (threadIdx.x == 0) {
    T.ok = ok; T.nrows = nrows; T.total = ok ? s_total : 0;
    T.xlo = x0; T.xhi = x1; T.zlo = zlo; T.nz = zok ? zhi - zlo + 1 : 0; T.pad = 0;
  }
  if (threadIdx.x < kHaloMaxZ) T.ylo[threadIdx.x] = s_ylo[threadIdx.x];
  if (threadIdx.x < kHaloMaxZ + 1) T.rowbase[threadIdx.x] = s_rowbase[threadIdx.x];
  for (int r = threadIdx.x; r < nrows; r += blockDim.x) T.gstart[r] = s_gs[r];
  for (int r = threadIdx.x; r <= nrows; r += blockDim.x) T.lbase[r] = s_lb[r];
  if (!ok) return;
  uint32_t* sr = src + (size_t)t * kHaloCap;
  for (int r = 0; r < nrows; ++r) {
    const uint32_t lb = s_lb[r], c = s_lb[r + 1] - lb, gs = s_gs[r];
    for (uint32_t k = threadIdx.x; k < c; k += blockDim.x) sr[lb + k] = gs + k;
  }
}

psb_status launch_halo(psb_grid g, const float4* xs, uint32_t n, int R, HaloTile* tiles,
                       uint32_t* src, hipStream_t s) {
  if (!n) return PSB_OK;
  GridDev gd = grid_dev(g->desc, g->desc.cell_size);
  gd.R = R;
  const uint32_t nt = (n + kHaloTile - 1) / kHaloTile;
  hipLaunchKernelGGL(k_halo, dim3(nt), dim3(kHaloTile), 0, s, xs, n, gd, g->start, tiles, src);
  PSB_HIP(hipGetLastError());
  return PSB_OK;
}

// start[0..n] = exclusive prefix sums of count[0..n) (start[n] = total);
// count is zeroed; bsum holds one entry per kScanTile counts
psb_status scan_exclusive(uint32_t* count, uint64_t n, uint32_t* bsum, uint32_t* start,
                          hipStream_t s) {
  const uint32_t nt = (uint32_t)((n + kScanTile - 1) / kScanTile);
  if (nt) hipLaunchKernelGGL(k_scan_reduce, dim3(nt), dim3(kBlock), 0, s, count, n, bsum);
  hipLaunchKernelGGL(k_scan_tiles<false>, dim3(1), dim3(kTilesPer), 0, s, bsum, bsum, nt, start, n);
  if (nt) hipLaunchKernelGGL(k_scan_apply<true>, dim3(nt), dim3(kBlock), 0, s, count, n, bsum, start,
                             (uint32_t*)nullptr);
  PSB_HIP(hipGetLastError());
  return PSB_OK;
}

psb_status grid_build(psb_grid g, const float4* pos, uint32_t n, const ReorderArrays* ra,
                      hipStream_t s, const StepReset* reset) {
  GridDev gd = grid_dev(g->desc, g->desc.cell_size);
  StepReset rs{};
  if (reset) {
    if (n && blocks_for(n) >= reset->scenes) rs = *reset;   // rides on the hashing pass
    else PSB_TRY(launch_pci_reset(reset->st, false, s, reset->scenes, reset->done, reset->es));
  }
  if (n) {
    hipLaunchKernelGGL(k_hash_count<SingleMap>, dim3(blocks_for(n)), dim3(kBlock), 0, s,
                       SingleMap{}, pos, n, gd, g->hash, g->slot, g->count, g->flags, g->tsum,
                       g->nscan, rs);
  }
  return grid_sort(g, n, ra, s);
}

psb_status grid_build_batch(psb_grid g, const BatchMap& map, uint32_t nblocks, uint32_t bsize,
                            const float4* pos, uint32_t n, const ReorderArrays* ra,
                            hipStream_t s, const StepReset* reset) {
  StepReset rs{};
  if (reset) {
    if (n && nblocks >= reset->scenes) rs = *reset;   // rides on the hashing pass
    else PSB_TRY(launch_pci_reset(reset->st, false, s, reset->scenes, reset->done, reset->es));
  }
  if (n) {
    GridDev none{};
    hipLaunchKernelGGL(k_hash_count<BatchMap>, dim3(nblocks), dim3(bsize), 0, s, map, pos, n,
                       none, g->hash, g->slot, g->count, g->flags, g->tsum, g->nscan, rs);
  }
  return grid_sort(g, n, ra, s);
}

psb_status launch_neighbors_batch(psb_grid g, const BatchMap& map, uint32_t nblocks,
                                  uint32_t bsize, const float4* xs, uint32_t n, float r2, int R,
                                  psb_neighbors nb, float* rho, float mc, uint32_t* flags,
                                  uint32_t* maxcnt, hipStream_t s, const Compact16& c16,
                                  ErrSlots es, const EpiArgs* ep) {
  if (!n) return PSB_OK;
  GridDev none{};
  dim3 gb(nblocks), tb(bsize);
  EpiArgs e{};
  if (ep && rho) e = *ep;
#define PSB_NB(D_, R_)                                                                       \
  hipLaunchKernelGGL((k_neighbors<D_, R_, BatchMap>), gb, tb, 0, s, map, xs, n, none, g->start, \
                     r2, nb.capacity, nb.count, nb.list, rho, mc, flags, maxcnt, c16, es, \
                     nullptr, e)
  if (rho) {
    if (R == 1) PSB_NB(true, 1); else if (R == 2) PSB_NB(true, 2); else PSB_NB(true, 0);
  } else {
    if (R == 1) PSB_NB(false, 1); else if (R == 2) PSB_NB(false, 2); else PSB_NB(false, 0);
  }
#undef PSB_NB
  PSB_HIP(hipGetLastError());
  return PSB_OK;
}

psb_status launch_neighbors(psb_grid g, const float4* xs, uint32_t n, float r2, int R,
                            psb_neighbors nb, float* rho, float mc, uint32_t* flags,
                            uint32_t* maxcnt, hipStream_t s, const Compact16& c16,
                            ErrSlots es, const HaloTile* tiles, const EpiArgs* ep) {
  if (!n) return PSB_OK;
  GridDev gd = grid_dev(g->desc, g->desc.cell_size);
  gd.R = R;
  dim3 gb(blocks_for(n)), tb(kBlock);
  EpiArgs e{};
  if (ep && rho) e = *ep;
  // Several lanes per particle, for the stencils that have that kernel, while
  // one leaves the chip short of waves.  Us, one lane -> kSplit, cells of half
  // the radius (cells of the radius); blocks and sheets as loaded (a lattice),
  // and after some hundred steps, when the lanes of a wave have rows of
  // different lengths:
  //   with the density sum     block           4 layers        2 layers
  //      4,096 loaded        27 -> 9 (34, 10)
  //     64,000 loaded        29 -> 19 (37, 24)  26 -> 20 (28, 21)  19 -> 19 (19, 20)
  //     64,000 moved         50 -> 27 (60, 28)  45 -> 24 (53, 25)  29 -> 18 (28, 18)
  //    125,000 loaded        33 -> 34 (42, 39)  28 -> 34 (33, 38)  22 -> 30 (23, 34)
  //    125,000 moved         56 -> 45 (67, 45)  50 -> 39 (58, 41)  30 -> 28 (31, 29)
  //    146,000 moved         64 -> 51 (77, 50)  52 -> 40 (66, 45)  32 -> 31 (32, 31)
  //   without
  //    148,000 loaded        35 -> 22 (46, 30)  29 -> 21 (36, 23)  24 -> 19 (25, 19)
  //    262,144 loaded        41 -> 34 (57, 42)  36 -> 32 (46, 37)  29 -> 29 (32, 30)
  //    512,000 loaded        72 -> 68 (99, 85)  63 -> 65 (76, 76)  48 -> 59 (47, 65)
  // With the sum the line lies at 147,456, and at 65,536 where the lists are long
  // enough for neighbour counts that do not fit the lanes' buffers: 145
  // neighbours 123 -> 67 at 47,000, 148 -> 151 at 97,000; 268 (cells of half the
  // radius; of the radius) 142 -> 63 (234, 92) at 8,000, 241 -> 231 (331, 273) at
  // 47,000, 259 -> 323 (356, 412) at 64,000.  Without it at 262,144 (268: 477 ->
  // 452).  Staged tiles keep the plain search, and so do particles whose index
  // takes more than 24 bits.
  const uint64_t per_cu = !rho ? 1024u : nb.capacity <= 192u ? 576u : 256u;
  if (!tiles && (R == 1 || R == 2) && n < 1u << 24 && n <= per_cu * (uint64_t)g->ctx->cus) {
#define PSB_NBS(D_, R_)                                                                           \
  hipLaunchKernelGGL((k_neighbors_split<D_, R_>), dim3(blocks_for(n, 64u)),                       \
                     dim3(64 * kSplit), 0, s, xs, n, gd, g->start, r2, nb.capacity, \
                     nb.count, nb.list, rho, mc, flags, maxcnt, c16, es, e)
    if (rho) { if (R == 1) PSB_NBS(true, 1); else PSB_NBS(true, 2); }
    else { if (R == 1) PSB_NBS(false, 1); else PSB_NBS(false, 2); }
#undef PSB_NBS
    PSB_HIP(hipGetLastError());
    return PSB_OK;
  }
#define PSB_NB(D_, R_)                                                                       \
  hipLaunchKernelGGL((k_neighbors<D_, R_, SingleMap>), gb, tb, 0, s, SingleMap{}, xs, n, gd,    \
                     g->start, r2, nb.capacity, nb.count, nb.list, rho, mc, flags, maxcnt, c16, es, \
                     tiles, e)
  if (rho) {
    if (R == 1) PSB_NB(true, 1); else if (R == 2) PSB_NB(true, 2); else PSB_NB(true, 0);
  } else {
    if (R == 1) PSB_NB(false, 1); else if (R == 2) PSB_NB(false, 2); else PSB_NB(false, 0);
  }
#undef PSB_NB
  PSB_HIP(hipGetLastError());
  return PSB_OK;
}

static psb_status grid_alloc(psb_grid g) {
  g->ncells = (uint64_t)g->desc.dims[0] * g->desc.dims[1] * g->desc.dims[2];
  g->nscan = (uint32_t)((g->ncells + kScanTile - 1) / kScanTile);
  const size_t cap = g->capacity ? g->capacity : 1;
  PSB_HIP(hipMalloc(&g->count, 4 * (g->nscan * (size_t)kScanTile)));
  PSB_HIP(hipMalloc(&g->start, 4 * (g->ncells + 1)));
  PSB_HIP(hipMalloc(&g->hash, 4 * cap));
  PSB_HIP(hipMalloc(&g->slot, 4 * cap));
  PSB_HIP(hipMalloc(&g->tmp, 4 * cap));
  PSB_HIP(hipMalloc(&g->perm, 4 * cap));
  PSB_HIP(hipMalloc(&g->bsum, 4 * (size_t)g->nscan));
  PSB_HIP(hipMalloc(&g->tsum, 4 * (size_t)kTileSlots * g->nscan));
  PSB_HIP(hipMemsetAsync(g->tsum, 0, 4 * (size_t)kTileSlots * g->nscan, g->ctx->stream));
  PSB_HIP(hipMalloc(&g->flags, 64));
  PSB_HIP(hipMemsetAsync(g->count, 0, 4 * (g->nscan * (size_t)kScanTile), g->ctx->stream));
  PSB_HIP(hipMemsetAsync(g->flags, 0, 64, g->ctx->stream));
  PSB_HIP(hipStreamSynchronize(g->ctx->stream));
  return PSB_OK;
}

psb_status grid_create(psb_context ctx, const psb_grid_desc& d, uint32_t capacity, psb_grid* out) {
  PSB_ARG(ctx && out, "null argument");
  PSB_ARG(d.cell_size > 0.f && d.dims[0] > 0 && d.dims[1] > 0 && d.dims[2] > 0, "bad grid");
  PSB_ARG((uint64_t)d.dims[0] * d.dims[1] * d.dims[2] < (1ull << 32) - 1, "grid too large");
  PSB_HIP(hipSetDevice(ctx->device));
  psb_grid g = new psb_grid_s();
  g->ctx = ctx;
  g->desc = d;
  g->capacity = capacity;
  psb_status st = grid_alloc(g);
  if (st != PSB_OK) { psb_finalize_grid(g); return st; }
  *out = g;
  return PSB_OK;
}

}  // namespace psb

using namespace psb;

extern "C" {

psb_status psb_create_grid(psb_context ctx, double xc, double yc, double zc, double length,
                           double width, double depth, float cell_size, uint32_t capacity,
                           psb_grid* out) {
  PSB_ARG(cell_size > 0.f && length > 0 && width > 0 && depth > 0, "bad grid extent");
  psb_grid_desc d{};
  // createGrid (UniformGrid.cu:19-29): Min = C - extent/2 (stored as float),
  // nbCells = ceil(extent / sizeCell)
  d.min[0] = (float)(xc - length / 2);
  d.min[1] = (float)(yc - width / 2);
  d.min[2] = (float)(zc - depth / 2);
  d.cell_size = cell_size;
  d.dims[0] = (int32_t)std::ceil(length / cell_size);
  d.dims[1] = (int32_t)std::ceil(width / cell_size);
  d.dims[2] = (int32_t)std::ceil(depth / cell_size);
  return grid_create(ctx, d, capacity, out);
}

psb_status psb_create_grid_desc(psb_context ctx, const psb_grid_desc* desc, uint32_t capacity,
                                psb_grid* out) {
  PSB_ARG(desc, "null desc");
  return grid_create(ctx, *desc, capacity, out);
}

psb_status psb_finalize_grid(psb_grid g) {
  if (!g) return PSB_OK;
  if (g->ctx) { hipSetDevice(g->ctx->device); hipStreamSynchronize(g->ctx->stream); }
  hipFree(g->count); hipFree(g->start); hipFree(g->hash); hipFree(g->slot);
  hipFree(g->tmp); hipFree(g->perm); hipFree(g->bsum); hipFree(g->tsum); hipFree(g->flags);
  delete g;
  return PSB_OK;
}

psb_status psb_grid_get_desc(psb_grid g, psb_grid_desc* out) {
  PSB_ARG(g && out, "null argument");
  *out = g->desc;
  return PSB_OK;
}

psb_status psb_store_particles(psb_grid g, const float* pos4, uint32_t n) {
  PSB_ARG(g && (pos4 || !n), "null argument");
  if (n > g->capacity) { set_error("n exceeds grid capacity"); return PSB_ERR_CAPACITY; }
  PSB_HIP(hipSetDevice(g->ctx->device));
  PSB_HIP(hipMemsetAsync(g->flags, 0, 4, g->ctx->stream));
  return grid_build(g, reinterpret_cast<const float4*>(pos4), n, nullptr, g->ctx->stream);
}

psb_status psb_grid_get_arrays(psb_grid g, const uint32_t** hash, const uint32_t** perm,
                               const uint32_t** cell_start, uint64_t* ncells) {
  PSB_ARG(g, "null grid");
  if (hash) *hash = g->hash;
  if (perm) *perm = g->perm;
  if (cell_start) *cell_start = g->start;
  if (ncells) *ncells = g->ncells;
  return PSB_OK;
}

psb_status psb_grid_reorder(psb_grid g, const float* src, float* dst, uint32_t n,
                            int32_t elem_floats) {
  PSB_ARG(g && src && dst, "null argument");
  PSB_ARG(elem_floats == 1 || elem_floats == 4, "elem_floats must be 1 or 4");
  PSB_ARG(n == g->n, "n differs from the last psb_store_particles");
  if (!n) return PSB_OK;
  if (elem_floats == 4)
    hipLaunchKernelGGL(k_gather<4>, dim3(blocks_for(n)), dim3(kBlock), 0, g->ctx->stream, src, dst,
                       g->perm, n);
  else
    hipLaunchKernelGGL(k_gather<1>, dim3(blocks_for(n)), dim3(kBlock), 0, g->ctx->stream, src, dst,
                       g->perm, n);
  PSB_HIP(hipGetLastError());
  return PSB_OK;
}

psb_status psb_search_neighbors(psb_grid g, const float* sorted_pos4, uint32_t n, float radius,
                                psb_neighbors nb, uint32_t* flags_out) {
  PSB_ARG(g && (sorted_pos4 || !n), "null argument");
  PSB_ARG(nb.count && nb.list && nb.capacity > 0, "bad neighbour buffers");
  PSB_ARG(nb.n == n, "neighbors.n must equal n (ELL stride)");
  PSB_ARG(n == g->n, "n differs from the last psb_store_particles");
  PSB_ARG(radius > 0.f, "radius must be > 0");
  psb_context ctx = g->ctx;
  PSB_HIP(hipSetDevice(ctx->device));
  PSB_HIP(hipMemsetAsync(ctx->d_flags, 0, 8, ctx->stream));
  GridDev gd = grid_dev(g->desc, radius);
  PSB_TRY(launch_neighbors(g, reinterpret_cast<const float4*>(sorted_pos4), n, radius * radius,
                           gd.R, nb, nullptr, 0.f, ctx->d_flags, nullptr, ctx->stream));
  PSB_TRY(launch_words_out(ctx->d_flags, 2, g->flags, 1, nullptr, 0, ctx->d_pinned, ctx->stream));
  PSB_HIP(hipStreamSynchronize(ctx->stream));
  if (flags_out) *flags_out = ctx->h_pinned[0] | ctx->h_pinned[2];
  return PSB_OK;
}

}  // extern "C"
