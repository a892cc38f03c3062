// ob_tiled3d.hip -- tile-sorted 3D charge deposition (Grid3D::binValue, Grid3D.cc:307-432)
// and potential gather for the kick (SpaceChargeCalc3D.cc:120-147).
//
// Scattering 27 FP64 atomics per particle in random particle order over a 64 MiB grid
// misses L2 on almost every update, and gathering 27 potential values per particle in
// particle order touches a different cache line per lane.  Instead, each SC step:
//   1. tile_hist    key = T x T x Tz box of the particle's TSC centre node; per-block LDS
//                   histogram, merged into global tile counts;
//   2. tile_scan    exclusive scan of the counts; work items of at most kChunk particles
//                   per tile;
//   3. tile_scatter counting-sort scatter of the bunch (6 coordinates, macrosize and the
//                   user index) into the spare buffers, ranges reserved per block;
//   4. tile_deposit one workgroup per work item accumulates its particles into an LDS
//                   block of the box plus a one-node halo, then adds the block to rho with
//                   atomics;
//   5. the kick     after the Poisson solve, workgroups copy the same block of phi into LDS
//                   and compute their particles' kicks from it.  It waits on the bunch and
//                   runs in the launch of the maps that follow it (tile_push in ob_push.hip).
// The blocks are small (~14 KiB for 8 x 8 x 16 boxes), so many workgroups share a CU.
// Weights, indices and the kick arithmetic are the reference's (same device helpers as
// the unsorted path); only the FP64 summation order of rho differs.
#include "ob_internal.hpp"
#include "ob_sc_device.hpp"
#include "ob_tiled3d.hpp"
#include "ob_tiled3d_device.hpp"

namespace ob {
namespace {

constexpr int kThreads = kTileThreads;
constexpr int kChunk = 1024;

// Particles of a work item at most.  A step of few particles has too few items of 1024 for 256
// CUs: at 50k particles on 32 x 32 x 32 nodes items of 256 take the deposit from 15.4 to 12.0
// us, the kick from 13.0 to 8.4 and a step from 72 to 63 (items of 512: 65); at 100k on 64 x 64
// x 64 nodes the step takes 85 with 256 or 512 and 90 with 1024, at 200k 104, 93 and 97, at
// 300k 124, 106 and 103 (a tile's copies then cost more than the CUs give).
int64_t tile_chunk(int64_t n) { return n <= 1 << 16 ? 256 : n <= 1 << 18 ? 512 : kChunk; }

constexpr int kMaxTiles = 16383;  // (ntiles + 1) 32-bit counters in 64 KiB of LDS (the scan: 2x)

__device__ __forceinline__ bool inside(const TileGeom& g, double x, double y, double z) {
  return !(x < g.xMin || x > g.xMax || y < g.yMin || y > g.yMax || z < g.zMin || z > g.zMax);
}

__device__ __forceinline__ uint32_t tile_key(const TileGeom& g, double x, double y, double z) {
  if (!inside(g, x, y, z)) return (uint32_t)g.ntiles;
  int iX, iY, iZ;
  double xF, yF, zF;
  node_ind_frac(x, g.xMin, g.dx, g.nx, iX, xF);
  node_ind_frac(y, g.yMin, g.dy, g.ny, iY, yF);
  grid3d_z_ind_frac(z, g.zMin, g.dz, g.nz, iZ, zF);
  return (uint32_t)(((iX / g.T) * g.ty + (iY / g.T)) * g.tz + iZ / g.Tz);
}

// Workgroups past hist_blocks clear rho, which the deposit needs, beside the histogram.  That
// saves the launch and its gap, not the stores: 4M particles on 256 x 256 x 128 nodes take 34.5
// us so, 25.0 without the clearing, whose own launch took 10.8; on 64 x 64 x 64 that one took
// 3.3 us.
__global__ __launch_bounds__(1024) void tile_hist(const double* __restrict__ cur, int64_t cap,
                                                      int64_t n, TileGeom g,
                                                      uint32_t* __restrict__ key,
                                                      uint32_t* __restrict__ counts,
                                                      uint32_t* __restrict__ cursor,
                                                      int hist_blocks,
                                                      double* __restrict__ rho) {
  extern __shared__ uint32_t lh[];
  if ((int)blockIdx.x >= hist_blocks) {
    const int64_t ng = (int64_t)g.nx * g.ny * g.nz;
    const int64_t step = (int64_t)(gridDim.x - hist_blocks) * 1024;
    for (int64_t c = (int64_t)(blockIdx.x - hist_blocks) * 1024 + threadIdx.x; c < ng; c += step)
      rho[c] = 0.0;
    return;
  }
  const int nb = g.ntiles + 1;
  if (cursor && blockIdx.x == 0)  // (scan in the scatter: its positions start at 0)
    for (int t = threadIdx.x; t < nb; t += blockDim.x) cursor[t] = 0;
  for (int t = threadIdx.x; t < nb; t += blockDim.x) lh[t] = 0;
  __syncthreads();
  const int64_t stride = (int64_t)hist_blocks * blockDim.x;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  // four particles per round: their 12 loads are in flight together
  constexpr int U = 4;
  for (; i + (U - 1) * stride < n; i += U * stride) {
    double x[U], y[U], z[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t j = i + u * stride;
      x[u] = cur[j];
      y[u] = cur[2 * cap + j];
      z[u] = cur[4 * cap + j];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t k = tile_key(g, x[u], y[u], z[u]);
      key[i + u * stride] = k;
      atomicAdd(&lh[k], 1u);
    }
  }
  for (; i < n; i += stride) {
    const uint32_t k = tile_key(g, cur[i], cur[2 * cap + i], cur[4 * cap + i]);
    key[i] = k;
    atomicAdd(&lh[k], 1u);
  }
  __syncthreads();
  for (int t = threadIdx.x; t < nb; t += blockDim.x)
    if (lh[t]) atomicAdd(&counts[t], lh[t]);
}

// One block.  counts[0..ntiles] (the last = particles outside the grid) -> offsets
// (exclusive) and cursor = offsets; work items of at most kChunk particles per tile, in tile
// order; counts are cleared for the next step.  The counts are staged through LDS: thread i
// loads tiles i, i + 1024, ... (coalesced, all its loads in flight together), the scan runs
// over contiguous ranges read back from LDS, and the stores go out tile-strided again, so
// neighbouring lanes write neighbouring offsets and items.  LDS: 2 * (ntiles + 2) counters.
__global__ __launch_bounds__(1024) void tile_scan(uint32_t* __restrict__ counts, int ntiles,
                                                  uint32_t* __restrict__ offsets,
                                                  uint32_t* __restrict__ cursor,
                                                  int4* __restrict__ items,
                                                  uint32_t* __restrict__ nitems,
                                                  uint32_t chunk) {
  extern __shared__ uint32_t ls[];
  const int nb = ntiles + 1;
  uint32_t* loff = ls;            // [nb + 1]: counts, then exclusive particle offsets
  uint32_t* litem = ls + nb + 1;  // [nb + 1]: exclusive item offsets
  constexpr int kPer = (kMaxTiles + 1) / 1024;
  uint32_t cv[kPer];
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int t = (int)threadIdx.x + u * 1024;
    cv[u] = counts[t < nb ? t : 0];
  }
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int t = (int)threadIdx.x + u * 1024;
    if (t < nb) loff[t] = cv[u];
  }
  __syncthreads();
  const int per = (nb + blockDim.x - 1) / blockDim.x;
  const int lo = min(nb, (int)threadIdx.x * per), hi = min(nb, lo + per);
  uint32_t off = 0, item = 0;
  for (int t = lo; t < hi; t++) {
    const uint32_t k = loff[t];
    off += k;
    if (t < ntiles) item += (k + chunk - 1) / chunk;
  }
  uint32_t total, total_items;
  block_scan2(off, item, total, total_items);
  // each thread rewrites only the entries it alone has read
  for (int t = lo; t < hi; t++) {
    const uint32_t k = loff[t];
    loff[t] = off;
    litem[t] = item;
    off += k;
    if (t < ntiles) item += (k + chunk - 1) / chunk;
  }
  if (threadIdx.x == 0) {
    loff[nb] = total;
    *nitems = total_items;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    const int t = (int)threadIdx.x + u * 1024;
    if (t >= nb) break;
    const uint32_t o = loff[t], e = loff[t + 1];
    offsets[t] = o;
    cursor[t] = o;
    counts[t] = 0;
    if (t < ntiles) {
      uint32_t j = litem[t];
      for (uint32_t b0 = o; b0 < e; b0 += chunk)
        items[j++] = make_int4(t, (int)b0, (int)min(e, b0 + chunk), 0);
    }
  }
}

// SCAN: few tiles (kScanTiles): every workgroup scans the counts itself and workgroup 0 writes
// the offsets and work items; cursor then counts from 0 in each tile and the deposit clears
// the counts.  Otherwise tile_scan has written offsets and cursor = offsets.  At 840 tiles
// (96 x 80 x 100 nodes, 700k particles) the scatter goes from 21.3 to 23.4 us and the scan's
// 5.0 us and the gap before it go; at 8192 tiles it would go from 153 to 267 us against the
// scan's 26, its LDS too large for the workgroups a CU needs.
constexpr int kScanTiles = 1024;
struct ScatterScan {
  const uint32_t* counts;
  uint32_t* offsets;
  int4* items;
  uint32_t* nitems;
  uint32_t chunk;
};
template <bool SCAN>
__global__ __launch_bounds__(kThreads) void tile_scatter(
    const double* __restrict__ cur, double* __restrict__ alt, int64_t cap, int64_t n,
    const uint32_t* __restrict__ key, int ntiles, uint32_t* __restrict__ cursor,
    const int32_t* __restrict__ perm, int32_t* __restrict__ perm_alt,
    const double* __restrict__ msize, double* __restrict__ msize_alt, int64_t per_block,
    ScatterScan sc) {
  extern __shared__ uint32_t sh[];
  const uint32_t chunk = sc.chunk;
  uint32_t* lc = sh;               // local counts, then running destinations
  const int nb = ntiles + 1;
  uint32_t* loff = sh + nb;        // SCAN: tile offsets
  for (int t = threadIdx.x; t < nb; t += blockDim.x) lc[t] = 0;
  if constexpr (SCAN) {
    const int per = (nb + kThreads - 1) / kThreads;
    const int a = min(nb, (int)threadIdx.x * per), e = min(nb, a + per);
    uint32_t off = 0, item = 0;
    for (int t = a; t < e; t++) {
      const uint32_t k = sc.counts[t];
      loff[t] = k;
      off += k;
      if (t < ntiles) item += (k + chunk - 1) / chunk;
    }
    uint32_t total, total_items;
    block_scan2(off, item, total, total_items);
    const bool writer = blockIdx.x == 0;
    for (int t = a; t < e; t++) {  // each thread rewrites only the entries it alone has read
      const uint32_t k = loff[t];
      loff[t] = off;
      if (writer) {
        sc.offsets[t] = off;
        if (t < ntiles)
          for (uint32_t b0 = 0; b0 < k; b0 += chunk)
            sc.items[item++] =
                make_int4(t, (int)(off + b0), (int)(off + min(k, b0 + chunk)), 0);
      }
      off += k;
    }
    if (writer && threadIdx.x == 0) *sc.nitems = total_items;
  }
  __syncthreads();
  const int64_t lo = (int64_t)blockIdx.x * per_block;
  const int64_t hi = min(n, lo + per_block);
  for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) atomicAdd(&lc[key[i]], 1u);
  __syncthreads();
  for (int t = threadIdx.x; t < nb; t += blockDim.x) {
    const uint32_t c = lc[t];
    lc[t] = c ? (SCAN ? loff[t] : 0u) + atomicAdd(&cursor[t], c) : 0u;
  }
  __syncthreads();
  // U particles per thread and round: all their loads are issued before any store
  constexpr int U = 4;
  for (int64_t i0 = lo + threadIdx.x; i0 < hi; i0 += U * (int64_t)blockDim.x) {
    double v[U][6], m[U];
    uint32_t kk[U];
    int32_t pp[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t i = i0 + u * (int64_t)blockDim.x;
      const int64_t j = i < hi ? i : lo;  // a masked lane reloads the first particle
      kk[u] = key[j];
#pragma unroll
      for (int k = 0; k < 6; k++) v[u][k] = cur[k * cap + j];
      pp[u] = perm[j];
      m[u] = msize ? msize[j] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t i = i0 + u * (int64_t)blockDim.x;
      if (i >= hi) break;
      const int64_t d = atomicAdd(&lc[kk[u]], 1u);
#pragma unroll
      for (int k = 0; k < 6; k++) alt[k * cap + d] = v[u][k];
      perm_alt[d] = pp[u];
      if (msize) msize_alt[d] = m[u];
    }
  }
}

// Grid3D::binValue for one particle into a z-fastest window (global rho or an LDS block).
__device__ __forceinline__ void deposit_particle(double* __restrict__ base, int64_t sx,
                                                 int64_t sy, int nz, int zoff, double m, double xF,
                                                 double yF, int iZ, double zF) {
  const double wx[3] = {0.5 * (0.5 - xF) * (0.5 - xF), 0.75 - xF * xF, 0.5 * (0.5 + xF) * (0.5 + xF)};
  const double wy[3] = {0.5 * (0.5 - yF) * (0.5 - yF), 0.75 - yF * yF, 0.5 * (0.5 + yF) * (0.5 + yF)};
  // base: node (iX-1, iY-1, 0) of the window; zoff: window z origin
  if (nz >= 3) {
    int iZm = iZ - 1, iZp = iZ + 1;
    if (iZm < 0) iZm = nz - 1;
    if (iZp >= nz) iZp = 0;
    const double wz[3] = {0.5 * (0.5 - zF) * (0.5 - zF), 0.75 - zF * zF,
                          0.5 * (0.5 + zF) * (0.5 + zF)};
    const int zz[3] = {iZm - zoff, iZ - zoff, iZp - zoff};
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        const double tmp = wy[c] * wz[a] * m;
#pragma unroll
        for (int d = 0; d < 3; d++) atomicAdd(base + d * sx + c * sy + zz[a], wx[d] * tmp);
      }
  } else if (nz == 2) {
    const double wz[2] = {1.0 - zF, zF};
    for (int a = 0; a < 2; a++)
      for (int c = 0; c < 3; c++) {
        const double tmp = wy[c] * wz[a] * m;
        for (int d = 0; d < 3; d++) atomicAdd(base + d * sx + c * sy + (a - zoff), wx[d] * tmp);
      }
  } else {
    for (int c = 0; c < 3; c++) {
      const double tmp = wy[c] * m;
      for (int d = 0; d < 3; d++) atomicAdd(base + d * sx + c * sy - zoff, wx[d] * tmp);
    }
  }
}

// LDS bank scheduling of the deposit: the 27 LDS atomics of a particle are at fixed word
// offsets from its first node's word, so lanes whose first words differ modulo kBankWords
// (8-byte words) hit distinct banks in all 27.  Half a work item at a time, the particles
// are ranked within their residue class, staged in LDS grouped by class, and deposited in
// rounds where lane l of each 32-lane group takes the next particle of class l (an idle
// lane when the class is used up).  In particle order, 64 lanes fall on the banks about as
// balls in bins.  Staging half an item keeps 4 workgroups per CU.
constexpr int kBankWords = 32;
constexpr int kDepU = kChunk / kThreads;  // particles per thread of a work item
constexpr int kDepStage = kChunk / 2;     // particles staged at a time
static_assert(kDepU % 2 == 0, "deposit halves");

// staging after the accumulation block: xF, yF, zF, m (doubles), first-node word << 16 |
// z index (int)
__host__ __device__ inline int tile_dep_acc_doubles(int cells) { return (cells + 1) & ~1; }

__global__ __launch_bounds__(kThreads) void tile_deposit(const double* __restrict__ cur,
                                                         int64_t cap,
                                                         const double* __restrict__ msize,
                                                         double macrosize, TileGeom g,
                                                         const int4* __restrict__ items,
                                                         const uint32_t* __restrict__ nitems,
                                                         double* __restrict__ rho,
                                                         uint32_t* __restrict__ counts) {
  if (counts && blockIdx.x == 0)  // (scan in the scatter: zero for the next step)
    for (int t = threadIdx.x; t <= g.ntiles; t += blockDim.x) counts[t] = 0;
  if (blockIdx.x >= *nitems) return;
  extern __shared__ double acc[];
  __shared__ uint32_t rcount[kBankWords], roff[kBankWords], rmax;
  const int4 it = items[blockIdx.x];
  const TileBox box(g, it.x);
  const int nz = g.nz, cells = box.cells();
  double* sxf = acc + tile_dep_acc_doubles(cells);
  double* syf = sxf + kDepStage;
  double* szf = syf + kDepStage;
  double* smm = szf + kDepStage;
  int* sbz = (int*)(smm + kDepStage);
  const int64_t gsx = (int64_t)g.ny * nz;
  const int np = it.z - it.y;  // at most kChunk
  // all of a thread's particle loads go out before the block is cleared
  double px[kDepU], py[kDepU], pz[kDepU], pm[kDepU];
#pragma unroll
  for (int u = 0; u < kDepU; u++) {
    const int j = (int)threadIdx.x + u * kThreads;
    const int64_t i = it.y + (j < np ? j : 0);
    px[u] = cur[i];
    py[u] = cur[2 * cap + i];
    pz[u] = cur[4 * cap + i];
    pm[u] = msize ? msize[i] : macrosize;
  }
  for (int c = threadIdx.x; c < cells; c += blockDim.x) acc[c] = 0.0;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    if (threadIdx.x < kBankWords) rcount[threadIdx.x] = 0u;
    __syncthreads();  // (h = 0: the block is clear)
    // rank each particle within its residue class (particles outside the block: global)
    constexpr int H = kDepU / 2;
    int bz[H];
    double xF[H], yF[H], zF[H];
    uint32_t res[H], rank[H];
#pragma unroll
    for (int v = 0; v < H; v++) {
      const int u = h * H + v;
      const int j = (int)threadIdx.x + u * kThreads;
      res[v] = kBankWords;  // none
      if (j >= np) continue;
      int iX, iY, iZ;
      node_ind_frac(px[u], g.xMin, g.dx, g.nx, iX, xF[v]);
      node_ind_frac(py[u], g.yMin, g.dy, g.ny, iY, yF[v]);
      grid3d_z_ind_frac(pz[u], g.zMin, g.dz, nz, iZ, zF[v]);
      const int zlo = nz >= 3 ? iZ - 1 : 0, zhi = nz >= 3 ? iZ + 1 : nz - 1;
      if (!box.holds(iX, iY, zlo, zhi)) {  // not in this tile's block (cannot happen for a
        // consistent sort): global
        deposit_particle(rho + (iX - 1) * gsx + (int64_t)(iY - 1) * nz, gsx, nz, nz, 0, pm[u],
                         xF[v], yF[v], iZ, zF[v]);
        continue;
      }
      const int b0 = box.idx(iX - 1, iY - 1, box.z0);  // < 2^15 (tile blocks <= 116 KiB)
      bz[v] = (b0 << 16) | iZ;
      const int w0 = b0 + (nz >= 3 ? iZ - 1 - box.z0 : -box.z0);
      res[v] = (uint32_t)w0 & (kBankWords - 1);
      rank[v] = atomicAdd(&rcount[res[v]], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // one wave: exclusive scan and maximum of the class counts
      const int l = threadIdx.x;
      const uint32_t c = l < kBankWords ? rcount[l] : 0u;
      uint32_t sc = c, mx = c;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(sc, o, 64);
        if (l >= o) sc += t;
        mx = max(mx, __shfl_xor(mx, o, 64));
      }
      if (l < kBankWords) roff[l] = sc - c;
      if (l == 0) rmax = mx;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < H; v++) {
      if (res[v] >= (uint32_t)kBankWords) continue;
      const uint32_t q = roff[res[v]] + rank[v];
      sxf[q] = xF[v];
      syf[q] = yF[v];
      szf[q] = zF[v];
      smm[q] = pm[h * H + v];
      sbz[q] = bz[v];
    }
    __syncthreads();
    const int l = (int)threadIdx.x & (kBankWords - 1);
    const int grp = (int)threadIdx.x / kBankWords, ngrp = kThreads / kBankWords;
    const uint32_t cl = rcount[l], ol = roff[l], rm = rmax;
    for (uint32_t k = grp; k < rm; k += ngrp) {
      if (k >= cl) continue;
      const uint32_t q = ol + k;
      const int b = sbz[q];
      deposit_particle(acc + (b >> 16), box.W * box.Wz, box.Wz, nz, box.z0, smm[q], sxf[q],
                       syf[q], b & 0xFFFF, szf[q]);
    }
    __syncthreads();  // every wave is done with the counters and the staging of this half
  }
  CellWalk w((int)threadIdx.x, box.W, box.Wz);
  for (int c = threadIdx.x; c < cells; c += kThreads, w.next()) {
    const double v = acc[c];
    if (v == 0.0) continue;
    const int gx = box.x0 + w.lx, gy = box.y0 + w.ly, gz = box.z0 + w.lz;
    if (gx < 0 || gx >= g.nx || gy < 0 || gy >= g.ny || gz < 0 || gz >= nz) continue;
    atomicAdd(rho + gx * gsx + (int64_t)gy * nz + gz, v);
  }
}

}  // namespace

TileGeom make_tile_geom(int nx, int ny, int nz, double xMin, double xMax, double yMin,
                        double yMax, double zMin, double zMax, double dx, double dy, double dz,
                        int lds_budget) {
  TileGeom g;
  g.nx = nx; g.ny = ny; g.nz = nz;
  g.xMin = xMin; g.xMax = xMax; g.yMin = yMin; g.yMax = yMax; g.zMin = zMin; g.zMax = zMax;
  g.dx = dx; g.dy = dy; g.dz = dz;
  g.T = g.Tz = g.zh = g.tx = g.ty = g.tz = g.ntiles = 0;
  // Small boxes first (many workgroups per CU); larger ones only to bound the tile count.
  static const int shapes[][2] = {{8, 16}, {8, 8},  {16, 16}, {8, 32}, {16, 32},
                                  {32, 32}, {6, 8}, {4, 8},   {4, 4},  {2, 2},  {1, 1}};
  for (const auto& sh : shapes) {
    const int T = sh[0];
    const int Tz = nz <= 2 ? nz : std::min(sh[1], nz);
    const int zh = nz >= 3 ? 1 : 0;
    const int64_t tx = (nx + T - 1) / T, ty = (ny + T - 1) / T, tz = (nz + Tz - 1) / Tz;
    const int64_t ntiles = tx * ty * tz;
    const int64_t lds = (int64_t)(T + 2) * (T + 2) * (Tz + 2 * zh) * 8;
    if (lds <= lds_budget && ntiles <= kMaxTiles) {
      g.T = T; g.Tz = Tz; g.zh = zh;
      g.tx = (int)tx; g.ty = (int)ty; g.tz = (int)tz; g.ntiles = (int)ntiles;
      break;
    }
  }
  return g;
}

size_t tile_deposit_lds_bytes(const TileGeom& g) {
  const int cells = (g.T + 2) * (g.T + 2) * (g.Tz + 2 * g.zh);
  return sizeof(double) * tile_dep_acc_doubles(cells) +
         (size_t)kDepStage * (4 * sizeof(double) + sizeof(int));
}

size_t tile_lds_bytes(const TileGeom& g) {
  return sizeof(double) * (g.T + 2) * (g.T + 2) * (g.Tz + 2 * g.zh);
}

void TileWork::reserve(int64_t n, int ntiles) {
  if (n > n_cap) {
    if (key) OB_HIP(hipFree(key));
    int64_t c = n_cap ? n_cap : 1 << 20;
    while (c < n) c *= 2;
    OB_HIP(hipMalloc((void**)&key, sizeof(uint32_t) * c));
    n_cap = c;
  }
  const int64_t want_items = n_cap / kChunk + ntiles + 2;  // (tile_chunk: at most 512 more)
  if (ntiles + 1 > t_cap || want_items > i_cap) {
    for (void* p : {(void*)counts, (void*)offsets, (void*)cursor, (void*)items, (void*)nitems})
      if (p) OB_HIP(hipFree(p));
    t_cap = std::max<int64_t>(ntiles + 1, t_cap);
    i_cap = std::max<int64_t>(want_items, i_cap);
    OB_HIP(hipMalloc((void**)&counts, sizeof(uint32_t) * t_cap));
    OB_HIP(hipMalloc((void**)&offsets, sizeof(uint32_t) * t_cap));
    OB_HIP(hipMalloc((void**)&cursor, sizeof(uint32_t) * t_cap));
    OB_HIP(hipMalloc((void**)&items, sizeof(int4) * i_cap));
    OB_HIP(hipMalloc((void**)&nitems, sizeof(uint32_t)));
    OB_HIP(hipMemset(counts, 0, sizeof(uint32_t) * t_cap));
  }
}

void TileWork::release() {
  for (void* p : {(void*)key, (void*)counts, (void*)offsets, (void*)cursor, (void*)items,
                  (void*)nitems})
    if (p) (void)hipFree(p);
  key = nullptr;
  counts = offsets = cursor = nullptr;
  items = nullptr;
  nitems = nullptr;
  n_cap = t_cap = i_cap = 0;
}

void sort_and_deposit_3d(ob_bunch* b, const TileGeom& g, double macrosize, double* rho,
                         TileWork& w) {
  static bool attr_done = false;
  if (!attr_done) {
    OB_HIP(hipFuncSetAttribute((const void*)tile_deposit,  // (plus its static class counters)
                               hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024));
    OB_HIP(hipFuncSetAttribute((const void*)tile_hist,
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    OB_HIP(hipFuncSetAttribute((const void*)tile_scatter<false>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    OB_HIP(hipFuncSetAttribute((const void*)tile_scan,
                               hipFuncAttributeMaxDynamicSharedMemorySize, 136 * 1024));
    attr_done = true;
  }
  const int64_t n = bunch_size(b);
  OB_REQUIRE((int64_t)(g.ntiles + 1) * 4 <= 150 * 1024, "tile sort: too many tiles for LDS");
  OB_REQUIRE(tile_deposit_lds_bytes(g) <= 159 * 1024, "tile deposit: tile block too large for LDS");
  OB_REQUIRE(g.nz < 65536, "tile deposit: more than 65535 z nodes");
  OB_REQUIRE(n < (int64_t)1 << 31, "tile sort: more than 2^31 particles");
  w.reserve(n, g.ntiles);
  hipStream_t s = stream();
  SortBuffers sb = bunch_sort_begin(b);
  const size_t hl = sizeof(uint32_t) * (g.ntiles + 1);
  const bool scan = n > 0 && g.ntiles <= kScanTiles;  // (no scatter without particles)
  // one workgroup of 1024 threads per CU: each merges up to ntiles + 1 counters into the
  // global counts, so fewer, larger workgroups mean fewer global atomics (measured 38 -> 32 us)
  int hb = (int)std::min<int64_t>((n + 1023) / 1024, device_cu_count());
  if (hb < 1) hb = 1;
  {
    ProfScope ps("tile_hist");
    // (four nodes per thread, at most one clearing workgroup per CU)
    const int64_t ng = (int64_t)g.nx * g.ny * g.nz;
    const int cb = (int)std::min<int64_t>((ng + 4095) / 4096, device_cu_count());
    hipLaunchKernelGGL(tile_hist, dim3(hb + cb), dim3(1024), hl, s, sb.cur, sb.cap, n, g, w.key,
                       w.counts, scan ? w.cursor : nullptr, hb, rho);
  }
  if (!scan) {
    ProfScope ps("tile_scan");
    hipLaunchKernelGGL(tile_scan, dim3(1), dim3(1024), sizeof(uint32_t) * 2 * (g.ntiles + 2), s,
                       w.counts, g.ntiles, w.offsets,
                       w.cursor, w.items, w.nitems, (uint32_t)tile_chunk(n));
  }
  // about 4096 workgroups: measured fastest for the scatter and for the deposit after it
  const int64_t per = std::max<int64_t>(512, (n + 4095) / 4096);
  const int sb_blocks = (int)((n + per - 1) / per);
  if (n) {
    ProfScope ps("tile_scatter");
    const ScatterScan sc{w.counts, w.offsets, w.items, w.nitems, (uint32_t)tile_chunk(n)};
    if (scan)
      hipLaunchKernelGGL(tile_scatter<true>, dim3(sb_blocks), dim3(kThreads), 2 * hl, s, sb.cur,
                         sb.alt, sb.cap, n, w.key, g.ntiles, w.cursor, sb.perm, sb.perm_alt,
                         sb.msize, sb.msize_alt, per, sc);
    else
      hipLaunchKernelGGL(tile_scatter<false>, dim3(sb_blocks), dim3(kThreads), hl, s, sb.cur,
                         sb.alt, sb.cap, n, w.key, g.ntiles, w.cursor, sb.perm, sb.perm_alt,
                         sb.msize, sb.msize_alt, per, sc);
  }
  OB_HIP(hipGetLastError());
  bunch_sort_commit(b);
  DeviceBunchView v = bunch_device_view(b);
  const int64_t max_items = n / tile_chunk(n) + g.ntiles + 1;
  {
    ProfScope ps("tile_deposit");
    hipLaunchKernelGGL(tile_deposit, dim3((unsigned)max_items), dim3(kThreads),
                       tile_deposit_lds_bytes(g),
                       s, v.c[0], (int64_t)(v.c[1] - v.c[0]), v.msize, macrosize, g, w.items,
                       w.nitems, rho, scan ? w.counts : nullptr);
  }
  OB_HIP(hipGetLastError());
}

void tile_kick_3d(ob_bunch* b, const TileGeom& g, const Kick3D& k, TileWork& w) {
  const int64_t n = bunch_size(b);
  if (n == 0) return;
  TileKick t{g, k, w.items, w.nitems, w.offsets, n, n / tile_chunk(n) + g.ntiles + 1};
  t.k.fx = k.trans_factor / g.dx;
  t.k.fy = k.trans_factor / g.dy;
  t.k.fz = k.long_factor / k.rdz;
  bunch_queue_tile_kick(b, t);
}

}  // namespace ob
