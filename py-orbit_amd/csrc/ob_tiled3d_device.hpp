// ob_tiled3d_device.hpp -- device side of the tile blocks: the deposit (ob_tiled3d.hip) and the
// kick, which runs in one launch with the maps after it (ob_push.hip).
#pragma once

#include "ob_sc_device.hpp"
#include "ob_tiled3d.hpp"

namespace ob {

constexpr int kTileThreads = 256;

// Cell c = (lx*W + ly)*Wz + lz of a tile block, advanced by kTileThreads cells per step with
// carries instead of a division per cell (the divisions are done once per thread).
struct CellWalk {
  int lx, ly, lz, sx, sy, sz, W, Wz;
  __device__ __forceinline__ CellWalk(int c, int W_, int Wz_) : W(W_), Wz(Wz_) {
    lz = c % Wz;
    const int r = c / Wz;
    ly = r % W;
    lx = r / W;
    sz = kTileThreads % Wz;
    const int sr = kTileThreads / Wz;
    sy = sr % W;
    sx = sr / W;
  }
  __device__ __forceinline__ void next() {
    lz += sz;
    int carry = lz >= Wz ? 1 : 0;
    lz -= carry * Wz;
    ly += sy + carry;  // < 2W
    carry = ly >= W ? 1 : 0;
    ly -= carry * W;
    lx += sx + carry;
  }
};

// Tile t's LDS block: nodes x0..x0+W-1, y0..y0+W-1, z0..z0+Wz-1, z fastest.
struct TileBox {
  int x0, y0, z0, W, Wz;
  __device__ __forceinline__ TileBox(const TileGeom& g, int t) {
    const int tzi = t % g.tz, r = t / g.tz;
    const int tyi = r % g.ty, txi = r / g.ty;
    W = g.T + 2;
    Wz = g.Tz + 2 * g.zh;
    x0 = txi * g.T - 1;
    y0 = tyi * g.T - 1;
    z0 = tzi * g.Tz - g.zh;
  }
  __device__ __forceinline__ int cells() const { return W * W * Wz; }
  __device__ __forceinline__ int idx(int gx, int gy, int gz) const {
    return ((gx - x0) * W + (gy - y0)) * Wz + (gz - z0);
  }
  // nodes gx-1..gx+1, gy-1..gy+1, zlo..zhi inside the block
  __device__ __forceinline__ bool holds(int gx, int gy, int zlo, int zhi) const {
    return gx - 1 >= x0 && gx + 1 < x0 + W && gy - 1 >= y0 && gy + 1 < y0 + W && zlo >= z0 &&
           zhi < z0 + Wz;
  }
};

// Grid3D::calcGradient (Grid3D.cc:438-532) in units of the grid steps: gx dx, gy dy, gz dz.  The
// steps are divided out of the kick's factors once on the host (as many roundings per
// particle, nine divisions fewer), and the 27 nodes are summed z, y, x with the partial sums
// shared by the three components: 90 fused operations instead of about 250 and the divisions,
// which bound the kick (120 us for 4M particles, whose bytes take 70).
__device__ __forceinline__ void tile_gradient(const Grid3View& a, int nz, int iX, int iY, int iZ,
                                              double xF, double yF, double zF, double& gx,
                                              double& gy, double& gz) {
  const double wx[3] = {0.5 * (0.5 - xF) * (0.5 - xF), 0.75 - xF * xF,
                        0.5 * (0.5 + xF) * (0.5 + xF)};
  const double wy[3] = {0.5 * (0.5 - yF) * (0.5 - yF), 0.75 - yF * yF,
                        0.5 * (0.5 + yF) * (0.5 + yF)};
  const double dx[3] = {xF - 0.5, -2. * xF, 0.5 + xF};
  const double dy[3] = {yF - 0.5, -2. * yF, 0.5 + yF};
  gx = gy = gz = 0.0;
  if (nz >= 3) {
    const double wz[3] = {0.5 * (0.5 - zF) * (0.5 - zF), 0.75 - zF * zF,
                          0.5 * (0.5 + zF) * (0.5 + zF)};
    const double dz[3] = {zF - 0.5, -2. * zF, 0.5 + zF};
    const int zm = iZ - 1 < 0 ? nz - 1 : -1, zp = iZ + 1 >= nz ? 1 - nz : 1;
    const double* s = a.at(iX - 1, iY - 1, iZ);
#pragma unroll
    for (int i = 0; i < 3; i++) {
      double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const double* n = s + i * a.sx + j * a.sy;
        const double m = n[zm], c = n[0], p = n[zp];
        const double v = fma(wz[2], p, fma(wz[1], c, wz[0] * m));
        const double d = fma(dz[2], p, fma(dz[1], c, dz[0] * m));
        sx = fma(wy[j], v, sx);
        sy = fma(dy[j], v, sy);
        sz = fma(wy[j], d, sz);
      }
      gx = fma(dx[i], sx, gx);
      gy = fma(wx[i], sy, gy);
      gz = fma(wx[i], sz, gz);
    }
  } else {  // two nodes (linear in z) or one (no z dependence)
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const double* n = a.at(iX - 1 + i, iY - 1 + j, 0);
        double v = n[0], d = 0.0;
        if (nz == 2) {
          const double p = n[1];
          d = p - v;
          v = fma(zF, p, (1.0 - zF) * v);
        }
        gx = fma(dx[i] * wy[j], v, gx);
        gy = fma(wx[i] * dy[j], v, gy);
        gz = fma(wx[i] * wy[j], d, gz);
      }
  }
}

// The SpaceChargeCalc3D kick of a particle, gathering phi from its tile's block, or from the
// whole grid if the block does not hold its 27 nodes.  BND: particles outside
// the boundary in k are not kicked.
template <bool BND>
__device__ __forceinline__ void tile_kick_particle(const TileGeom& g, const Kick3D& k,
                                                   const double* lds, const TileBox& box,
                                                   double x, double y, double z, double& xp,
                                                   double& yp, double& dE) {
  if (BND && !boundary_inside(k.bnd_type, k.bnd, x, y)) return;
  const double zr = (z - k.zc) * k.gamma + k.zc;
  int iX, iY, iZ;
  double xF, yF, zF;
  node_ind_frac(x, g.xMin, g.dx, g.nx, iX, xF);
  node_ind_frac(y, g.yMin, g.dy, g.ny, iY, yF);
  grid3d_z_ind_frac(zr, k.rzMin, k.rdz, g.nz, iZ, zF);
  const int zlo = g.nz >= 3 ? iZ - 1 : 0, zhi = g.nz >= 3 ? iZ + 1 : g.nz - 1;
  double gx, gy, gz;
  if (box.holds(iX, iY, zlo, zhi)) {
    const Grid3View v{lds, (int64_t)box.W * box.Wz, box.Wz, box.x0, box.y0, box.z0};
    tile_gradient(v, g.nz, iX, iY, iZ, xF, yF, zF, gx, gy, gz);
  } else {
    const Grid3View v{k.phi, (int64_t)g.ny * g.nz, g.nz, 0, 0, 0};
    tile_gradient(v, g.nz, iX, iY, iZ, xF, yF, zF, gx, gy, gz);
  }
  xp += -gx * k.fx;
  yp += -gy * k.fy;
  dE += -gz * k.fz;
}

}  // namespace ob
