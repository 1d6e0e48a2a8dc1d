// fd_tile.h -- tile bookkeeping shared by the y-streaming FD stencil kernels.
#pragma once
#include "klrtm_internal.h"
#include "fd_kernels.h"

namespace klrtm {

inline void grid_of(IsoArgs &a) {
  a.nbz = div_up(a.nz, a.tz);
  a.nbx = div_up(a.nx, a.tx);
  a.nby = div_up(a.ny, a.ychunk);
}

}  // namespace klrtm

#ifdef __HIPCC__
namespace klrtm {

struct TileCoord {
  int tz, tx, iz, ix, y0, y1;
  bool act;  // the cell lies inside the grid
  size_t col;
};
// Consecutive logical tiles run together on one XCD (xcd_remap); z tiles vary fastest, so the
// co-resident set is a patch of whole z columns over neighbouring x: the z and x halos a block
// reads are mostly its neighbours' rows, already in that XCD's L2.
__device__ __forceinline__ TileCoord tile_coord(const IsoArgs &a) {
  TileCoord c;
  int t = xcd_remap(blockIdx.x, gridDim.x);
  const int bz = t % a.nbz;
  t /= a.nbz;
  const int bx = t % a.nbx;
  const int by = t / a.nbx;
  c.tz = threadIdx.x % a.tz, c.tx = threadIdx.x / a.tz;
  c.iz = bz * a.tz + c.tz, c.ix = bx * a.tx + c.tx;
  c.y0 = by * a.ychunk, c.y1 = min(a.ny, c.y0 + a.ychunk);
  c.act = c.iz < a.nz && c.ix < a.nx;
  c.col = (size_t)c.ix * a.nz + c.iz;
  return c;
}
// Byte offsets of a thread's cell and of its halo loads inside a plane (out of range where there is
// nothing to load): z halos of the own row, x halos of the own column.
struct TileOffsets {
  uint32_t c, z0, z1, x0, x1;
};
template<int R>
__device__ __forceinline__ TileOffsets tile_offsets(const TileCoord &c, const IsoArgs &a) {
  TileOffsets o;
  const int nx = a.nx, nz = a.nz;
  o.c = c.act ? (uint32_t)c.col * 4u : OOR;
  o.z0 = (c.tz < R && c.ix < nx && c.iz - R >= 0) ? (uint32_t)(c.col - R) * 4u : OOR;
  o.z1 = (c.tz >= a.tz - R && c.ix < nx && c.iz + R < nz) ? (uint32_t)(c.col + R) * 4u : OOR;
  o.x0 = (c.tx < R && c.iz < nz && c.ix - R >= 0) ? (uint32_t)(c.col - (size_t)R * nz) * 4u : OOR;
  o.x1 = (c.tx >= a.tx - R && c.iz < nz && c.ix + R < nx) ? (uint32_t)(c.col + (size_t)R * nz) * 4u : OOR;
  return o;
}

// PML layer slots of a thread's column: state byte offset at y = 0 and stride per plane of the z and of the x
// layers (0 outside them), their position's round coefficients for the own axis (scale 1) and the cross axes
// (pml3d_scaler), and the cells of the first layer of each pair.
struct LayerSlots {
  bool zin, xin, any;  // (any: some cell of the block lies in a z or x layer)
  uint32_t zo, zs, xo, xs;
  float zc[2][3], xc[2][3];
  uint32_t first[3];  // per axis z, x, y
};
__device__ __forceinline__ LayerSlots layer_slots(const TileCoord &c, const IsoArgs &a) {
  LayerSlots s;
  const PmlDesc &P = a.pml;
  const int nx = a.nx, ny = a.ny, nz = a.nz, ix = c.ix, iz = c.iz;
  s.zo = s.xo = s.zs = s.xs = 0;
  s.zin = s.xin = s.any = false;
#pragma unroll
  for(int k = 0; k < 2; k++) {
    s.zc[k][0] = s.zc[k][1] = s.xc[k][0] = s.xc[k][1] = 0.f;
    s.zc[k][2] = s.xc[k][2] = 1.f;
  }
  const int fa[3] = {FZ1, FX1, FY1};
#pragma unroll
  for(int k = 0; k < 3; k++) s.first[k] = P.q[fa[k]][0][0] ? face_cells_dev(P, fa[k], nx, ny, nz) : 0u;
  if(!a.has_pml) return s;
  if(c.act) {
    // (faces are picked with selects: indexing the argument struct with a lane value would copy it to
    // scratch memory)
    const bool z1 = P.q[FZ1][0][0] && iz < P.w[FZ1], z2 = !z1 && P.q[FZ2][0][0] && iz >= nz - P.w[FZ2];
    if(z1 || z2) {
      const int w = z1 ? P.w[FZ1] : P.w[FZ2], j = z1 ? iz : iz - (nz - w);
  #pragma unroll
      for(int k = 0; k < 2; k++) {
        const float *t = (z1 ? P.abc[FZ1][k] : P.abc[FZ2][k]) + 3 * j;
        s.zc[k][0] = t[0], s.zc[k][1] = t[1], s.zc[k][2] = t[2];
      }
      s.zin = true;
      s.zo = ((z2 ? s.first[0] : 0u) + (uint32_t)ix * w + j) * 4u;  // ((iy*nx + ix)*w + j)
      s.zs = (uint32_t)nx * w * 4u;
    }
    const bool x1 = P.q[FX1][0][0] && ix < P.w[FX1], x2 = !x1 && P.q[FX2][0][0] && ix >= nx - P.w[FX2];
    if(x1 || x2) {
      const int w = x1 ? P.w[FX1] : P.w[FX2], j = x1 ? ix : ix - (nx - w);
  #pragma unroll
      for(int k = 0; k < 2; k++) {
        const float *t = (x1 ? P.abc[FX1][k] : P.abc[FX2][k]) + 3 * j;
        s.xc[k][0] = t[0], s.xc[k][1] = t[1], s.xc[k][2] = t[2];
      }
      s.xin = true;
      s.xo = ((x2 ? s.first[1] : 0u) + (uint32_t)j * nz + iz) * 4u;  // ((iy*w + j)*nz + iz)
      s.xs = (uint32_t)w * nz * 4u;
    }
  }
  s.any = __builtin_amdgcn_readfirstlane(__syncthreads_or(s.zin || s.xin)) != 0;
  return s;
}

}  // namespace klrtm
#endif
