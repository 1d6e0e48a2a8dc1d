// fd_div_kernels.hip -- divergence pass of the first-derivative form of the FD step.
#include "fd_layers.h"

namespace klrtm {

// ---------------------------------------------------------------------------
// Divergence + PML round 2 + pb -= vel*div (x, z, then y as the reference)
// (+ update2nd in MODE_STEP).  Dx needs x-neighbours of px, Dz z-neighbours of
// pz, Dy y-neighbours of py: two LDS tiles and one register queue.
template<int MODE, bool RHO>
struct DivPlane {
  float qa;            // py at y+R
  float cz, hz0, hz1;  // pz at y and its z halos
  float cx, hx0, hx1;  // px at y and its x halos
  float w, v, u, rho;  // w0, vel, w1, density at y
  LayerState q;
};

template<int R, int MODE, bool RHO>
__global__ void __launch_bounds__(512) div_kernel(const float *__restrict__ px, const float *__restrict__ py,
                                                  const float *__restrict__ pz, const float *__restrict__ w1,
                                                  float *__restrict__ w0, const float *__restrict__ vel,
                                                  const IsoArgs a) {
  extern __shared__ float s[];
  constexpr int SZ = TILE_Z + 2 * R, SX = TILE_Z;    // row pitches of the z-haloed (pz) and x-haloed (px) tiles
  const int ny = a.ny, nz = a.nz;
  const size_t nxz = (size_t)a.nx * nz;
  const uint32_t pbytes = (uint32_t)(nxz * 4);
  const TileCoord c = tile_coord(a);
  const TileOffsets o = tile_offsets<R>(c, a);
  const int TZ = a.tz, TX = a.tx;
  const int tile = TX * SZ + (TX + 2 * R) * SX;  // TX rows of the first tile, TX+2R rows of the second
  const LayerSlots sl = layer_slots(c, a);
  const LayerOps L(a, sl, 1, c);
  auto prs = [&](const float *base, int y) { return buf_rsrc(base + (size_t)y * nxz, pbytes); };
  float q[2 * R + 1];
#pragma unroll
  for(int k = 0; k < 2 * R; k++) {
    const int yy = c.y0 - R + k;
    q[k] = (c.act && yy >= 0 && yy < ny) ? py[(size_t)yy * nxz + c.col] : 0.f;
  }
  float *zrow0 = s + c.tx * SZ + c.tz + R;                 // LDS tiles of even planes
  float *xrow0 = s + TX * SZ + (c.tx + R) * SX + c.tz;
  int slot = 0;
  // irregular z grid: this block's per-iz first-derivative weights, after the tiles
  const bool irr = a.zc1 != nullptr;
  float *zct = s + 2 * tile + c.tz * (R + 1);
  if(irr) {
    if(c.tx == 0) {
      const float *g = a.zc1 + (size_t)min(c.iz, nz - 1) * ZC1_STRIDE;
#pragma unroll
      for(int m = 1; m <= R; m++) zct[m] = g[m];
    }
    lds_barrier();
  }
  auto segment = [&](auto zx_tag, auto y_tag, int ya, int yb, int fy, int jy0) __attribute__((always_inline)) {
    constexpr bool ZX = decltype(zx_tag)::value, YL = decltype(y_tag)::value;
    typedef DivPlane<MODE, RHO> Plane;
    auto fetch = [&](Plane &N, int y) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t rz = prs(pz, y), rx = prs(px, y);
      const size_t pl = (size_t)y * nxz;
      N.qa = at_ld(py + (size_t)min(y + R, ny - 1) * nxz, L.col);
      N.cz = buf_ld(rz, o.c, 0), N.hz0 = buf_ld(rz, o.z0, 0), N.hz1 = buf_ld(rz, o.z1, 0);
      N.cx = buf_ld(rx, o.c, 0), N.hx0 = buf_ld(rx, o.x0, 0), N.hx1 = buf_ld(rx, o.x1, 0);
      N.w = at_ld(w0 + pl, L.col);
      N.v = at_ld(vel + pl, L.col);
      if(MODE == MODE_STEP) N.u = at_ld(w1 + pl, L.col);
      if(RHO) N.rho = at_ld(a.rho + pl, L.col);
      L.load<1, ZX, YL>(N.q, y, fy, y - jy0);
      L.load<0, ZX, YL>(N.q, y, fy, y - jy0);
      L.load<2, ZX, YL>(N.q, y, fy, y - jy0);
    };
    auto plane = [&](Plane &C, int y) __attribute__((always_inline)) {
      q[2 * R] = c.act && y + R < ny ? C.qa : 0.f;  // zero beyond the grid (those lanes feed the tile's edge)
      float *zrow = zrow0 + slot, *xrow = xrow0 + slot;  // the tiles of even and odd planes in turn
      slot = tile - slot;
      zrow[0] = C.cz;
      if(c.tz < R) zrow[-R] = C.hz0;
      if(c.tz >= TZ - R) zrow[R] = C.hz1;
      xrow[0] = C.cx;
      if(c.tx < R) xrow[-R * SX] = C.hx0;
      if(c.tx >= TX - R) xrow[R * SX] = C.hx1;
      lds_barrier();
      float dxv = 0.f;
#pragma unroll
      for(int m = 1; m <= R; m++) {
        dxv = fmaf(-a.cx[m], xrow[-m * SX], dxv);
        dxv = fmaf(a.cx[m], xrow[m * SX], dxv);
      }
      float dzv = 0.f;
      if(opaque(irr)) {
#pragma unroll
        for(int m = R; m >= 1; m--) dzv = fmaf(-zct[m], zrow[-m], dzv);
#pragma unroll
        for(int m = 1; m <= R; m++) dzv = fmaf(zct[m], zrow[m], dzv);
        asm volatile("");
      } else {
#pragma unroll
        for(int m = R; m >= 1; m--) dzv = fmaf(-a.cz[m], zrow[-m], dzv);
#pragma unroll
        for(int m = 1; m <= R; m++) dzv = fmaf(a.cz[m], zrow[m], dzv);
      }
      float dyv = 0.f;
#pragma unroll
      for(int m = 1; m <= R; m++) {
        dyv = fmaf(-a.cy[m], q[R - m], dyv);
        dyv = fmaf(a.cy[m], q[R + m], dyv);
      }
      dxv = L.damp<1, ZX, YL>(dxv, C.q, fy, y - jy0);
      dzv = L.damp<0, ZX, YL>(dzv, C.q, fy, y - jy0);
      dyv = L.damp<2, ZX, YL>(dyv, C.q, fy, y - jy0);
      float w;
      if(RHO) {  // out -= d*vel*rho (bgprtm/FdEngine_fd.cpp:409-412, 435-438, 461-464)
        w = fmaf(-(dxv * C.v), C.rho, C.w);
        w = fmaf(-(dzv * C.v), C.rho, w);
        w = fmaf(-(dyv * C.v), C.rho, w);
      } else {
        w = fmaf(-dxv, C.v, C.w);
        w = fmaf(-dzv, C.v, w);
        w = fmaf(-dyv, C.v, w);
      }
      if(MODE == MODE_STEP) w = (C.u + C.u) - w;
      if(c.act) at_st(w0 + (size_t)y * nxz, L.col, w);
      L.store<ZX, YL>(C.q, y, fy, y - jy0);
#pragma unroll
      for(int k = 0; k < 2 * R; k++) q[k] = q[k + 1];
    };
    stream_planes<Plane>(ya, yb, fetch, plane);
  };
  run_segments(c, a, sl.any, segment);
}

template<int R, int MODE, bool RHO>
static int launch_div_rm(const float *px, const float *py, const float *pz, const float *w1, float *w0, const float *vel,
                         IsoArgs a) {
  LaunchTimer tm(MODE == MODE_STEP ? "fd_div_step" : "fd_div");
  grid_of(a);
  size_t lds = 2 * sizeof(float) * ((size_t)a.tx * (TILE_Z + 2 * R) + (size_t)(a.tx + 2 * R) * TILE_Z);
  if(a.zc1) lds += sizeof(float) * (size_t)a.tz * (R + 1);
  hipLaunchKernelGGL((div_kernel<R, MODE, RHO>), dim3(a.nbz * a.nbx * a.nby), dim3(a.tz * a.tx), lds, stream(), px, py, pz, w1, w0, vel, a);
  return check_launch("div_kernel");
}
template<int R>
static int launch_div_r(int mode, const float *px, const float *py, const float *pz, const float *w1, float *w0,
                        const float *vel, const IsoArgs &a) {
  if(mode == MODE_STEP)
    return a.rho ? launch_div_rm<R, MODE_STEP, true>(px, py, pz, w1, w0, vel, a)
                 : launch_div_rm<R, MODE_STEP, false>(px, py, pz, w1, w0, vel, a);
  return a.rho ? launch_div_rm<R, MODE_KERNEL, true>(px, py, pz, w1, w0, vel, a)
               : launch_div_rm<R, MODE_KERNEL, false>(px, py, pz, w1, w0, vel, a);
}
int launch_div(int R, int mode, const float *px, const float *py, const float *pz, const float *w1, float *w0,
               const float *vel, const IsoArgs &a) {
  switch(R) {
  case 4: return launch_div_r<4>(mode, px, py, pz, w1, w0, vel, a);
  case 5: return launch_div_r<5>(mode, px, py, pz, w1, w0, vel, a);
  case 6: return launch_div_r<6>(mode, px, py, pz, w1, w0, vel, a);
  case 7: return launch_div_r<7>(mode, px, py, pz, w1, w0, vel, a);
  case 8: return launch_div_r<8>(mode, px, py, pz, w1, w0, vel, a);
  default: set_error("FD half order %d not supported (4..8)", R); return KLRTM_EINVAL;
  }
}

}  // namespace klrtm
