// fd_grad_kernels.hip -- gradient pass of the first-derivative form of the FD step.
#include "fd_layers.h"

namespace klrtm {

// ---------------------------------------------------------------------------
// Gradient + PML round 1 + scalar operator.  Writes px, py (= pr), pz.
template<int MODEL, bool RHO>
struct GradPlane {
  float qa;                  // u at y+R (own column)
  float hz0, hz1, hx0, hx1;  // z and x halos of u at y+R
  float e, d, ax, ay, rho;   // model parameters at y
  LayerState q;
};

template<int R, int MODEL, bool RHO>
__global__ void __launch_bounds__(512) grad_kernel(const float *__restrict__ u, float *__restrict__ px,
                                                   float *__restrict__ py, float *__restrict__ pz,
                                                   const float *__restrict__ eps, const float *__restrict__ del,
                                                   const float *__restrict__ pjx, const float *__restrict__ pjy,
                                                   const IsoArgs a) {
  extern __shared__ float s[];
  constexpr int S = TILE_Z + 2 * R;
  const int ny = a.ny, nz = a.nz;
  const size_t nxz = (size_t)a.nx * nz;
  const uint32_t pbytes = (uint32_t)(nxz * 4);
  const TileCoord c = tile_coord(a);
  const TileOffsets o = tile_offsets<R>(c, a);
  const LayerSlots sl = layer_slots(c, a);
  const LayerOps L(a, sl, 0, c);
  // (ny > 1: a 2D grid has kernels of its own.  Asked for again because a branch of its own keeps gy's last products in
  // its block, and with them what the compiler contracts there: the bits of the step)
  const bool st_y = c.act && ny > 1;
  auto prs = [&](const float *base, int y) { return buf_rsrc(base + (size_t)y * nxz, pbytes); };
  float q[2 * R + 1];
#pragma unroll
  for(int k = 0; k < 2 * R; k++) {
    const int yy = c.y0 - R + k;
    q[k] = (c.act && yy >= 0 && yy < ny) ? u[(size_t)yy * nxz + c.col] : 0.f;
  }
  // ring of NP plane tiles: plane p sits in slot p % NP
  constexpr int NP = R + 2;
  const int slot = (a.tx + 2 * R) * S;
  float *srow0 = s + (c.tx + R) * S + c.tz + R;
  const bool lz0 = c.tz < R, lz1 = c.tz >= a.tz - R, lx0 = c.tx < R, lx1 = c.tx >= a.tx - R;
  auto tile_put = [&](float *row, float v, float hz0, float hz1, float hx0, float hx1) __attribute__((always_inline)) {
    row[0] = v;
    if(lz0) row[-R] = hz0;
    if(lz1) row[R] = hz1;
    if(lx0) row[-R * S] = hx0;
    if(lx1) row[R * S] = hx1;
  };
  // planes y0 .. y0+R-1 of the chunk, all loads in flight together
  {
    float h[4][R];
#pragma unroll
    for(int k = 0; k < R; k++) {
      const __amdgpu_buffer_rsrc_t ru = prs(u, min(c.y0 + k, ny - 1));
      h[0][k] = buf_ld(ru, o.z0, 0), h[1][k] = buf_ld(ru, o.z1, 0);
      h[2][k] = buf_ld(ru, o.x0, 0), h[3][k] = buf_ld(ru, o.x1, 0);
    }
#pragma unroll
    for(int k = 0; k < R; k++)
      tile_put(srow0 + ((c.y0 + k) % NP) * slot, q[R + k], h[0][k], h[1][k], h[2][k], h[3][k]);
  }
  int ps = c.y0 % NP;  // slot of the current plane
  // irregular z grid: this block's per-iz first-derivative weights, after the ring
  const bool irr = a.zc1 != nullptr;
  float *zct = s + NP * slot + c.tz * (R + 1);
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
    typedef GradPlane<MODEL, RHO> Plane;
    auto fetch = [&](Plane &N, int y) __attribute__((always_inline)) {
      const int yr = min(y + R, ny - 1);
      const __amdgpu_buffer_rsrc_t ru = prs(u, yr);
      const size_t pl = (size_t)y * nxz;
      N.qa = at_ld(u + (size_t)yr * nxz, L.col);
      if(MODEL != KLRTM_ISO) {
        N.e = at_ld(eps + pl, L.col);
        N.d = at_ld(del + pl, L.col);
      }
      if(MODEL == KLRTM_TTI) {
        N.ax = at_ld(pjx + pl, L.col);
        N.ay = at_ld(pjy + pl, L.col);
      }
      if(RHO) N.rho = at_ld(a.rho + pl, L.col);
      N.hz0 = buf_ld(ru, o.z0, 0), N.hz1 = buf_ld(ru, o.z1, 0);
      N.hx0 = buf_ld(ru, o.x0, 0), N.hx1 = buf_ld(ru, o.x1, 0);
      L.load<0, ZX, YL>(N.q, y, fy, y - jy0);
      L.load<1, ZX, YL>(N.q, y, fy, y - jy0);
      L.load<2, ZX, YL>(N.q, y, fy, y - jy0);
    };
    // plane y+R goes into the slot of plane y-2, which nobody reads any more (every wave has passed the
    // barrier of y-1), then plane y is computed (beyond the grid's last plane the slot is written, not read)
    auto plane = [&](Plane &C, int y) __attribute__((always_inline)) {
      q[2 * R] = c.act && y + R < ny ? C.qa : 0.f;  // zero beyond the grid (those lanes feed the tile's edge)
      tile_put(srow0 + (ps >= 2 ? ps - 2 : ps + NP - 2) * slot, q[2 * R], C.hz0, C.hz1, C.hx0, C.hx1);
      const float *srow = srow0 + ps * slot;
      ps = ps + 1 == NP ? 0 : ps + 1;
      lds_barrier();
      // z: vz accumulates (-c_m) u[-m] for m=R..1, then c_m u[+m] (bgprtm/FdEngine_fd.cpp:394-403)
      float gz = 0.f;
      if(opaque(irr)) {
#pragma unroll
        for(int m = R; m >= 1; m--) gz = fmaf(-zct[m], srow[-m], gz);
#pragma unroll
        for(int m = 1; m <= R; m++) gz = fmaf(zct[m], srow[m], gz);
        asm volatile("");  // keeps the branches apart (a common weight load would be a flat access)
      } else {
#pragma unroll
        for(int m = R; m >= 1; m--) gz = fmaf(-a.cz[m], srow[-m], gz);
#pragma unroll
        for(int m = 1; m <= R; m++) gz = fmaf(a.cz[m], srow[m], gz);
      }
      // x: vx -= c u[-m]; vx += c u[+m] (bgprtm/FdEngine_fd.cpp:420-431)
      float gx = 0.f;
#pragma unroll
      for(int m = 1; m <= R; m++) {
        gx = fmaf(-a.cx[m], srow[-m * S], gx);
        gx = fmaf(a.cx[m], srow[m * S], gx);
      }
      float gy = 0.f;
#pragma unroll
      for(int m = 1; m <= R; m++) {
        gy = fmaf(-a.cy[m], q[R - m], gy);
        gy = fmaf(a.cy[m], q[R + m], gy);
      }
      gz = L.damp<0, ZX, YL>(gz, C.q, fy, y - jy0);
      gx = L.damp<1, ZX, YL>(gx, C.q, fy, y - jy0);
      gy = L.damp<2, ZX, YL>(gy, C.q, fy, y - jy0);
      if(RHO) {  // KernelCPU::divideRho before the scalar operator (bgprtm/KernelCPU.cpp:103, 340-349)
        gx /= C.rho;
        gy /= C.rho;
        gz /= C.rho;
      }
      if(MODEL == KLRTM_VTI) scalar_vti(C.e, C.d, gx, gy, gz);
      else if(MODEL == KLRTM_TTI) scalar_tti(C.e, C.d, C.ax, C.ay, gx, gy, gz);
      if(c.act) {
        const size_t pl = (size_t)y * nxz;
        at_st(px + pl, L.col, gx);
        at_st(pz + pl, L.col, gz);
      }
      if(st_y) at_st(py + (size_t)y * nxz, L.col, gy);
      L.store<ZX, YL>(C.q, y, fy, y - jy0);
#pragma unroll
      for(int k = 0; k < 2 * R; k++) q[k] = q[k + 1];
    };
    stream_planes<Plane>(ya, yb, fetch, plane);
  };
  run_segments(c, a, sl.any, segment);
}

template<int R, int MODEL, bool RHO>
static int launch_grad_rm(const float *u, float *px, float *py, float *pz, const float *eps, const float *del,
                          const float *pjx, const float *pjy, IsoArgs a) {
  LaunchTimer tm("fd_grad");
  grid_of(a);
  size_t lds = sizeof(float) * (size_t)(R + 2) * (a.tx + 2 * R) * (TILE_Z + 2 * R);  // the ring of plane tiles
  if(a.zc1) lds += sizeof(float) * (size_t)a.tz * (R + 1);
  hipLaunchKernelGGL((grad_kernel<R, MODEL, RHO>), dim3(a.nbz * a.nbx * a.nby), dim3(a.tz * a.tx), lds, stream(), u, px, py, pz, eps, del, pjx, pjy, a);
  return check_launch("grad_kernel");
}
template<int R>
static int launch_grad_r(int model, const float *u, float *px, float *py, float *pz, const float *eps,
                         const float *del, const float *pjx, const float *pjy, const IsoArgs &a) {
  if(a.rho) {
    if(model == KLRTM_VTI) return launch_grad_rm<R, KLRTM_VTI, true>(u, px, py, pz, eps, del, pjx, pjy, a);
    if(model == KLRTM_TTI) return launch_grad_rm<R, KLRTM_TTI, true>(u, px, py, pz, eps, del, pjx, pjy, a);
    return launch_grad_rm<R, KLRTM_ISO, true>(u, px, py, pz, eps, del, pjx, pjy, a);
  }
  if(model == KLRTM_VTI) return launch_grad_rm<R, KLRTM_VTI, false>(u, px, py, pz, eps, del, pjx, pjy, a);
  if(model == KLRTM_TTI) return launch_grad_rm<R, KLRTM_TTI, false>(u, px, py, pz, eps, del, pjx, pjy, a);
  return launch_grad_rm<R, KLRTM_ISO, false>(u, px, py, pz, eps, del, pjx, pjy, a);
}
int launch_grad(int R, int model, const float *u, float *px, float *py, float *pz, const float *eps, const float *del,
                const float *pjx, const float *pjy, const IsoArgs &a) {
  switch(R) {
  case 4: return launch_grad_r<4>(model, u, px, py, pz, eps, del, pjx, pjy, a);
  case 5: return launch_grad_r<5>(model, u, px, py, pz, eps, del, pjx, pjy, a);
  case 6: return launch_grad_r<6>(model, u, px, py, pz, eps, del, pjx, pjy, a);
  case 7: return launch_grad_r<7>(model, u, px, py, pz, eps, del, pjx, pjy, a);
  case 8: return launch_grad_r<8>(model, u, px, py, pz, eps, del, pjx, pjy, a);
  default: set_error("FD half order %d not supported (4..8)", R); return KLRTM_EINVAL;
  }
}

}  // namespace klrtm
