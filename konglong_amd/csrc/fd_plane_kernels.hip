// fd_plane_kernels.hip -- the first-derivative form of the FD step (gradient and divergence pass) on a 2D grid.
//
// One plane, no y derivative: a thread per cell of a (TZ x TX) tile, z and x halos in LDS, one barrier.  As a volume of
// one plane the streaming kernels filled their ring of planes, loaded the plane twice and ran one or two workgroups a
// CU (grad_kernel, div_kernel); here 47 to 73 VGPRs leave three or four, bound by HBM and L2.  A step of both passes,
// 2000 x 1000 / 3000 x 4000 cells: VTI FD8 100 / 512 -> 37 / 193 us, TTI FD16 203 / 1096 -> 41 / 220 us.
#include "fd_layers.h"

namespace klrtm {

// a zero that the compiler does not know: what it contracts stays what it is with a y derivative
__device__ __forceinline__ float opaque_zero() {
  float v = 0.f;
  asm volatile("" : "+v"(v));
  return v;
}

// damping state of one derivative axis (0 z, 1 x) of the plane: LayerState slots [AX]
template<int AX, bool ZX>
__device__ __forceinline__ void plane_store(const LayerOps &L, const LayerState &q) {
  typedef LayerComp<AX> K;
  if(!ZX) return;
  if(AX == 0 ? L.zin : L.zcr) at_st(L.base<0>(K::z), L.zcell(0), q.z[AX]);
  if(AX == 1 ? L.xin : L.xcr) at_st(L.base<1>(K::x), L.xcell(0), q.x[AX]);
}

// per-iz first-derivative weights of the block's rows (irregular z grid), read after the next barrier
template<int R>
__device__ __forceinline__ void plane_weights(float *zct, const TileCoord &c, const IsoArgs &a) {
  if(c.tx) return;
  const float *g = a.zc1 + (size_t)min(c.iz, a.nz - 1) * ZC1_STRIDE;
#pragma unroll
  for(int m = 1; m <= R; m++) zct[m] = g[m];
}
template<int R>
__device__ __forceinline__ float plane_dz(const float *row, const float *zct, bool irr, const IsoArgs &a) {
  float g = 0.f;
  if(irr) {
#pragma unroll
    for(int m = R; m >= 1; m--) g = fmaf(-zct[m], row[-m], g);
#pragma unroll
    for(int m = 1; m <= R; m++) g = fmaf(zct[m], row[m], g);
  } else {
#pragma unroll
    for(int m = R; m >= 1; m--) g = fmaf(-a.cz[m], row[-m], g);
#pragma unroll
    for(int m = 1; m <= R; m++) g = fmaf(a.cz[m], row[m], g);
  }
  return g;
}
template<int R>
__device__ __forceinline__ float plane_dx(const float *row, int pitch, const IsoArgs &a) {
  float g = 0.f;
#pragma unroll
  for(int m = 1; m <= R; m++) {
    g = fmaf(-a.cx[m], row[-m * pitch], g);
    g = fmaf(a.cx[m], row[m * pitch], g);
  }
  return g;
}

template<int R, int MODEL, bool RHO>
__global__ void __launch_bounds__(512) grad_plane_kernel(const float *__restrict__ u, float *__restrict__ px,
                                                         float *__restrict__ pz, const float *__restrict__ eps,
                                                         const float *__restrict__ del, const float *__restrict__ pjx,
                                                         const IsoArgs a) {
  extern __shared__ float s[];
  constexpr int S = TILE_Z + 2 * R;
  const TileCoord c = tile_coord(a);
  const TileOffsets o = tile_offsets<R>(c, a);
  const LayerSlots sl = layer_slots(c, a);
  const LayerOps L(a, sl, 0, c);
  float *row = s + (c.tx + R) * S + c.tz + R, *zct = s + (a.tx + 2 * R) * S + c.tz * (R + 1);
  const bool irr = a.zc1 != nullptr;
  auto body = [&](auto zx_tag) __attribute__((always_inline)) {
    constexpr bool ZX = decltype(zx_tag)::value;
    const __amdgpu_buffer_rsrc_t ru = buf_rsrc(u, (uint32_t)((size_t)a.nx * a.nz * 4));
    const float ctr = buf_ld(ru, o.c, 0), hz0 = buf_ld(ru, o.z0, 0), hz1 = buf_ld(ru, o.z1, 0), hx0 = buf_ld(ru, o.x0, 0),
                hx1 = buf_ld(ru, o.x1, 0);
    float e = 0.f, d = 0.f, ax = 0.f, rho = 1.f;
    if(MODEL != KLRTM_ISO) e = at_ld(eps, L.col), d = at_ld(del, L.col);
    if(MODEL == KLRTM_TTI) ax = at_ld(pjx, L.col);
    if(RHO) rho = at_ld(a.rho, L.col);
    LayerState q;
    L.load<0, ZX, false>(q, 0, FY1, 0);
    L.load<1, ZX, false>(q, 0, FY1, 0);
    row[0] = ctr;
    if(c.tz < R) row[-R] = hz0;
    if(c.tz >= a.tz - R) row[R] = hz1;
    if(c.tx < R) row[-R * S] = hx0;
    if(c.tx >= a.tx - R) row[R * S] = hx1;
    if(irr) plane_weights<R>(zct, c, a);
    lds_barrier();
    float gz = plane_dz<R>(row, zct, irr, a), gx = plane_dx<R>(row, S, a), gy = opaque_zero();
    gz = L.damp<0, ZX, false>(gz, q, FY1, 0);
    gx = L.damp<1, ZX, false>(gx, q, FY1, 0);
    if(RHO) gx /= rho, gz /= rho;
    if(MODEL == KLRTM_VTI) scalar_vti(e, d, gx, gy, gz);
    else if(MODEL == KLRTM_TTI) scalar_tti(e, d, ax, opaque_zero(), gx, gy, gz);
    if(c.act) at_st(px, L.col, gx), at_st(pz, L.col, gz);
    plane_store<0, ZX>(L, q);
    plane_store<1, ZX>(L, q);
  };
  if(sl.any) body(std::true_type());
  else body(std::false_type());
}

template<int R, int MODE, bool RHO>
__global__ void __launch_bounds__(512) div_plane_kernel(const float *__restrict__ px, const float *__restrict__ pz,
                                                        const float *__restrict__ w1, float *__restrict__ w0,
                                                        const float *__restrict__ vel, const IsoArgs a) {
  extern __shared__ float s[];
  constexpr int SZ = TILE_Z + 2 * R, SX = TILE_Z;  // row pitches of the z-haloed (pz) and x-haloed (px) tiles
  const TileCoord c = tile_coord(a);
  const TileOffsets o = tile_offsets<R>(c, a);
  const LayerSlots sl = layer_slots(c, a);
  const LayerOps L(a, sl, 1, c);
  float *zrow = s + c.tx * SZ + c.tz + R, *xrow = s + a.tx * SZ + (c.tx + R) * SX + c.tz;
  float *zct = s + a.tx * SZ + (a.tx + 2 * R) * SX + c.tz * (R + 1);
  const bool irr = a.zc1 != nullptr;
  auto body = [&](auto zx_tag) __attribute__((always_inline)) {
    constexpr bool ZX = decltype(zx_tag)::value;
    const uint32_t pbytes = (uint32_t)((size_t)a.nx * a.nz * 4);
    const __amdgpu_buffer_rsrc_t rz = buf_rsrc(pz, pbytes), rx = buf_rsrc(px, pbytes);
    const float cz = buf_ld(rz, o.c, 0), hz0 = buf_ld(rz, o.z0, 0), hz1 = buf_ld(rz, o.z1, 0);
    const float cx = buf_ld(rx, o.c, 0), hx0 = buf_ld(rx, o.x0, 0), hx1 = buf_ld(rx, o.x1, 0);
    const float w00 = at_ld(w0, L.col), v = at_ld(vel, L.col);
    float u = 0.f, rho = 1.f;
    if(MODE == MODE_STEP) u = at_ld(w1, L.col);
    if(RHO) rho = at_ld(a.rho, L.col);
    LayerState q;
    L.load<1, ZX, false>(q, 0, FY1, 0);
    L.load<0, ZX, false>(q, 0, FY1, 0);
    zrow[0] = cz;
    if(c.tz < R) zrow[-R] = hz0;
    if(c.tz >= a.tz - R) zrow[R] = hz1;
    xrow[0] = cx;
    if(c.tx < R) xrow[-R * SX] = hx0;
    if(c.tx >= a.tx - R) xrow[R * SX] = hx1;
    if(irr) plane_weights<R>(zct, c, a);
    lds_barrier();
    float dxv = plane_dx<R>(xrow, SX, a), dzv = plane_dz<R>(zrow, zct, irr, a);
    dxv = L.damp<1, ZX, false>(dxv, q, FY1, 0);
    dzv = L.damp<0, ZX, false>(dzv, q, FY1, 0);
    float w;
    if(RHO) {
      w = fmaf(-(dxv * v), rho, w00);
      w = fmaf(-(dzv * v), rho, w);
    } else {
      w = fmaf(-dxv, v, w00);
      w = fmaf(-dzv, v, w);
    }
    if(MODE == MODE_STEP) w = (u + u) - w;
    if(c.act) at_st(w0, L.col, w);
    plane_store<0, ZX>(L, q);
    plane_store<1, ZX>(L, q);
  };
  if(sl.any) body(std::true_type());
  else body(std::false_type());
}

template<int R, int MODEL>
static int launch_grad_plane_rm(const float *u, float *px, float *pz, const float *eps, const float *del, const float *pjx,
                                IsoArgs a) {
  LaunchTimer tm("fd_grad");
  grid_of(a);
  size_t lds = sizeof(float) * (size_t)(a.tx + 2 * R) * (TILE_Z + 2 * R);
  if(a.zc1) lds += sizeof(float) * (size_t)a.tz * (R + 1);
  const dim3 grid(a.nbz * a.nbx), block(a.tz * a.tx);
  if(a.rho)
    hipLaunchKernelGGL((grad_plane_kernel<R, MODEL, true>), grid, block, lds, stream(), u, px, pz, eps, del, pjx, a);
  else
    hipLaunchKernelGGL((grad_plane_kernel<R, MODEL, false>), grid, block, lds, stream(), u, px, pz, eps, del, pjx, a);
  return check_launch("grad_plane_kernel");
}
template<int R>
static int launch_grad_plane_r(int model, const float *u, float *px, float *pz, const float *eps, const float *del,
                               const float *pjx, const IsoArgs &a) {
  if(model == KLRTM_VTI) return launch_grad_plane_rm<R, KLRTM_VTI>(u, px, pz, eps, del, pjx, a);
  if(model == KLRTM_TTI) return launch_grad_plane_rm<R, KLRTM_TTI>(u, px, pz, eps, del, pjx, a);
  return launch_grad_plane_rm<R, KLRTM_ISO>(u, px, pz, eps, del, pjx, a);
}
int launch_grad_plane(int R, int model, const float *u, float *px, float *pz, const float *eps, const float *del,
                      const float *pjx, const IsoArgs &a) {
  switch(R) {
  case 4: return launch_grad_plane_r<4>(model, u, px, pz, eps, del, pjx, a);
  case 5: return launch_grad_plane_r<5>(model, u, px, pz, eps, del, pjx, a);
  case 6: return launch_grad_plane_r<6>(model, u, px, pz, eps, del, pjx, a);
  case 7: return launch_grad_plane_r<7>(model, u, px, pz, eps, del, pjx, a);
  case 8: return launch_grad_plane_r<8>(model, u, px, pz, eps, del, pjx, a);
  default: set_error("FD half order %d not supported (4..8)", R); return KLRTM_EINVAL;
  }
}

template<int R, int MODE>
static int launch_div_plane_rm(const float *px, const float *pz, const float *w1, float *w0, const float *vel, IsoArgs a) {
  LaunchTimer tm(MODE == MODE_STEP ? "fd_div_step" : "fd_div");
  grid_of(a);
  size_t lds = sizeof(float) * ((size_t)a.tx * (TILE_Z + 2 * R) + (size_t)(a.tx + 2 * R) * TILE_Z);
  if(a.zc1) lds += sizeof(float) * (size_t)a.tz * (R + 1);
  const dim3 grid(a.nbz * a.nbx), block(a.tz * a.tx);
  if(a.rho) hipLaunchKernelGGL((div_plane_kernel<R, MODE, true>), grid, block, lds, stream(), px, pz, w1, w0, vel, a);
  else hipLaunchKernelGGL((div_plane_kernel<R, MODE, false>), grid, block, lds, stream(), px, pz, w1, w0, vel, a);
  return check_launch("div_plane_kernel");
}
template<int R>
static int launch_div_plane_r(int mode, const float *px, const float *pz, const float *w1, float *w0, const float *vel,
                              const IsoArgs &a) {
  return mode == MODE_STEP ? launch_div_plane_rm<R, MODE_STEP>(px, pz, w1, w0, vel, a)
                           : launch_div_plane_rm<R, MODE_KERNEL>(px, pz, w1, w0, vel, a);
}
int launch_div_plane(int R, int mode, const float *px, const float *pz, const float *w1, float *w0, const float *vel,
                     const IsoArgs &a) {
  switch(R) {
  case 4: return launch_div_plane_r<4>(mode, px, pz, w1, w0, vel, a);
  case 5: return launch_div_plane_r<5>(mode, px, pz, w1, w0, vel, a);
  case 6: return launch_div_plane_r<6>(mode, px, pz, w1, w0, vel, a);
  case 7: return launch_div_plane_r<7>(mode, px, pz, w1, w0, vel, a);
  case 8: return launch_div_plane_r<8>(mode, px, pz, w1, w0, vel, a);
  default: set_error("FD half order %d not supported (4..8)", R); return KLRTM_EINVAL;
  }
}

}  // namespace klrtm
