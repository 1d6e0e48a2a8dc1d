// fd_layers.h -- shared parts of the first-derivative form of the FD step (VTI, TTI, and ISO with density) on gfx950.
//
// grad: gradient + PML round 1 + ScalarVTI/ScalarTTI
//       (bgprtm/KernelCPU.cpp:93-119,176-297, bgprtm/FdEngine_fd.cpp:388-470).
// div:  divergence + PML round 2 + pb -= vel*div (+ update2nd).
//
// Both stream along y like the Laplacian step: a block owns a (TZ x TX) tile of the (z,x) plane, keeps the
// 2R+1 y-neighbours of its column in registers and stages the plane's z/x halos in LDS.  They are bound by
// HBM (gradient 8-24 bytes in and 12 out per cell, divergence 24-28 in and 4 out, plus 8 bytes per damped cell
// and component), which takes memory requests in flight and lines read once, not arithmetic.  The first form
// copied one prefetched plane between registers and read the PML state where it was used: two thirds of the
// wave cycles waited for loads.  Here
//  * the loads of plane y+1, PML state included, go out unconditionally before plane y is computed, into the
//    other of two register sets;
//  * the gradient loads halos R planes ahead, with the own column's sample of the same plane, when neighbour
//    blocks load the same lines (R+2 plane tiles in LDS);
//  * LDS pitches are constants (an address register and an add per x tap otherwise), blocks that touch no
//    layer run code without any, and nothing is loaded or stored with the streaming cache policy: a tile's
//    rows end inside 128-byte lines that its z neighbour reads too (VTI 301x277x333: 20 % less time a step).
// MI355X, a whole step before and after: TTI FD16 600x600x400 5.46 -> 3.68 ms (14.6 GB moved at 3.9 TB/s, 7.8 GB
// needed), TTI FD16 300^3 1.19 -> 0.69 ms, VTI FD8 301x277x333 0.96 -> 0.62 ms.
#pragma once
#include "fd_tile.h"
#include "stencil_common.h"
#include <algorithm>
#include <type_traits>

namespace klrtm {

// state of one plane's PML layers: [component slot] of the z, x and y layers
struct LayerState {
  float z[3], x[3], y[3];
};

// One derivative axis' damping: slot k of every layer is the state component that acts on derivative axis
// AX (0 z, 1 x, 2 y).  FdEngine::pml1_{z,x,y}bnd order: the own axis, then the cross axes; component 0 is the
// own axis', 1 and 2 the cross axes' (bgprtm/FdEngine.cpp:301-350).
template<int AX> struct LayerComp;
template<> struct LayerComp<0> { static constexpr int z = 0, x = 1, y = 1; };
template<> struct LayerComp<1> { static constexpr int z = 1, x = 0, y = 2; };
template<> struct LayerComp<2> { static constexpr int z = 2, x = 2, y = 0; };

// a launch-uniform flag that the compiler may not hoist out of the plane loop (it would copy the loop)
__device__ __forceinline__ bool opaque(bool f) {
  int v = __builtin_amdgcn_readfirstlane((int)f);
  asm volatile("" : "+s"(v));
  return v != 0;
}

// one dword at a wave-uniform base plus a 32-bit byte offset (scalar base, vector offset addressing)
__device__ __forceinline__ float at_ld(const float *base, uint32_t off) { return *(const float *)((const char *)base + off); }
__device__ __forceinline__ void at_st(float *base, uint32_t off, float v) { *(float *)((char *)base + off) = v; }

// The damping rounds of one plane for one block.  State is loaded through global accesses (two SGPRs a
// stream where a buffer resource takes four: the resources of nine streams spilled SGPRs into every plane);
// a lane outside the layer loads the layer's first cell, unused, and its stores are masked.
struct LayerOps {
  const IsoArgs &a;
  const LayerSlots &s;
  int round;
  bool cross;               // pml3d: the cross axes damp too
  bool zin, xin, act;       // thread in a z layer, in an x layer, inside the grid
  bool zcr, xcr, acr;       // the same where the cross axes damp
  uint32_t col;  // byte offset of the thread's cell inside a plane (the first cell for inactive threads)
  uint32_t nxz;
  float *any;  // state of some layer, loaded (unused) for an axis without layers
  __device__ __forceinline__ LayerOps(const IsoArgs &a_, const LayerSlots &s_, int round_, const TileCoord &c)
      : a(a_), s(s_), round(round_), cross(a_.pml.pml3d != 0), zin(s_.zin), xin(s_.xin), act(c.act),
        zcr(zin && cross), xcr(xin && cross), acr(c.act && cross), col(c.act ? (uint32_t)c.col * 4u : 0u), nxz((uint32_t)a_.nx * (uint32_t)a_.nz),
        any(nullptr) {
#pragma unroll
    for(int f = 0; f < 6; f++)
      if(!any) any = a_.pml.q[f][round_][0];
  }
  template<int AX3> __device__ __forceinline__ float *base(int comp) const {
    constexpr int f1 = AX3 == 0 ? FZ1 : AX3 == 1 ? FX1 : FY1;
    const int k = cross ? comp : 0;  // without pml3d only component 0 exists; the others are never stored
    float *q = a.pml.q[f1][round][k] ? a.pml.q[f1][round][k] : a.pml.q[f1 + 1][round][k];
    return q ? q : any;
  }
  // (0 outside the layers)
  __device__ __forceinline__ uint32_t zcell(int y) const { return s.zo + (uint32_t)y * s.zs; }
  __device__ __forceinline__ uint32_t xcell(int y) const { return s.xo + (uint32_t)y * s.xs; }
  __device__ __forceinline__ float *yplane(int comp, int fy, int j) const {
    return base<2>(comp) + ((fy == FY2 ? (size_t)s.first[2] : 0) + (size_t)j * nxz);
  }
  template<int AX, bool ZX, bool YL>
  __device__ __forceinline__ void load(LayerState &q, int y, int fy, int j) const {
    typedef LayerComp<AX> K;
    if(ZX) q.z[AX] = at_ld(base<0>(K::z), zcell(y));
    if(ZX) q.x[AX] = at_ld(base<1>(K::x), xcell(y));
    if(YL) q.y[AX] = at_ld(yplane(K::y, fy, j), col);
  }
  template<bool ZX, bool YL>
  __device__ __forceinline__ void store(const LayerState &q, int y, int fy, int j) const {
    if(ZX) {
      if(zin) at_st(base<0>(0), zcell(y), q.z[0]);
      if(zcr) at_st(base<0>(1), zcell(y), q.z[1]), at_st(base<0>(2), zcell(y), q.z[2]);
    }
    if(ZX) {
      if(xin) at_st(base<1>(0), xcell(y), q.x[1]);
      if(xcr) at_st(base<1>(1), xcell(y), q.x[0]), at_st(base<1>(2), xcell(y), q.x[2]);
    }
    if(YL) {
      if(act) at_st(yplane(0, fy, j), col, q.y[2]);
      if(acr) at_st(yplane(1, fy, j), col, q.y[0]), at_st(yplane(2, fy, j), col, q.y[1]);
    }
  }
  __device__ __forceinline__ static float one(float t0, float t1, float t2, float p, float &q) {
    const float qi = t0 * q - t1 * p;
    q = qi;
    return qi + p * t2;
  }
  template<int AX>
  __device__ __forceinline__ float zlayer(float p, LayerState &q) const {
    constexpr int k = AX == 0 ? 0 : 1;
    const float r = one(s.zc[k][0], s.zc[k][1], s.zc[k][2], p, q.z[AX]);
    return (AX == 0 ? zin : zcr) ? r : p;
  }
  template<int AX>
  __device__ __forceinline__ float xlayer(float p, LayerState &q) const {
    constexpr int k = AX == 1 ? 0 : 1;
    const float r = one(s.xc[k][0], s.xc[k][1], s.xc[k][2], p, q.x[AX]);
    return (AX == 1 ? xin : xcr) ? r : p;
  }
  template<int AX>
  __device__ __forceinline__ float ylayer(float p, LayerState &q, int fy, int j) const {
    const cfloat *t = (const cfloat *)a.pml.abc[fy][AX == 2 ? 0 : 1] + 3 * j;
    const float r = one(t[0], t[1], t[2], p, q.y[AX]);
    return AX == 2 || cross ? r : p;
  }
  template<int AX, bool ZX, bool YL>
  __device__ __forceinline__ float damp(float p, LayerState &q, int fy, int j) const {
    if(AX == 0) {
      if(ZX) p = zlayer<AX>(p, q);
      if(ZX) p = xlayer<AX>(p, q);
      if(YL) p = ylayer<AX>(p, q, fy, j);
    } else if(AX == 1) {
      if(ZX) p = xlayer<AX>(p, q);
      if(ZX) p = zlayer<AX>(p, q);
      if(YL) p = ylayer<AX>(p, q, fy, j);
    } else {
      if(YL) p = ylayer<AX>(p, q, fy, j);
      if(ZX) p = zlayer<AX>(p, q);
      if(ZX) p = xlayer<AX>(p, q);
    }
    return p;
  }
};

// Runs body(plane set, y) over the planes of one y segment: the loads of plane y+1 go out before plane y is
// computed, into the other of two register sets (at the segment end the last plane is fetched again, unused).
template<class Plane, class Fetch, class Body>
__device__ __forceinline__ void stream_planes(int ya, int yb, const Fetch &fetch, const Body &body) {
  Plane A{}, B{};
  fetch(A, ya);
  for(int y = ya;;) {
    fetch(B, min(y + 1, yb - 1)), body(A, y);
    if(++y >= yb) break;
    fetch(A, min(y + 1, yb - 1)), body(B, y);
    if(++y >= yb) break;
  }
}

// The y segments of a block, layer 1 [0, wy1), interior, layer 2 [ny - wy2, ny): seg(z/x layer tag, y layer tag,
// first plane, end, y face, first plane of the layer) for each that is not empty.  A block that touches no z or
// x layer runs code without them.  (Written out: in a loop over the segments the compiler keeps the registers
// of all variants alive.)
template<class Seg>
__device__ __forceinline__ void run_segments(const TileCoord &c, const IsoArgs &a, bool zx, const Seg &seg) {
  const PmlDesc &P = a.pml;
  const int wy1 = (a.has_pml && P.q[FY1][0][0]) ? P.w[FY1] : 0;
  const int wy2 = (a.has_pml && P.q[FY2][0][0]) ? P.w[FY2] : 0;
  const int s1e = min(c.y1, max(c.y0, wy1)), s3b = max(s1e, min(c.y1, a.ny - wy2));
  auto run = [&](auto zxt) __attribute__((always_inline)) {
    if(c.y0 < s1e) seg(zxt, std::true_type(), c.y0, s1e, FY1, 0);
    if(s1e < s3b) seg(zxt, std::false_type(), s1e, s3b, FY1, 0);
    if(s3b < c.y1) seg(zxt, std::true_type(), s3b, c.y1, FY2, a.ny - wy2);
  };
  if(zx) run(std::true_type());
  else run(std::false_type());
}

}  // namespace klrtm
