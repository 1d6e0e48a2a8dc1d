// convae.hip -- learned snapshot compressor: a 3D convolutional autoencoder on 32^3 blocks.
//
// Replaces the source-wavefield compression of bgprtm's snapshot cache
// (WaveFieldCompress, bgprtm/WaveFieldCompress.cpp:25-279, called from
// bgprtm/Propagator.cpp:1233-1243) by an autoencoder trained on snapshots the
// propagator itself generates; WaveFieldCompress stays the fallback.  A 32^3
// block is divided by its scale s = rms(block) + floor * rms(volume) and
// encoded by four 3x3x3 convolutions
//   1 -> 16 (stride 2, 16^3), 16 -> 32 (stride 2, 8^3), 32 -> 32, 32 -> 4
// to a 4 x 8^3 latent (2048 values: 16x fewer than the block) stored as BF16
// with s in FP32, and decoded by four more
//   4 -> 32, nearest x2 + 32 -> 32 (16^3), nearest x2 + 32 -> 16 (32^3), 16 -> 1,
// with GELU after every layer except the latent and the output.  Zero padding
// at every grid edge; block cells outside the volume are zero.
//
// Tensors are channels-last, [block][position][channel] in FP32, position
// p = (iy*D + ix)*D + iz on a layer's D^3 grid.  Every convolution -- forward,
// data gradient and weight gradient -- is an implicit GEMM on the matrix cores,
// v_mfma_f32_32x32x16_bf16 (BF16 operands rounded from the FP32 tensors and
// weights, FP32 accumulation).  Operand layouts of that instruction (lane l):
//   A: A[l % 32][(l / 32)*8 + t]   B: B[(l / 32)*8 + t][l % 32]   (t < 8)
//   C: register r holds C[(r / 4)*8 + (l / 32)*4 + r % 4][l % 32]
// Forward and data gradient: M = 32 output positions of one block, N = 32
// output channels (padded), K = 27 taps x gathered channels, the A operand
// gathered from the input tensor per tap (im2col on the fly, zero outside the
// grid), the B operand from weights pre-arranged in fragment order after every
// update; the upsampling layers' and the output layer's forward have kernels of
// their own (cae_up_kernel, cae_last_kernel).  Weight gradient: M = 16 output
// channels, N = 16 input channels (or taps), K = 32 positions, on
// v_mfma_f32_16x16x32_bf16 from operands transposed into LDS as runs of 8
// positions; partial sums of the workgroups are added in a fixed order
// (cae_wgrad_up_kernel, cae_wgrad_vec_kernel, cae_wgrad_tile_kernel).
// Training minimises the mean squared reconstruction error with Adam.
#include "klrtm_internal.h"
#include "convae.h"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <type_traits>
#include <vector>

namespace klrtm {

typedef __bf16 cae_bf16x8 __attribute__((ext_vector_type(8)));
typedef float cae_f32x16 __attribute__((ext_vector_type(16)));

// layer table: input / output channels, input / output grid side, kind, GELU after
enum { K_SAME = 0, K_DOWN = 1, K_UP = 2 };
static const int kCin[CAE_LAYERS] = {1, 16, 32, 32, 4, 32, 32, 16};
static const int kCout[CAE_LAYERS] = {16, 32, 32, 4, 32, 32, 16, 1};
static const int kDin[CAE_LAYERS] = {32, 16, 8, 8, 8, 8, 16, 32};
static const int kDout[CAE_LAYERS] = {16, 8, 8, 8, 8, 16, 32, 32};
static const int kKind[CAE_LAYERS] = {K_DOWN, K_DOWN, K_SAME, K_SAME, K_SAME, K_UP, K_UP, K_SAME};
static const int kGelu[CAE_LAYERS] = {1, 1, 1, 0, 1, 1, 1, 0};

// gather modes of the implicit GEMM: the gathered-tensor cell q of output position p and tap offset d
// (per axis), on grids of side Dout (GEMM output) and Dg (gathered tensor)
enum { G_SAME = 0, G_DOWN = 1, G_BSAME = 2, G_BDOWN = 3 };

__device__ __forceinline__ int gather1(int mode, int p, int d, int Dout, int Dg) {
  int q;
  switch(mode) {
  case G_SAME: q = p + d; break;                                   // y[p] += w[d] x[p + d]
  case G_DOWN: q = 2 * p + d; break;                               // y[p] += w[d] x[2p + d]
  case G_BSAME: q = p - d; break;                                  // dx[p] += w[d]^T dy[p - d]
  default: q = p - d; return q >= 0 && !(q & 1) && (q >> 1) < Dg ? q >> 1 : -1;  // dx[p] += w[d]^T dy[(p - d)/2]
  }
  return q >= 0 && q < Dg ? q : -1;
}

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
  return 0.5f * (1.f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

enum { E_FWD = 0, E_BWD = 1, E_PLAIN = 2 };

__global__ void cae_zero_kernel(float *__restrict__ p, size_t n) {
  for(size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0.f;
}
static void cae_zero(float *p, size_t n) {
  hipLaunchKernelGGL(cae_zero_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096)), dim3(256), 0, stream(), p, n);
}

// out[b][p][n] (n < nout) = sum_{tap, c} B[(tap, c)][n] * G[b][q(p, tap)][c]; E_FWD adds the bias, keeps
// the pre-activation in z (when set) and stores act(v) in out; E_BWD multiplies by gelu'(zg[b][p][n])
// when zg is set (the gradient through the previous layer's GELU); E_PLAIN stores v.
template<int CG, int MODE, int EPI>
__global__ void __launch_bounds__(256) cae_conv_kernel(const float *__restrict__ G, const cae_bf16x8 *__restrict__ wf,
                                                       int ks, int nout, int lgo, int lgg, const float *__restrict__ bias,
                                                       int act, float *__restrict__ z, float *__restrict__ out,
                                                       const float *__restrict__ zg) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int Dout = 1 << lgo, Dg = 1 << lgg;
  const long Pout = 1L << (3 * lgo), Pg = 1L << (3 * lgg);
  const long p0 = ((long)blockIdx.x * 4 + wv) * 32;
  const long b = blockIdx.y;
  if(p0 >= Pout) return;
  const long p = p0 + (lane & 31);
  const int pz = (int)(p & (Dout - 1)), px = (int)((p >> lgo) & (Dout - 1)), py = (int)(p >> (2 * lgo));
  const int half = lane >> 5;
  const float *Gb = G + (size_t)b * Pg * CG;
  cae_f32x16 acc = {};
  for(int s = 0; s < ks; s++) {
    cae_bf16x8 a;
    const int k0 = s * 16 + half * 8;
    if(CG >= 16) {
      const int tap = k0 / CG, c0 = k0 - tap * CG;
      long q = -1;
      if(tap < 27) {
        const int qy = gather1(MODE, py, tap / 9 - 1, Dout, Dg), qx = gather1(MODE, px, (tap / 3) % 3 - 1, Dout, Dg),
                  qz = gather1(MODE, pz, tap % 3 - 1, Dout, Dg);
        if(qy >= 0 && qx >= 0 && qz >= 0) q = ((((long)qy << lgg) + qx) << lgg) + qz;
      }
      float4 v0 = {0.f, 0.f, 0.f, 0.f}, v1 = {0.f, 0.f, 0.f, 0.f};
      if(q >= 0) {
        const float4 *src = (const float4 *)(Gb + q * CG + c0);
        v0 = src[0], v1 = src[1];
      }
      a[0] = (__bf16)v0.x, a[1] = (__bf16)v0.y, a[2] = (__bf16)v0.z, a[3] = (__bf16)v0.w;
      a[4] = (__bf16)v1.x, a[5] = (__bf16)v1.y, a[6] = (__bf16)v1.z, a[7] = (__bf16)v1.w;
    } else {
#pragma unroll
      for(int t = 0; t < 8; t++) {
        const int k = k0 + t, tap = k / CG, c = k - tap * CG;
        float v = 0.f;
        if(tap < 27) {
          const int qy = gather1(MODE, py, tap / 9 - 1, Dout, Dg), qx = gather1(MODE, px, (tap / 3) % 3 - 1, Dout, Dg),
                    qz = gather1(MODE, pz, tap % 3 - 1, Dout, Dg);
          if(qy >= 0 && qx >= 0 && qz >= 0) v = Gb[(((((long)qy << lgg) + qx) << lgg) + qz) * CG + c];
        }
        a[t] = (__bf16)v;
      }
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, wf[(size_t)s * 64 + lane], acc, 0, 0, 0);
  }
  const int n = lane & 31;
  if(n >= nout) return;
  const float bn = EPI == E_FWD ? bias[n] : 0.f;
#pragma unroll
  for(int r = 0; r < 16; r++) {
    const long pp = p0 + (r >> 2) * 8 + half * 4 + (r & 3);
    const size_t o = ((size_t)b * Pout + pp) * nout + n;
    float v = acc[r];
    if(EPI == E_FWD) {
      v = v + bn;
      if(z) z[o] = v;
      out[o] = act ? gelu(v) : v;
    } else if(EPI == E_BWD) {
      out[o] = zg ? v * gelu_grad(zg[o]) : v;
    } else {
      out[o] = v;
    }
  }
}

// ---- nearest x2 upsampling + 3x3x3 convolution, 32 -> COUT channels -----------------------------------
//
// A fine cell f = 2i + a (phase a in {0,1}^3) sees, along each axis, the coarse cells i + t + a - 1 with t = 0 or 1:
// tap d in {0, 1, 2} falls on t = (d > a).  Its 27 products are added in tap order, one v_mfma_f32_16x16x32_bf16 (a
// tap's 32 channels) each: the same bits as two v_mfma_f32_32x32x16_bf16 a tap, the steps of the implicit GEMM.
// (Sums of the weights that share a coarse cell would take 8 products instead of 27, but they do not fit BF16: one
// rounded term moved a decoded volume by 0.8 %, two terms lose 2^-17 of each sum.)
// One workgroup owns TY x TX x Dc coarse cells, staged with their halo as BF16 in LDS (pitch 80 bytes a cell: the
// 16 cells of a fragment read fall on distinct banks).  A wave keeps the 27 weight fragments of 16 output channels in
// registers while it walks the tile's cells for one ay, one ax after the other, and forms both az at once: of a row
// of taps it reads six coarse fragments and uses each for up to four of the 18 products.
// 128 blocks: 178 us for layer 6 (46 us the matrix products, about 80 the vector instructions of 67 M exact GELUs,
// 268 MB written) and 45 us for layer 5; gathering the taps per fine cell from L2, as the other layers do, the two
// took 1364 us.
// Operand layouts (lane l):
//   A: A[l % 16][(l / 16)*8 + t]   B: B[(l / 16)*8 + t][l % 16]   C: register r holds C[(l / 16)*4 + r][l % 16]
typedef float cae_f32x4 __attribute__((ext_vector_type(4)));
constexpr int CAE_UP_TY = 2, CAE_UP_TX = 8, CAE_UP_PITCH = 80;

template<int COUT, int LGD>
__global__ void __launch_bounds__(256, 2) cae_up_kernel(const float *__restrict__ X, const cae_bf16x8 *__restrict__ wu,
                                                        const float *__restrict__ bias, float *__restrict__ z,
                                                        float *__restrict__ out) {
  constexpr int Dc = 1 << LGD, Df = 2 * Dc, TY = CAE_UP_TY, TX = CAE_UP_TX;
  constexpr int SZ = Dc + 2, SX = (TX + 2) * SZ, CELLS = (TY + 2) * SX;  // LDS strides in cells
  constexpr int NXT = Dc / TX, NYT = Dc / TY;
  __shared__ __attribute__((aligned(16))) char lds[CELLS * CAE_UP_PITCH];
  const int tile = blockIdx.x, y0 = (tile / NXT) * TY, x0 = (tile % NXT) * TX;
  static_assert(NYT * TY == Dc && NXT * TX == Dc, "whole tiles");
  const size_t b = blockIdx.y;
  const float *Xb = X + b * ((size_t)32 << (3 * LGD));
  // stage the tile: four channels per thread and step, eight steps' loads in flight
  typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
  constexpr int U = 8;
  for(int e0 = threadIdx.x; e0 < CELLS * 8; e0 += 256 * U) {
    float4 v[U];
#pragma unroll
    for(int u = 0; u < U; u++) {
      const int e = e0 + 256 * u, cell = e >> 3, c4 = (e & 7) * 4;
      const int ly = cell / SX, r = cell - ly * SX, lx = r / SZ, lz = r - lx * SZ;
      const int y = y0 + ly - 1, x = x0 + lx - 1, zz = lz - 1;
      v[u] = float4{0.f, 0.f, 0.f, 0.f};
      if(e < CELLS * 8 && (unsigned)y < (unsigned)Dc && (unsigned)x < (unsigned)Dc && (unsigned)zz < (unsigned)Dc)
        v[u] = *(const float4 *)(Xb + (size_t)(((y << LGD) + x) << LGD) * 32 + zz * 32 + c4);
    }
#pragma unroll
    for(int u = 0; u < U; u++) {
      const int e = e0 + 256 * u;
      bf4 h;
      h[0] = (__bf16)v[u].x, h[1] = (__bf16)v[u].y, h[2] = (__bf16)v[u].z, h[3] = (__bf16)v[u].w;
      if(e < CELLS * 8) *(bf4 *)(lds + (e >> 3) * CAE_UP_PITCH + (e & 7) * 8) = h;
    }
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, n = lane & 15;
  // wave = (ay, half of the channels) of 32 channels, (ay, every second row of cells) of 16
  constexpr int NT = COUT / 16, RPM = Dc == 8 ? 2 : 1, MT = TY * TX / RPM;  // 16 cells: one row of 16 or two of 8
  const int ay = w & 1, h = NT == 2 ? w >> 1 : 0;
  cae_bf16x8 B[27];
#pragma unroll
  for(int t = 0; t < 27; t++) B[t] = wu[(t * NT + h) * 64 + lane];
  const float bn = bias[h * 16 + n];
  // a workgroup of several for a tile takes one ax and every (parts / 2)-th of the wave's rows
  const int parts = gridDim.z, part = blockIdx.z, rs = parts > 2 ? parts >> 1 : 1;
  const int m0 = (NT == 2 ? 0 : w >> 1) + (3 - NT) * (part >> 1), dm = (3 - NT) * rs;
  __syncthreads();
  auto phases = [&](auto ax_tag) __attribute__((always_inline)) {
    constexpr int ax = decltype(ax_tag)::value;
    for(int m = m0; m < MT; m += dm) {
      const int row = m * RPM + (Dc == 8 ? n >> 3 : 0), ly = row / TX, lx = row % TX, lz = n & (Dc - 1);
      const char *base = lds + ((ly + ay) * SX + (lx + ax) * SZ + lz) * CAE_UP_PITCH + q * 16;
      cae_f32x4 acc[2] = {};
#pragma unroll
      for(int dy = 0; dy < 3; dy++) {
        const char *by = base + (dy == 0 || (dy == 1 && ay) ? 0 : SX * CAE_UP_PITCH);
        cae_bf16x8 A[2][3];  // coarse x offset t, z offset - 1
#pragma unroll
        for(int t = 0; t < 2; t++)
#pragma unroll
          for(int o = 0; o < 3; o++) A[t][o] = *(const cae_bf16x8 *)(by + (t * SZ + o) * CAE_UP_PITCH);
#pragma unroll
        for(int dx = 0; dx < 3; dx++)
#pragma unroll
          for(int dz = 0; dz < 3; dz++)
#pragma unroll
            for(int az = 0; az < 2; az++)
              acc[az] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[dx > ax][(dz > az) + az], B[(dy * 3 + dx) * 3 + dz],
                                                                acc[az], 0, 0, 0);
      }
#pragma unroll
      for(int r = 0; r < 4; r++) {
        const int mr = q * 4 + r, rr = m * RPM + (Dc == 8 ? mr >> 3 : 0);
        const int cy = y0 + rr / TX, cx = x0 + rr % TX, cz = mr & (Dc - 1);
#pragma unroll
        for(int az = 0; az < 2; az++) {
          const size_t f = ((size_t)(2 * cy + ay) * Df + (2 * cx + ax)) * Df + (2 * cz + az);
          const size_t o = (b * ((size_t)1 << (3 * LGD + 3)) + f) * COUT + h * 16 + n;
          const float v = acc[az][r] + bn;
          if(z) z[o] = v;
          out[o] = gelu(v);
        }
      }
    }
  };
  if(parts == 1 || !(part & 1)) phases(std::integral_constant<int, 0>());
  if(parts == 1 || part & 1) phases(std::integral_constant<int, 1>());
}

// weight fragments of an upsampling layer: wu[tap][half of the channels][lane], k = input channel
__global__ void cae_wup_kernel(const float *__restrict__ W, int cout, cae_bf16x8 *__restrict__ wu) {
  const int nt = cout / 16, i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= 27 * nt * 64) return;
  const int l = i & 63, co = (i >> 6) % nt * 16 + (l & 15), tap = (i >> 6) / nt;
  cae_bf16x8 v;
#pragma unroll
  for(int j = 0; j < 8; j++) v[j] = (__bf16)W[((size_t)co * 32 + (l >> 4) * 8 + j) * 27 + tap];
  wu[i] = v;
}

// ---- the output layer: 3x3x3 convolution of 16 channels to one on the 32^3 grid ------------------------
//
// The cells are the columns, 16 along z, and the weights row 0 of the other operand: a v_mfma_f32_16x16x32_bf16 adds
// two taps' channels, in tap order and with the bits of the implicit GEMM's one tap a step (a 28th tap is zero on
// both sides).  15 of 16 rows are padding; sums over each cell's products with all taps, which need none, round
// every tap's product sum to FP32 before it is added.
// 128 blocks: 71 us, bound by the LDS reads (48 us) and the 268 MB read (55 us at the copy rate); as an ordinary
// implicit GEMM, which gathers every cell's channels 27 times from L2, 513 us.
// A workgroup owns 8 rows (and one more on each side) and walks along y with three planes and the next one as BF16
// in LDS, channel halves apart: [half][row][z], 16 bytes each, so a fragment read is contiguous.
constexpr int CAE_LT = 14;  // steps of two taps
__global__ void cae_wtap_kernel(const float *__restrict__ W, cae_bf16x8 *__restrict__ wt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= CAE_LT * 64) return;
  const int l = i & 63, q = l >> 4, tap = (i >> 6) * 2 + (q >> 1);
  cae_bf16x8 v;
#pragma unroll
  for(int j = 0; j < 8; j++) v[j] = (__bf16)((l & 15) == 0 && tap < 27 ? W[((q & 1) * 8 + j) * 27 + tap] : 0.f);
  wt[i] = v;
}
__global__ void __launch_bounds__(256) cae_last_kernel(const float *__restrict__ X, const cae_bf16x8 *__restrict__ wt,
                                                       const float *__restrict__ bias, float *__restrict__ out) {
  constexpr int ROWS = 10, SX = 34, HALF = ROWS * SX, PLANE = 2 * HALF;  // in 16-byte units
  __shared__ cae_bf16x8 T[4 * PLANE];                                    // plane y in slot y & 3
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, n = lane & 15;
  const int x0 = (blockIdx.x & 3) * 8, planes = 128 / gridDim.x, y0 = (blockIdx.x >> 2) * planes;
  const size_t b = blockIdx.y;
  const float *Xb = X + b * (32768 * 16);
  cae_bf16x8 W[CAE_LT];
#pragma unroll
  for(int s = 0; s < CAE_LT; s++) W[s] = wt[s * 64 + lane];
  const float b0 = bias[0];
  const cae_bf16x8 zero = {};
  // 640 items a plane: 8 channels of one cell
  constexpr int NI = 3;
  float4 v[NI][2];
  auto load = [&](int y) __attribute__((always_inline)) {
#pragma unroll
    for(int k = 0; k < NI; k++) {
      const int e = tid + k * 256, hf = e & 1, z = (e >> 1) & 31, x = x0 + (e >> 6) - 1;
      v[k][0] = v[k][1] = float4{0.f, 0.f, 0.f, 0.f};
      if(e < ROWS * 64 && (unsigned)x < 32u && (unsigned)y < 32u) {
        const float4 *src = (const float4 *)(Xb + (((size_t)y * 32 + x) * 32 + z) * 16 + hf * 8);
        v[k][0] = src[0], v[k][1] = src[1];
      }
    }
  };
  auto put = [&](int y) __attribute__((always_inline)) {
#pragma unroll
    for(int k = 0; k < NI; k++) {
      const int e = tid + k * 256, hf = e & 1, z = (e >> 1) & 31, r = e >> 6;
      if(e >= ROWS * 64) continue;
      cae_bf16x8 a;
      a[0] = (__bf16)v[k][0].x, a[1] = (__bf16)v[k][0].y, a[2] = (__bf16)v[k][0].z, a[3] = (__bf16)v[k][0].w;
      a[4] = (__bf16)v[k][1].x, a[5] = (__bf16)v[k][1].y, a[6] = (__bf16)v[k][1].z, a[7] = (__bf16)v[k][1].w;
      T[(y & 3) * PLANE + hf * HALF + r * SX + z + 1] = a;
    }
  };
  // the cells beside z = 0 and 31 stay zero
  for(int e = tid; e < 4 * 2 * ROWS * 2; e += 256) T[(e >> 1) * SX + (e & 1) * (SX - 1)] = zero;
  load(y0 - 1), put(y0 - 1);
  load(y0), put(y0);
  load(y0 + 1);
  for(int y = y0; y < y0 + planes; y++) {
    put(y + 1);  // into the slot of plane y - 3, which every wave left before the barrier of y - 1
    if(y + 1 < y0 + planes) load(y + 2);
    __syncthreads();
    // four runs of 16 cells a wave, rows lx, lx + 2, ..: this lane's channel half of cell z0 + n, tap offset (-1, -1, -1)
    const int lx = w >> 1, z0 = (w & 1) * 16;
    const cae_bf16x8 *base = T + (q & 1) * HALF + lx * SX + z0 + n;
    cae_f32x4 acc[4] = {};
    cae_bf16x8 keep[4];  // a pair two rows on is the next run's pair three steps before
#pragma unroll
    for(int s = 0; s < CAE_LT; s++) {
      const bool first = s == 0 || s == 5 || s == 9, again = s == 3 || s == 8 || s == 12;
      const int t0 = 2 * s, t1 = 2 * s + 1;
      auto off = [&](int t) { return ((y + t / 9 - 1) & 3) * PLANE + t / 3 % 3 * SX + t % 3; };
      const cae_bf16x8 *p = base + (q >> 1 && t1 < 27 ? off(t1) : off(t0));
#pragma unroll
      for(int u = 0; u < 4; u++) {
        cae_bf16x8 a = again && u < 3 ? keep[u + 1] : p[2 * u * SX];
        if(first) keep[u] = a;
        if(t1 == 27) a = q >> 1 ? zero : a;
        acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W[s], a, acc[u], 0, 0, 0);
      }
    }
    if(lane < 16) {
#pragma unroll
      for(int u = 0; u < 4; u++) out[b * 32768 + ((size_t)y * 32 + x0 + lx + 2 * u) * 32 + z0 + lane] = acc[u][0] + b0;
    }
  }
}

// ---- weight gradients of the upsampling layers ---------------------------------------------------------
//
// dW[co][ci][d] = sum over phases a of G[a][t(a, d)][co][ci], where
//   G[a][t][co][ci] = sum_i dZ[2i + a][co] X[i + t + a - 1][ci]
// runs over coarse cells i: 64 products a coarse cell instead of 8 * 27, with the same BF16 operands and FP32 sums.
// K = positions, so both operands lie in LDS as runs of 8 z positions of one channel: chunk[row][z / 8][channel],
// X three times, shifted by -1, 0, +1 in z, dZ split by phase.  Rows of a fragment's 16 channels are 256 contiguous
// bytes.  A workgroup walks tiles of TY x TX coarse rows; the next tile's loads are in flight during the products.
// Wave = (ay, ax, half of the input channels): 16 accumulators, 14 LDS reads for 16 products.  blockIdx.y = 16 output
// channels.  Sums of a workgroup go to its slot of `part`; cae_wred_kernel and cae_wup_sum_kernel add them in a fixed
// order.
constexpr int CAE_UPG = 64 * 16 * 32;  // products of one workgroup

template<int COUT, int LGD>
__global__ void __launch_bounds__(512) cae_wgrad_up_kernel(const float *__restrict__ X, const float *__restrict__ dZ,
                                                           int ntask, float *__restrict__ part) {
  constexpr int Dc = 1 << LGD, Df = 2 * Dc, NCH = Dc / 8, TY = 2, TX = Dc == 8 ? 4 : 2, SX = TX + 2;
  constexpr int HROWS = (TY + 2) * SX, ROWS = TY * TX, KS = ROWS * NCH / 4, NXT = Dc / TX, TILES = NXT * (Dc / TY);
  __shared__ __attribute__((aligned(16))) char xs[3 * HROWS * NCH * 32 * 16], zs[ROWS * 8 * NCH * 16 * 16];
  typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
  const int tid = threadIdx.x, c0 = blockIdx.y * 16;
  // staging: X, one chunk (with one cell more on both ends) of two channels; dZ, eight fine cells of two channels
  const int xc = tid & 15, xch = (tid >> 4) % NCH, xrow = (tid >> 4) / NCH;
  const int zc = tid & 7, zh = (tid >> 3) & 1, zch = (tid >> 4) % NCH, zph = (tid >> 4) / NCH & 3, zrow = (tid >> 4) / NCH >> 2;
  static_assert(HROWS * NCH * 16 <= 512 && ROWS * 4 * NCH * 16 == 512, "one item per thread");
  float2 xv[10], zv[8];
  auto load = [&](int task) __attribute__((always_inline)) {
    const size_t b = task / TILES;
    const int tile = task % TILES, y0 = tile / NXT * TY, x0 = tile % NXT * TX;
    const int y = y0 + xrow / SX - 1, x = x0 + xrow % SX - 1;
    const bool in = xrow < HROWS && (unsigned)y < (unsigned)Dc && (unsigned)x < (unsigned)Dc;
    const float *sx = X + ((b << (3 * LGD)) + (size_t)(((y << LGD) + x) << LGD) + xch * 8) * 32 + xc * 2;
#pragma unroll
    for(int k = 0; k < 10; k++) {
      const bool ok = in && (k > 0 || xch > 0) && (k < 9 || xch < NCH - 1);
      xv[k] = float2{0.f, 0.f};
      if(ok) xv[k] = *(const float2 *)(sx + (k - 1) * 32);
    }
    const int fy = 2 * (y0 + zrow / TX) + (zph >> 1), fx = 2 * (x0 + zrow % TX) + (zph & 1);
    const float *sz = dZ + ((b << (3 * LGD + 3)) + (size_t)(fy * Df + fx) * Df + zch * 16 + zh * 8) * COUT + c0 + zc * 2;
#pragma unroll
    for(int k = 0; k < 8; k++) zv[k] = *(const float2 *)(sz + k * COUT);
  };
  const int lane = tid & 63, w = tid >> 6, q = lane >> 4, n = lane & 15;
  const int ay = w >> 2, ax = (w >> 1) & 1, h = w & 1;
  cae_f32x4 acc[2][8] = {};
  int task = blockIdx.x;
  load(task);
  while(task < ntask) {
    __syncthreads();  // the previous tile's products are done with the chunks
    if(xrow < HROWS) {
#pragma unroll
      for(int o = 0; o < 3; o++) {
        cae_bf16x8 u, v;
#pragma unroll
        for(int k = 0; k < 8; k++) u[k] = (__bf16)xv[o + k].x, v[k] = (__bf16)xv[o + k].y;
        char *d = xs + (((o * HROWS + xrow) * NCH + xch) * 32 + xc * 2) * 16;
        *(cae_bf16x8 *)d = u, *(cae_bf16x8 *)(d + 16) = v;
      }
    }
#pragma unroll
    for(int az = 0; az < 2; az++) {
      bf4 u, v;
#pragma unroll
      for(int k = 0; k < 4; k++) u[k] = (__bf16)zv[2 * k + az].x, v[k] = (__bf16)zv[2 * k + az].y;
      char *d = zs + (((zrow * 8 + zph * 2 + az) * NCH + zch) * 16 + zc * 2) * 16 + zh * 8;
      *(bf4 *)d = u, *(bf4 *)(d + 16) = v;
    }
    __syncthreads();
    task += gridDim.x;
    if(task < ntask) load(task);
#pragma unroll
    for(int ks = 0; ks < KS; ks++) {
      // lane quarter q: chunk ks*4 + q of the tile
      const int row = (ks * 4 + q) / NCH, ch = q % NCH, ly = row / TX, lx = row % TX;
      cae_bf16x8 a[2];
#pragma unroll
      for(int az = 0; az < 2; az++)
        a[az] = *(const cae_bf16x8 *)(zs + (((row * 8 + ay * 4 + ax * 2 + az) * NCH + ch) * 16 + n) * 16);
#pragma unroll
      for(int ty = 0; ty < 2; ty++)
#pragma unroll
        for(int tx = 0; tx < 2; tx++)
#pragma unroll
          for(int o = 0; o < 3; o++) {  // z offset o - 1: tap o - az of phase az
            const int hr = (ly + ty + ay) * SX + lx + tx + ax;
            const cae_bf16x8 v = *(const cae_bf16x8 *)(xs + (((o * HROWS + hr) * NCH + ch) * 32 + h * 16 + n) * 16);
#pragma unroll
            for(int az = 0; az < 2; az++) {
              const int t = o - az;
              if(t < 0 || t > 1) continue;
              acc[az][(ty * 2 + tx) * 2 + t] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[az], v, acc[az][(ty * 2 + tx) * 2 + t], 0, 0, 0);
            }
          }
    }
  }
  // part[slot][(a, t)][co][ci]
  float *o = part + (size_t)blockIdx.x * (CAE_UPG / 16 * COUT);
#pragma unroll
  for(int az = 0; az < 2; az++)
#pragma unroll
    for(int t = 0; t < 8; t++)
#pragma unroll
      for(int r = 0; r < 4; r++)
        o[(((ay * 4 + ax * 2 + az) * 8 + t) * COUT + c0 + q * 4 + r) * 32 + h * 16 + n] = acc[az][t][r];
}

// sum of nslot partial results of n values (n a multiple of 32) in a fixed order.  R_PITCH27: value i is
// [i / 32][i % 32] of rows of 27 values in out; R_TAPS: [tap][pair] of n / 27 pairs, out is [pair][tap].
enum { R_PLAIN = 0, R_PITCH27 = 1, R_TAPS = 2 };
template<int MODE>
__global__ void __launch_bounds__(256) cae_wred_kernel(const float *__restrict__ part, int nslot, int n,
                                                       float *__restrict__ out) {
  __shared__ float s[256];
  const int l = threadIdx.x & 31, g = threadIdx.x >> 5, i = blockIdx.x * 32 + l;
  float v = 0.f;
#pragma unroll 8
  for(int k = g; k < nslot; k += 8) v += part[(size_t)k * n + i];
  s[threadIdx.x] = v;
  __syncthreads();
  if(g) return;
#pragma unroll
  for(int k = 1; k < 8; k++) v += s[k * 32 + l];
  if(MODE == R_PLAIN) out[i] = v;
  else if(MODE == R_TAPS) out[i % (n / 27) * 27 + i / (n / 27)] = v;
  else if(l < 27) out[blockIdx.x * 27 + l] = v;
}

// dW[co][ci][tap] from G[(a, t)][co][ci]
__global__ void cae_wup_sum_kernel(const float *__restrict__ G, int cout, float *__restrict__ dW) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= cout * 32 * 27) return;
  const int tap = i % 27, c = i / 27, d[3] = {tap / 9, tap / 3 % 3, tap % 3};
  float s = 0.f;
#pragma unroll
  for(int a = 0; a < 8; a++) {
    int t = 0;
    for(int k = 0; k < 3; k++) t = t * 2 + (d[k] > (a >> (2 - k) & 1));
    s += G[(size_t)(a * 8 + t) * cout * 32 + c];
  }
  dW[i] = s;
}

// ---- weight gradients of the layers with one channel on one side ----------------------------------------
//
// 1 -> 16 (stride 2) and 16 -> 1: dW[m][tap] = sum_p V[p][m] S[.][tap] with V the 16-channel tensor on a grid of side
// D and S the 1-channel tensor on the 32^3 grid, at 2p + d (STRIDE 2) or p - d (STRIDE 1).  M = 16 channels, N = 27
// taps in two halves, K = positions.  V is read once, straight into the operand; S lies in LDS three times, at the
// three z offsets, as runs of 8 positions.  A workgroup walks slabs of 4 planes.  `part` as above: [slot][16][32].
// 64 blocks: 8 us and 22 us, the latter for reading 134 MB of V (gathered per tap and padded to 32 channels: 541 us
// and 1450 us).
// (S may be the caller's tensor, aligned to its elements only: the hardware's wide loads accept that)
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
template<int LGP, int STRIDE>
__global__ void __launch_bounds__(256) cae_wgrad_vec_kernel(const float *__restrict__ V, const float *__restrict__ S,
                                                            int ntask, float *__restrict__ part) {
  constexpr int D = 1 << LGP, NCH = D / 8, TY = 4, SLABS = D / TY, RPK = 4 / NCH, W = 8 * STRIDE;
  constexpr int SY = STRIDE * TY + 3 - STRIDE, SX = STRIDE * D + 3 - STRIDE, NR = SY * SX;
  static_assert(STRIDE * D == 32, "S is on the 32^3 grid");
  __shared__ __attribute__((aligned(16))) char ss[3 * NR * NCH * 16];
  static_assert(sizeof(ss) >= 4 * 512 * 4, "holds the waves' sums");
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, n = lane & 15;
  int toff[2];
#pragma unroll
  for(int h = 0; h < 2; h++) {
    const int tap = min(h * 16 + n, 26), dy = tap / 9 - 1, dx = tap / 3 % 3 - 1, dz = tap % 3;
    toff[h] = (dz * NR + (STRIDE == 1 ? (1 - dy) * SX + 1 - dx : (1 + dy) * SX + 1 + dx)) * NCH * 16;
  }
  cae_f32x4 acc[2] = {};
  for(int task = blockIdx.x; task < ntask; task += gridDim.x) {
    const size_t b = task / SLABS;
    const int y0 = task % SLABS * TY;
    const float *Sb = S + b * 32768;
    __syncthreads();  // the previous slab's products are done with S
    for(int e = threadIdx.x; e < NR * NCH; e += 256) {
      const int ch = e % NCH, row = e / NCH, y = y0 * STRIDE + row / SX - 1, x = row % SX - 1;
      float v[W + 2];  // cells ch*W - 1 ...
#pragma unroll
      for(int k = 0; k < W + 2; k++) v[k] = 0.f;
      if((unsigned)y < 32u && (unsigned)x < 32u) {
        const float *src = Sb + (y * 32 + x) * 32 + ch * W;
#pragma unroll
        for(int k = 0; k < W; k += 4) {
          const f4u f = *(const f4u *)(src + k);
          v[k + 1] = f.x, v[k + 2] = f.y, v[k + 3] = f.z, v[k + 4] = f.w;
        }
        if(ch > 0) v[0] = src[-1];
        if(ch < NCH - 1) v[W + 1] = src[W];
      }
#pragma unroll
      for(int o = 0; o < 3; o++) {
        cae_bf16x8 u;
#pragma unroll
        for(int k = 0; k < 8; k++) u[k] = (__bf16)v[STRIDE == 1 ? k + 2 - o : 2 * k + o];
        *(cae_bf16x8 *)(ss + ((o * NR + row) * NCH + ch) * 16) = u;
      }
    }
    __syncthreads();
    const float *Vb = V + ((b << (3 * LGP)) + ((size_t)y0 << (2 * LGP))) * 16;
#pragma unroll 4
    for(int k = 0; k < TY * D / RPK; k += 4) {
      const int row = (k + w) * RPK + q / NCH, ch = q % NCH, ly = row >> LGP, x = row & (D - 1);
      const float *src = Vb + ((row << LGP) + ch * 8) * 16 + n;
      cae_bf16x8 a;
#pragma unroll
      for(int t = 0; t < 8; t++) a[t] = (__bf16)src[t * 16];
      const char *base = ss + ((STRIDE * ly * SX + STRIDE * x) * NCH + ch) * 16;
#pragma unroll
      for(int h = 0; h < 2; h++)
        acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, *(const cae_bf16x8 *)(base + toff[h]), acc[h], 0, 0, 0);
    }
  }
  __syncthreads();
  float *red = (float *)ss;
#pragma unroll
  for(int h = 0; h < 2; h++)
#pragma unroll
    for(int r = 0; r < 4; r++) red[w * 512 + (q * 4 + r) * 32 + h * 16 + n] = acc[h][r];
  __syncthreads();
  for(int i = threadIdx.x; i < 512; i += 256)
    part[(size_t)blockIdx.x * 512 + i] = red[i] + red[512 + i] + red[1024 + i] + red[1536 + i];
}

// ---- weight gradients of the layers on the 8^3 grid ----------------------------------------------------
//
// dW[co][ci][tap] = sum_p dZ[p][co] X[STRIDE*p + d(tap)][ci] over the positions p of the 8^3 output grid.  As in
// cae_wgrad_up_kernel both operands lie in LDS as runs of 8 z positions (here a whole row) of one channel, X three
// times at the three z offsets.  A workgroup walks tiles of two planes; a wave owns 16 output channels, 16 input
// channels and NT taps.  Columns past CIN and rows past COUT repeat the last channel and are not stored.
// `part` is [slot][tap][co][ci].  64 blocks, one tile a workgroup: 12 us for 32 -> 32 and 10 us for 16 -> 32, bound by
// the latency of one load, two barriers and the store of 108 KB of sums (32 taps and channels gathered per position from
// L2 and added with atomics: 155 and 145 us).
template<int CIN, int COUT, int STRIDE>
__global__ void __launch_bounds__(512) cae_wgrad_tile_kernel(const float *__restrict__ X, const float *__restrict__ dZ,
                                                             int ntask, float *__restrict__ part) {
  constexpr int NI = (CIN + 15) / 16, NO = (COUT + 15) / 16, TG = 8 / (NI * NO), NT = (27 + TG - 1) / TG;
  constexpr int DG = 8 * STRIDE, HX = STRIDE * 8 + 3 - STRIDE, HR = (STRIDE * 2 + 3 - STRIDE) * HX;
  __shared__ __attribute__((aligned(16))) char xs[3 * HR * CIN * 16], zs[16 * COUT * 16];
  const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, n = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), h = w % NI, c = w / NI % NO, g = w / (NI * NO);
  int toff[NT];
#pragma unroll
  for(int i = 0; i < NT; i++) {
    const int tap = min(g * NT + i, 26), dy = tap / 9, dx = tap / 3 % 3, dz = tap % 3;
    toff[i] = (dz * HR + dy * HX + dx) * CIN * 16;
  }
  const int ca = min(c * 16 + n, COUT - 1), cb = min(h * 16 + n, CIN - 1);
  cae_f32x4 acc[NT] = {};
  for(int task = blockIdx.x; task < ntask; task += gridDim.x) {
    const size_t b = task >> 2;
    const int y0 = (task & 3) * 2;
    __syncthreads();  // the previous tile's products are done with the rows
    for(int e = tid; e < HR * (CIN / 2); e += 512) {
      const int cp = e % (CIN / 2), row = e / (CIN / 2), y = STRIDE * y0 + row / HX - 1, x = row % HX - 1;
      const bool in = (unsigned)y < (unsigned)DG && (unsigned)x < (unsigned)DG;
      const float *src = X + ((b * DG + (in ? y : 0)) * DG + (in ? x : 0)) * DG * CIN + cp * 2;
      float2 v[DG];
#pragma unroll
      for(int k = 0; k < DG; k++) {
        v[k] = *(const float2 *)(src + k * CIN);
        if(!in) v[k] = float2{0.f, 0.f};
      }
#pragma unroll
      for(int o = 0; o < 3; o++) {
        cae_bf16x8 s0, s1;
#pragma unroll
        for(int k = 0; k < 8; k++) {
          const int z = STRIDE * k + o - 1;
          const float2 f = z >= 0 && z < DG ? v[z < 0 ? 0 : z >= DG ? DG - 1 : z] : float2{0.f, 0.f};
          s0[k] = (__bf16)f.x, s1[k] = (__bf16)f.y;
        }
        char *d = xs + ((o * HR + row) * CIN + cp * 2) * 16;
        *(cae_bf16x8 *)d = s0, *(cae_bf16x8 *)(d + 16) = s1;
      }
    }
    for(int e = tid; e < 16 * (COUT / 2); e += 512) {
      const int cp = e % (COUT / 2), row = e / (COUT / 2);
      const float *src = dZ + ((b * 64 + y0 * 8 + row) * 8) * COUT + cp * 2;
      cae_bf16x8 s0, s1;
#pragma unroll
      for(int k = 0; k < 8; k++) {
        const float2 f = *(const float2 *)(src + k * COUT);
        s0[k] = (__bf16)f.x, s1[k] = (__bf16)f.y;
      }
      char *d = zs + (row * COUT + cp * 2) * 16;
      *(cae_bf16x8 *)d = s0, *(cae_bf16x8 *)(d + 16) = s1;
    }
    __syncthreads();
#pragma unroll
    for(int ks = 0; ks < 4; ks++) {
      const int row = ks * 4 + q, ly = row >> 3, lx = row & 7;
      const cae_bf16x8 a = *(const cae_bf16x8 *)(zs + (row * COUT + ca) * 16);
      const char *base = xs + ((STRIDE * ly * HX + STRIDE * lx) * CIN + cb) * 16;
#pragma unroll
      for(int i = 0; i < NT; i++)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, *(const cae_bf16x8 *)(base + toff[i]), acc[i], 0, 0, 0);
    }
  }
  float *o = part + (size_t)blockIdx.x * (27 * COUT * CIN);
  const int ci = h * 16 + n;
#pragma unroll
  for(int i = 0; i < NT; i++)
#pragma unroll
    for(int r = 0; r < 4; r++) {
      const int co = c * 16 + q * 4 + r;
      if(g * NT + i < 27 && co < COUT && ci < CIN) o[((g * NT + i) * COUT + co) * CIN + ci] = acc[i][r];
    }
}

// db[c] += sum over a chunk of positions of dZ[b][p][c]
__global__ void cae_bgrad_kernel(const float *__restrict__ dZ, long n, int cout, float *__restrict__ db) {
  __shared__ float s[32];
  if(threadIdx.x < 32) s[threadIdx.x] = 0.f;
  __syncthreads();
  const long e0 = (long)blockIdx.x * 8192;
  float acc = 0.f;
  int c = -1;
  // cout divides 256: a thread's elements share one channel
  for(long e = e0 + threadIdx.x; e < e0 + 8192 && e < n; e += 256) acc += dZ[e], c = (int)(e % cout);
  if(c >= 0) atomicAdd(&s[c], acc);
  __syncthreads();
  if(threadIdx.x < cout) atomicAdd(&db[threadIdx.x], s[threadIdx.x]);
}

// dX[b][q][c] = (sum of dU over the 8 fine cells of coarse cell q) * gelu'(zg[b][q][c]) (zg optional):
// the data gradient of nearest x2 upsampling
__global__ void cae_downsum_kernel(const float *__restrict__ dU, int C, int lgc, const float *__restrict__ zg,
                                   float *__restrict__ dX, long total) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= total) return;
  const int c = (int)(i % C);
  const long cell = i / C;
  const long Pc = 1L << (3 * lgc);
  const long b = cell / Pc, q = cell - b * Pc;
  const int Dc = 1 << lgc, lgf = lgc + 1;
  const int qz = (int)(q & (Dc - 1)), qx = (int)((q >> lgc) & (Dc - 1)), qy = (int)(q >> (2 * lgc));
  const float *U = dU + (size_t)b * (Pc << 3) * C;
  float s = 0.f;
#pragma unroll
  for(int e = 0; e < 8; e++) {
    const long f = ((((long)(2 * qy + (e >> 2)) << lgf) + (2 * qx + ((e >> 1) & 1))) << lgf) + 2 * qz + (e & 1);
    s += U[f * C + c];
  }
  dX[i] = zg ? s * gelu_grad(zg[i]) : s;
}

// loss: d = y - x, dY = 2 d / n, sum d^2 into *loss
__global__ void cae_mse_kernel(const float *__restrict__ y, const float *__restrict__ x, long n, float inv_n,
                               float *__restrict__ dy, float *__restrict__ loss) {
  __shared__ float s[256];
  float acc = 0.f;
  for(long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
    const float d = y[i] - x[i];
    dy[i] = 2.f * d * inv_n;
    acc += d * d;
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1) {
    if(threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if(threadIdx.x == 0) atomicAdd(loss, s[0] * inv_n);
}

__global__ void cae_adam_kernel(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                                float *__restrict__ v, long n, float lr, float b1, float b2, float c1, float c2,
                                float eps) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi, vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi, v[i] = vi;
  p[i] = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// weight fragments of one layer: forward B[(tap, ci)][co], backward B[(tap, co)][ci], W[co][ci][tap]
__global__ void cae_wfrag_kernel(const float *__restrict__ W, int cin, int cout, int ksf, int ksb,
                                 cae_bf16x8 *__restrict__ wf, cae_bf16x8 *__restrict__ wb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int nf = ksf * 64, nb = ksb * 64;
  if(i >= nf + nb) return;
  const bool fwd = i < nf;
  const int j = fwd ? i : i - nf, s = j / 64, l = j % 64, nn = l & 31;
  const int g = fwd ? cin : cout;  // channels of the gathered tensor
  cae_bf16x8 v;
#pragma unroll
  for(int t = 0; t < 8; t++) {
    const int k = s * 16 + (l >> 5) * 8 + t, tap = k / g, c = k - tap * g;
    float w = 0.f;
    if(tap < 27) {
      const int co = fwd ? nn : c, ci = fwd ? c : nn;
      if(co < cout && ci < cin) w = W[((size_t)co * cin + ci) * 27 + tap];
    }
    v[t] = (__bf16)w;
  }
  if(fwd) wf[j] = v;
  else wb[j] = v;
}

// ---- blocks of a volume ----------------------------------------------------------------------------

// sum of squares of a volume in a fixed order: per-workgroup partials (grid-stride, tree in LDS), then
// one workgroup adds the partials in index order into *ss, so the result does not depend on scheduling
__global__ void cae_sumsq_part_kernel(const float *__restrict__ v, size_t n, float *__restrict__ part) {
  __shared__ float s[256];
  float acc = 0.f;
  for(size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) acc += v[i] * v[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1) {
    if(threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if(threadIdx.x == 0) part[blockIdx.x] = s[0];
}
__global__ void cae_sumsq_final_kernel(const float *__restrict__ part, int np, float *__restrict__ ss) {
  __shared__ float s[256];
  float acc = 0.f;
  for(int i = threadIdx.x; i < np; i += 256) acc += part[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1) {
    if(threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if(threadIdx.x == 0) *ss = s[0];
}
constexpr int CAE_PARTS = 1024;
static void cae_sumsq(const float *v, size_t n, float *part, float *ss) {
  const int np = (int)std::min<size_t>((n + 255) / 256, CAE_PARTS);
  hipLaunchKernelGGL(cae_sumsq_part_kernel, dim3(np), dim3(256), 0, stream(), v, n, part);
  hipLaunchKernelGGL(cae_sumsq_final_kernel, dim3(1), dim3(256), 0, stream(), part, np, ss);
}

struct CaeBlocks {
  int nx, ny, nz, nbx, nbz;
  long b0;  // first block of this chunk
};

__device__ __forceinline__ void cae_block_origin(const CaeBlocks &g, long b, int &oy, int &ox, int &oz) {
  const int bz = (int)(b % g.nbz);
  const long t = b / g.nbz;
  oz = bz * 32, ox = (int)(t % g.nbx) * 32, oy = (int)(t / g.nbx) * 32;
}

// one workgroup per block: gather the block (zero outside the volume), its scale
// s = sqrt(mean square) + floor * rms(volume) (rms from the sum of squares *ss over n cells), out = x / s
__global__ void __launch_bounds__(256) cae_gather_kernel(const float *__restrict__ vol, const CaeBlocks g,
                                                         const float *__restrict__ ss, float nvol, float floor_frac,
                                                         float *__restrict__ out, float *__restrict__ scale) {
  __shared__ float red[256];
  const long b = g.b0 + blockIdx.x;
  int oy, ox, oz;
  cae_block_origin(g, b, oy, ox, oz);
  float *o = out + (size_t)blockIdx.x * 32768;
  float acc = 0.f;
  for(int e = threadIdx.x; e < 32768; e += 256) {
    const int lz = e & 31, lx = (e >> 5) & 31, ly = e >> 10;
    const int iy = oy + ly, ix = ox + lx, iz = oz + lz;
    float v = 0.f;
    if(iy < g.ny && ix < g.nx && iz < g.nz) v = vol[((size_t)iy * g.nx + ix) * g.nz + iz];
    o[e] = v;
    acc += v * v;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1) {
    if(threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  const float s = sqrtf(red[0] * (1.f / 32768.f)) + floor_frac * sqrtf(*ss / nvol);
  const float inv = s > 0.f ? 1.f / s : 0.f;
  for(int e = threadIdx.x; e < 32768; e += 256) o[e] = o[e] * inv;
  if(threadIdx.x == 0) scale[blockIdx.x] = s;
}

// training samples: block i of the batch from snapshot snap[i] of the bank at origin org[i] (inside)
__global__ void __launch_bounds__(256) cae_sample_kernel(const float *__restrict__ bank, int nx, int ny, int nz,
                                                         const int4 *__restrict__ org, const float *__restrict__ ss,
                                                         float nvol, float floor_frac, float *__restrict__ out) {
  __shared__ float red[256];
  const int4 o4 = org[blockIdx.x];
  const float *vol = bank + (size_t)o4.w * nx * ny * nz;
  float *o = out + (size_t)blockIdx.x * 32768;
  float acc = 0.f;
  for(int e = threadIdx.x; e < 32768; e += 256) {
    const int lz = e & 31, lx = (e >> 5) & 31, ly = e >> 10;
    const float v = vol[((size_t)(o4.x + ly) * nx + (o4.y + lx)) * nz + o4.z + lz];
    o[e] = v;
    acc += v * v;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for(int w = 128; w > 0; w >>= 1) {
    if(threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  const float s = sqrtf(red[0] * (1.f / 32768.f)) + floor_frac * sqrtf(ss[o4.w] / nvol);
  const float inv = s > 0.f ? 1.f / s : 0.f;
  for(int e = threadIdx.x; e < 32768; e += 256) o[e] = o[e] * inv;
}

// latent (FP32, [block][512][4]) <-> BF16 code
__global__ void cae_latent_store_kernel(const float *__restrict__ lat, long n, uint16_t *__restrict__ code) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) code[i] = __builtin_bit_cast(uint16_t, (__bf16)lat[i]);
}
__global__ void cae_latent_load_kernel(const uint16_t *__restrict__ code, long n, float *__restrict__ lat) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) lat[i] = __uint_as_float((unsigned)code[i] << 16);
}

// decoded blocks ([block][32^3]) times their scale, written back into the volume (cropped)
__global__ void cae_scatter_kernel(const float *__restrict__ rec, const CaeBlocks g, const float *__restrict__ scale,
                                   float *__restrict__ vol) {
  const long b = g.b0 + blockIdx.y;
  int oy, ox, oz;
  cae_block_origin(g, b, oy, ox, oz);
  const float s = scale[b];
  const float *r = rec + (size_t)blockIdx.y * 32768;
  for(int e = blockIdx.x * 256 + threadIdx.x; e < 32768; e += gridDim.x * 256) {
    const int lz = e & 31, lx = (e >> 5) & 31, ly = e >> 10;
    const int iy = oy + ly, ix = ox + lx, iz = oz + lz;
    if(iy < g.ny && ix < g.nx && iz < g.nz) vol[((size_t)iy * g.nx + ix) * g.nz + iz] = r[e] * s;
  }
}

// ---- host side -------------------------------------------------------------------------------------

// partial weight gradients: 256 workgroups of an upsampling layer (one per CU)
constexpr int CAE_PART = 256 * CAE_UPG;

static int lg2(int d) {
  int l = 0;
  while((1 << l) < d) l++;
  return l;
}
static int ksteps(int ch) { return (ch * 27 + 15) / 16; }
// the upsampling layers and the output layer have fragments of their own for the forward pass
static int fwd_ksteps(int l) { return kKind[l] == K_UP || l == CAE_LAYERS - 1 ? 0 : ksteps(kCin[l]); }

CaeWork::~CaeWork() {
  for(int l = 0; l < CAE_LAYERS; l++) (void)hipFree(z[l]), (void)hipFree(a[l]);
  for(void *p : {(void *)g0, (void *)g1, (void *)g2, (void *)x, (void *)scale, (void *)ss, (void *)part, (void *)wpart, org})
    (void)hipFree(p);
}

ConvAE::~ConvAE() {
  for(void *p : {(void *)d_param, (void *)d_grad, (void *)d_m, (void *)d_v, d_wf, d_wb, (void *)d_loss}) (void)hipFree(p);
  for(void *p : d_wu) (void)hipFree(p);
}

size_t cae_param_count() {
  size_t n = 0;
  for(int l = 0; l < CAE_LAYERS; l++) n += (size_t)kCout[l] * kCin[l] * 27 + kCout[l];
  return n;
}

int cae_create(ConvAE **out, unsigned seed) {
  ConvAE *c = new ConvAE();
  size_t off = 0, foff = 0, boff = 0;
  for(int l = 0; l < CAE_LAYERS; l++) {
    c->w_off[l] = off;
    off += (size_t)kCout[l] * kCin[l] * 27;
    c->b_off[l] = off;
    off += kCout[l];
    c->wf_off[l] = foff, c->wb_off[l] = boff;
    foff += (size_t)fwd_ksteps(l) * 64;
    boff += (size_t)ksteps(kCout[l]) * 64;
  }
  c->nparam = off;
  // He initialisation for the GELU layers, Glorot for the linear ones; zero biases
  std::vector<float> h(off, 0.f);
  std::mt19937 rng(seed);
  for(int l = 0; l < CAE_LAYERS; l++) {
    const float fan_in = 27.f * kCin[l], fan_out = 27.f * kCout[l];
    const float sd = kGelu[l] ? sqrtf(2.f / fan_in) : sqrtf(2.f / (fan_in + fan_out));
    std::normal_distribution<float> nd(0.f, sd);
    for(size_t i = 0; i < (size_t)kCout[l] * kCin[l] * 27; i++) h[c->w_off[l] + i] = nd(rng);
  }
  hipError_t e = hipMalloc(&c->d_param, off * 4);
  if(e == hipSuccess) e = hipMalloc(&c->d_grad, off * 4);
  if(e == hipSuccess) e = hipMalloc(&c->d_m, off * 4);
  if(e == hipSuccess) e = hipMalloc(&c->d_v, off * 4);
  if(e == hipSuccess) e = hipMalloc(&c->d_wf, foff * sizeof(cae_bf16x8));
  if(e == hipSuccess) e = hipMalloc(&c->d_wb, boff * sizeof(cae_bf16x8));
  for(int l = 0; l < CAE_LAYERS && e == hipSuccess; l++)
    if(kKind[l] == K_UP) e = hipMalloc(&c->d_wu[l], (size_t)27 * (kCout[l] / 16) * 64 * sizeof(cae_bf16x8));
    else if(l == CAE_LAYERS - 1) e = hipMalloc(&c->d_wu[l], (size_t)CAE_LT * 64 * sizeof(cae_bf16x8));
  if(e == hipSuccess) e = hipMalloc(&c->d_loss, sizeof(float) * 2);
  if(e == hipSuccess) e = hipMemcpy(c->d_param, h.data(), off * 4, hipMemcpyHostToDevice);
  if(e == hipSuccess) e = hipMemset(c->d_m, 0, off * 4);
  if(e == hipSuccess) e = hipMemset(c->d_v, 0, off * 4);
  if(e != hipSuccess) {
    set_error("autoencoder allocation failed: %s", hipGetErrorString(e));
    delete c;
    return KLRTM_ENOMEM;
  }
  int rc = cae_refresh(*c);
  if(rc) {
    delete c;
    return rc;
  }
  *out = c;
  return KLRTM_OK;
}

// weight fragments from the FP32 weights
int cae_refresh(ConvAE &c) {
  for(int l = 0; l < CAE_LAYERS; l++) {
    const int ksf = fwd_ksteps(l), ksb = ksteps(kCout[l]), n = (ksf + ksb) * 64;
    hipLaunchKernelGGL(cae_wfrag_kernel, dim3((n + 255) / 256), dim3(256), 0, stream(), c.d_param + c.w_off[l], kCin[l],
                       kCout[l], ksf, ksb, (cae_bf16x8 *)c.d_wf + c.wf_off[l], (cae_bf16x8 *)c.d_wb + c.wb_off[l]);
    if(kKind[l] == K_UP)
      hipLaunchKernelGGL(cae_wup_kernel, dim3((27 * 64 * (kCout[l] / 16) + 255) / 256), dim3(256), 0, stream(), c.d_param + c.w_off[l], kCout[l],
                         (cae_bf16x8 *)c.d_wu[l]);
    else if(l == CAE_LAYERS - 1)
      hipLaunchKernelGGL(cae_wtap_kernel, dim3((CAE_LT * 64 + 255) / 256), dim3(256), 0, stream(), c.d_param + c.w_off[l], (cae_bf16x8 *)c.d_wu[l]);
  }
  return check_launch("cae_wfrag_kernel");
}

// work buffers for nb blocks (training keeps the pre-activations and gradients too)
int cae_reserve(CaeWork &w, int nb, bool train) {
  if(nb <= w.cap && (!train || w.train)) return KLRTM_OK;
  nb = std::max(nb, w.cap);
  train = train || w.train;
  for(int l = 0; l < CAE_LAYERS; l++) {
    (void)hipFree(w.z[l]), (void)hipFree(w.a[l]);
    w.z[l] = w.a[l] = nullptr;
  }
  for(float **p : {&w.g0, &w.g1, &w.g2, &w.x, &w.scale, &w.ss, &w.part, &w.wpart}) (void)hipFree(*p), *p = nullptr;
  (void)hipFree(w.org);
  w.org = nullptr;
  w.cap = 0, w.train = false;
  size_t gmax = 0, umax = 0;
  for(int l = 0; l < CAE_LAYERS; l++) {
    const size_t no = (size_t)nb * kCout[l] * ((size_t)kDout[l] * kDout[l] * kDout[l]);
    KL_HIP(hipMalloc(&w.a[l], no * 4));
    if(train && kGelu[l]) KL_HIP(hipMalloc(&w.z[l], no * 4));  // (read by the gradient through the activation only)
    // gradient buffers: this layer's output gradient, its input gradient, and for upsampling layers
    // the input gradient on the fine grid
    const size_t ni = (size_t)nb * kCin[l] * ((size_t)kDin[l] * kDin[l] * kDin[l]);
    const size_t nu = kKind[l] == K_UP ? (size_t)nb * kCin[l] * ((size_t)kDout[l] * kDout[l] * kDout[l]) : 0;
    gmax = std::max(gmax, std::max(no, ni));
    umax = std::max(umax, nu);
  }
  KL_HIP(hipMalloc(&w.x, (size_t)nb * 32768 * 4));
  KL_HIP(hipMalloc(&w.scale, (size_t)nb * 4));
  KL_HIP(hipMalloc(&w.ss, 1024 * 4));
  KL_HIP(hipMalloc(&w.part, CAE_PARTS * 4));
  KL_HIP(hipMalloc(&w.org, (size_t)nb * sizeof(int4)));
  if(train) {
    KL_HIP(hipMalloc(&w.g0, gmax * 4));
    KL_HIP(hipMalloc(&w.g1, gmax * 4));
    KL_HIP(hipMalloc(&w.g2, umax * 4));
    KL_HIP(hipMalloc(&w.wpart, ((size_t)CAE_PART + CAE_UPG * 2) * 4));
  }
  w.cap = nb, w.train = train;
  return KLRTM_OK;
}

template<int CG, int MODE, int EPI>
static void conv_launch(const float *G, const void *wf, int ks, int nout, int lgo, int lgg, const float *bias, int act,
                        float *z, float *out, const float *zg, int nb) {
  const long P = 1L << (3 * lgo);
  const dim3 grid((unsigned)((P + 127) / 128), (unsigned)nb);
  hipLaunchKernelGGL((cae_conv_kernel<CG, MODE, EPI>), grid, dim3(256), 0, stream(), G, (const cae_bf16x8 *)wf, ks, nout,
                     lgo, lgg, bias, act, z, out, zg);
}

// Workgroups that share a tile of the upsampling layers, and slabs along y of the output layer's columns, for a launch
// of wg tiles: up to two workgroups a CU, past which the repeated staging costs more than it hides.  1, 8, 27 and 64
// blocks, us with 1 / 2 / 4 / 8 parts: layer 6 34 22 16 14, 39 28 24 30, 47 56 70 96, 91 109 148 226; layer 5 29 19 13 10,
// 30 19 14 11, 32 21 17 22, 36 28 31 35; output layer 50 27 15 9, 50 27 16 11, 51 29 23 27, 54 41 48 48.
static int cae_parts(long wg) {
  int parts = 1;
  while(parts < 8 && 2 * wg * parts <= 512) parts *= 2;
  return parts;
}

// forward of layer l over nb blocks: out = act(conv(in) + b), pre-activation kept in z when set
static int layer_fwd(const ConvAE &c, int l, const float *in, float *z, float *out, int nb) {
  const int lgo = lg2(kDout[l]), lgg = lg2(kDin[l]), ks = ksteps(kCin[l]);
  const void *wf = (const cae_bf16x8 *)c.d_wf + c.wf_off[l];
  const float *bias = c.d_param + c.b_off[l];
  const cae_bf16x8 *wu = (const cae_bf16x8 *)c.d_wu[l];
  if(kKind[l] == K_UP) {
    const int tiles = (kDin[l] / CAE_UP_TY) * (kDin[l] / CAE_UP_TX);
    const dim3 grid((unsigned)tiles, (unsigned)nb, (unsigned)cae_parts((long)tiles * nb));
    if(kCout[l] == 32 && kDin[l] == 8)
      hipLaunchKernelGGL((cae_up_kernel<32, 3>), grid, dim3(256), 0, stream(), in, wu, bias, z, out);
    else if(kCout[l] == 16 && kDin[l] == 16)
      hipLaunchKernelGGL((cae_up_kernel<16, 4>), grid, dim3(256), 0, stream(), in, wu, bias, z, out);
    else {
      set_error("autoencoder layer %d has no forward kernel", l);
      return KLRTM_EINVAL;
    }
    return check_launch("cae_up_kernel");
  }
  if(l == CAE_LAYERS - 1) {  // (no activation: nothing reads its pre-activation)
    hipLaunchKernelGGL(cae_last_kernel, dim3(4 * (unsigned)cae_parts(4L * nb), (unsigned)nb), dim3(256), 0, stream(), in, wu,
                       bias, out);
    return check_launch("cae_last_kernel");
  }
  const int mode = kKind[l] == K_DOWN ? G_DOWN : G_SAME;
#define CAE_F(CG, M) conv_launch<CG, M, E_FWD>(in, wf, ks, kCout[l], lgo, lgg, bias, kGelu[l], z, out, nullptr, nb)
  switch(kCin[l] * 8 + mode) {
  case 1 * 8 + G_DOWN: CAE_F(1, G_DOWN); break;
  case 16 * 8 + G_DOWN: CAE_F(16, G_DOWN); break;
  case 32 * 8 + G_SAME: CAE_F(32, G_SAME); break;
  case 4 * 8 + G_SAME: CAE_F(4, G_SAME); break;
  default: set_error("autoencoder layer %d has no forward kernel", l); return KLRTM_EINVAL;
  }
#undef CAE_F
  return check_launch("cae_conv_kernel");
}

// data gradient of layer l: din (gradient of the previous layer's pre-activation, or of the input for
// l == 0) from dz (gradient of this layer's pre-activation)
static int layer_dgrad(const ConvAE &c, const CaeWork &w, int l, const float *dz, float *din, float *scratch, int nb) {
  const float *zg = l > 0 && kGelu[l - 1] ? w.z[l - 1] : nullptr;
  const void *wb = (const cae_bf16x8 *)c.d_wb + c.wb_off[l];
  const int ks = ksteps(kCout[l]);
  const int lgi = lg2(kDin[l]), lgo = lg2(kDout[l]);
  if(kKind[l] == K_UP) {
    // on the fine grid, then summed onto the coarse one
#define CAE_U(CG) conv_launch<CG, G_BSAME, E_PLAIN>(dz, wb, ks, kCin[l], lgo, lgo, nullptr, 0, nullptr, scratch, nullptr, nb)
    switch(kCout[l]) {
    case 32: CAE_U(32); break;
    case 16: CAE_U(16); break;
    default: set_error("autoencoder layer %d has no gradient kernel", l); return KLRTM_EINVAL;
    }
#undef CAE_U
    const long total = (long)nb * kCin[l] * (1L << (3 * lgi));
    hipLaunchKernelGGL(cae_downsum_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream(), scratch, kCin[l],
                       lgi, zg, din, total);
    return check_launch("cae_downsum_kernel");
  }
  const int mode = kKind[l] == K_DOWN ? G_BDOWN : G_BSAME;
#define CAE_B(CG, M) conv_launch<CG, M, E_BWD>(dz, wb, ks, kCin[l], lgi, lgo, nullptr, 0, nullptr, din, zg, nb)
  switch(kCout[l] * 8 + mode) {
  case 32 * 8 + G_BDOWN: CAE_B(32, G_BDOWN); break;
  case 16 * 8 + G_BDOWN: CAE_B(16, G_BDOWN); break;
  case 32 * 8 + G_BSAME: CAE_B(32, G_BSAME); break;
  case 4 * 8 + G_BSAME: CAE_B(4, G_BSAME); break;
  case 1 * 8 + G_BSAME: CAE_B(1, G_BSAME); break;
  default: set_error("autoencoder layer %d has no gradient kernel", l); return KLRTM_EINVAL;
  }
#undef CAE_B
  return check_launch("cae_conv_kernel");
}

// weight and bias gradients of layer l into d_grad (cleared before) from its input and its pre-activation gradient
static int layer_wgrad(ConvAE &c, CaeWork &w, int l, const float *in, const float *dz, int nb) {
  const long P = 1L << (3 * lg2(kDout[l]));
  float *dW = c.d_grad + c.w_off[l];
  const long n = (long)nb * P * kCout[l];
  hipLaunchKernelGGL(cae_bgrad_kernel, dim3((unsigned)((n + 8191) / 8192)), dim3(256), 0, stream(), dz, n, kCout[l],
                     c.d_grad + c.b_off[l]);
  if(kKind[l] == K_UP) {
    const int ng = CAE_UPG / 16 * kCout[l], tiles = kDin[l] == 8 ? 8 : 64, ntask = nb * tiles;
    const int slots = std::min(ntask, CAE_PART / ng);
    const dim3 grid((unsigned)slots, (unsigned)(kCout[l] / 16));
    float *G = w.wpart + CAE_PART;
    if(kCout[l] == 32 && kDin[l] == 8)
      hipLaunchKernelGGL((cae_wgrad_up_kernel<32, 3>), grid, dim3(512), 0, stream(), in, dz, ntask, w.wpart);
    else if(kCout[l] == 16 && kDin[l] == 16)
      hipLaunchKernelGGL((cae_wgrad_up_kernel<16, 4>), grid, dim3(512), 0, stream(), in, dz, ntask, w.wpart);
    else {
      set_error("autoencoder layer %d has no weight-gradient kernel", l);
      return KLRTM_EINVAL;
    }
    hipLaunchKernelGGL(cae_wred_kernel<R_PLAIN>, dim3((unsigned)(ng / 32)), dim3(256), 0, stream(), w.wpart, slots, ng, G);
    hipLaunchKernelGGL(cae_wup_sum_kernel, dim3((unsigned)((kCout[l] * 32 * 27 + 255) / 256)), dim3(256), 0, stream(), G,
                       kCout[l], dW);
    return check_launch("cae_wgrad_up_kernel");
  }
  if(kCin[l] == 1 || kCout[l] == 1) {
    const bool first = kCin[l] == 1;
    const int ntask = nb * (first ? 4 : 8), slots = std::min(ntask, 1024);
    if(first)
      hipLaunchKernelGGL((cae_wgrad_vec_kernel<4, 2>), dim3((unsigned)slots), dim3(256), 0, stream(), dz, in, ntask, w.wpart);
    else
      hipLaunchKernelGGL((cae_wgrad_vec_kernel<5, 1>), dim3((unsigned)slots), dim3(256), 0, stream(), in, dz, ntask, w.wpart);
    hipLaunchKernelGGL(cae_wred_kernel<R_PITCH27>, dim3(16), dim3(256), 0, stream(), w.wpart, slots, 512, dW);
    return check_launch("cae_wgrad_vec_kernel");
  }
  const int nw = 27 * kCout[l] * kCin[l], ntask = nb * 4, slots = std::min(ntask, 256);
#define CAE_W(CI, CO, S) \
  hipLaunchKernelGGL((cae_wgrad_tile_kernel<CI, CO, S>), dim3((unsigned)slots), dim3(512), 0, stream(), in, dz, ntask, w.wpart)
  if(kCin[l] == 16 && kCout[l] == 32 && kKind[l] == K_DOWN && kDout[l] == 8) CAE_W(16, 32, 2);
  else if(kCin[l] == 32 && kCout[l] == 32 && kKind[l] == K_SAME && kDout[l] == 8) CAE_W(32, 32, 1);
  else if(kCin[l] == 32 && kCout[l] == 4 && kKind[l] == K_SAME && kDout[l] == 8) CAE_W(32, 4, 1);
  else if(kCin[l] == 4 && kCout[l] == 32 && kKind[l] == K_SAME && kDout[l] == 8) CAE_W(4, 32, 1);
  else {
    set_error("autoencoder layer %d has no weight-gradient kernel", l);
    return KLRTM_EINVAL;
  }
#undef CAE_W
  hipLaunchKernelGGL(cae_wred_kernel<R_TAPS>, dim3((unsigned)(nw / 32)), dim3(256), 0, stream(), w.wpart, slots, nw, dW);
  return check_launch("cae_wgrad_tile_kernel");
}

// forward of layers [l0, l1) from in; pre-activations kept when training
static int run_layers(const ConvAE &c, CaeWork &w, int l0, int l1, const float *in, int nb, bool train) {
  int rc;
  for(int l = l0; l < l1; l++) {
    if((rc = layer_fwd(c, l, l == l0 ? in : w.a[l - 1], train ? w.z[l] : nullptr, w.a[l], nb))) return rc;
  }
  return KLRTM_OK;
}

// gradient of the mean squared error of the reconstruction of x (nb blocks) into d_grad (cleared
// first); the loss goes to d_loss[0]
int cae_loss_grad(ConvAE &c, const float *x, int nb) {
  CaeWork &w = c.w;
  int rc;
  if((rc = cae_reserve(w, nb, true))) return rc;
  if((rc = run_layers(c, w, 0, CAE_LAYERS, x, nb, true))) return rc;
  cae_zero(c.d_grad, c.nparam);
  cae_zero(c.d_loss, 1);
  const long n = (long)nb * 32768;
  hipLaunchKernelGGL(cae_mse_kernel, dim3(256), dim3(256), 0, stream(), w.a[CAE_LAYERS - 1], x, n, 1.f / (float)n, w.g0,
                     c.d_loss);
  float *dz = w.g0, *din = w.g1;
  for(int l = CAE_LAYERS - 1; l >= 0; l--) {
    const float *in = l == 0 ? x : w.a[l - 1];
    if((rc = layer_wgrad(c, w, l, in, dz, nb))) return rc;
    if(l == 0) break;
    if((rc = layer_dgrad(c, w, l, dz, din, w.g2, nb))) return rc;
    std::swap(dz, din);
  }
  return check_launch("cae_loss_grad");
}

int cae_adam(ConvAE &c, float lr) {
  c.step++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - powf(b1, (float)c.step), c2 = 1.f - powf(b2, (float)c.step);
  hipLaunchKernelGGL(cae_adam_kernel, dim3((unsigned)((c.nparam + 255) / 256)), dim3(256), 0, stream(), c.d_param,
                     c.d_grad, c.d_m, c.d_v, (long)c.nparam, lr, b1, b2, c1, c2, 1e-8f);
  int rc = check_launch("cae_adam_kernel");
  return rc ? rc : cae_refresh(c);
}

size_t cae_code_bytes(int nx, int ny, int nz) {
  const size_t nb = (size_t)((nx + 31) / 32) * ((ny + 31) / 32) * ((nz + 31) / 32);
  return ((nb * 2048 * 2 + 255) & ~(size_t)255) + nb * 4;
}

static CaeBlocks blocks_of(int nx, int ny, int nz) {
  CaeBlocks g;
  g.nx = nx, g.ny = ny, g.nz = nz, g.nbx = (nx + 31) / 32, g.nbz = (nz + 31) / 32, g.b0 = 0;
  return g;
}

int cae_encode(const ConvAE &c, CaeWork &w, const float *vol, int nx, int ny, int nz, float floor_frac, void *code) {
  CaeBlocks g = blocks_of(nx, ny, nz);
  const long nb = (long)g.nbx * g.nbz * ((ny + 31) / 32);
  uint16_t *lat = (uint16_t *)code;
  float *scale = (float *)((char *)code + ((nb * 2048 * 2 + 255) & ~(size_t)255));
  const size_t n = (size_t)nx * ny * nz;
  int rc;
  if((rc = cae_reserve(w, CAE_CHUNK, false))) return rc;
  LaunchTimer tm("cae_encode");
  cae_sumsq(vol, n, w.part, w.ss);
  for(long b0 = 0; b0 < nb; b0 += CAE_CHUNK) {
    const int cnt = (int)std::min<long>(CAE_CHUNK, nb - b0);
    g.b0 = b0;
    hipLaunchKernelGGL(cae_gather_kernel, dim3(cnt), dim3(256), 0, stream(), vol, g, w.ss, (float)n, floor_frac, w.x,
                       scale + b0);
    if((rc = run_layers(c, w, 0, 4, w.x, cnt, false))) return rc;
    const long nl = (long)cnt * 2048;
    hipLaunchKernelGGL(cae_latent_store_kernel, dim3((unsigned)((nl + 255) / 256)), dim3(256), 0, stream(), w.a[3], nl,
                       lat + b0 * 2048);
  }
  return check_launch("cae_encode");
}

int cae_decode(const ConvAE &c, CaeWork &w, const void *code, float *vol, int nx, int ny, int nz) {
  CaeBlocks g = blocks_of(nx, ny, nz);
  const long nb = (long)g.nbx * g.nbz * ((ny + 31) / 32);
  const uint16_t *lat = (const uint16_t *)code;
  const float *scale = (const float *)((const char *)code + ((nb * 2048 * 2 + 255) & ~(size_t)255));
  int rc;
  if((rc = cae_reserve(w, CAE_CHUNK, false))) return rc;
  LaunchTimer tm("cae_decode");
  for(long b0 = 0; b0 < nb; b0 += CAE_CHUNK) {
    const int cnt = (int)std::min<long>(CAE_CHUNK, nb - b0);
    g.b0 = b0;
    const long nl = (long)cnt * 2048;
    hipLaunchKernelGGL(cae_latent_load_kernel, dim3((unsigned)((nl + 255) / 256)), dim3(256), 0, stream(),
                       lat + b0 * 2048, nl, w.x);
    if((rc = run_layers(c, w, 4, CAE_LAYERS, w.x, cnt, false))) return rc;
    hipLaunchKernelGGL(cae_scatter_kernel, dim3(32, cnt), dim3(256), 0, stream(), w.a[CAE_LAYERS - 1], g, scale, vol);
  }
  return check_launch("cae_decode");
}

// training on random 32^3 blocks of a bank of nsnap snapshots [nsnap][ny][nx][nz] (device)
int cae_train(ConvAE &c, const float *bank, int nsnap, int nx, int ny, int nz, float floor_frac, int steps, int batch,
              float lr, unsigned seed, float *loss_first, float *loss_last) {
  KL_REQUIRE(bank && nsnap > 0 && nsnap <= 1024 && nx >= 32 && ny >= 32 && nz >= 32 && batch > 0 && steps > 0,
             KLRTM_EINVAL, "bad training set");
  CaeWork &w = c.w;
  int rc;
  if((rc = cae_reserve(w, batch, true))) return rc;
  const size_t n = (size_t)nx * ny * nz;
  for(int s = 0; s < nsnap; s++) cae_sumsq(bank + s * n, n, w.part, w.ss + s);
  std::mt19937 rng(seed);
  std::vector<int4> org(batch);
  LaunchTimer tm("cae_train");
  for(int it = 0; it < steps; it++) {
    for(int i = 0; i < batch; i++) {
      org[i].x = (int)(rng() % (unsigned)(ny - 31));
      org[i].y = (int)(rng() % (unsigned)(nx - 31));
      org[i].z = (int)(rng() % (unsigned)(nz - 31));
      org[i].w = (int)(rng() % (unsigned)nsnap);
    }
    KL_HIP(hipMemcpyAsync(w.org, org.data(), sizeof(int4) * batch, hipMemcpyHostToDevice, stream()));
    hipLaunchKernelGGL(cae_sample_kernel, dim3(batch), dim3(256), 0, stream(), bank, nx, ny, nz, (const int4 *)w.org, w.ss,
                       (float)n, floor_frac, w.x);
    if((rc = cae_loss_grad(c, w.x, batch))) return rc;
    if(it == 0 && loss_first) KL_HIP(hipMemcpyAsync(&c.h_loss[0], c.d_loss, 4, hipMemcpyDeviceToHost, stream()));
    if((rc = cae_adam(c, lr))) return rc;
    // the host copy of the samples' origins must not be overwritten before the upload has run
    KL_HIP(hipStreamSynchronize(stream()));
  }
  if(loss_first) *loss_first = c.h_loss[0];
  if(loss_last) {
    KL_HIP(hipStreamSynchronize(stream()));
    KL_HIP(hipMemcpy(&c.h_loss[1], c.d_loss, 4, hipMemcpyDeviceToHost));
    *loss_last = c.h_loss[1];
  }
  return KLRTM_OK;
}

}  // namespace klrtm

using namespace klrtm;

extern "C" {

int klrtm_convae_create(klrtm_convae **out, unsigned seed) {
  KL_REQUIRE(out, KLRTM_EINVAL, "null argument");
  ConvAE *c = nullptr;
  int rc = cae_create(&c, seed);
  *out = reinterpret_cast<klrtm_convae *>(c);
  return rc;
}
int klrtm_convae_destroy(klrtm_convae *c) {
  delete reinterpret_cast<ConvAE *>(c);
  return KLRTM_OK;
}
size_t klrtm_convae_param_count(void) { return cae_param_count(); }
int klrtm_convae_get_params(klrtm_convae *h, float *params) {
  KL_REQUIRE(h && params, KLRTM_EINVAL, "null argument");
  ConvAE &c = *reinterpret_cast<ConvAE *>(h);
  KL_HIP(hipStreamSynchronize(stream()));  // the copy runs on the null stream, the kernels on the library's
  KL_HIP(hipMemcpy(params, c.d_param, c.nparam * 4, hipMemcpyDeviceToHost));
  return KLRTM_OK;
}
int klrtm_convae_set_params(klrtm_convae *h, const float *params) {
  KL_REQUIRE(h && params, KLRTM_EINVAL, "null argument");
  ConvAE &c = *reinterpret_cast<ConvAE *>(h);
  KL_HIP(hipStreamSynchronize(stream()));
  KL_HIP(hipMemcpy(c.d_param, params, c.nparam * 4, hipMemcpyHostToDevice));
  return cae_refresh(c);
}
int klrtm_convae_forward(klrtm_convae *h, const float *x, int nb, float *latent, float *recon) {
  KL_REQUIRE(h && x && nb > 0, KLRTM_EINVAL, "bad argument");
  ConvAE &c = *reinterpret_cast<ConvAE *>(h);
  int rc;
  if((rc = cae_reserve(c.w, nb, false)) || (rc = run_layers(c, c.w, 0, CAE_LAYERS, x, nb, false))) return rc;
  if(latent) KL_HIP(hipMemcpyAsync(latent, c.w.a[3], (size_t)nb * 2048 * 4, hipMemcpyDeviceToDevice, stream()));
  if(recon) KL_HIP(hipMemcpyAsync(recon, c.w.a[CAE_LAYERS - 1], (size_t)nb * 32768 * 4, hipMemcpyDeviceToDevice, stream()));
  return KLRTM_OK;
}
int klrtm_convae_loss_grad(klrtm_convae *h, const float *x, int nb, float *grad, float *loss) {
  KL_REQUIRE(h && x && nb > 0, KLRTM_EINVAL, "bad argument");
  ConvAE &c = *reinterpret_cast<ConvAE *>(h);
  int rc = cae_loss_grad(c, x, nb);
  if(rc) return rc;
  KL_HIP(hipStreamSynchronize(stream()));
  if(grad) KL_HIP(hipMemcpy(grad, c.d_grad, c.nparam * 4, hipMemcpyDeviceToHost));
  if(loss) KL_HIP(hipMemcpy(loss, c.d_loss, 4, hipMemcpyDeviceToHost));
  return KLRTM_OK;
}
int klrtm_convae_adam_step(klrtm_convae *h, float lr) {
  KL_REQUIRE(h, KLRTM_EINVAL, "null argument");
  return cae_adam(*reinterpret_cast<ConvAE *>(h), lr);
}
int klrtm_convae_train(klrtm_convae *h, const float *bank, int nsnap, int nx, int ny, int nz, float floor_frac, int steps,
                       int batch, float lr, unsigned seed, float *loss_first, float *loss_last) {
  KL_REQUIRE(h, KLRTM_EINVAL, "null argument");
  return cae_train(*reinterpret_cast<ConvAE *>(h), bank, nsnap, nx, ny, nz, floor_frac, steps, batch, lr, seed,
                   loss_first, loss_last);
}
size_t klrtm_convae_code_bytes(int nx, int ny, int nz) { return cae_code_bytes(nx, ny, nz); }
int klrtm_convae_encode(klrtm_convae *h, const float *vol, int nx, int ny, int nz, float floor_frac, void *code) {
  KL_REQUIRE(h && vol && code && nx > 0 && ny > 0 && nz > 0, KLRTM_EINVAL, "bad argument");
  ConvAE &c = *reinterpret_cast<ConvAE *>(h);
  return cae_encode(c, c.w, vol, nx, ny, nz, floor_frac, code);
}
int klrtm_convae_decode(klrtm_convae *h, const void *code, float *vol, int nx, int ny, int nz) {
  KL_REQUIRE(h && vol && code && nx > 0 && ny > 0 && nz > 0, KLRTM_EINVAL, "bad argument");
  ConvAE &c = *reinterpret_cast<ConvAE *>(h);
  return cae_decode(c, c.w, code, vol, nx, ny, nz);
}

}  // extern "C"
