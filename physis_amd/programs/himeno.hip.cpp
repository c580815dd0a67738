// Generated by physisc-hip from himeno.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

// ---------------------------------------------- stencil jacobi_kernel
struct __PSStencil_jacobi_kernel {
  __PSDomain dom;
  __PSGrid *p0;
  int __p0_index;
  __PSGrid *p1;
  int __p1_index;
  __PSGrid *a0;
  int __a0_index;
  __PSGrid *a1;
  int __a1_index;
  __PSGrid *a2;
  int __a2_index;
  __PSGrid *a3;
  int __a3_index;
  __PSGrid *b0;
  int __b0_index;
  __PSGrid *b1;
  int __b1_index;
  __PSGrid *b2;
  int __b2_index;
  __PSGrid *c0;
  int __c0_index;
  __PSGrid *c1;
  int __c1_index;
  __PSGrid *c2;
  int __c2_index;
  __PSGrid *bnd;
  int __bnd_index;
  __PSGrid *wrk1;
  int __wrk1_index;
  float omega;
  float *__reduce_out;  // PSStencilMapReduce target
  int __reduce_op;
};

static struct __PSStencil_jacobi_kernel __PSStencilMap_jacobi_kernel(
    __PSDomain __dom, __PSGrid *p0, __PSGrid *p1, __PSGrid *a0, __PSGrid *a1, __PSGrid *a2, __PSGrid *a3, __PSGrid *b0, __PSGrid *b1, __PSGrid *b2, __PSGrid *c0, __PSGrid *c1, __PSGrid *c2, __PSGrid *bnd, __PSGrid *wrk1, float omega) {
  struct __PSStencil_jacobi_kernel __s = {__dom, p0, __PSGridGetID(p0), p1, __PSGridGetID(p1), a0, __PSGridGetID(a0), a1, __PSGridGetID(a1), a2, __PSGridGetID(a2), a3, __PSGridGetID(a3), b0, __PSGridGetID(b0), b1, __PSGridGetID(b1), b2, __PSGridGetID(b2), c0, __PSGridGetID(c0), c1, __PSGridGetID(c1), c2, __PSGridGetID(c2), bnd, __PSGridGetID(bnd), wrk1, __PSGridGetID(wrk1), omega, NULL, 0};
  return __s;
}

static struct __PSStencil_jacobi_kernel __PSStencilMapReduce_jacobi_kernel(
    float *__v, int __op, __PSDomain __dom, __PSGrid *p0, __PSGrid *p1, __PSGrid *a0, __PSGrid *a1, __PSGrid *a2, __PSGrid *a3, __PSGrid *b0, __PSGrid *b1, __PSGrid *b2, __PSGrid *c0, __PSGrid *c1, __PSGrid *c2, __PSGrid *bnd, __PSGrid *wrk1, float omega) {
  struct __PSStencil_jacobi_kernel __s = __PSStencilMap_jacobi_kernel(__dom, p0, p1, a0, a1, a2, a3, b0, b1, b2, c0, c1, c2, bnd, wrk1, omega);
  __s.__reduce_out = __v;
  __s.__reduce_op = __op;
  return __s;
}

// Stencil analysis of jacobi_kernel (2.5D run kernel):
//   p0  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,1) 1:(0,1,0) 2:(1,0,0) 3:(0,1,1) 4:(0,-1,1) 5:(0,1,-1) 6:(0,-1,-1) 7:(1,1,0) 8:(1,-1,0) 9:(-1,1,0) 10:(-1,-1,0) 11:(1,0,1) 12:(1,0,-1) 13:(-1,0,1) 14:(-1,0,-1) 15:(0,0,-1) 16:(0,-1,0) 17:(-1,0,0) 18:(0,0,0)
//   p1  not read, emitted
//   a0  direct (centre only)
//   a1  direct (centre only)
//   a2  direct (centre only)
//   a3  direct (centre only)
//   b0  direct (centre only)
//   b1  direct (centre only)
//   b2  direct (centre only)
//   c0  direct (centre only)
//   c1  direct (centre only)
//   c2  direct (centre only)
//   bnd  direct (centre only)
//   wrk1  direct (centre only)
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_jacobi_kernel {
  float p0[19];
  const float *p0_p;
  int p0_dim[3];
  float p1_v;
  bool p1_e;
  const float *p1_p;
  int p1_dim[3];
  float a0_c;
  const float *a0_p;
  int a0_dim[3];
  float a1_c;
  const float *a1_p;
  int a1_dim[3];
  float a2_c;
  const float *a2_p;
  int a2_dim[3];
  float a3_c;
  const float *a3_p;
  int a3_dim[3];
  float b0_c;
  const float *b0_p;
  int b0_dim[3];
  float b1_c;
  const float *b1_p;
  int b1_dim[3];
  float b2_c;
  const float *b2_p;
  int b2_dim[3];
  float c0_c;
  const float *c0_p;
  int c0_dim[3];
  float c1_c;
  const float *c1_p;
  int c1_dim[3];
  float c2_c;
  const float *c2_p;
  int c2_dim[3];
  float bnd_c;
  const float *bnd_p;
  int bnd_dim[3];
  float wrk1_c;
  const float *wrk1_p;
  int wrk1_dim[3];
};

__device__ __forceinline__ float jacobi_kernel(
    int i, int j, int k, __PSCtx_jacobi_kernel &__ctx, float omega) {
  float s0, ss;
  s0 = __ctx.a0_c * __ctx.p0[0] + __ctx.a1_c * __ctx.p0[1] + __ctx.a2_c * __ctx.p0[2] + __ctx.b0_c * (__ctx.p0[3] - __ctx.p0[4] - __ctx.p0[5] + __ctx.p0[6]) + __ctx.b1_c * (__ctx.p0[7] - __ctx.p0[8] - __ctx.p0[9] + __ctx.p0[10]) + __ctx.b2_c * (__ctx.p0[11] - __ctx.p0[12] - __ctx.p0[13] + __ctx.p0[14]) + __ctx.c0_c * __ctx.p0[15] + __ctx.c1_c * __ctx.p0[16] + __ctx.c2_c * __ctx.p0[17] + __ctx.wrk1_c;
  ss = (s0 * __ctx.a3_c - __ctx.p0[18]) * __ctx.bnd_c;
  float v = __ctx.p0[18] + omega * ss;
  (__ctx.p1_v = (v), __ctx.p1_e = true);
  return ss * ss;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_jacobi_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev p0, __PSGrid3DFloat_dev p1, __PSGrid3DFloat_dev a0, __PSGrid3DFloat_dev a1, __PSGrid3DFloat_dev a2, __PSGrid3DFloat_dev a3, __PSGrid3DFloat_dev b0, __PSGrid3DFloat_dev b1, __PSGrid3DFloat_dev b2, __PSGrid3DFloat_dev c0, __PSGrid3DFloat_dev c1, __PSGrid3DFloat_dev c2, __PSGrid3DFloat_dev bnd, __PSGrid3DFloat_dev wrk1, float omega, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, false, float, RAGGED> S_p0;
  __shared__ __attribute__((aligned(16))) float p0_lds[S_p0::kLdsElems];
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, sh.tiles_y);
  const int x0 = (sh.x_first_tile + tc.bx) * TX;
  const int y0 = dom.local_min[1] + tc.by * TY;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  float __racc = 0;
  if constexpr (RED >= 0) __racc = physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::identity();
  if (zb < ze) {
    const int yrow = y0 - HY + wave;
    const bool computes = wave >= HY && wave < BY - HY && yrow < dom.local_max[1];
    const int xs = x0 + lane * VX;
    // centre-only grids are read at the nearest compute row, so halo
    // waves repeat their neighbours' addresses and every wave issues
    // the same loads
    const int drow = wave < HY ? y0 : (wave >= BY - HY ? y0 + TY - 1 : yrow);
    const int p0_nxy = p0.dim[0] * p0.dim[1];
    const physis_hip::BufWin<float> p0_w = physis_hip::BufWin<float>::Make(p0.p, p0_nxy * p0.dim[2], (long)(zb + -2) * p0_nxy, (long)(ze + 2) * p0_nxy);
    S_p0 p0_st[PD];
    const typename S_p0::Addr p0_ra = S_p0::Prepare(p0.dim, x0, yrow, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      p0_st[0].Load(p0_w, p0.p, p0.dim, p0_ra, zb + -1 + k);
      p0_st[0].Store(p0_lds + k * S_p0::kPlane, wave, lane, p0_ra);
    }
#pragma unroll
    for (int k = 0; k < PD; ++k)
      p0_st[k].Load(p0_w, p0.p, p0.dim, p0_ra, zb + 2 + k);
    int p0_base = 0;
    const int p1_enx = p1.dim[0], p1_enxy = p1.dim[0] * p1.dim[1];
    const physis_hip::BufWin<float> p1_ew = physis_hip::BufWin<float>::Make(p1.p, p1_enxy * p1.dim[2], (long)zb * p1_enxy, (long)ze * p1_enxy);
    const int a0_nx = a0.dim[0], a0_nxy = a0.dim[0] * a0.dim[1];
    const physis_hip::BufWin<float> a0_w = physis_hip::BufWin<float>::Make(a0.p, a0_nxy * a0.dim[2], (long)zb * a0_nxy, (long)ze * a0_nxy);
    float a0_dv[2][VX];
    a0_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a0_nx + zb * a0_nxy, a0_dv[0]);
    const int a1_nx = a1.dim[0], a1_nxy = a1.dim[0] * a1.dim[1];
    const physis_hip::BufWin<float> a1_w = physis_hip::BufWin<float>::Make(a1.p, a1_nxy * a1.dim[2], (long)zb * a1_nxy, (long)ze * a1_nxy);
    float a1_dv[2][VX];
    a1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a1_nx + zb * a1_nxy, a1_dv[0]);
    const int a2_nx = a2.dim[0], a2_nxy = a2.dim[0] * a2.dim[1];
    const physis_hip::BufWin<float> a2_w = physis_hip::BufWin<float>::Make(a2.p, a2_nxy * a2.dim[2], (long)zb * a2_nxy, (long)ze * a2_nxy);
    float a2_dv[2][VX];
    a2_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a2_nx + zb * a2_nxy, a2_dv[0]);
    const int a3_nx = a3.dim[0], a3_nxy = a3.dim[0] * a3.dim[1];
    const physis_hip::BufWin<float> a3_w = physis_hip::BufWin<float>::Make(a3.p, a3_nxy * a3.dim[2], (long)zb * a3_nxy, (long)ze * a3_nxy);
    float a3_dv[2][VX];
    a3_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a3_nx + zb * a3_nxy, a3_dv[0]);
    const int b0_nx = b0.dim[0], b0_nxy = b0.dim[0] * b0.dim[1];
    const physis_hip::BufWin<float> b0_w = physis_hip::BufWin<float>::Make(b0.p, b0_nxy * b0.dim[2], (long)zb * b0_nxy, (long)ze * b0_nxy);
    float b0_dv[2][VX];
    b0_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * b0_nx + zb * b0_nxy, b0_dv[0]);
    const int b1_nx = b1.dim[0], b1_nxy = b1.dim[0] * b1.dim[1];
    const physis_hip::BufWin<float> b1_w = physis_hip::BufWin<float>::Make(b1.p, b1_nxy * b1.dim[2], (long)zb * b1_nxy, (long)ze * b1_nxy);
    float b1_dv[2][VX];
    b1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * b1_nx + zb * b1_nxy, b1_dv[0]);
    const int b2_nx = b2.dim[0], b2_nxy = b2.dim[0] * b2.dim[1];
    const physis_hip::BufWin<float> b2_w = physis_hip::BufWin<float>::Make(b2.p, b2_nxy * b2.dim[2], (long)zb * b2_nxy, (long)ze * b2_nxy);
    float b2_dv[2][VX];
    b2_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * b2_nx + zb * b2_nxy, b2_dv[0]);
    const int c0_nx = c0.dim[0], c0_nxy = c0.dim[0] * c0.dim[1];
    const physis_hip::BufWin<float> c0_w = physis_hip::BufWin<float>::Make(c0.p, c0_nxy * c0.dim[2], (long)zb * c0_nxy, (long)ze * c0_nxy);
    float c0_dv[2][VX];
    c0_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c0_nx + zb * c0_nxy, c0_dv[0]);
    const int c1_nx = c1.dim[0], c1_nxy = c1.dim[0] * c1.dim[1];
    const physis_hip::BufWin<float> c1_w = physis_hip::BufWin<float>::Make(c1.p, c1_nxy * c1.dim[2], (long)zb * c1_nxy, (long)ze * c1_nxy);
    float c1_dv[2][VX];
    c1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c1_nx + zb * c1_nxy, c1_dv[0]);
    const int c2_nx = c2.dim[0], c2_nxy = c2.dim[0] * c2.dim[1];
    const physis_hip::BufWin<float> c2_w = physis_hip::BufWin<float>::Make(c2.p, c2_nxy * c2.dim[2], (long)zb * c2_nxy, (long)ze * c2_nxy);
    float c2_dv[2][VX];
    c2_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c2_nx + zb * c2_nxy, c2_dv[0]);
    const int bnd_nx = bnd.dim[0], bnd_nxy = bnd.dim[0] * bnd.dim[1];
    const physis_hip::BufWin<float> bnd_w = physis_hip::BufWin<float>::Make(bnd.p, bnd_nxy * bnd.dim[2], (long)zb * bnd_nxy, (long)ze * bnd_nxy);
    float bnd_dv[2][VX];
    bnd_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * bnd_nx + zb * bnd_nxy, bnd_dv[0]);
    const int wrk1_nx = wrk1.dim[0], wrk1_nxy = wrk1.dim[0] * wrk1.dim[1];
    const physis_hip::BufWin<float> wrk1_w = physis_hip::BufWin<float>::Make(wrk1.p, wrk1_nxy * wrk1.dim[2], (long)zb * wrk1_nxy, (long)ze * wrk1_nxy);
    float wrk1_dv[2][VX];
    wrk1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * wrk1_nx + zb * wrk1_nxy, wrk1_dv[0]);
    __syncthreads();
    __PSCtx_jacobi_kernel ctx;
    ctx.p0_p = p0.p;
    for (int d = 0; d < 3; ++d) ctx.p0_dim[d] = p0.dim[d];
    ctx.p1_p = p1.p;
    for (int d = 0; d < 3; ++d) ctx.p1_dim[d] = p1.dim[d];
    ctx.a0_p = a0.p;
    for (int d = 0; d < 3; ++d) ctx.a0_dim[d] = a0.dim[d];
    ctx.a1_p = a1.p;
    for (int d = 0; d < 3; ++d) ctx.a1_dim[d] = a1.dim[d];
    ctx.a2_p = a2.p;
    for (int d = 0; d < 3; ++d) ctx.a2_dim[d] = a2.dim[d];
    ctx.a3_p = a3.p;
    for (int d = 0; d < 3; ++d) ctx.a3_dim[d] = a3.dim[d];
    ctx.b0_p = b0.p;
    for (int d = 0; d < 3; ++d) ctx.b0_dim[d] = b0.dim[d];
    ctx.b1_p = b1.p;
    for (int d = 0; d < 3; ++d) ctx.b1_dim[d] = b1.dim[d];
    ctx.b2_p = b2.p;
    for (int d = 0; d < 3; ++d) ctx.b2_dim[d] = b2.dim[d];
    ctx.c0_p = c0.p;
    for (int d = 0; d < 3; ++d) ctx.c0_dim[d] = c0.dim[d];
    ctx.c1_p = c1.p;
    for (int d = 0; d < 3; ++d) ctx.c1_dim[d] = c1.dim[d];
    ctx.c2_p = c2.p;
    for (int d = 0; d < 3; ++d) ctx.c2_dim[d] = c2.dim[d];
    ctx.bnd_p = bnd.p;
    for (int d = 0; d < 3; ++d) ctx.bnd_dim[d] = bnd.dim[d];
    ctx.wrk1_p = wrk1.p;
    for (int d = 0; d < 3; ++d) ctx.wrk1_dim[d] = wrk1.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.p0_dim[0] & 3) == 0);
      __builtin_assume((ctx.p1_dim[0] & 3) == 0);
      __builtin_assume((ctx.a0_dim[0] & 3) == 0);
      __builtin_assume((ctx.a1_dim[0] & 3) == 0);
      __builtin_assume((ctx.a2_dim[0] & 3) == 0);
      __builtin_assume((ctx.a3_dim[0] & 3) == 0);
      __builtin_assume((ctx.b0_dim[0] & 3) == 0);
      __builtin_assume((ctx.b1_dim[0] & 3) == 0);
      __builtin_assume((ctx.b2_dim[0] & 3) == 0);
      __builtin_assume((ctx.c0_dim[0] & 3) == 0);
      __builtin_assume((ctx.c1_dim[0] & 3) == 0);
      __builtin_assume((ctx.c2_dim[0] & 3) == 0);
      __builtin_assume((ctx.bnd_dim[0] & 3) == 0);
      __builtin_assume((ctx.wrk1_dim[0] & 3) == 0);
    }
    constexpr int U = 2;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        a0_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a0_nx + (z + 1) * a0_nxy, a0_dv[nxt]);
        a1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a1_nx + (z + 1) * a1_nxy, a1_dv[nxt]);
        a2_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a2_nx + (z + 1) * a2_nxy, a2_dv[nxt]);
        a3_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * a3_nx + (z + 1) * a3_nxy, a3_dv[nxt]);
        b0_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * b0_nx + (z + 1) * b0_nxy, b0_dv[nxt]);
        b1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * b1_nx + (z + 1) * b1_nxy, b1_dv[nxt]);
        b2_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * b2_nx + (z + 1) * b2_nxy, b2_dv[nxt]);
        c0_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c0_nx + (z + 1) * c0_nxy, c0_dv[nxt]);
        c1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c1_nx + (z + 1) * c1_nxy, c1_dv[nxt]);
        c2_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c2_nx + (z + 1) * c2_nxy, c2_dv[nxt]);
        bnd_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * bnd_nx + (z + 1) * bnd_nxy, bnd_dv[nxt]);
        wrk1_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * wrk1_nx + (z + 1) * wrk1_nxy, wrk1_dv[nxt]);
        if (computes && z < ze) {
          float p0_r0[VX + 2];
          S_p0::template ReadRow<-1, 1>(p0_lds + physis_hip::RingSlot<4>(p0_base, 2) * S_p0::kPlane, wave + 0, lane, p0_r0);
          float p0_r1[VX + 2];
          S_p0::template ReadRow<-1, 1>(p0_lds + physis_hip::RingSlot<4>(p0_base, 1) * S_p0::kPlane, wave + 1, lane, p0_r1);
          float p0_r2[VX + 2];
          S_p0::template ReadRow<-1, 1>(p0_lds + physis_hip::RingSlot<4>(p0_base, 1) * S_p0::kPlane, wave + 0, lane, p0_r2);
          float p0_r3[VX + 0];
          S_p0::template ReadRow<0, 0>(p0_lds + physis_hip::RingSlot<4>(p0_base, 2) * S_p0::kPlane, wave + 1, lane, p0_r3);
          float p0_r4[VX + 0];
          S_p0::template ReadRow<0, 0>(p0_lds + physis_hip::RingSlot<4>(p0_base, 2) * S_p0::kPlane, wave + -1, lane, p0_r4);
          float p0_r5[VX + 0];
          S_p0::template ReadRow<0, 0>(p0_lds + physis_hip::RingSlot<4>(p0_base, 0) * S_p0::kPlane, wave + 1, lane, p0_r5);
          float p0_r6[VX + 0];
          S_p0::template ReadRow<0, 0>(p0_lds + physis_hip::RingSlot<4>(p0_base, 0) * S_p0::kPlane, wave + -1, lane, p0_r6);
          float p0_r7[VX + 2];
          S_p0::template ReadRow<-1, 1>(p0_lds + physis_hip::RingSlot<4>(p0_base, 1) * S_p0::kPlane, wave + -1, lane, p0_r7);
          float p0_r8[VX + 2];
          S_p0::template ReadRow<-1, 1>(p0_lds + physis_hip::RingSlot<4>(p0_base, 0) * S_p0::kPlane, wave + 0, lane, p0_r8);
          float p1_out[VX];
          unsigned p1_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.p0[0] = p0_r0[i + 1];
              ctx.p0[1] = p0_r1[i + 1];
              ctx.p0[2] = p0_r2[i + 2];
              ctx.p0[3] = p0_r3[i + 0];
              ctx.p0[4] = p0_r4[i + 0];
              ctx.p0[5] = p0_r5[i + 0];
              ctx.p0[6] = p0_r6[i + 0];
              ctx.p0[7] = p0_r1[i + 2];
              ctx.p0[8] = p0_r7[i + 2];
              ctx.p0[9] = p0_r1[i + 0];
              ctx.p0[10] = p0_r7[i + 0];
              ctx.p0[11] = p0_r0[i + 2];
              ctx.p0[12] = p0_r8[i + 2];
              ctx.p0[13] = p0_r0[i + 0];
              ctx.p0[14] = p0_r8[i + 0];
              ctx.p0[15] = p0_r8[i + 1];
              ctx.p0[16] = p0_r7[i + 1];
              ctx.p0[17] = p0_r2[i + 0];
              ctx.p0[18] = p0_r2[i + 1];
              ctx.p1_e = false;
              ctx.a0_c = a0_dv[cur][i];
              ctx.a1_c = a1_dv[cur][i];
              ctx.a2_c = a2_dv[cur][i];
              ctx.a3_c = a3_dv[cur][i];
              ctx.b0_c = b0_dv[cur][i];
              ctx.b1_c = b1_dv[cur][i];
              ctx.b2_c = b2_dv[cur][i];
              ctx.c0_c = c0_dv[cur][i];
              ctx.c1_c = c1_dv[cur][i];
              ctx.c2_c = c2_dv[cur][i];
              ctx.bnd_c = bnd_dv[cur][i];
              ctx.wrk1_c = wrk1_dv[cur][i];
              const float __r = jacobi_kernel(x, yrow, z, ctx, omega);
              if constexpr (RED >= 0) __racc = __in ? physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(__racc, __r) : __racc;
              p1_out[i] = ctx.p1_v;
              p1_mask |= (__in && ctx.p1_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(p1_ew, xs + yrow * p1_enx + z * p1_enxy, p1_out, p1_mask);
        }
        p0_st[k % PD].Store(p0_lds + physis_hip::RingSlot<4>(p0_base, 3) * S_p0::kPlane, wave, lane, p0_ra);
        __syncthreads();
        p0_st[k % PD].Load(p0_w, p0.p, p0.dim, p0_ra, z + 2 + PD);
        p0_base = physis_hip::RingSlot<4>(p0_base, 1);
      }
    }
  }
  if constexpr (RED >= 0) {
    __shared__ float __lds_red[BY];
    const float __r = physis_hip::BlockReduce<float, RED < 0 ? 0 : RED, 64 * BY>(__racc, __lds_red);
    if (threadIdx.x == 0) __red[blockIdx.x] = __r;
  }
}

template <int VX>
static physis_hip::RunShape __PSShape_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_jacobi_kernel<VX, 8, -1>, 64 * 8);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 8 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.p0, s.p1, s.a0, s.a1, s.a2, s.a3, s.b0, s.b1, s.b2, s.c0, s.c1, s.c2, s.bnd, s.wrk1}, 2));
}

template <int VX>
static int __PSLaunch_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_jacobi_kernel<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 8);
  {
  switch (red ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRun_jacobi_kernel<VX, 8, PS_MAX>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRun_jacobi_kernel<VX, 8, PS_MIN>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRun_jacobi_kernel<VX, 8, PS_SUM>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRun_jacobi_kernel<VX, 8, PS_PROD>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRun_jacobi_kernel<VX, 8, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s) {
  return (s.p0->dim[0] % 4 == 0 && s.p1->dim[0] % 4 == 0 && s.a0->dim[0] % 4 == 0 && s.a1->dim[0] % 4 == 0 && s.a2->dim[0] % 4 == 0 && s.a3->dim[0] % 4 == 0 && s.b0->dim[0] % 4 == 0 && s.b1->dim[0] % 4 == 0 && s.b2->dim[0] % 4 == 0 && s.c0->dim[0] % 4 == 0 && s.c1->dim[0] % 4 == 0 && s.c2->dim[0] % 4 == 0 && s.bnd->dim[0] % 4 == 0 && s.wrk1->dim[0] % 4 == 0) ? __PSShape_jacobi_kernel<4>(s).blocks
         : (s.dom.local_max[0] <= s.p0->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_jacobi_kernel<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_jacobi_kernel<1>(s).blocks;
}

static int __PSRun_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.p0, PS_FLOAT);
  physis_hip::CheckGrid3D(s.p1, PS_FLOAT);
  physis_hip::CheckGrid3D(s.a0, PS_FLOAT);
  physis_hip::CheckGrid3D(s.a1, PS_FLOAT);
  physis_hip::CheckGrid3D(s.a2, PS_FLOAT);
  physis_hip::CheckGrid3D(s.a3, PS_FLOAT);
  physis_hip::CheckGrid3D(s.b0, PS_FLOAT);
  physis_hip::CheckGrid3D(s.b1, PS_FLOAT);
  physis_hip::CheckGrid3D(s.b2, PS_FLOAT);
  physis_hip::CheckGrid3D(s.c0, PS_FLOAT);
  physis_hip::CheckGrid3D(s.c1, PS_FLOAT);
  physis_hip::CheckGrid3D(s.c2, PS_FLOAT);
  physis_hip::CheckGrid3D(s.bnd, PS_FLOAT);
  physis_hip::CheckGrid3D(s.wrk1, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.p1);
  return (s.p0->dim[0] % 4 == 0 && s.p1->dim[0] % 4 == 0 && s.a0->dim[0] % 4 == 0 && s.a1->dim[0] % 4 == 0 && s.a2->dim[0] % 4 == 0 && s.a3->dim[0] % 4 == 0 && s.b0->dim[0] % 4 == 0 && s.b1->dim[0] % 4 == 0 && s.b2->dim[0] % 4 == 0 && s.c0->dim[0] % 4 == 0 && s.c1->dim[0] % 4 == 0 && s.c2->dim[0] % 4 == 0 && s.bnd->dim[0] % 4 == 0 && s.wrk1->dim[0] % 4 == 0) ? __PSLaunch_jacobi_kernel<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.p0->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_jacobi_kernel<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_jacobi_kernel<1>(s, stream, red);
}

// Two-sweep run kernel of jacobi_kernel over a domain strictly inside
// the grid: one pass over src computes u' = jacobi_kernel(src) on the
// tile and a one-point halo (bg's own values outside the domain) and
// u'' = jacobi_kernel(u') two planes behind; dst <- u'', and bg <- u'
// when store_mid.  red1 / red2: per-block partials of the two sweeps.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, int RED, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_jacobi_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, __PSGrid3DFloat_dev bg, int store_mid, __PSGrid3DFloat_dev a0, __PSGrid3DFloat_dev a1, __PSGrid3DFloat_dev a2, __PSGrid3DFloat_dev a3, __PSGrid3DFloat_dev b0, __PSGrid3DFloat_dev b1, __PSGrid3DFloat_dev b2, __PSGrid3DFloat_dev c0, __PSGrid3DFloat_dev c1, __PSGrid3DFloat_dev c2, __PSGrid3DFloat_dev bnd, __PSGrid3DFloat_dev wrk1, float omega, physis_hip::RunShape sh, float *__restrict__ red1, float *__restrict__ red2) {
  constexpr int PD = 2, TX = 64 * VX, TY = BY - 4;
  typedef physis_hip::Stage<float, VX, BY, 2, 2, 4, false, float, RAGGED> SA;
  typedef physis_hip::Stage<float, VX, BY, 1, 1, 4, false> SB;
  __shared__ __attribute__((aligned(16))) float a_lds[SA::kLdsElems];
  __shared__ __attribute__((aligned(16))) float b_lds[SB::kLdsElems];
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, sh.tiles_y);
  const int x0 = (sh.x_first_tile + tc.bx) * TX;
  const int y0 = dom.local_min[1] + tc.by * TY;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  float acc1 = 0, acc2 = 0;
  if constexpr (RED >= 0) acc1 = acc2 = physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::identity();
  if (zb < ze) {
    const int yrow = y0 - 2 + wave;
    const bool mid_row = wave >= 1 && wave < BY - 1;
    const bool out_row = wave >= 2 && wave < BY - 2 && yrow < dom.local_max[1];
    const int xs = x0 + lane * VX;
    const int nx = src.dim[0], nxy = src.dim[0] * src.dim[1];
    const int n = nxy * src.dim[2];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) __builtin_assume((nx & 3) == 0);
    // u' halo columns x0 - 1 and x0 + TX of rows y0 - 1 .. y0 + TY: one
    // point per lane of wave 0 (which otherwise only loads)
    const bool hlane = wave == 0 && lane < 2 * (BY - 2);
    const int hr = 1 + (lane >> 1);
    const int px = (lane & 1) ? TX : -1;
    const int hx = x0 + px, hy = y0 - 2 + hr;
    const bool yin = yrow >= dom.local_min[1] && yrow < dom.local_max[1];
    const bool hin = hy >= dom.local_min[1] && hy < dom.local_max[1] &&
                     hx >= dom.local_min[0] && hx < dom.local_max[0];
    bool xin_all = true;
#pragma unroll
    for (int i = 0; i < VX; ++i)
      xin_all = xin_all && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
    const auto zin = [&](int z) { return z >= dom.local_min[2] && z < dom.local_max[2]; };
    const physis_hip::BufWin<float> aw = physis_hip::BufWin<float>::Make(src.p, n, (long)(zb - 3) * nxy, (long)(ze + 3) * nxy);
    const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, (long)zb * nxy, (long)ze * nxy);
    const physis_hip::BufWin<float> bw = physis_hip::BufWin<float>::Make(bg.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> mw = physis_hip::BufWin<float>::Make(bg.p, n, (long)zb * nxy, (long)ze * nxy);
    const physis_hip::BufWin<float> a0_w = physis_hip::BufWin<float>::Make(a0.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> a1_w = physis_hip::BufWin<float>::Make(a1.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> a2_w = physis_hip::BufWin<float>::Make(a2.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> a3_w = physis_hip::BufWin<float>::Make(a3.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> b0_w = physis_hip::BufWin<float>::Make(b0.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> b1_w = physis_hip::BufWin<float>::Make(b1.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> b2_w = physis_hip::BufWin<float>::Make(b2.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> c0_w = physis_hip::BufWin<float>::Make(c0.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> c1_w = physis_hip::BufWin<float>::Make(c1.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> c2_w = physis_hip::BufWin<float>::Make(c2.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> bnd_w = physis_hip::BufWin<float>::Make(bnd.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    const physis_hip::BufWin<float> wrk1_w = physis_hip::BufWin<float>::Make(wrk1.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    SA st[PD], pro[3];
    const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Load(aw, src.p, src.dim, ra, zb - 2 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      st[k].Load(aw, src.p, src.dim, ra, zb + 1 + k);
    float a0_c1[4][VX];
    float a1_c1[4][VX];
    float a2_c1[4][VX];
    float a3_c1[4][VX];
    float b0_c1[4][VX];
    float b1_c1[4][VX];
    float b2_c1[4][VX];
    float c0_c1[4][VX];
    float c1_c1[4][VX];
    float c2_c1[4][VX];
    float bnd_c1[4][VX];
    float wrk1_c1[4][VX];
    float bg_c1[4][VX];
    // loads of plane z for u': the lane's VX points on mid rows, its halo
    // point in wave 0; emitted-grid values only where a point lies
    // outside the domain
    auto load1 = [&](int z, int slot) {
      if (wave == 0) {
        const int o = hlane ? hx + hy * nx + z * nxy : physis_hip::kDrop;
        const int ob = hlane && !(hin && zin(z)) ? o : physis_hip::kDrop;
        a0_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&a0_c1[slot][0]));
        a1_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&a1_c1[slot][0]));
        a2_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&a2_c1[slot][0]));
        a3_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&a3_c1[slot][0]));
        b0_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&b0_c1[slot][0]));
        b1_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&b1_c1[slot][0]));
        b2_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&b2_c1[slot][0]));
        c0_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&c0_c1[slot][0]));
        c1_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&c1_c1[slot][0]));
        c2_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&c2_c1[slot][0]));
        bnd_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&bnd_c1[slot][0]));
        wrk1_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&wrk1_c1[slot][0]));
        bw.template Load<1>(ob, *reinterpret_cast<float (*)[1]>(&bg_c1[slot][0]));
      } else {
        const int o = mid_row ? xs + yrow * nx + z * nxy : physis_hip::kDrop;
        const int ob = mid_row && !(yin && xin_all && zin(z)) ? o : physis_hip::kDrop;
        a0_w.template Load<VX>(o, a0_c1[slot]);
        a1_w.template Load<VX>(o, a1_c1[slot]);
        a2_w.template Load<VX>(o, a2_c1[slot]);
        a3_w.template Load<VX>(o, a3_c1[slot]);
        b0_w.template Load<VX>(o, b0_c1[slot]);
        b1_w.template Load<VX>(o, b1_c1[slot]);
        b2_w.template Load<VX>(o, b2_c1[slot]);
        c0_w.template Load<VX>(o, c0_c1[slot]);
        c1_w.template Load<VX>(o, c1_c1[slot]);
        c2_w.template Load<VX>(o, c2_c1[slot]);
        bnd_w.template Load<VX>(o, bnd_c1[slot]);
        wrk1_w.template Load<VX>(o, wrk1_c1[slot]);
        bw.template Load<VX>(ob, bg_c1[slot]);
      }
    };
    load1(zb - 1, 0);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Store(a_lds + k * SA::kPlane, wave, lane, ra);
    __syncthreads();
    __PSCtx_jacobi_kernel ctx;
    ctx.p0_p = src.p;
    for (int d = 0; d < 3; ++d) ctx.p0_dim[d] = src.dim[d];
    ctx.p1_p = dst.p;
    for (int d = 0; d < 3; ++d) ctx.p1_dim[d] = dst.dim[d];
    ctx.a0_p = a0.p;
    for (int d = 0; d < 3; ++d) ctx.a0_dim[d] = a0.dim[d];
    ctx.a1_p = a1.p;
    for (int d = 0; d < 3; ++d) ctx.a1_dim[d] = a1.dim[d];
    ctx.a2_p = a2.p;
    for (int d = 0; d < 3; ++d) ctx.a2_dim[d] = a2.dim[d];
    ctx.a3_p = a3.p;
    for (int d = 0; d < 3; ++d) ctx.a3_dim[d] = a3.dim[d];
    ctx.b0_p = b0.p;
    for (int d = 0; d < 3; ++d) ctx.b0_dim[d] = b0.dim[d];
    ctx.b1_p = b1.p;
    for (int d = 0; d < 3; ++d) ctx.b1_dim[d] = b1.dim[d];
    ctx.b2_p = b2.p;
    for (int d = 0; d < 3; ++d) ctx.b2_dim[d] = b2.dim[d];
    ctx.c0_p = c0.p;
    for (int d = 0; d < 3; ++d) ctx.c0_dim[d] = c0.dim[d];
    ctx.c1_p = c1.p;
    for (int d = 0; d < 3; ++d) ctx.c1_dim[d] = c1.dim[d];
    ctx.c2_p = c2.p;
    for (int d = 0; d < 3; ++d) ctx.c2_dim[d] = c2.dim[d];
    ctx.bnd_p = bnd.p;
    for (int d = 0; d < 3; ++d) ctx.bnd_dim[d] = bnd.dim[d];
    ctx.wrk1_p = wrk1.p;
    for (int d = 0; d < 3; ++d) ctx.wrk1_dim[d] = wrk1.dim[d];
    for (int sc = zb - 1; sc <= ze + 1; sc += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = sc + k;
        const int abase = k, bbase = k;
        const int cur = k, nxt = (k + 1) & 3;
        const int old = (k + 2) & 3;
        if (s > ze + 1) break;  // uniform over the block
        load1(s + 1, nxt);
        if (mid_row && s <= ze) {
          float a_r0[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 0, lane, a_r0);
          float a_r1[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 1, lane, a_r1);
          float a_r2[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 0, lane, a_r2);
          float a_r3[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 1, lane, a_r3);
          float a_r4[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + -1, lane, a_r4);
          float a_r5[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 1, lane, a_r5);
          float a_r6[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + -1, lane, a_r6);
          float a_r7[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + -1, lane, a_r7);
          float a_r8[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 0, lane, a_r8);
          float uo[VX];
          unsigned m = 0;
          const bool own = out_row && s >= zb && s < ze;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.p0[0] = a_r0[i + 1];
            ctx.p0[1] = a_r1[i + 1];
            ctx.p0[2] = a_r2[i + 2];
            ctx.p0[3] = a_r3[i + 0];
            ctx.p0[4] = a_r4[i + 0];
            ctx.p0[5] = a_r5[i + 0];
            ctx.p0[6] = a_r6[i + 0];
            ctx.p0[7] = a_r1[i + 2];
            ctx.p0[8] = a_r7[i + 2];
            ctx.p0[9] = a_r1[i + 0];
            ctx.p0[10] = a_r7[i + 0];
            ctx.p0[11] = a_r0[i + 2];
            ctx.p0[12] = a_r8[i + 2];
            ctx.p0[13] = a_r0[i + 0];
            ctx.p0[14] = a_r8[i + 0];
            ctx.p0[15] = a_r8[i + 1];
            ctx.p0[16] = a_r7[i + 1];
            ctx.p0[17] = a_r2[i + 0];
            ctx.p0[18] = a_r2[i + 1];
            ctx.a0_c = a0_c1[cur][i];
            ctx.a1_c = a1_c1[cur][i];
            ctx.a2_c = a2_c1[cur][i];
            ctx.a3_c = a3_c1[cur][i];
            ctx.b0_c = b0_c1[cur][i];
            ctx.b1_c = b1_c1[cur][i];
            ctx.b2_c = b2_c1[cur][i];
            ctx.c0_c = c0_c1[cur][i];
            ctx.c1_c = c1_c1[cur][i];
            ctx.c2_c = c2_c1[cur][i];
            ctx.bnd_c = bnd_c1[cur][i];
            ctx.wrk1_c = wrk1_c1[cur][i];
            ctx.p1_e = false;
            const bool in = yin && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0] && zin(s);
            const float r = jacobi_kernel(xs + i, yrow, s, ctx, omega);
            if constexpr (RED >= 0) acc1 = in && own ? physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(acc1, r) : acc1;
            uo[i] = in ? ctx.p1_v : bg_c1[cur][i];
            m |= in ? 1u << i : 0u;
          }
          float *brow = b_lds + physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + wave * SB::kRow + SB::kPad + lane * VX;
#pragma unroll
          for (int i = 0; i < VX; ++i) brow[i] = uo[i];
          if (store_mid && own)
            physis_hip::StoreMasked<float, VX>(mw, xs + yrow * nx + s * nxy, uo, m);
        }
        if (hlane && s <= ze) {
          ctx.p0[0] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[1] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[2] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.p0[3] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[4] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[5] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[6] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[7] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
          ctx.p0[8] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.p0[9] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.p0[10] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
          ctx.p0[11] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.p0[12] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.p0[13] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
          ctx.p0[14] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
          ctx.p0[15] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[16] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
          ctx.p0[17] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
          ctx.p0[18] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.a0_c = a0_c1[cur][0];
          ctx.a1_c = a1_c1[cur][0];
          ctx.a2_c = a2_c1[cur][0];
          ctx.a3_c = a3_c1[cur][0];
          ctx.b0_c = b0_c1[cur][0];
          ctx.b1_c = b1_c1[cur][0];
          ctx.b2_c = b2_c1[cur][0];
          ctx.c0_c = c0_c1[cur][0];
          ctx.c1_c = c1_c1[cur][0];
          ctx.c2_c = c2_c1[cur][0];
          ctx.bnd_c = bnd_c1[cur][0];
          ctx.wrk1_c = wrk1_c1[cur][0];
          ctx.p1_e = false;
          (void)jacobi_kernel(hx, hy, s, ctx, omega);
          b_lds[physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + hr * SB::kRow + SB::kPad + px] = hin && zin(s) ? ctx.p1_v : bg_c1[cur][0];
        }
        if (out_row && s - 2 >= zb) {
          float b_r0[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 0, lane, b_r0);
          float b_r1[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 1, lane, b_r1);
          float b_r2[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 0, lane, b_r2);
          float b_r3[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 1, lane, b_r3);
          float b_r4[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + -1, lane, b_r4);
          float b_r5[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 1, lane, b_r5);
          float b_r6[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + -1, lane, b_r6);
          float b_r7[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + -1, lane, b_r7);
          float b_r8[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 0, lane, b_r8);
          float uu[VX];
          unsigned m = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.p0[0] = b_r0[i + 1];
            ctx.p0[1] = b_r1[i + 1];
            ctx.p0[2] = b_r2[i + 2];
            ctx.p0[3] = b_r3[i + 0];
            ctx.p0[4] = b_r4[i + 0];
            ctx.p0[5] = b_r5[i + 0];
            ctx.p0[6] = b_r6[i + 0];
            ctx.p0[7] = b_r1[i + 2];
            ctx.p0[8] = b_r7[i + 2];
            ctx.p0[9] = b_r1[i + 0];
            ctx.p0[10] = b_r7[i + 0];
            ctx.p0[11] = b_r0[i + 2];
            ctx.p0[12] = b_r8[i + 2];
            ctx.p0[13] = b_r0[i + 0];
            ctx.p0[14] = b_r8[i + 0];
            ctx.p0[15] = b_r8[i + 1];
            ctx.p0[16] = b_r7[i + 1];
            ctx.p0[17] = b_r2[i + 0];
            ctx.p0[18] = b_r2[i + 1];
            ctx.a0_c = a0_c1[old][i];
            ctx.a1_c = a1_c1[old][i];
            ctx.a2_c = a2_c1[old][i];
            ctx.a3_c = a3_c1[old][i];
            ctx.b0_c = b0_c1[old][i];
            ctx.b1_c = b1_c1[old][i];
            ctx.b2_c = b2_c1[old][i];
            ctx.c0_c = c0_c1[old][i];
            ctx.c1_c = c1_c1[old][i];
            ctx.c2_c = c2_c1[old][i];
            ctx.bnd_c = bnd_c1[old][i];
            ctx.wrk1_c = wrk1_c1[old][i];
            ctx.p1_e = false;
            const bool in = xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
            const float r = jacobi_kernel(xs + i, yrow, s - 2, ctx, omega);
            if constexpr (RED >= 0) acc2 = in ? physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(acc2, r) : acc2;
            uu[i] = ctx.p1_v;
            m |= in ? 1u << i : 0u;
          }
          physis_hip::StoreMasked<float, VX>(dw, xs + yrow * nx + (s - 2) * nxy, uu, m);
        }
        st[k % PD].Store(a_lds + physis_hip::RingSlot<4>(abase, 3) * SA::kPlane, wave, lane, ra);
        __syncthreads();
        st[k % PD].Load(aw, src.p, src.dim, ra, s + 2 + PD);
      }
    }
  }
  if constexpr (RED >= 0) {
    __shared__ float lds_r1[BY], lds_r2[BY];
    const float r1 = physis_hip::BlockReduce<float, RED < 0 ? 0 : RED, 64 * BY>(acc1, lds_r1);
    const float r2 = physis_hip::BlockReduce<float, RED < 0 ? 0 : RED, 64 * BY>(acc2, lds_r2);
    if (threadIdx.x == 0) {
      if (red1) red1[blockIdx.x] = r1;
      if (red2) red2[blockIdx.x] = r2;
    }
  } else {
    (void)acc1; (void)acc2; (void)red1; (void)red2;
  }
}

static constexpr int __PS2VX_jacobi_kernel = 1, __PS2BY_jacobi_kernel = 12;
template <int VX, int BY>
static physis_hip::RunShape __PSShape2_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_jacobi_kernel<VX, BY, -1, false>, 64 * BY);
  return physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.p0, s.p1, s.a0, s.a1, s.a2, s.a3, s.b0, s.b1, s.b2, s.c0, s.c1, s.c2, s.bnd, s.wrk1}, 3));
}

static int __PSBlocks2_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s) {
  return __PSShape2_jacobi_kernel<__PS2VX_jacobi_kernel, __PS2BY_jacobi_kernel>(s).blocks;
}

template <bool RAGGED>
static void __PSLaunch2R_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  constexpr int VX = __PS2VX_jacobi_kernel, BY = __PS2BY_jacobi_kernel;
  const physis_hip::RunShape sh = __PSShape2_jacobi_kernel<VX, BY>(s);
  if (sh.blocks == 0) return;
  const dim3 grid(sh.blocks), block(64 * BY);
  switch (red1 || red2 ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRun2_jacobi_kernel<VX, BY, PS_MAX, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red1, (float *)red2);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRun2_jacobi_kernel<VX, BY, PS_MIN, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red1, (float *)red2);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRun2_jacobi_kernel<VX, BY, PS_SUM, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red1, (float *)red2);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRun2_jacobi_kernel<VX, BY, PS_PROD, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red1, (float *)red2);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRun2_jacobi_kernel<VX, BY, -1, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.p1), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.a0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.a3), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.b2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c0), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.bnd), physis_hip::DevView<__PSGrid3DFloat_dev>(s.wrk1), s.omega, sh, (float *)red1, (float *)red2);
  }
}

static void __PSLaunch2_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  if (s.p0->dim[0] % __PS2VX_jacobi_kernel == 0)
    __PSLaunch2R_jacobi_kernel<false>(s, src, dst, store_mid, stream, red1, red2);
  else
    __PSLaunch2R_jacobi_kernel<__PS2VX_jacobi_kernel != 1>(s, src, dst, store_mid, stream, red1, red2);
}

// The pair (s0, s1) is jacobi_kernel(a -> b), jacobi_kernel(b -> a) over one domain strictly
// inside the grids, with the same centre-only grids (neither a nor b) and
// scalars: it may run as two-sweep passes.
static bool __PSFusable2_jacobi_kernel(const struct __PSStencil_jacobi_kernel &s0, const struct __PSStencil_jacobi_kernel &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.p0, *b = s0.p1;
  if (off || !a || !b || a == b || s1.p0 != b || s1.p1 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != s1.dom.local_min[d] ||
        s0.dom.local_max[d] != s1.dom.local_max[d]) return false;
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  }
  if (s0.a0 != s1.a0 || !s0.a0 || s0.a0 == a || s0.a0 == b || s0.a0->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.a0->dim[d] != a->dim[d]) return false;
  if (s0.a1 != s1.a1 || !s0.a1 || s0.a1 == a || s0.a1 == b || s0.a1->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.a1->dim[d] != a->dim[d]) return false;
  if (s0.a2 != s1.a2 || !s0.a2 || s0.a2 == a || s0.a2 == b || s0.a2->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.a2->dim[d] != a->dim[d]) return false;
  if (s0.a3 != s1.a3 || !s0.a3 || s0.a3 == a || s0.a3 == b || s0.a3->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.a3->dim[d] != a->dim[d]) return false;
  if (s0.b0 != s1.b0 || !s0.b0 || s0.b0 == a || s0.b0 == b || s0.b0->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.b0->dim[d] != a->dim[d]) return false;
  if (s0.b1 != s1.b1 || !s0.b1 || s0.b1 == a || s0.b1 == b || s0.b1->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.b1->dim[d] != a->dim[d]) return false;
  if (s0.b2 != s1.b2 || !s0.b2 || s0.b2 == a || s0.b2 == b || s0.b2->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.b2->dim[d] != a->dim[d]) return false;
  if (s0.c0 != s1.c0 || !s0.c0 || s0.c0 == a || s0.c0 == b || s0.c0->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.c0->dim[d] != a->dim[d]) return false;
  if (s0.c1 != s1.c1 || !s0.c1 || s0.c1 == a || s0.c1 == b || s0.c1->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.c1->dim[d] != a->dim[d]) return false;
  if (s0.c2 != s1.c2 || !s0.c2 || s0.c2 == a || s0.c2 == b || s0.c2->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.c2->dim[d] != a->dim[d]) return false;
  if (s0.bnd != s1.bnd || !s0.bnd || s0.bnd == a || s0.bnd == b || s0.bnd->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.bnd->dim[d] != a->dim[d]) return false;
  if (s0.wrk1 != s1.wrk1 || !s0.wrk1 || s0.wrk1 == a || s0.wrk1 == b || s0.wrk1->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.wrk1->dim[d] != a->dim[d]) return false;
  if (__builtin_memcmp(&s0.omega, &s1.omega, sizeof(s0.omega))) return false;
  if ((s0.__reduce_out == NULL) != (s1.__reduce_out == NULL) ||
      (s0.__reduce_out && s0.__reduce_op != s1.__reduce_op)) return false;
  return physis_hip::WindowsFit({a, b, s0.a0, s0.a1, s0.a2, s0.a3, s0.b0, s0.b1, s0.b2, s0.c0, s0.c1, s0.c2, s0.bnd, s0.wrk1}, 3);
}

static void __PSStencilRun_0(int iter, struct __PSStencil_jacobi_kernel s0, struct __PSStencil_jacobi_kernel s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("jacobi_kernel, jacobi_kernel");
  physis_hip::RunTimer timer(stream);
  physis_hip::ReduceSlots __slots;
  const bool __fuse = iter >= 2 && __PSFusable2_jacobi_kernel(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.p0->num_elms * sizeof(float), (iter) % 2 != 0);
  physis_hip::MapReducer red0(s0.__reduce_out, s0.__reduce_op, PS_FLOAT,
      s0.__reduce_out ? (!__fuse ? __PSBlocks_jacobi_kernel(s0) : __PSBlocks2_jacobi_kernel(s0)) : 0, iter, __slots);
  physis_hip::MapReducer red1(s1.__reduce_out, s1.__reduce_op, PS_FLOAT,
      s1.__reduce_out ? (!__fuse ? __PSBlocks_jacobi_kernel(s1) : __PSBlocks2_jacobi_kernel(s1)) : 0, iter, __slots);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.p0, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.p1, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.p0);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.p1);
    const size_t bytes = (size_t)s0.p0->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const int passes = iter;
    __PSGrid3DFloat_dev vt2 = va;
    physis_hip::CopyShell(vt.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    if (passes % 2) {
      vt2.p = (float *)__PSHipScratch(9, bytes);
      physis_hip::CopyShell(vt2.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    }
    __PSGrid3DFloat_dev src = va;
    for (int j = 0, i = 0; j < passes; ++j) {
      __PSGrid3DFloat_dev dst = (j % 2 == (passes % 2 ? 0 : 1)) ? va : vt;
      if (passes % 2 && j < 2) dst = j == 0 ? vt : vt2;
      const int pairs = 1;
      __PSLaunch2_jacobi_kernel(s0, src, dst, (j == passes - 1), stream, red0.Slot(i), red1.Slot(i));
      i += pairs;
      red0.After(i - 1);
      red1.After(i - 1);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_jacobi_kernel(s0, stream, red0.Slot(i));
    __PSRun_jacobi_kernel(s1, stream, red1.Slot(i));
    red0.After(i);
    red1.After(i);
  }
  red0.Finish(stream);
  red1.Finish(stream);
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void himeno_run(int nn, PSGrid3DFloat p0, PSGrid3DFloat p1, PSGrid3DFloat a0, PSGrid3DFloat a1, PSGrid3DFloat a2, PSGrid3DFloat a3, PSGrid3DFloat b0, PSGrid3DFloat b1, PSGrid3DFloat b2, PSGrid3DFloat c0, PSGrid3DFloat c1, PSGrid3DFloat c2, PSGrid3DFloat bnd, PSGrid3DFloat wrk1, float omega) {
  PSDomain3D inner = PSDomain3DNew(1, PSGridDim(p0, 0) - 1, 1, PSGridDim(p0, 1) - 1, 1, PSGridDim(p0, 2) - 1);
  __PSStencilRun_0(nn / 2, __PSStencilMap_jacobi_kernel(inner, p0, p1, a0, a1, a2, a3, b0, b1, b2, c0, c1, c2, bnd, wrk1, omega), __PSStencilMap_jacobi_kernel(inner, p1, p0, a0, a1, a2, a3, b0, b1, b2, c0, c1, c2, bnd, wrk1, omega));
}

}  // extern "C"

static void __PSStencilRun_1(int iter, struct __PSStencil_jacobi_kernel s0, struct __PSStencil_jacobi_kernel s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("jacobi_kernel, jacobi_kernel");
  physis_hip::RunTimer timer(stream);
  physis_hip::ReduceSlots __slots;
  const bool __fuse = iter >= 2 && __PSFusable2_jacobi_kernel(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.p0->num_elms * sizeof(float), (iter) % 2 != 0);
  physis_hip::MapReducer red0(s0.__reduce_out, s0.__reduce_op, PS_FLOAT,
      s0.__reduce_out ? (!__fuse ? __PSBlocks_jacobi_kernel(s0) : __PSBlocks2_jacobi_kernel(s0)) : 0, iter, __slots);
  physis_hip::MapReducer red1(s1.__reduce_out, s1.__reduce_op, PS_FLOAT,
      s1.__reduce_out ? (!__fuse ? __PSBlocks_jacobi_kernel(s1) : __PSBlocks2_jacobi_kernel(s1)) : 0, iter, __slots);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.p0, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.p1, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.p0);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.p1);
    const size_t bytes = (size_t)s0.p0->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const int passes = iter;
    __PSGrid3DFloat_dev vt2 = va;
    physis_hip::CopyShell(vt.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    if (passes % 2) {
      vt2.p = (float *)__PSHipScratch(9, bytes);
      physis_hip::CopyShell(vt2.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    }
    __PSGrid3DFloat_dev src = va;
    for (int j = 0, i = 0; j < passes; ++j) {
      __PSGrid3DFloat_dev dst = (j % 2 == (passes % 2 ? 0 : 1)) ? va : vt;
      if (passes % 2 && j < 2) dst = j == 0 ? vt : vt2;
      const int pairs = 1;
      __PSLaunch2_jacobi_kernel(s0, src, dst, (j == passes - 1), stream, red0.Slot(i), red1.Slot(i));
      i += pairs;
      red0.After(i - 1);
      red1.After(i - 1);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_jacobi_kernel(s0, stream, red0.Slot(i));
    __PSRun_jacobi_kernel(s1, stream, red1.Slot(i));
    red0.After(i);
    red1.After(i);
  }
  red0.Finish(stream);
  red1.Finish(stream);
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void himeno_run_gosa(int nn, PSGrid3DFloat p0, PSGrid3DFloat p1, PSGrid3DFloat a0, PSGrid3DFloat a1, PSGrid3DFloat a2, PSGrid3DFloat a3, PSGrid3DFloat b0, PSGrid3DFloat b1, PSGrid3DFloat b2, PSGrid3DFloat c0, PSGrid3DFloat c1, PSGrid3DFloat c2, PSGrid3DFloat bnd, PSGrid3DFloat wrk1, float omega, float * gosa_even, float * gosa_odd) {
  PSDomain3D inner = PSDomain3DNew(1, PSGridDim(p0, 0) - 1, 1, PSGridDim(p0, 1) - 1, 1, PSGridDim(p0, 2) - 1);
  __PSStencilRun_1(nn / 2, __PSStencilMapReduce_jacobi_kernel(gosa_even, PS_SUM, inner, p0, p1, a0, a1, a2, a3, b0, b1, b2, c0, c1, c2, bnd, wrk1, omega), __PSStencilMapReduce_jacobi_kernel(gosa_odd, PS_SUM, inner, p1, p0, a0, a1, a2, a3, b0, b1, b2, c0, c1, c2, bnd, wrk1, omega));
}

}  // extern "C"

