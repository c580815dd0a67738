// Generated by physisc-hip from udt7.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

extern "C" {

struct Point { float p; float q; };

DeclareGrid3D(Point, struct Point);

}  // extern "C"

// ---------------------------------------------- point type Point (struct Point)
// Type info of the reference's REF target (reference_runtime_builder.cc:
// 959-1065): one entry per member, scalar size, array rank and extents.
static __PSGridTypeMemberInfo __PSTypeMembers_Point[] = {
  {PS_FLOAT, sizeof(float), 0, {0}},
  {PS_FLOAT, sizeof(float), 0, {0}},
};
static __PSGridTypeInfo __PSTypeInfo_Point = {PS_USER, sizeof(struct Point), 2, __PSTypeMembers_Point};

// Device view: the first component plane of each member (component c
// of an array member, row-major, c * n elements further).
struct __PSUdtView_Point {
  float *m_p;
  float *m_q;
  long n;
  int dim[3];
};

static inline __PSUdtView_Point __PSUdtViewOf_Point(__PSGrid *g) {
  __PSUdtView_Point v;
  v.m_p = (float *)__PSGridUserMember(g, 0);
  v.m_q = (float *)__PSGridUserMember(g, 1);
  v.n = (long)g->num_elms;
  for (int d = 0; d < 3; ++d) v.dim[d] = g->dim[d];
  return v;
}

__device__ __forceinline__ struct Point __PSUdtLoad_Point(const __PSUdtView_Point &v, long off) {
  struct Point r{};
  if (off < 0) return r;
  r.p = v.m_p[off];
  r.q = v.m_q[off];
  return r;
}

__device__ __forceinline__ void __PSUdtStore_Point(const __PSUdtView_Point &v, long off, const struct Point &r) {
  v.m_p[off] = r.p;
  v.m_q[off] = r.q;
}

__device__ __forceinline__ struct Point __PSUdtMake_Point(float m0, float m1) {
  struct Point r;
  r.p = m0;
  r.q = m1;
  return r;
}

// ---------------------------------------------- stencil udt7_kernel
struct __PSStencil_udt7_kernel {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  float ce;
  float cw;
  float cn;
  float cs;
  float ct;
  float cb;
  float cc;
};

static struct __PSStencil_udt7_kernel __PSStencilMap_udt7_kernel(
    __PSDomain __dom, __PSGrid *g, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_udt7_kernel __s = {__dom, g, __PSGridGetID(g), ce, cw, cn, cs, ct, cb, cc};
  return __s;
}

// Stencil analysis of udt7_kernel (2.5D run kernel):
//   g  split into one grid per member it uses
//   g__p  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,1,0) 4:(0,-1,0) 5:(0,0,-1) 6:(0,0,1)
//   g__q  not read, emitted
//   two-sweep fusion of map pairs: no (a grid of user-defined points)
struct __PSCtx_udt7_kernel {
  float g__p[7];
  const float *g__p_p;
  int g__p_dim[3];
  float g__q_v;
  bool g__q_e;
  const float *g__q_p;
  int g__q_dim[3];
};

__device__ __forceinline__ void udt7_kernel(
    const int x, const int y, const int z, __PSCtx_udt7_kernel &__ctx, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  float v = cc * __ctx.g__p[0] + cw * __ctx.g__p[1] + ce * __ctx.g__p[2] + cs * __ctx.g__p[3] + cn * __ctx.g__p[4] + cb * __ctx.g__p[5] + ct * __ctx.g__p[6];
  (__ctx.g__q_v = (v), __ctx.g__q_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_udt7_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev g__p, __PSGrid3DFloat_dev g__q, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, false, float, RAGGED> S_g__p;
  __shared__ __attribute__((aligned(16))) float g__p_lds[S_g__p::kLdsElems];
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, sh.tiles_y);
  const int x0 = (sh.x_first_tile + tc.bx) * TX;
  const int y0 = dom.local_min[1] + tc.by * TY;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  if (zb < ze) {
    const int yrow = y0 - HY + wave;
    const bool computes = wave >= HY && wave < BY - HY && yrow < dom.local_max[1];
    const int xs = x0 + lane * VX;
    const int g__p_nxy = g__p.dim[0] * g__p.dim[1];
    const physis_hip::BufWin<float> g__p_w = physis_hip::BufWin<float>::Make(g__p.p, g__p_nxy * g__p.dim[2], (long)(zb + -2) * g__p_nxy, (long)(ze + 2) * g__p_nxy);
    S_g__p g__p_st[PD];
    const typename S_g__p::Addr g__p_ra = S_g__p::Prepare(g__p.dim, x0, yrow, lane);
    S_g__p g__p_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_pro[k].Load(g__p_w, g__p.p, g__p.dim, g__p_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g__p_st[k].Load(g__p_w, g__p.p, g__p.dim, g__p_ra, zb + 2 + k);
    int g__p_base = 0;
    const int g__q_enx = g__q.dim[0], g__q_enxy = g__q.dim[0] * g__q.dim[1];
    const physis_hip::BufWin<float> g__q_ew = physis_hip::BufWin<float>::Make(g__q.p, g__q_enxy * g__q.dim[2], (long)zb * g__q_enxy, (long)ze * g__q_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_pro[k].Store(g__p_lds + k * S_g__p::kPlane, wave, lane, g__p_ra);
    __syncthreads();
    __PSCtx_udt7_kernel ctx;
    ctx.g__p_p = g__p.p;
    for (int d = 0; d < 3; ++d) ctx.g__p_dim[d] = g__p.dim[d];
    ctx.g__q_p = g__q.p;
    for (int d = 0; d < 3; ++d) ctx.g__q_dim[d] = g__q.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g__p_dim[0] & 3) == 0);
      __builtin_assume((ctx.g__q_dim[0] & 3) == 0);
    }
    constexpr int U = 4;
    (void)g__p_base;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        const int g__p_base = k % 4;
        if (computes && z < ze) {
          float g__p_r0[VX + 2];
          S_g__p::template ReadRow<-1, 1>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 1) * S_g__p::kPlane, wave + 0, lane, g__p_r0);
          float g__p_r1[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 1) * S_g__p::kPlane, wave + 1, lane, g__p_r1);
          float g__p_r2[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 1) * S_g__p::kPlane, wave + -1, lane, g__p_r2);
          float g__p_r3[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 0) * S_g__p::kPlane, wave + 0, lane, g__p_r3);
          float g__p_r4[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 2) * S_g__p::kPlane, wave + 0, lane, g__p_r4);
          float g__q_out[VX];
          unsigned g__q_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g__p[0] = g__p_r0[i + 1];
              ctx.g__p[1] = g__p_r0[i + 0];
              ctx.g__p[2] = g__p_r0[i + 2];
              ctx.g__p[3] = g__p_r1[i + 0];
              ctx.g__p[4] = g__p_r2[i + 0];
              ctx.g__p[5] = g__p_r3[i + 0];
              ctx.g__p[6] = g__p_r4[i + 0];
              ctx.g__q_e = false;
              udt7_kernel(x, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
              g__q_out[i] = ctx.g__q_v;
              g__q_mask |= (__in && ctx.g__q_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g__q_ew, xs + yrow * g__q_enx + z * g__q_enxy, g__q_out, g__q_mask);
        }
        g__p_st[k % PD].Store(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 3) * S_g__p::kPlane, wave, lane, g__p_ra);
        __syncthreads();
        g__p_st[k % PD].Load(g__p_w, g__p.p, g__p.dim, g__p_ra, z + 2 + PD);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_udt7_kernel(const struct __PSStencil_udt7_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_udt7_kernel<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g}, 2));
}

template <int VX>
static int __PSLaunch_udt7_kernel(const struct __PSStencil_udt7_kernel &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_udt7_kernel<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_udt7_kernel<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g, 1, 0), s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_udt7_kernel(const struct __PSStencil_udt7_kernel &s) {
  return (s.g->dim[0] % 4 == 0) ? __PSShape_udt7_kernel<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_udt7_kernel<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_udt7_kernel<1>(s).blocks;
}

static int __PSRun_udt7_kernel(const struct __PSStencil_udt7_kernel &s, hipStream_t stream, void *red) {
  physis_hip::CheckUserGrid3D(s.g);
  physis_hip::CheckEmitDomain(s.dom, s.g);
  return (s.g->dim[0] % 4 == 0) ? __PSLaunch_udt7_kernel<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_udt7_kernel<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_udt7_kernel<1>(s, stream, red);
}

// ---------------------------------------------- stencil udt7_whole_kernel
struct __PSStencil_udt7_whole_kernel {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  float ce;
  float cw;
  float cn;
  float cs;
  float ct;
  float cb;
  float cc;
};

static struct __PSStencil_udt7_whole_kernel __PSStencilMap_udt7_whole_kernel(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_udt7_whole_kernel __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), ce, cw, cn, cs, ct, cb, cc};
  return __s;
}

// Stencil analysis of udt7_whole_kernel (2.5D run kernel):
//   g  split into one grid per member it uses
//   g2  split into one grid per member it uses
//   g__p  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,1,0) 4:(0,-1,0) 5:(0,0,-1) 6:(0,0,1)
//   g2__p  not read, emitted
//   g2__q  not read, emitted
//   two-sweep fusion of map pairs: no (a grid of user-defined points)
struct __PSCtx_udt7_whole_kernel {
  float g__p[7];
  const float *g__p_p;
  int g__p_dim[3];
  float g2__p_v;
  bool g2__p_e;
  const float *g2__p_p;
  int g2__p_dim[3];
  float g2__q_v;
  bool g2__q_e;
  const float *g2__q_p;
  int g2__q_dim[3];
};

__device__ __forceinline__ void udt7_whole_kernel(
    const int x, const int y, const int z, __PSCtx_udt7_whole_kernel &__ctx, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct Point c = __PSUdtMake_Point(__ctx.g__p[0], 0);
  struct Point w = __PSUdtMake_Point(__ctx.g__p[1], 0);
  struct Point e = __PSUdtMake_Point(__ctx.g__p[2], 0);
  struct Point s = __PSUdtMake_Point(__ctx.g__p[3], 0);
  struct Point n = __PSUdtMake_Point(__ctx.g__p[4], 0);
  struct Point b = __PSUdtMake_Point(__ctx.g__p[5], 0);
  struct Point t = __PSUdtMake_Point(__ctx.g__p[6], 0);
  struct Point v;
  v.p = c.p;
  v.q = cc * c.p + cw * w.p + ce * e.p + cs * s.p + cn * n.p + cb * b.p + ct * t.p;
  ((__ctx.g2__p_v = ((v).p), __ctx.g2__p_e = true), (__ctx.g2__q_v = ((v).q), __ctx.g2__q_e = true));
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_udt7_whole_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev g__p, __PSGrid3DFloat_dev g2__p, __PSGrid3DFloat_dev g2__q, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, false, float, RAGGED> S_g__p;
  __shared__ __attribute__((aligned(16))) float g__p_lds[S_g__p::kLdsElems];
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, sh.tiles_y);
  const int x0 = (sh.x_first_tile + tc.bx) * TX;
  const int y0 = dom.local_min[1] + tc.by * TY;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  if (zb < ze) {
    const int yrow = y0 - HY + wave;
    const bool computes = wave >= HY && wave < BY - HY && yrow < dom.local_max[1];
    const int xs = x0 + lane * VX;
    const int g__p_nxy = g__p.dim[0] * g__p.dim[1];
    const physis_hip::BufWin<float> g__p_w = physis_hip::BufWin<float>::Make(g__p.p, g__p_nxy * g__p.dim[2], (long)(zb + -2) * g__p_nxy, (long)(ze + 2) * g__p_nxy);
    S_g__p g__p_st[PD];
    const typename S_g__p::Addr g__p_ra = S_g__p::Prepare(g__p.dim, x0, yrow, lane);
    S_g__p g__p_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_pro[k].Load(g__p_w, g__p.p, g__p.dim, g__p_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g__p_st[k].Load(g__p_w, g__p.p, g__p.dim, g__p_ra, zb + 2 + k);
    int g__p_base = 0;
    const int g2__p_enx = g2__p.dim[0], g2__p_enxy = g2__p.dim[0] * g2__p.dim[1];
    const physis_hip::BufWin<float> g2__p_ew = physis_hip::BufWin<float>::Make(g2__p.p, g2__p_enxy * g2__p.dim[2], (long)zb * g2__p_enxy, (long)ze * g2__p_enxy);
    const int g2__q_enx = g2__q.dim[0], g2__q_enxy = g2__q.dim[0] * g2__q.dim[1];
    const physis_hip::BufWin<float> g2__q_ew = physis_hip::BufWin<float>::Make(g2__q.p, g2__q_enxy * g2__q.dim[2], (long)zb * g2__q_enxy, (long)ze * g2__q_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_pro[k].Store(g__p_lds + k * S_g__p::kPlane, wave, lane, g__p_ra);
    __syncthreads();
    __PSCtx_udt7_whole_kernel ctx;
    ctx.g__p_p = g__p.p;
    for (int d = 0; d < 3; ++d) ctx.g__p_dim[d] = g__p.dim[d];
    ctx.g2__p_p = g2__p.p;
    for (int d = 0; d < 3; ++d) ctx.g2__p_dim[d] = g2__p.dim[d];
    ctx.g2__q_p = g2__q.p;
    for (int d = 0; d < 3; ++d) ctx.g2__q_dim[d] = g2__q.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g__p_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2__p_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2__q_dim[0] & 3) == 0);
    }
    constexpr int U = 4;
    (void)g__p_base;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        const int g__p_base = k % 4;
        if (computes && z < ze) {
          float g__p_r0[VX + 2];
          S_g__p::template ReadRow<-1, 1>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 1) * S_g__p::kPlane, wave + 0, lane, g__p_r0);
          float g__p_r1[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 1) * S_g__p::kPlane, wave + 1, lane, g__p_r1);
          float g__p_r2[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 1) * S_g__p::kPlane, wave + -1, lane, g__p_r2);
          float g__p_r3[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 0) * S_g__p::kPlane, wave + 0, lane, g__p_r3);
          float g__p_r4[VX + 0];
          S_g__p::template ReadRow<0, 0>(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 2) * S_g__p::kPlane, wave + 0, lane, g__p_r4);
          float g2__p_out[VX];
          unsigned g2__p_mask = 0;
          float g2__q_out[VX];
          unsigned g2__q_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g__p[0] = g__p_r0[i + 1];
              ctx.g__p[1] = g__p_r0[i + 0];
              ctx.g__p[2] = g__p_r0[i + 2];
              ctx.g__p[3] = g__p_r1[i + 0];
              ctx.g__p[4] = g__p_r2[i + 0];
              ctx.g__p[5] = g__p_r3[i + 0];
              ctx.g__p[6] = g__p_r4[i + 0];
              ctx.g2__p_e = false;
              ctx.g2__q_e = false;
              udt7_whole_kernel(x, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
              g2__p_out[i] = ctx.g2__p_v;
              g2__p_mask |= (__in && ctx.g2__p_e) ? 1u << i : 0u;
              g2__q_out[i] = ctx.g2__q_v;
              g2__q_mask |= (__in && ctx.g2__q_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2__p_ew, xs + yrow * g2__p_enx + z * g2__p_enxy, g2__p_out, g2__p_mask);
          physis_hip::StoreMasked<float, VX>(g2__q_ew, xs + yrow * g2__q_enx + z * g2__q_enxy, g2__q_out, g2__q_mask);
        }
        g__p_st[k % PD].Store(g__p_lds + physis_hip::RingSlot<4>(g__p_base, 3) * S_g__p::kPlane, wave, lane, g__p_ra);
        __syncthreads();
        g__p_st[k % PD].Load(g__p_w, g__p.p, g__p.dim, g__p_ra, z + 2 + PD);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_udt7_whole_kernel(const struct __PSStencil_udt7_whole_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_udt7_whole_kernel<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_udt7_whole_kernel(const struct __PSStencil_udt7_whole_kernel &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_udt7_whole_kernel<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_udt7_whole_kernel<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g2, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g2, 1, 0), s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_udt7_whole_kernel(const struct __PSStencil_udt7_whole_kernel &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_udt7_whole_kernel<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_udt7_whole_kernel<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_udt7_whole_kernel<1>(s).blocks;
}

static int __PSRun_udt7_whole_kernel(const struct __PSStencil_udt7_whole_kernel &s, hipStream_t stream, void *red) {
  physis_hip::CheckUserGrid3D(s.g);
  physis_hip::CheckUserGrid3D(s.g2);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_udt7_whole_kernel<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_udt7_whole_kernel<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_udt7_whole_kernel<1>(s, stream, red);
}

extern "C" {

PSGrid3DPoint udt7_new(int nx, int ny, int nz) {
  return physis_hip::NewUserGrid(&__PSTypeInfo_Point, 3, nx, ny, nz);
}

void udt7_copyin(PSGrid3DPoint g, struct Point * in) {
  __PSGridCopyin(g, in, NULL);
}

void udt7_copyout(PSGrid3DPoint g, struct Point * out) {
  __PSGridCopyout(g, out, NULL);
}

void udt7_free(PSGrid3DPoint g) {
  __PSGridFree(g, NULL);
}

}  // extern "C"

static void __PSStencilRun_0(int iter, struct __PSStencil_udt7_kernel s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("udt7_kernel");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_udt7_kernel(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void udt7_run(PSGrid3DPoint g, int count, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  PSDomain3D dom = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1, 1, PSGridDim(g, 2) - 1);
  __PSStencilRun_0(count, __PSStencilMap_udt7_kernel(dom, g, ce, cw, cn, cs, ct, cb, cc));
}

}  // extern "C"

static void __PSStencilRun_1(int iter, struct __PSStencil_udt7_whole_kernel s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("udt7_whole_kernel");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_udt7_whole_kernel(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void udt7_whole_run(PSGrid3DPoint g, PSGrid3DPoint g2, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  PSDomain3D dom = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1, 1, PSGridDim(g, 2) - 1);
  __PSStencilRun_1(1, __PSStencilMap_udt7_whole_kernel(dom, g, g2, ce, cw, cn, cs, ct, cb, cc));
}

}  // extern "C"

