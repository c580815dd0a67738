// Generated by physisc-hip from redblack7.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

// ---------------------------------------------- stencil redblack7_kernel
struct __PSStencil_redblack7_kernel {
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
  int __rb;  // -1 all points, 0 red, 1 black, 2 red then black
};

static struct __PSStencil_redblack7_kernel __PSStencilMap_redblack7_kernel(
    __PSDomain __dom, __PSGrid *g, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_redblack7_kernel __s = {__dom, g, __PSGridGetID(g), ce, cw, cn, cs, ct, cb, cc, -1};
  return __s;
}

static struct __PSStencil_redblack7_kernel __PSStencilMapRed_redblack7_kernel(
    __PSDomain __dom, __PSGrid *g, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_redblack7_kernel __s = __PSStencilMap_redblack7_kernel(__dom, g, ce, cw, cn, cs, ct, cb, cc);
  __s.__rb = 0;
  return __s;
}

static struct __PSStencil_redblack7_kernel __PSStencilMapBlack_redblack7_kernel(
    __PSDomain __dom, __PSGrid *g, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_redblack7_kernel __s = __PSStencilMap_redblack7_kernel(__dom, g, ce, cw, cn, cs, ct, cb, cc);
  __s.__rb = 1;
  return __s;
}

static struct __PSStencil_redblack7_kernel __PSStencilMapRedBlack_redblack7_kernel(
    __PSDomain __dom, __PSGrid *g, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_redblack7_kernel __s = __PSStencilMap_redblack7_kernel(__dom, g, ce, cw, cn, cs, ct, cb, cc);
  __s.__rb = 2;
  return __s;
}

// Stencil analysis of redblack7_kernel (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic, emitted
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,-1,0) 4:(0,1,0) 5:(0,0,-1) 6:(0,0,1)
//   red-black: in-place colour sweep reads only the other colour
//   two-sweep fusion of map pairs: red-black: one pass per iteration (red, then black) over a domain inside the grid
struct __PSCtx_redblack7_kernel {
  float g[7];
  float g_v;
  bool g_e;
  const float *g_p;
  int g_dim[3];
};

__device__ __forceinline__ void redblack7_kernel(
    const int x, const int y, const int z, __PSCtx_redblack7_kernel &__ctx, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  float c, w, e, n, s, b, t;
  c = __ctx.g[0];
  w = __ctx.g[1];
  e = __ctx.g[2];
  n = __ctx.g[3];
  s = __ctx.g[4];
  b = __ctx.g[5];
  t = __ctx.g[6];
  (__ctx.g_v = (cc * c + cw * w + ce * e + cs * s + cn * n + cb * b + ct * t), __ctx.g_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_redblack7_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev g, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh, float *__restrict__ __red, int __rb) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, false, float, RAGGED> S_g;
  __shared__ __attribute__((aligned(16))) float g_lds[S_g::kLdsElems];
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
    const int g_nxy = g.dim[0] * g.dim[1];
    const physis_hip::BufWin<float> g_w = physis_hip::BufWin<float>::Make(g.p, g_nxy * g.dim[2], (long)(zb + -2) * g_nxy, (long)(ze + 2) * g_nxy);
    S_g g_st[PD];
    const typename S_g::Addr g_ra = S_g::Prepare(g.dim, x0, yrow, lane);
    S_g g_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Load(g_w, g.p, g.dim, g_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g_st[k].Load(g_w, g.p, g.dim, g_ra, zb + 2 + k);
    int g_base = 0;
    const int g_enx = g.dim[0], g_enxy = g.dim[0] * g.dim[1];
    const physis_hip::BufWin<float> g_ew = physis_hip::BufWin<float>::Make(g.p, g_enxy * g.dim[2], (long)zb * g_enxy, (long)ze * g_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_redblack7_kernel ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
    }
    constexpr int U = 4;
    (void)g_base;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        const int g_base = k % 4;
        if (computes && z < ze) {
          float g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r2);
          float g_r3[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r4);
          float g_out[VX];
          unsigned g_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0] &&
                (__rb < 0 || ((x + yrow + z + __rb) & 1) == 0);
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 0];
              ctx.g[2] = g_r0[i + 2];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g[5] = g_r3[i + 0];
              ctx.g[6] = g_r4[i + 0];
              ctx.g_e = false;
              redblack7_kernel(x, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
              g_out[i] = ctx.g_v;
              g_mask |= (__in && ctx.g_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g_ew, xs + yrow * g_enx + z * g_enxy, g_out, g_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<4>(g_base, 3) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 2 + PD);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_redblack7_kernel<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g}, 2));
}

template <int VX>
static int __PSLaunch_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_redblack7_kernel<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  for (int __c = s.__rb == 2 ? 0 : s.__rb; __c <= (s.__rb == 2 ? 1 : s.__rb); ++__c) {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_redblack7_kernel<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh, (float *)NULL, __c);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s) {
  return (s.g->dim[0] % 4 == 0) ? __PSShape_redblack7_kernel<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, true)) ? __PSShape_redblack7_kernel<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_redblack7_kernel<1>(s).blocks;
}

static int __PSRun_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g);
  return (s.g->dim[0] % 4 == 0) ? __PSLaunch_redblack7_kernel<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, true)) ? __PSLaunch_redblack7_kernel<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_redblack7_kernel<1>(s, stream, red);
}

// Two-sweep run kernel of redblack7_kernel (temporal blocking): one pass over src
// computes u' = redblack7_kernel(src) on the tile and a one-point halo and
// u'' = redblack7_kernel(u') three planes behind; dst <- u'', mid <- u' when
// mid is not NULL.  Two planes per barrier: an interval computes u' of
// planes s0 and s0 + 1 and u'' of s0 - 3 and s0 - 2 from rings of six
// slots (source plane p in slot (p - zb + 2) % 6, u'(p) in slot
// (p - zb + 1) % 6), then stores source planes s0 + 3 and s0 + 4.
// Red-black: one pass is one iteration (red sweep u', black sweep
// u''); dom is the map's domain, gd the whole grid the pass tiles.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_redblack7_kernel(
    __PSDomain dom, __PSDomain gd, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ mid, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh) {
  constexpr int PD = 2, TX = 64 * VX, TY = BY - 4;
  typedef physis_hip::Stage<float, VX, BY, 2, 2, 6, false, float, RAGGED> SA;
  typedef physis_hip::Stage<float, VX, BY, 1, 1, 6, false> SB;
  __shared__ __attribute__((aligned(16))) float a_lds[SA::kLdsElems];
  __shared__ __attribute__((aligned(16))) float b_lds[SB::kLdsElems];
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, sh.tiles_y);
  const int x0 = (sh.x_first_tile + tc.bx) * TX;
  const int y0 = gd.local_min[1] + tc.by * TY;
  const int zb = gd.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, gd.local_max[2]);
  if (zb >= ze) return;  // uniform over the block
  const int yrow = y0 - 2 + wave;
  const bool mid_row = wave >= 1 && wave < BY - 1;
  const bool out_row = wave >= 2 && wave < BY - 2 && yrow < gd.local_max[1];
  const int xs = x0 + lane * VX;
  const int nx = src.dim[0], nxy = src.dim[0] * src.dim[1];
  const int n = nxy * src.dim[2];
  // tiles start at multiples of TX
  __builtin_assume((xs & (VX - 1)) == 0);
  if constexpr (!RAGGED) __builtin_assume((nx & (VX - 1)) == 0);
  const physis_hip::BufWin<float> aw = physis_hip::BufWin<float>::Make(src.p, n, (long)(zb - 3) * nxy, (long)(ze + 3) * nxy);
  const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, (long)zb * nxy, (long)ze * nxy);
  const physis_hip::BufWin<float> mw = physis_hip::BufWin<float>::Make(mid ? mid : dst.p, n, (long)zb * nxy, (long)ze * nxy);
  SA st[PD], pro[4];
  const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    pro[k].Load(aw, src.p, src.dim, ra, zb - 2 + k);
#pragma unroll
  for (int k = 0; k < PD; ++k)
    st[k].Load(aw, src.p, src.dim, ra, zb + 2 + k);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    pro[k].Store(a_lds + k * SA::kPlane, wave, lane, ra);
  __syncthreads();
  __PSCtx_redblack7_kernel ctx;
  ctx.g_p = src.p;
  ctx.g_p = dst.p;
  for (int d = 0; d < 3; ++d) {
    ctx.g_dim[d] = src.dim[d];
    ctx.g_dim[d] = src.dim[d];
  }
  auto __uprime = [&](const int s, const int sm, const int sc, const int sp, const int bo) {
    if (mid_row && s <= ze) {
      float a_r0[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sc * SA::kPlane, wave + 0, lane, a_r0);
      float a_r1[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sc * SA::kPlane, wave + -1, lane, a_r1);
      float a_r2[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sc * SA::kPlane, wave + 1, lane, a_r2);
      float a_r3[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sm * SA::kPlane, wave + 0, lane, a_r3);
      float a_r4[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sp * SA::kPlane, wave + 0, lane, a_r4);
      float uo[VX];
      auto __half = [&](auto __odd) {
      constexpr int __p = decltype(__odd)::value ? 1 : 0;
#pragma unroll
      for (int i = 1 - __p; i < VX; i += 2) uo[i] = a_r0[i + 1];
      __builtin_assume(((yrow + s + 0) & 1) == __p);
#pragma unroll
      for (int i = __p; i < VX; i += 2) {
        ctx.g[0] = a_r0[i + 1];
        ctx.g[1] = a_r0[i + 0];
        ctx.g[2] = a_r0[i + 2];
        ctx.g[3] = a_r1[i + 0];
        ctx.g[4] = a_r2[i + 0];
        ctx.g[5] = a_r3[i + 0];
        ctx.g[6] = a_r4[i + 0];
        ctx.g_e = false;
        redblack7_kernel(xs + i, yrow, s, ctx, ce, cw, cn, cs, ct, cb, cc);
        uo[i] = ((xs + i) >= dom.local_min[0] && (xs + i) < dom.local_max[0] && yrow >= dom.local_min[1] && yrow < dom.local_max[1] && s >= dom.local_min[2] && s < dom.local_max[2] && (((xs + i) + yrow + s + 0) & 1) == 0) ? ctx.g_v : a_r0[i + 1];
      }
      };
      if ((yrow + s + 0) & 1)
        __half(physis_hip::Flag<true>{});
      else
        __half(physis_hip::Flag<false>{});
      SB::WriteRow(b_lds + bo * SB::kPlane, wave, lane, uo);
      if (mid && out_row && s >= zb && s < ze) {
        unsigned m = 0;
#pragma unroll
        for (int i = 0; i < VX; ++i)
          if (xs + i >= dom.local_min[0] && xs + i < dom.local_max[0]) m |= 1u << i;
        physis_hip::StoreMasked<float, VX>(mw, xs + yrow * nx + s * nxy, uo, m);
      }
    }
    if (wave == 0 && lane < 2 * (BY - 2) && s <= ze) {
      const int hr = 1 + (lane >> 1);
      const int px = (lane & 1) ? TX : -1;
      ctx.g[0] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[1] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g[2] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g[3] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[4] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[5] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[6] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g_e = false;
      redblack7_kernel(x0 + px, y0 - 2 + hr, s, ctx, ce, cw, cn, cs, ct, cb, cc);
      const float old = a_lds[sc * SA::kPlane + hr * SA::kRow + SA::kPad + px];
      const float now = ctx.g_v;
      b_lds[bo * SB::kPlane + hr * SB::kRow + SB::kPad + px] = ((x0 + px) >= dom.local_min[0] && (x0 + px) < dom.local_max[0] && (y0 - 2 + hr) >= dom.local_min[1] && (y0 - 2 + hr) < dom.local_max[1] && s >= dom.local_min[2] && s < dom.local_max[2] && (((x0 + px) + (y0 - 2 + hr) + s + 0) & 1) == 0) ? now : old;
    }
  };
  auto __udouble = [&](const int z, const int sm, const int sc, const int sp) {
    if (out_row && z >= zb && z < ze) {
      float b_r0[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sc * SB::kPlane, wave + 0, lane, b_r0);
      float b_r1[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sc * SB::kPlane, wave + -1, lane, b_r1);
      float b_r2[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sc * SB::kPlane, wave + 1, lane, b_r2);
      float b_r3[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sm * SB::kPlane, wave + 0, lane, b_r3);
      float b_r4[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sp * SB::kPlane, wave + 0, lane, b_r4);
      float uu[VX];
      unsigned m = 0;
      auto __half = [&](auto __odd) {
      constexpr int __p = decltype(__odd)::value ? 1 : 0;
#pragma unroll
      for (int i = 1 - __p; i < VX; i += 2) uu[i] = b_r0[i + 1];
      __builtin_assume(((yrow + z + 1) & 1) == __p);
#pragma unroll
      for (int i = __p; i < VX; i += 2) {
        ctx.g[0] = b_r0[i + 1];
        ctx.g[1] = b_r0[i + 0];
        ctx.g[2] = b_r0[i + 2];
        ctx.g[3] = b_r1[i + 0];
        ctx.g[4] = b_r2[i + 0];
        ctx.g[5] = b_r3[i + 0];
        ctx.g[6] = b_r4[i + 0];
        ctx.g_e = false;
        redblack7_kernel(xs + i, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
        uu[i] = ((xs + i) >= dom.local_min[0] && (xs + i) < dom.local_max[0] && yrow >= dom.local_min[1] && yrow < dom.local_max[1] && z >= dom.local_min[2] && z < dom.local_max[2] && (((xs + i) + yrow + z + 1) & 1) == 0) ? ctx.g_v : b_r0[i + 1];
      }
      };
      if ((yrow + z + 1) & 1)
        __half(physis_hip::Flag<true>{});
      else
        __half(physis_hip::Flag<false>{});
#pragma unroll
      for (int i = 0; i < VX; ++i)
        m |= (xs + i >= gd.local_min[0] && xs + i < gd.local_max[0]) ? 1u << i : 0u;
      physis_hip::StoreMasked<float, VX>(dw, xs + yrow * nx + z * nxy, uu, m);
    }
  };
  for (int t3 = 0;; t3 += 3) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int s0 = zb - 1 + 2 * (t3 + j);
      if (s0 - 3 > ze - 1) return;  // uniform over the block: every u'' done
      __uprime(s0, (2 * j) % 6, (2 * j + 1) % 6, (2 * j + 2) % 6, (2 * j) % 6);
      __uprime(s0 + 1, (2 * j + 1) % 6, (2 * j + 2) % 6, (2 * j + 3) % 6, (2 * j + 1) % 6);
      __udouble(s0 - 3, (2 * j + 2) % 6, (2 * j + 3) % 6, (2 * j + 4) % 6);
      __udouble(s0 - 2, (2 * j + 3) % 6, (2 * j + 4) % 6, (2 * j + 5) % 6);
      st[0].Store(a_lds + ((2 * j + 4) % 6) * SA::kPlane, wave, lane, ra);
      st[1].Store(a_lds + ((2 * j + 5) % 6) * SA::kPlane, wave, lane, ra);
      __syncthreads();
      st[0].Load(aw, src.p, src.dim, ra, s0 + 5);
      st[1].Load(aw, src.p, src.dim, ra, s0 + 6);
    }
  }
}

template <int VX>
static void __PSLaunch2V_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  constexpr int BY = 12;
  const __PSDomain gd = physis_hip::WholeDomain(s.g);
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_redblack7_kernel<VX, BY, false>, 64 * BY);
  const physis_hip::RunShape sh = physis_hip::PlanRun(gd, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g}, 3), 4);
  if (sh.blocks == 0) return;
  if (s.g->dim[0] % VX == 0)
    hipLaunchKernelGGL((__PSStencilRun2_redblack7_kernel<VX, BY, false>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, gd, src, dst, mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh);
  else
    hipLaunchKernelGGL((__PSStencilRun2_redblack7_kernel<VX, BY, true>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, gd, src, dst, mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh);
}

static void __PSLaunch2_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  if (physis_hip::PairVX(s.g->dim, false, true) == 4)
    __PSLaunch2V_redblack7_kernel<4>(s, src, dst, mid, stream);
  else
    __PSLaunch2V_redblack7_kernel<2>(s, src, dst, mid, stream);
}

// The red-black map s0 may run as one pass per iteration: both colours, a domain
// strictly inside the grid.
static bool __PSFusableRB_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s0) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g;
  if (off || !a || s0.__rb != 2 || a->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  if (!physis_hip::PassesPay(a->dim, false, true, true)) return false;
  return physis_hip::WindowsFit({a}, 3) &&
         physis_hip::HaveScratch((size_t)a->num_elms * sizeof(float), false);
}

// Resident-tile pass of redblack7_kernel: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_redblack7_kernel(
    __PSDomain dom, __PSDomain gd, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, float ce, float cw, float cn, float cs, float ct, float cb, float cc, int tiles_x, int tiles_y, physis_hip::TileReds red) {
  __shared__ float lds[2][TILE::kElems];
  constexpr int K = TILE::K, RX = TILE::RX, RY = TILE::RY;
  int b = physis_hip::XcdLogicalBlock(blockIdx.x, gridDim.x);
  const int x0 = gd.local_min[0] + (b % tiles_x) * TILE::TX;
  b /= tiles_x;
  const int y0 = gd.local_min[1] + (b % tiles_y) * TILE::TY;
  const int z0 = gd.local_min[2] + (b / tiles_y) * TILE::TZ;
  const int nx = src.dim[0], nxy = src.dim[0] * src.dim[1];
  const int n = nxy * src.dim[2];
  const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, 0, n);
  const physis_hip::BufWin<float> bw = physis_hip::BufWin<float>::Make(bg ? bg : dst.p, n, 0, n);
  physis_hip::TilePoint pt[K];
#pragma unroll
  for (int k = 0; k < K; ++k)
    pt[k] = physis_hip::OwnedPoint<TILE>(k, x0, y0, z0);
  physis_hip::LoadTile<TILE, false>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  __PSCtx_redblack7_kernel ctx;
  ctx.g_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
#pragma unroll
  for (int t = 1; t <= TILE::T; ++t) {
    const float *const cur = lds[(t - 1) & 1];
    float *const nxt = lds[t & 1];
#pragma unroll
    for (int k = 0; k < TILE::Count(t); ++k) {
      const physis_hip::TilePoint &p = pt[k];
      if (p.at < 0) continue;
      ctx.g[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g[1] = cur[p.at + -1 + RX * (0 + RY * (0))];
      ctx.g[2] = cur[p.at + 1 + RX * (0 + RY * (0))];
      ctx.g[3] = cur[p.at + 0 + RX * (-1 + RY * (0))];
      ctx.g[4] = cur[p.at + 0 + RX * (1 + RY * (0))];
      ctx.g[5] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g[6] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g_e = false;
      redblack7_kernel(p.x, p.y, p.z, ctx, ce, cw, cn, cs, ct, cb, cc);
      const int off = p.x + nx * p.y + nxy * p.z;
      const bool upd = p.x >= dom.local_min[0] && p.x < dom.local_max[0] &&
          p.y >= dom.local_min[1] && p.y < dom.local_max[1] &&
          p.z >= dom.local_min[2] && p.z < dom.local_max[2] &&
          ((p.x + p.y + p.z + t - 1) & 1) == 0;
      const float v[1] = {upd ? ctx.g_v : cur[p.at]};
      if (t < TILE::T) nxt[p.at] = v[0];
      const bool keep = p.x < nx && p.y < src.dim[1] && p.z < src.dim[2];
      if (k < TILE::Owned(0)) {
        if (t == TILE::T)
          dw.template Store<1>(keep ? off : physis_hip::kDrop, v);
        if (t == TILE::T - 1 && store_mid)
          bw.template Store<1>(keep ? off : physis_hip::kDrop, v);
      }
    }
    if (t < TILE::T) __syncthreads();
  }
  (void)red;
}

template <typename TILE>
static void __PSLaunchTile_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = physis_hip::WholeDomain(s.g);
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_redblack7_kernel<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, d, src, dst, bg, store_mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_redblack7_kernel(const struct __PSStencil_redblack7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(physis_hip::WholeDomain(s.g)))
    __PSLaunchTile_redblack7_kernel<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_redblack7_kernel<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

static void __PSStencilRun_0(int iter, struct __PSStencil_redblack7_kernel s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("redblack7_kernel");
  physis_hip::RunTimer timer(stream);
  int i0 = 0;
  if (iter >= 1 && __PSFusableRB_redblack7_kernel(s0)) {
    physis_hip::CheckGrid3D(s0.g, PS_FLOAT);
    const __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g);
    const size_t bytes = (size_t)s0.g->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    __PSGrid3DFloat_dev src = va;
    const bool __small = physis_hip::TilesBeatPairs(s0.g->dim, false, true);
    // (the last iteration may be left to the colour sweeps below)
    const int last = physis_hip::RedBlackLastAsSweeps(s0.g->dim, iter) ? 1 : 0;
    iter -= last;
    // two iterations a resident-tile pass, an even number of times, so that
    // the count of passes is odd when iter is
    const int two = __small ? iter / 2 & ~1 : 0;
    for (int i = 0, j = 0; i < iter; ++j) {
      const __PSGrid3DFloat_dev dst = (j % 2 == 0) ? vt : va;
      const int its = j < two ? 2 : 1;
      if (!__small)
        __PSLaunch2_redblack7_kernel(s0, src, dst, NULL, stream);
      else if (its == 2)
        __PSLaunchT_redblack7_kernel<4>(s0, src, dst, NULL, 0, stream, {});
      else
        __PSLaunchT_redblack7_kernel<2>(s0, src, dst, NULL, 0, stream, {});
      src = dst;
      i += its;
    }
    if (iter % 2) physis_hip::CopyDevice(va.p, vt.p, bytes, stream);
    i0 = iter;
    iter += last;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_redblack7_kernel(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void redblack7_run(PSGrid3DFloat g, int count, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  PSDomain3D dom = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1, 1, PSGridDim(g, 2) - 1);
  __PSStencilRun_0(count, __PSStencilMapRedBlack_redblack7_kernel(dom, g, ce, cw, cn, cs, ct, cb, cc));
}

}  // extern "C"

