// Generated by physisc-hip from diffusion7.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

// ---------------------------------------------- stencil diffusion7_kernel
struct __PSStencil_diffusion7_kernel {
  __PSDomain dom;
  __PSGrid *g1;
  int __g1_index;
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

static struct __PSStencil_diffusion7_kernel __PSStencilMap_diffusion7_kernel(
    __PSDomain __dom, __PSGrid *g1, __PSGrid *g2, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_diffusion7_kernel __s = {__dom, g1, __PSGridGetID(g1), g2, __PSGridGetID(g2), ce, cw, cn, cs, ct, cb, cc};
  return __s;
}

// Stencil analysis of diffusion7_kernel (2.5D run kernel):
//   g1  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,-1,0) 4:(0,1,0) 5:(0,0,-1) 6:(0,0,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes
struct __PSCtx_diffusion7_kernel {
  float g1[7];
  const float *g1_p;
  int g1_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void diffusion7_kernel(
    const int x, const int y, const int z, __PSCtx_diffusion7_kernel &__ctx, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  int nx, ny, nz;
  nx = __ctx.g1_dim[0];
  ny = __ctx.g1_dim[1];
  nz = __ctx.g1_dim[2];
  float c, w, e, n, s, b, t;
  c = __ctx.g1[0];
  if (x == 0)
    w = __ctx.g1[0];
  else
    w = __ctx.g1[1];
  if (x == nx - 1)
    e = __ctx.g1[0];
  else
    e = __ctx.g1[2];
  if (y == 0)
    n = __ctx.g1[0];
  else
    n = __ctx.g1[3];
  if (y == ny - 1)
    s = __ctx.g1[0];
  else
    s = __ctx.g1[4];
  if (z == 0)
    b = __ctx.g1[0];
  else
    b = __ctx.g1[5];
  if (z == nz - 1)
    t = __ctx.g1[0];
  else
    t = __ctx.g1[6];
  (__ctx.g2_v = (cc * c + cw * w + ce * e + cs * s + cn * n + cb * b + ct * t), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_diffusion7_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev g1, __PSGrid3DFloat_dev g2, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, false, float, RAGGED> S_g1;
  __shared__ __attribute__((aligned(16))) float g1_lds[S_g1::kLdsElems];
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
    const int g1_nxy = g1.dim[0] * g1.dim[1];
    const physis_hip::BufWin<float> g1_w = physis_hip::BufWin<float>::Make(g1.p, g1_nxy * g1.dim[2], (long)(zb + -2) * g1_nxy, (long)(ze + 2) * g1_nxy);
    S_g1 g1_st[PD];
    const typename S_g1::Addr g1_ra = S_g1::Prepare(g1.dim, x0, yrow, lane);
    S_g1 g1_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1_pro[k].Load(g1_w, g1.p, g1.dim, g1_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g1_st[k].Load(g1_w, g1.p, g1.dim, g1_ra, zb + 2 + k);
    int g1_base = 0;
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1_pro[k].Store(g1_lds + k * S_g1::kPlane, wave, lane, g1_ra);
    __syncthreads();
    __PSCtx_diffusion7_kernel ctx;
    ctx.g1_p = g1.p;
    for (int d = 0; d < 3; ++d) ctx.g1_dim[d] = g1.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g1_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
    }
    constexpr int U = 4;
    (void)g1_base;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        const int g1_base = k % 4;
        if (computes && z < ze) {
          float g1_r0[VX + 2];
          S_g1::template ReadRow<-1, 1>(g1_lds + physis_hip::RingSlot<4>(g1_base, 1) * S_g1::kPlane, wave + 0, lane, g1_r0);
          float g1_r1[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 1) * S_g1::kPlane, wave + -1, lane, g1_r1);
          float g1_r2[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 1) * S_g1::kPlane, wave + 1, lane, g1_r2);
          float g1_r3[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 0) * S_g1::kPlane, wave + 0, lane, g1_r3);
          float g1_r4[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 2) * S_g1::kPlane, wave + 0, lane, g1_r4);
          float g2_out[VX];
          unsigned g2_mask = 0;
          auto __pts = [&](auto __interior) {
            if constexpr (decltype(__interior)::value) {
              __builtin_assume(yrow >= 1); __builtin_assume(yrow <= ctx.g1_dim[1] - 2); __builtin_assume(yrow != 0); __builtin_assume(yrow != ctx.g1_dim[1] - 1); __builtin_assume(yrow >= 1); __builtin_assume(yrow <= ctx.g2_dim[1] - 2); __builtin_assume(yrow != 0); __builtin_assume(yrow != ctx.g2_dim[1] - 1); __builtin_assume(z >= 1); __builtin_assume(z <= ctx.g1_dim[2] - 2); __builtin_assume(z != 0); __builtin_assume(z != ctx.g1_dim[2] - 1); __builtin_assume(z >= 1); __builtin_assume(z <= ctx.g2_dim[2] - 2); __builtin_assume(z != 0); __builtin_assume(z != ctx.g2_dim[2] - 1); 
            }
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g1[0] = g1_r0[i + 1];
              ctx.g1[1] = g1_r0[i + 0];
              ctx.g1[2] = g1_r0[i + 2];
              ctx.g1[3] = g1_r1[i + 0];
              ctx.g1[4] = g1_r2[i + 0];
              ctx.g1[5] = g1_r3[i + 0];
              ctx.g1[6] = g1_r4[i + 0];
              ctx.g2_e = false;
              diffusion7_kernel(x, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          };
          if (yrow >= 1 && yrow <= ctx.g1_dim[1] - 2 && yrow >= 1 && yrow <= ctx.g2_dim[1] - 2 && z >= 1 && z <= ctx.g1_dim[2] - 2 && z >= 1 && z <= ctx.g2_dim[2] - 2)
            __pts(physis_hip::Flag<true>{});
          else
            __pts(physis_hip::Flag<false>{});
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g1_st[k % PD].Store(g1_lds + physis_hip::RingSlot<4>(g1_base, 3) * S_g1::kPlane, wave, lane, g1_ra);
        __syncthreads();
        g1_st[k % PD].Load(g1_w, g1.p, g1.dim, g1_ra, z + 2 + PD);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_diffusion7_kernel<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g1, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_diffusion7_kernel<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_diffusion7_kernel<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s) {
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_diffusion7_kernel<4>(s).blocks
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_diffusion7_kernel<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_diffusion7_kernel<1>(s).blocks;
}

static int __PSRun_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g1, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_diffusion7_kernel<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_diffusion7_kernel<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_diffusion7_kernel<1>(s, stream, red);
}

// Two-sweep run kernel of diffusion7_kernel (temporal blocking): one pass over src
// computes u' = diffusion7_kernel(src) on the tile and a one-point halo and
// u'' = diffusion7_kernel(u') three planes behind; dst <- u'', mid <- u' when
// mid is not NULL.  Two planes per barrier: an interval computes u' of
// planes s0 and s0 + 1 and u'' of s0 - 3 and s0 - 2 from rings of six
// slots (source plane p in slot (p - zb + 2) % 6, u'(p) in slot
// (p - zb + 1) % 6), then stores source planes s0 + 3 and s0 + 4.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_diffusion7_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ mid, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh) {
  constexpr int PD = 2, TX = 64 * VX, TY = BY - 4;
  typedef physis_hip::Stage<float, VX, BY, 2, 2, 6, false, float, RAGGED> SA;
  typedef physis_hip::Stage<float, VX, BY, 1, 1, 6, false> SB;
  __shared__ __attribute__((aligned(16))) float a_lds[SA::kLdsElems];
  __shared__ __attribute__((aligned(16))) float b_lds[SB::kLdsElems];
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, sh.tiles_y);
  const int x0 = (sh.x_first_tile + tc.bx) * TX;
  const int y0 = dom.local_min[1] + tc.by * TY;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  if (zb >= ze) return;  // uniform over the block
  const int yrow = y0 - 2 + wave;
  const bool mid_row = wave >= 1 && wave < BY - 1;
  const bool out_row = wave >= 2 && wave < BY - 2 && yrow < dom.local_max[1];
  const int xs = x0 + lane * VX;
  const int nx = src.dim[0], nxy = src.dim[0] * src.dim[1];
  const int n = nxy * src.dim[2];
  // tiles start at multiples of TX
  __builtin_assume((xs & (VX - 1)) == 0);
  if constexpr (!RAGGED) __builtin_assume((nx & (VX - 1)) == 0);
  const physis_hip::BufWin<float> aw = physis_hip::BufWin<float>::Make(src.p, n, (long)(zb - 3) * nxy, (long)(ze + 3) * nxy);
  const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, (long)zb * nxy, (long)ze * nxy);
  const physis_hip::BufWin<float> mw = physis_hip::BufWin<float>::Make(mid ? mid : dst.p, n, (long)zb * nxy, (long)ze * nxy);
  SA st[PD];
  const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    st[0].Load(aw, src.p, src.dim, ra, zb - 2 + k);
    st[0].Store(a_lds + k * SA::kPlane, wave, lane, ra);
  }
#pragma unroll
  for (int k = 0; k < PD; ++k)
    st[k].Load(aw, src.p, src.dim, ra, zb + 2 + k);
  __syncthreads();
  __PSCtx_diffusion7_kernel ctx;
  ctx.g1_p = src.p;
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) {
    ctx.g1_dim[d] = src.dim[d];
    ctx.g2_dim[d] = src.dim[d];
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
      auto __pts = [&](auto __interior) {
        if constexpr (decltype(__interior)::value) {
          __builtin_assume(yrow >= 1); __builtin_assume(yrow <= ctx.g1_dim[1] - 2); __builtin_assume(yrow != 0); __builtin_assume(yrow != ctx.g1_dim[1] - 1); __builtin_assume(s >= 1); __builtin_assume(s <= ctx.g1_dim[2] - 2); __builtin_assume(s != 0); __builtin_assume(s != ctx.g1_dim[2] - 1); 
        }
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g1[0] = a_r0[i + 1];
        ctx.g1[1] = a_r0[i + 0];
        ctx.g1[2] = a_r0[i + 2];
        ctx.g1[3] = a_r1[i + 0];
        ctx.g1[4] = a_r2[i + 0];
        ctx.g1[5] = a_r3[i + 0];
        ctx.g1[6] = a_r4[i + 0];
        ctx.g2_e = false;
        diffusion7_kernel(xs + i, yrow, s, ctx, ce, cw, cn, cs, ct, cb, cc);
        uo[i] = ctx.g2_v;
      }
      };
      if (yrow >= 1 && yrow <= ctx.g1_dim[1] - 2 && s >= 1 && s <= ctx.g1_dim[2] - 2)
        __pts(physis_hip::Flag<true>{});
      else
        __pts(physis_hip::Flag<false>{});
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
      ctx.g1[0] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[1] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g1[2] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g1[3] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[4] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[5] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[6] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g2_e = false;
      diffusion7_kernel(x0 + px, y0 - 2 + hr, s, ctx, ce, cw, cn, cs, ct, cb, cc);
      b_lds[bo * SB::kPlane + hr * SB::kRow + SB::kPad + px] = ctx.g2_v;
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
      auto __pts = [&](auto __interior) {
        if constexpr (decltype(__interior)::value) {
          __builtin_assume(yrow >= 1); __builtin_assume(yrow <= ctx.g1_dim[1] - 2); __builtin_assume(yrow != 0); __builtin_assume(yrow != ctx.g1_dim[1] - 1); __builtin_assume(z >= 1); __builtin_assume(z <= ctx.g1_dim[2] - 2); __builtin_assume(z != 0); __builtin_assume(z != ctx.g1_dim[2] - 1); 
        }
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g1[0] = b_r0[i + 1];
        ctx.g1[1] = b_r0[i + 0];
        ctx.g1[2] = b_r0[i + 2];
        ctx.g1[3] = b_r1[i + 0];
        ctx.g1[4] = b_r2[i + 0];
        ctx.g1[5] = b_r3[i + 0];
        ctx.g1[6] = b_r4[i + 0];
        ctx.g2_e = false;
        diffusion7_kernel(xs + i, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
        uu[i] = ctx.g2_v;
        m |= (xs + i >= dom.local_min[0] && xs + i < dom.local_max[0]) ? 1u << i : 0u;
      }
      };
      if (yrow >= 1 && yrow <= ctx.g1_dim[1] - 2 && z >= 1 && z <= ctx.g1_dim[2] - 2)
        __pts(physis_hip::Flag<true>{});
      else
        __pts(physis_hip::Flag<false>{});
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
static void __PSLaunch2V_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  constexpr int BY = 12;
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_diffusion7_kernel<VX, BY, false>, 64 * BY);
  const physis_hip::RunShape sh = physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g1}, 3), 4);
  if (sh.blocks == 0) return;
  if (s.g1->dim[0] % VX == 0)
    hipLaunchKernelGGL((__PSStencilRun2_diffusion7_kernel<VX, BY, false>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh);
  else
    hipLaunchKernelGGL((__PSStencilRun2_diffusion7_kernel<VX, BY, true>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh);
}

static void __PSLaunch2_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  if (physis_hip::PairVX(s.g1->dim, false, false) == 4)
    __PSLaunch2V_diffusion7_kernel<4>(s, src, dst, mid, stream);
  else
    __PSLaunch2V_diffusion7_kernel<2>(s, src, dst, mid, stream);
}

// The pair (s0, s1) is diffusion7_kernel(a -> b), diffusion7_kernel(b -> a) over the whole grid with the
// same scalars: it may run as two-sweep passes.
static bool __PSFusable2_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s0, const struct __PSStencil_diffusion7_kernel &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g1, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g1 != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != 0 || s0.dom.local_max[d] != a->dim[d]) return false;
    if (s1.dom.local_min[d] != 0 || s1.dom.local_max[d] != a->dim[d]) return false;
  }
  if (__builtin_memcmp(&s0.ce, &s1.ce, sizeof(s0.ce))) return false;
  if (__builtin_memcmp(&s0.cw, &s1.cw, sizeof(s0.cw))) return false;
  if (__builtin_memcmp(&s0.cn, &s1.cn, sizeof(s0.cn))) return false;
  if (__builtin_memcmp(&s0.cs, &s1.cs, sizeof(s0.cs))) return false;
  if (__builtin_memcmp(&s0.ct, &s1.ct, sizeof(s0.ct))) return false;
  if (__builtin_memcmp(&s0.cb, &s1.cb, sizeof(s0.cb))) return false;
  if (__builtin_memcmp(&s0.cc, &s1.cc, sizeof(s0.cc))) return false;
  if (!physis_hip::PassesPay(a->dim, false, false, true)) return false;
  return physis_hip::WindowsFit({a}, 3);
}

// Resident-tile pass of diffusion7_kernel: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_diffusion7_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, float ce, float cw, float cn, float cs, float ct, float cb, float cc, int tiles_x, int tiles_y, physis_hip::TileReds red) {
  __shared__ float lds[2][TILE::kElems];
  constexpr int K = TILE::K, RX = TILE::RX, RY = TILE::RY;
  int b = physis_hip::XcdLogicalBlock(blockIdx.x, gridDim.x);
  const int x0 = dom.local_min[0] + (b % tiles_x) * TILE::TX;
  b /= tiles_x;
  const int y0 = dom.local_min[1] + (b % tiles_y) * TILE::TY;
  const int z0 = dom.local_min[2] + (b / tiles_y) * TILE::TZ;
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
  __PSCtx_diffusion7_kernel ctx;
  ctx.g1_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g1_dim[d] = src.dim[d];
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = src.dim[d];
#pragma unroll
  for (int t = 1; t <= TILE::T; ++t) {
    const float *const cur = lds[(t - 1) & 1];
    float *const nxt = lds[t & 1];
#pragma unroll
    for (int k = 0; k < TILE::Count(t); ++k) {
      const physis_hip::TilePoint &p = pt[k];
      if (p.at < 0) continue;
      ctx.g1[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g1[1] = cur[p.at + -1 + RX * (0 + RY * (0))];
      ctx.g1[2] = cur[p.at + 1 + RX * (0 + RY * (0))];
      ctx.g1[3] = cur[p.at + 0 + RX * (-1 + RY * (0))];
      ctx.g1[4] = cur[p.at + 0 + RX * (1 + RY * (0))];
      ctx.g1[5] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g1[6] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g2_e = false;
      diffusion7_kernel(p.x, p.y, p.z, ctx, ce, cw, cn, cs, ct, cb, cc);
      const int off = p.x + nx * p.y + nxy * p.z;
      const float v[1] = {ctx.g2_v};
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
static void __PSLaunchTile_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_diffusion7_kernel<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_diffusion7_kernel(const struct __PSStencil_diffusion7_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_diffusion7_kernel<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_diffusion7_kernel<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil diffusion7_periodic_kernel
struct __PSStencil_diffusion7_periodic_kernel {
  __PSDomain dom;
  __PSGrid *g1;
  int __g1_index;
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

static struct __PSStencil_diffusion7_periodic_kernel __PSStencilMap_diffusion7_periodic_kernel(
    __PSDomain __dom, __PSGrid *g1, __PSGrid *g2, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  struct __PSStencil_diffusion7_periodic_kernel __s = {__dom, g1, __PSGridGetID(g1), g2, __PSGridGetID(g2), ce, cw, cn, cs, ct, cb, cc};
  return __s;
}

// Stencil analysis of diffusion7_periodic_kernel (2.5D run kernel):
//   g1  staged x[-1,1] y[-1,1] z[-1,1] periodic
//     offsets 0:(0,0,0) 1:(-1,0,0)p 2:(1,0,0)p 3:(0,-1,0)p 4:(0,1,0)p 5:(0,0,-1)p 6:(0,0,1)p
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes
struct __PSCtx_diffusion7_periodic_kernel {
  float g1[7];
  const float *g1_p;
  int g1_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void diffusion7_periodic_kernel(
    const int x, const int y, const int z, __PSCtx_diffusion7_periodic_kernel &__ctx, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  float c, w, e, n, s, b, t;
  c = __ctx.g1[0];
  w = __ctx.g1[1];
  e = __ctx.g1[2];
  n = __ctx.g1[3];
  s = __ctx.g1[4];
  b = __ctx.g1[5];
  t = __ctx.g1[6];
  (__ctx.g2_v = (cc * c + cw * w + ce * e + cs * s + cn * n + cb * b + ct * t), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_diffusion7_periodic_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev g1, __PSGrid3DFloat_dev g2, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, true, float, RAGGED> S_g1;
  __shared__ __attribute__((aligned(16))) float g1_lds[S_g1::kLdsElems];
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
    const int g1_nxy = g1.dim[0] * g1.dim[1];
    const physis_hip::BufWin<float> g1_w = physis_hip::BufWin<float>::Make(g1.p, g1_nxy * g1.dim[2], (long)(zb + -2) * g1_nxy, (long)(ze + 2) * g1_nxy);
    S_g1 g1_st[PD];
    const typename S_g1::Addr g1_ra = S_g1::Prepare(g1.dim, x0, yrow, lane);
    S_g1 g1_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1_pro[k].Load(g1_w, g1.p, g1.dim, g1_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g1_st[k].Load(g1_w, g1.p, g1.dim, g1_ra, zb + 2 + k);
    int g1_base = 0;
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1_pro[k].Store(g1_lds + k * S_g1::kPlane, wave, lane, g1_ra);
    __syncthreads();
    __PSCtx_diffusion7_periodic_kernel ctx;
    ctx.g1_p = g1.p;
    for (int d = 0; d < 3; ++d) ctx.g1_dim[d] = g1.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g1_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
    }
    constexpr int U = 4;
    (void)g1_base;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        const int g1_base = k % 4;
        if (computes && z < ze) {
          float g1_r0[VX + 2];
          S_g1::template ReadRow<-1, 1>(g1_lds + physis_hip::RingSlot<4>(g1_base, 1) * S_g1::kPlane, wave + 0, lane, g1_r0);
          float g1_r1[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 1) * S_g1::kPlane, wave + -1, lane, g1_r1);
          float g1_r2[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 1) * S_g1::kPlane, wave + 1, lane, g1_r2);
          float g1_r3[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 0) * S_g1::kPlane, wave + 0, lane, g1_r3);
          float g1_r4[VX + 0];
          S_g1::template ReadRow<0, 0>(g1_lds + physis_hip::RingSlot<4>(g1_base, 2) * S_g1::kPlane, wave + 0, lane, g1_r4);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g1[0] = g1_r0[i + 1];
              ctx.g1[1] = g1_r0[i + 0];
              ctx.g1[2] = g1_r0[i + 2];
              ctx.g1[3] = g1_r1[i + 0];
              ctx.g1[4] = g1_r2[i + 0];
              ctx.g1[5] = g1_r3[i + 0];
              ctx.g1[6] = g1_r4[i + 0];
              ctx.g2_e = false;
              diffusion7_periodic_kernel(x, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g1_st[k % PD].Store(g1_lds + physis_hip::RingSlot<4>(g1_base, 3) * S_g1::kPlane, wave, lane, g1_ra);
        __syncthreads();
        g1_st[k % PD].Load(g1_w, g1.p, g1.dim, g1_ra, z + 2 + PD);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_diffusion7_periodic_kernel<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g1, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_diffusion7_periodic_kernel<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_diffusion7_periodic_kernel<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s) {
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_diffusion7_periodic_kernel<4>(s).blocks
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSShape_diffusion7_periodic_kernel<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_diffusion7_periodic_kernel<1>(s).blocks;
}

static int __PSRun_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g1, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_diffusion7_periodic_kernel<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSLaunch_diffusion7_periodic_kernel<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_diffusion7_periodic_kernel<1>(s, stream, red);
}

// Two-sweep run kernel of diffusion7_periodic_kernel (temporal blocking): one pass over src
// computes u' = diffusion7_periodic_kernel(src) on the tile and a one-point halo and
// u'' = diffusion7_periodic_kernel(u') three planes behind; dst <- u'', mid <- u' when
// mid is not NULL.  Two planes per barrier: an interval computes u' of
// planes s0 and s0 + 1 and u'' of s0 - 3 and s0 - 2 from rings of six
// slots (source plane p in slot (p - zb + 2) % 6, u'(p) in slot
// (p - zb + 1) % 6), then stores source planes s0 + 3 and s0 + 4.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_diffusion7_periodic_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ mid, float ce, float cw, float cn, float cs, float ct, float cb, float cc, physis_hip::RunShape sh) {
  constexpr int PD = 2, TX = 64 * VX, TY = BY - 4;
  typedef physis_hip::Stage<float, VX, BY, 2, 2, 6, true, float, RAGGED> SA;
  typedef physis_hip::Stage<float, VX, BY, 1, 1, 6, false> SB;
  __shared__ __attribute__((aligned(16))) float a_lds[SA::kLdsElems];
  __shared__ __attribute__((aligned(16))) float b_lds[SB::kLdsElems];
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, sh.tiles_y);
  const int x0 = (sh.x_first_tile + tc.bx) * TX;
  const int y0 = dom.local_min[1] + tc.by * TY;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  if (zb >= ze) return;  // uniform over the block
  const int yrow = y0 - 2 + wave;
  const bool mid_row = wave >= 1 && wave < BY - 1;
  const bool out_row = wave >= 2 && wave < BY - 2 && yrow < dom.local_max[1];
  const int xs = x0 + lane * VX;
  const int nx = src.dim[0], nxy = src.dim[0] * src.dim[1];
  const int n = nxy * src.dim[2];
  // tiles start at multiples of TX
  __builtin_assume((xs & (VX - 1)) == 0);
  if constexpr (!RAGGED) __builtin_assume((nx & (VX - 1)) == 0);
  const physis_hip::BufWin<float> aw = physis_hip::BufWin<float>::Make(src.p, n, (long)(zb - 3) * nxy, (long)(ze + 3) * nxy);
  const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, (long)zb * nxy, (long)ze * nxy);
  const physis_hip::BufWin<float> mw = physis_hip::BufWin<float>::Make(mid ? mid : dst.p, n, (long)zb * nxy, (long)ze * nxy);
  SA st[PD];
  const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    st[0].Load(aw, src.p, src.dim, ra, zb - 2 + k);
    st[0].Store(a_lds + k * SA::kPlane, wave, lane, ra);
  }
#pragma unroll
  for (int k = 0; k < PD; ++k)
    st[k].Load(aw, src.p, src.dim, ra, zb + 2 + k);
  __syncthreads();
  __PSCtx_diffusion7_periodic_kernel ctx;
  ctx.g1_p = src.p;
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) {
    ctx.g1_dim[d] = src.dim[d];
    ctx.g2_dim[d] = src.dim[d];
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
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g1[0] = a_r0[i + 1];
        ctx.g1[1] = a_r0[i + 0];
        ctx.g1[2] = a_r0[i + 2];
        ctx.g1[3] = a_r1[i + 0];
        ctx.g1[4] = a_r2[i + 0];
        ctx.g1[5] = a_r3[i + 0];
        ctx.g1[6] = a_r4[i + 0];
        ctx.g2_e = false;
        diffusion7_periodic_kernel(xs + i, yrow, s, ctx, ce, cw, cn, cs, ct, cb, cc);
        uo[i] = ctx.g2_v;
      }
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
      ctx.g1[0] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[1] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g1[2] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g1[3] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[4] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[5] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g1[6] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g2_e = false;
      diffusion7_periodic_kernel(x0 + px, y0 - 2 + hr, s, ctx, ce, cw, cn, cs, ct, cb, cc);
      b_lds[bo * SB::kPlane + hr * SB::kRow + SB::kPad + px] = ctx.g2_v;
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
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g1[0] = b_r0[i + 1];
        ctx.g1[1] = b_r0[i + 0];
        ctx.g1[2] = b_r0[i + 2];
        ctx.g1[3] = b_r1[i + 0];
        ctx.g1[4] = b_r2[i + 0];
        ctx.g1[5] = b_r3[i + 0];
        ctx.g1[6] = b_r4[i + 0];
        ctx.g2_e = false;
        diffusion7_periodic_kernel(xs + i, yrow, z, ctx, ce, cw, cn, cs, ct, cb, cc);
        uu[i] = ctx.g2_v;
        m |= (xs + i >= dom.local_min[0] && xs + i < dom.local_max[0]) ? 1u << i : 0u;
      }
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
static void __PSLaunch2V_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  constexpr int BY = 12;
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_diffusion7_periodic_kernel<VX, BY, false>, 64 * BY);
  const physis_hip::RunShape sh = physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g1}, 3), 4);
  if (sh.blocks == 0) return;
  if (s.g1->dim[0] % VX == 0)
    hipLaunchKernelGGL((__PSStencilRun2_diffusion7_periodic_kernel<VX, BY, false>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh);
  else
    hipLaunchKernelGGL((__PSStencilRun2_diffusion7_periodic_kernel<VX, BY, true>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, sh);
}

static void __PSLaunch2_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  if (physis_hip::PairVX(s.g1->dim, true, false) == 4)
    __PSLaunch2V_diffusion7_periodic_kernel<4>(s, src, dst, mid, stream);
  else
    __PSLaunch2V_diffusion7_periodic_kernel<2>(s, src, dst, mid, stream);
}

// The pair (s0, s1) is diffusion7_periodic_kernel(a -> b), diffusion7_periodic_kernel(b -> a) over the whole grid with the
// same scalars: it may run as two-sweep passes.
static bool __PSFusable2_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s0, const struct __PSStencil_diffusion7_periodic_kernel &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g1, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g1 != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != 0 || s0.dom.local_max[d] != a->dim[d]) return false;
    if (s1.dom.local_min[d] != 0 || s1.dom.local_max[d] != a->dim[d]) return false;
  }
  if (__builtin_memcmp(&s0.ce, &s1.ce, sizeof(s0.ce))) return false;
  if (__builtin_memcmp(&s0.cw, &s1.cw, sizeof(s0.cw))) return false;
  if (__builtin_memcmp(&s0.cn, &s1.cn, sizeof(s0.cn))) return false;
  if (__builtin_memcmp(&s0.cs, &s1.cs, sizeof(s0.cs))) return false;
  if (__builtin_memcmp(&s0.ct, &s1.ct, sizeof(s0.ct))) return false;
  if (__builtin_memcmp(&s0.cb, &s1.cb, sizeof(s0.cb))) return false;
  if (__builtin_memcmp(&s0.cc, &s1.cc, sizeof(s0.cc))) return false;
  if (!physis_hip::PassesPay(a->dim, true, false, true)) return false;
  return physis_hip::WindowsFit({a}, 3);
}

// Resident-tile pass of diffusion7_periodic_kernel: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_diffusion7_periodic_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, float ce, float cw, float cn, float cs, float ct, float cb, float cc, int tiles_x, int tiles_y, physis_hip::TileReds red) {
  __shared__ float lds[2][TILE::kElems];
  constexpr int K = TILE::K, RX = TILE::RX, RY = TILE::RY;
  int b = physis_hip::XcdLogicalBlock(blockIdx.x, gridDim.x);
  const int x0 = dom.local_min[0] + (b % tiles_x) * TILE::TX;
  b /= tiles_x;
  const int y0 = dom.local_min[1] + (b % tiles_y) * TILE::TY;
  const int z0 = dom.local_min[2] + (b / tiles_y) * TILE::TZ;
  const int nx = src.dim[0], nxy = src.dim[0] * src.dim[1];
  const int n = nxy * src.dim[2];
  const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, 0, n);
  const physis_hip::BufWin<float> bw = physis_hip::BufWin<float>::Make(bg ? bg : dst.p, n, 0, n);
  physis_hip::TilePoint pt[K];
#pragma unroll
  for (int k = 0; k < K; ++k)
    pt[k] = physis_hip::OwnedPoint<TILE>(k, x0, y0, z0);
  physis_hip::LoadTile<TILE, true>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  __PSCtx_diffusion7_periodic_kernel ctx;
  ctx.g1_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g1_dim[d] = src.dim[d];
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = src.dim[d];
#pragma unroll
  for (int t = 1; t <= TILE::T; ++t) {
    const float *const cur = lds[(t - 1) & 1];
    float *const nxt = lds[t & 1];
#pragma unroll
    for (int k = 0; k < TILE::Count(t); ++k) {
      const physis_hip::TilePoint &p = pt[k];
      if (p.at < 0) continue;
      ctx.g1[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g1[1] = cur[p.at + -1 + RX * (0 + RY * (0))];
      ctx.g1[2] = cur[p.at + 1 + RX * (0 + RY * (0))];
      ctx.g1[3] = cur[p.at + 0 + RX * (-1 + RY * (0))];
      ctx.g1[4] = cur[p.at + 0 + RX * (1 + RY * (0))];
      ctx.g1[5] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g1[6] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g2_e = false;
      diffusion7_periodic_kernel(p.x, p.y, p.z, ctx, ce, cw, cn, cs, ct, cb, cc);
      const int off = p.x + nx * p.y + nxy * p.z;
      const float v[1] = {ctx.g2_v};
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
static void __PSLaunchTile_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_diffusion7_periodic_kernel<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.ce, s.cw, s.cn, s.cs, s.ct, s.cb, s.cc, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_diffusion7_periodic_kernel(const struct __PSStencil_diffusion7_periodic_kernel &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_diffusion7_periodic_kernel<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_diffusion7_periodic_kernel<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

static void __PSStencilRun_0(int iter, struct __PSStencil_diffusion7_kernel s0, struct __PSStencil_diffusion7_kernel s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("diffusion7_kernel, diffusion7_kernel");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_diffusion7_kernel(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.g1->num_elms * sizeof(float), false);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.g1, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.g2, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g1);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g2);
    const size_t bytes = (size_t)s0.g1->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const bool __small = physis_hip::TilesBeatPairs(s0.g1->dim, false, false);
    const int passes = !physis_hip::TilesBeatPairs(s0.g1->dim, false, false) ? iter : iter == 2 ? 2 : (iter + 1) / 2;
    __PSGrid3DFloat_dev src = va;
    for (int j = 0; j < passes; ++j) {
      const __PSGrid3DFloat_dev dst = passes % 2 && j == 0 ? vb
          : ((passes - 1 - j) % 2 == 0) ? va : vt;
      const int pairs = __small && iter > 2 && (j || iter % 2 == 0) ? 2 : 1;
      if (__small && pairs == 2)
        __PSLaunchT_diffusion7_kernel<4>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else if (__small)
        __PSLaunchT_diffusion7_kernel<2>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else
        __PSLaunch2_diffusion7_kernel(s0, src, dst, (j == passes - 1) ? vb.p : NULL, stream);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_diffusion7_kernel(s0, stream, NULL);
    __PSRun_diffusion7_kernel(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void diffusion7_run(PSGrid3DFloat g1, PSGrid3DFloat g2, int count, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  PSDomain3D dom = PSDomain3DNew(0, PSGridDim(g1, 0), 0, PSGridDim(g1, 1), 0, PSGridDim(g1, 2));
  __PSStencilRun_0(count / 2, __PSStencilMap_diffusion7_kernel(dom, g1, g2, ce, cw, cn, cs, ct, cb, cc), __PSStencilMap_diffusion7_kernel(dom, g2, g1, ce, cw, cn, cs, ct, cb, cc));
}

}  // extern "C"

static void __PSStencilRun_1(int iter, struct __PSStencil_diffusion7_periodic_kernel s0, struct __PSStencil_diffusion7_periodic_kernel s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("diffusion7_periodic_kernel, diffusion7_periodic_kernel");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_diffusion7_periodic_kernel(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.g1->num_elms * sizeof(float), false);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.g1, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.g2, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g1);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g2);
    const size_t bytes = (size_t)s0.g1->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const bool __small = physis_hip::TilesBeatPairs(s0.g1->dim, true, false);
    const int passes = !physis_hip::TilesBeatPairs(s0.g1->dim, true, false) ? iter : iter == 2 ? 2 : (iter + 1) / 2;
    __PSGrid3DFloat_dev src = va;
    for (int j = 0; j < passes; ++j) {
      const __PSGrid3DFloat_dev dst = passes % 2 && j == 0 ? vb
          : ((passes - 1 - j) % 2 == 0) ? va : vt;
      const int pairs = __small && iter > 2 && (j || iter % 2 == 0) ? 2 : 1;
      if (__small && pairs == 2)
        __PSLaunchT_diffusion7_periodic_kernel<4>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else if (__small)
        __PSLaunchT_diffusion7_periodic_kernel<2>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else
        __PSLaunch2_diffusion7_periodic_kernel(s0, src, dst, (j == passes - 1) ? vb.p : NULL, stream);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_diffusion7_periodic_kernel(s0, stream, NULL);
    __PSRun_diffusion7_periodic_kernel(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void diffusion7_periodic_run(PSGrid3DFloat g1, PSGrid3DFloat g2, int count, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  PSDomain3D dom = PSDomain3DNew(0, PSGridDim(g1, 0), 0, PSGridDim(g1, 1), 0, PSGridDim(g1, 2));
  __PSStencilRun_1(count / 2, __PSStencilMap_diffusion7_periodic_kernel(dom, g1, g2, ce, cw, cn, cs, ct, cb, cc), __PSStencilMap_diffusion7_periodic_kernel(dom, g2, g1, ce, cw, cn, cs, ct, cb, cc));
}

}  // extern "C"

static void __PSStencilRun_2(int iter, struct __PSStencil_diffusion7_periodic_kernel s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("diffusion7_periodic_kernel");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_diffusion7_periodic_kernel(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_3(int iter, struct __PSStencil_diffusion7_kernel s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("diffusion7_kernel");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_diffusion7_kernel(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void diffusion7_sweep_domain(PSGrid3DFloat g1, PSGrid3DFloat g2, int x0, int x1, int y0, int y1, int z0, int z1, int periodic, float ce, float cw, float cn, float cs, float ct, float cb, float cc) {
  PSDomain3D dom = PSDomain3DNew(x0, x1, y0, y1, z0, z1);
  if (periodic)
    __PSStencilRun_2(1, __PSStencilMap_diffusion7_periodic_kernel(dom, g1, g2, ce, cw, cn, cs, ct, cb, cc));
  else
    __PSStencilRun_3(1, __PSStencilMap_diffusion7_kernel(dom, g1, g2, ce, cw, cn, cs, ct, cb, cc));
}

}  // extern "C"

