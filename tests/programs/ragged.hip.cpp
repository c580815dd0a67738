// Generated by physisc-hip from ragged.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

// ---------------------------------------------- stencil corners
struct __PSStencil_corners {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_corners __PSStencilMap_corners(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_corners __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of corners (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,0,0) 2:(1,-1,0) 3:(-1,1,0) 4:(1,1,1) 5:(-1,-1,-1) 6:(1,0,-1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_corners {
  float g[7];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void corners(
    const int x, const int y, const int z, __PSCtx_corners &__ctx) {
  float v = 0.5f * __ctx.g[0] + __ctx.g[1] + 2.0f * __ctx.g[2] + 3.0f * __ctx.g[3] + 4.0f * __ctx.g[4] + 5.0f * __ctx.g[5] + 6.0f * __ctx.g[6];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_corners(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_corners ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
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
          float g_r0[VX + 1];
          S_g::template ReadRow<0, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r2);
          float g_r3[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 1, lane, g_r3);
          float g_r4[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + -1, lane, g_r4);
          float g_r5[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r5);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[1] = g_r0[i + 1];
              ctx.g[2] = g_r1[i + 0];
              ctx.g[3] = g_r2[i + 0];
              ctx.g[4] = g_r3[i + 0];
              ctx.g[5] = g_r4[i + 0];
              ctx.g[6] = g_r5[i + 0];
              ctx.g2_e = false;
              corners(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_corners(const struct __PSStencil_corners &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_corners<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_corners(const struct __PSStencil_corners &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_corners<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_corners<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_corners(const struct __PSStencil_corners &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_corners<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_corners<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_corners<1>(s).blocks;
}

static int __PSRun_corners(const struct __PSStencil_corners &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_corners<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_corners<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_corners<1>(s, stream, red);
}

// Two-sweep run kernel of corners over a domain strictly inside
// the grid: one pass over src computes u' = corners(src) on the
// tile and a one-point halo (bg's own values outside the domain) and
// u'' = corners(u') two planes behind; dst <- u'', and bg <- u'
// when store_mid.  red1 / red2: per-block partials of the two sweeps.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, int RED, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_corners(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, __PSGrid3DFloat_dev bg, int store_mid, physis_hip::RunShape sh, float *__restrict__ red1, float *__restrict__ red2) {
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
    SA st[PD], pro[3];
    const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Load(aw, src.p, src.dim, ra, zb - 2 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      st[k].Load(aw, src.p, src.dim, ra, zb + 1 + k);
    float bg_c1[4][VX];
    // loads of plane z for u': the lane's VX points on mid rows, its halo
    // point in wave 0; emitted-grid values only where a point lies
    // outside the domain
    auto load1 = [&](int z, int slot) {
      if (wave == 0) {
        const int o = hlane ? hx + hy * nx + z * nxy : physis_hip::kDrop;
        const int ob = hlane && !(hin && zin(z)) ? o : physis_hip::kDrop;
        bw.template Load<1>(ob, *reinterpret_cast<float (*)[1]>(&bg_c1[slot][0]));
      } else {
        const int o = mid_row ? xs + yrow * nx + z * nxy : physis_hip::kDrop;
        const int ob = mid_row && !(yin && xin_all && zin(z)) ? o : physis_hip::kDrop;
        bw.template Load<VX>(ob, bg_c1[slot]);
      }
    };
    load1(zb - 1, 0);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Store(a_lds + k * SA::kPlane, wave, lane, ra);
    __syncthreads();
    __PSCtx_corners ctx;
    ctx.g_p = src.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
    ctx.g2_p = dst.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
    for (int sc = zb - 1; sc <= ze + 1; sc += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = sc + k;
        const int abase = k, bbase = k;
        const int cur = k, nxt = (k + 1) & 3;
        if (s > ze + 1) break;  // uniform over the block
        load1(s + 1, nxt);
        if (mid_row && s <= ze) {
          float a_r0[VX + 1];
          SA::template ReadRow<0, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 0, lane, a_r0);
          float a_r1[VX + 0];
          SA::template ReadRow<1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + -1, lane, a_r1);
          float a_r2[VX + 0];
          SA::template ReadRow<-1, -1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 1, lane, a_r2);
          float a_r3[VX + 0];
          SA::template ReadRow<1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 1, lane, a_r3);
          float a_r4[VX + 0];
          SA::template ReadRow<-1, -1>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + -1, lane, a_r4);
          float a_r5[VX + 0];
          SA::template ReadRow<1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 0, lane, a_r5);
          float uo[VX];
          unsigned m = 0;
          const bool own = out_row && s >= zb && s < ze;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = a_r0[i + 0];
            ctx.g[1] = a_r0[i + 1];
            ctx.g[2] = a_r1[i + 0];
            ctx.g[3] = a_r2[i + 0];
            ctx.g[4] = a_r3[i + 0];
            ctx.g[5] = a_r4[i + 0];
            ctx.g[6] = a_r5[i + 0];
            ctx.g2_e = false;
            const bool in = yin && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0] && zin(s);
            corners(xs + i, yrow, s, ctx);
            uo[i] = in ? ctx.g2_v : bg_c1[cur][i];
            m |= in ? 1u << i : 0u;
          }
          float *brow = b_lds + physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + wave * SB::kRow + SB::kPad + lane * VX;
#pragma unroll
          for (int i = 0; i < VX; ++i) brow[i] = uo[i];
          if (store_mid && own)
            physis_hip::StoreMasked<float, VX>(mw, xs + yrow * nx + s * nxy, uo, m);
        }
        if (hlane && s <= ze) {
          ctx.g[0] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[1] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.g[2] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[3] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[4] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[5] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[6] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.g2_e = false;
          corners(hx, hy, s, ctx);
          b_lds[physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + hr * SB::kRow + SB::kPad + px] = hin && zin(s) ? ctx.g2_v : bg_c1[cur][0];
        }
        if (out_row && s - 2 >= zb) {
          float b_r0[VX + 1];
          SB::template ReadRow<0, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 0, lane, b_r0);
          float b_r1[VX + 0];
          SB::template ReadRow<1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + -1, lane, b_r1);
          float b_r2[VX + 0];
          SB::template ReadRow<-1, -1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 1, lane, b_r2);
          float b_r3[VX + 0];
          SB::template ReadRow<1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 1, lane, b_r3);
          float b_r4[VX + 0];
          SB::template ReadRow<-1, -1>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + -1, lane, b_r4);
          float b_r5[VX + 0];
          SB::template ReadRow<1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 0, lane, b_r5);
          float uu[VX];
          unsigned m = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = b_r0[i + 0];
            ctx.g[1] = b_r0[i + 1];
            ctx.g[2] = b_r1[i + 0];
            ctx.g[3] = b_r2[i + 0];
            ctx.g[4] = b_r3[i + 0];
            ctx.g[5] = b_r4[i + 0];
            ctx.g[6] = b_r5[i + 0];
            ctx.g2_e = false;
            const bool in = xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
            corners(xs + i, yrow, s - 2, ctx);
            uu[i] = ctx.g2_v;
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

static constexpr int __PS2VX_corners = 4, __PS2BY_corners = 16;
template <int VX, int BY>
static physis_hip::RunShape __PSShape2_corners(const struct __PSStencil_corners &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_corners<VX, BY, -1, false>, 64 * BY);
  return physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g, s.g2}, 3));
}

static int __PSBlocks2_corners(const struct __PSStencil_corners &s) {
  return __PSShape2_corners<__PS2VX_corners, __PS2BY_corners>(s).blocks;
}

template <bool RAGGED>
static void __PSLaunch2R_corners(const struct __PSStencil_corners &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  constexpr int VX = __PS2VX_corners, BY = __PS2BY_corners;
  const physis_hip::RunShape sh = __PSShape2_corners<VX, BY>(s);
  if (sh.blocks == 0) return;
  const dim3 grid(sh.blocks), block(64 * BY);
  {
      hipLaunchKernelGGL((__PSStencilRun2_corners<VX, BY, -1, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, sh, (float *)red1, (float *)red2);
  }
}

static void __PSLaunch2_corners(const struct __PSStencil_corners &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  if (s.g->dim[0] % __PS2VX_corners == 0)
    __PSLaunch2R_corners<false>(s, src, dst, store_mid, stream, red1, red2);
  else
    __PSLaunch2R_corners<__PS2VX_corners != 1>(s, src, dst, store_mid, stream, red1, red2);
}

// The pair (s0, s1) is corners(a -> b), corners(b -> a) over one domain strictly
// inside the grids, with the same centre-only grids (neither a nor b) and
// scalars: it may run as two-sweep passes.
static bool __PSFusable2_corners(const struct __PSStencil_corners &s0, const struct __PSStencil_corners &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != s1.dom.local_min[d] ||
        s0.dom.local_max[d] != s1.dom.local_max[d]) return false;
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  }
  if (!physis_hip::DomainPassesPay(s0.dom, a->dim[0], a->num_elms, true)) return false;
  return physis_hip::WindowsFit({a, b}, 3);
}

// Resident-tile pass of corners: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_corners(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, int tiles_x, int tiles_y, physis_hip::TileReds red) {
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
  float bg_c[K][1];
  bool in[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const physis_hip::TilePoint &p = pt[k];
    in[k] = p.at >= 0 && p.x >= dom.local_min[0] && p.x < dom.local_max[0] &&
            p.y >= dom.local_min[1] && p.y < dom.local_max[1] &&
            p.z >= dom.local_min[2] && p.z < dom.local_max[2];
    const bool grid = p.at >= 0 && p.x >= 0 && p.x < nx && p.y >= 0 &&
                      p.y < src.dim[1] && p.z >= 0 && p.z < src.dim[2];
    const int off = p.x + nx * p.y + nxy * p.z;
    bw.template Load<1>(grid && !in[k] ? off : physis_hip::kDrop, bg_c[k]);
  }
  physis_hip::LoadTile<TILE, false>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  __PSCtx_corners ctx;
  ctx.g_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
#pragma unroll
  for (int t = 1; t <= TILE::T; ++t) {
    const float *const cur = lds[(t - 1) & 1];
    float *const nxt = lds[t & 1];
#pragma unroll
    for (int k = 0; k < TILE::Count(t); ++k) {
      const physis_hip::TilePoint &p = pt[k];
      if (p.at < 0) continue;
      ctx.g[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g[1] = cur[p.at + 1 + RX * (0 + RY * (0))];
      ctx.g[2] = cur[p.at + 1 + RX * (-1 + RY * (0))];
      ctx.g[3] = cur[p.at + -1 + RX * (1 + RY * (0))];
      ctx.g[4] = cur[p.at + 1 + RX * (1 + RY * (1))];
      ctx.g[5] = cur[p.at + -1 + RX * (-1 + RY * (-1))];
      ctx.g[6] = cur[p.at + 1 + RX * (0 + RY * (-1))];
      ctx.g2_e = false;
      corners(p.x, p.y, p.z, ctx);
      const int off = p.x + nx * p.y + nxy * p.z;
      const bool keep = in[k];
      const float v[1] = {ctx.g2_v};
      if (t < TILE::T) {
        if (keep)
          nxt[p.at] = v[0];
        else if (t == 1)
          nxt[p.at] = bg_c[k][0];
      }
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
static void __PSLaunchTile_corners(const struct __PSStencil_corners &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_corners<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_corners(const struct __PSStencil_corners &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_corners<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_corners<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil corners_double
struct __PSStencil_corners_double {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_corners_double __PSStencilMap_corners_double(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_corners_double __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of corners_double (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,0,0) 2:(1,-1,0) 3:(-1,1,0) 4:(1,1,1) 5:(-1,-1,-1) 6:(1,0,-1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (not float grids)
struct __PSCtx_corners_double {
  double g[7];
  const double *g_p;
  int g_dim[3];
  double g2_v;
  bool g2_e;
  const double *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void corners_double(
    const int x, const int y, const int z, __PSCtx_corners_double &__ctx) {
  double v = 0.5 * __ctx.g[0] + __ctx.g[1] + 2.0 * __ctx.g[2] + 3.0 * __ctx.g[3] + 4.0 * __ctx.g[4] + 5.0 * __ctx.g[5] + 6.0 * __ctx.g[6];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_corners_double(
    __PSDomain dom, __PSGrid3DDouble_dev g, __PSGrid3DDouble_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<double, VX, BY, 1, HY, 4, false, double, RAGGED> S_g;
  __shared__ __attribute__((aligned(16))) double g_lds[S_g::kLdsElems];
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
    const physis_hip::BufWin<double> g_w = physis_hip::BufWin<double>::Make(g.p, g_nxy * g.dim[2], (long)(zb + -2) * g_nxy, (long)(ze + 2) * g_nxy);
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<double> g2_ew = physis_hip::BufWin<double>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_corners_double ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
    }
    constexpr int U = 2;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        if (computes && z < ze) {
          double g_r0[VX + 1];
          S_g::template ReadRow<0, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          double g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r1);
          double g_r2[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r2);
          double g_r3[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 1, lane, g_r3);
          double g_r4[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + -1, lane, g_r4);
          double g_r5[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r5);
          double g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[1] = g_r0[i + 1];
              ctx.g[2] = g_r1[i + 0];
              ctx.g[3] = g_r2[i + 0];
              ctx.g[4] = g_r3[i + 0];
              ctx.g[5] = g_r4[i + 0];
              ctx.g[6] = g_r5[i + 0];
              ctx.g2_e = false;
              corners_double(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<double, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<4>(g_base, 3) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 2 + PD);
        g_base = physis_hip::RingSlot<4>(g_base, 1);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_corners_double(const struct __PSStencil_corners_double &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_corners_double<VX, 8, -1>, 64 * 8);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 8 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_corners_double(const struct __PSStencil_corners_double &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_corners_double<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 8);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_corners_double<VX, 8, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DDouble_dev>(s.g), physis_hip::DevView<__PSGrid3DDouble_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_corners_double(const struct __PSStencil_corners_double &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_corners_double<4>(s).blocks
         : __PSShape_corners_double<1>(s).blocks;
}

static int __PSRun_corners_double(const struct __PSStencil_corners_double &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_DOUBLE);
  physis_hip::CheckGrid3D(s.g2, PS_DOUBLE);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_corners_double<4>(s, stream, red)
         : __PSLaunch_corners_double<1>(s, stream, red);
}

// ---------------------------------------------- stencil corners2d
struct __PSStencil_corners2d {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_corners2d __PSStencilMap_corners2d(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_corners2d __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of corners2d (2.5D run kernel over the rows view nx x 1 x ny of its 2-D grids, y marched as z):
//   g  staged x[-1,1] y[-0,0] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,0,-1) 2:(-1,0,1) 3:(1,0,0)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_corners2d {
  float g[4];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void corners2d(
    const int x, const int y, __PSCtx_corners2d &__ctx) {
  float v = 0.5f * __ctx.g[0] + 2.0f * __ctx.g[1] + 3.0f * __ctx.g[2] + 4.0f * __ctx.g[3];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_corners2d(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 0;
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_corners2d ctx;
    ctx.g_p = g.p;
    ctx.g_dim[0] = g.dim[0];
    ctx.g_dim[1] = g.dim[2];
    ctx.g_dim[2] = 1;
    ctx.g2_p = g2.p;
    ctx.g2_dim[0] = g2.dim[0];
    ctx.g2_dim[1] = g2.dim[2];
    ctx.g2_dim[2] = 1;
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
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
          float g_r0[VX + 1];
          S_g::template ReadRow<0, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r2);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[1] = g_r1[i + 0];
              ctx.g[2] = g_r2[i + 0];
              ctx.g[3] = g_r0[i + 1];
              ctx.g2_e = false;
              corners2d(x, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_corners2d(const struct __PSStencil_corners2d &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_corners2d<VX, 1, -1>, 64 * 1);
  return physis_hip::PlanRun(physis_hip::RowDomain(s.dom), 64 * physis_hip::FormVX(VX), 1 - 2 * 0, per_cu, physis_hip::WindowChunkLimitRows({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_corners2d(const struct __PSStencil_corners2d &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_corners2d<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 1);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_corners2d<VX, 1, -1>), grid, block, 0, stream, physis_hip::RowDomain(s.dom), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_corners2d(const struct __PSStencil_corners2d &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_corners2d<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSShape_corners2d<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_corners2d<1>(s).blocks;
}

static int __PSRun_corners2d(const struct __PSStencil_corners2d &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_corners2d<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSLaunch_corners2d<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_corners2d<1>(s, stream, red);
}

// Rows pass of corners2d: T sweeps of src into dst, the one before the
// last into bg when store_mid.
template <int T>
__global__ __launch_bounds__(64) void __PSStencilRunR_corners2d(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, physis_hip::RunShape sh) {
  constexpr int PD = 3;
  const int lane = threadIdx.x;
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, 1);
  const int xs = (sh.x_first_tile + tc.bx) * physis_hip::kRowsTX -
                 physis_hip::kRowsHalo + lane * 4;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  if (zb >= ze) return;
  const int nx = src.dim[0], n = nx * src.dim[2];
  const physis_hip::BufWin<float> aw = physis_hip::BufWin<float>::Make(src.p, n, (long)(zb - T - 1) * nx, (long)(ze + T + 1) * nx);
  const physis_hip::BufWin<float> bw = physis_hip::BufWin<float>::Make(bg, n, (long)(zb - T - 1) * nx, (long)(ze + T + 1) * nx);
  const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, (long)zb * nx, (long)ze * nx);
  const physis_hip::BufWin<float> mw = physis_hip::BufWin<float>::Make(bg, n, (long)zb * nx, (long)ze * nx);
  unsigned xm = 0;  // the lane's points inside the domain's columns
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (xs + i >= dom.local_min[0] && xs + i < dom.local_max[0]) xm |= 1u << i;
  const bool xin = __all(xm == 15u);
  const unsigned om = lane >= 1 && lane <= 62 ? xm : 0u;
  const auto zin = [&](int z) { return z >= dom.local_min[2] && z < dom.local_max[2]; };
  float ld[PD][4], lb[PD][4];
  // row z of src, and of b one row behind where the domain leaves points out
  const auto load = [&](int z, int k) {
    aw.template Load<4>(xs + z * nx, ld[k]);
    bw.template Load<4>(xm == 15u && zin(z - 1) ? physis_hip::kDrop
                                                : xs + (z - 1) * nx, lb[k]);
  };
  physis_hip::RowRegs q[T][3];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int i = 0; i < 6; ++i) q[t][k].v[i] = 0.0f;
  __PSCtx_corners2d ctx;
  ctx.g_p = src.p;
  ctx.g_dim[0] = nx;
  ctx.g_dim[1] = src.dim[2];
  ctx.g_dim[2] = 1;
  ctx.g2_p = dst.p;
  ctx.g2_dim[0] = nx;
  ctx.g2_dim[1] = src.dim[2];
  ctx.g2_dim[2] = 1;
#pragma unroll
  for (int k = 0; k < PD; ++k) load(zb - T + k, k);
  for (int sc = zb - T; sc < ze + T; sc += 3) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int s = sc + k;
      q[0][k].Set(ld[k]);
      float b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = lb[k][i];
      load(s + PD, k);
#pragma unroll
      for (int t = 1; t <= T; ++t) {
        const int z = s - t;
        float v[4];
        const auto pts = [&](auto inside) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            ctx.g[0] = q[t - 1][(k + 2) % 3].v[1 + i + 0];
            ctx.g[1] = q[t - 1][(k + 1) % 3].v[1 + i + 1];
            ctx.g[2] = q[t - 1][(k + 0) % 3].v[1 + i + -1];
            ctx.g[3] = q[t - 1][(k + 2) % 3].v[1 + i + 1];
            ctx.g2_e = false;
            corners2d(xs + i, z, ctx);
            v[i] = ctx.g2_v;
            if constexpr (!decltype(inside)::value)
              if (!((xm >> i) & 1u && zin(z)))
                v[i] = t == 1 ? b[i] : q[t == 1 ? 0 : t - 2][(k + 1) % 3].v[1 + i];
          }
        };
        if (xin && zin(z))
          pts(physis_hip::Flag<true>{});
        else
          pts(physis_hip::Flag<false>{});
        if (t < T) q[t == T ? 0 : t][k].Set(v);
        if (om && z >= zb && z < ze) {
          if (t == T)
            physis_hip::StoreMasked<float, 4>(dw, xs + z * nx, v, om);
          else if (t == T - 1 && store_mid)
            physis_hip::StoreMasked<float, 4>(mw, xs + z * nx, v, om);
        }
      }
    }
  }
}

template <int T>
static void __PSLaunchR_corners2d(const struct __PSStencil_corners2d &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream) {
  const __PSDomain d = physis_hip::RowDomain(s.dom);
  static int per_cu = physis_hip::BlocksPerCU((const void *)__PSStencilRunR_corners2d<T>, 64);
  const physis_hip::RunShape sh = physis_hip::PlanRun(d, physis_hip::kRowsTX, 1, per_cu,
      physis_hip::WindowChunkLimitRows({s.g, s.g2}, T + 1), 2 * T + 3);
  if (sh.blocks == 0) return;
  hipLaunchKernelGGL(__PSStencilRunR_corners2d<T>, dim3(sh.blocks), dim3(64), 0, stream, d, src, dst, bg, store_mid, sh);
}

// The pair (s0, s1) is corners2d(a -> b), corners2d(b -> a) over one domain strictly
// inside the grids, with the same scalars: it may run as rows passes.
static bool __PSFusable2_corners2d(const struct __PSStencil_corners2d &s0, const struct __PSStencil_corners2d &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 2 || b->num_dims != 2) return false;
  for (int d = 0; d < 2; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != s1.dom.local_min[d] ||
        s0.dom.local_max[d] != s1.dom.local_max[d]) return false;
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  }
  return physis_hip::WindowsFit({a, b}, 5, true);
}

// ---------------------------------------------- stencil wrap2
struct __PSStencil_wrap2 {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_wrap2 __PSStencilMap_wrap2(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_wrap2 __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of wrap2 (2.5D run kernel):
//   g  staged x[-2,2] y[-1,1] z[-1,1] periodic
//     offsets 0:(0,0,0) 1:(2,-1,0)p 2:(-2,1,0)p 3:(1,0,1)p 4:(-1,0,-1)p
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (halo wider than one point)
struct __PSCtx_wrap2 {
  float g[5];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void wrap2(
    const int x, const int y, const int z, __PSCtx_wrap2 &__ctx) {
  float v = 0.5f * __ctx.g[0] + 2.0f * __ctx.g[1] + 3.0f * __ctx.g[2] + 4.0f * __ctx.g[3] + 5.0f * __ctx.g[4];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_wrap2(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 2, HY, 4, true, float, RAGGED> S_g;
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_wrap2 ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
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
          float g_r0[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<2, 2>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<-2, -2>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r2);
          float g_r3[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r4);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[1] = g_r1[i + 0];
              ctx.g[2] = g_r2[i + 0];
              ctx.g[3] = g_r3[i + 0];
              ctx.g[4] = g_r4[i + 0];
              ctx.g2_e = false;
              wrap2(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_wrap2(const struct __PSStencil_wrap2 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_wrap2<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_wrap2(const struct __PSStencil_wrap2 &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_wrap2<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_wrap2<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_wrap2(const struct __PSStencil_wrap2 &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_wrap2<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSShape_wrap2<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_wrap2<1>(s).blocks;
}

static int __PSRun_wrap2(const struct __PSStencil_wrap2 &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_wrap2<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSLaunch_wrap2<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_wrap2<1>(s, stream, red);
}

// ---------------------------------------------- stencil inner
struct __PSStencil_inner {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  float w;
};

static struct __PSStencil_inner __PSStencilMap_inner(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float w) {
  struct __PSStencil_inner __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), w};
  return __s;
}

// Stencil analysis of inner (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,-1,0) 2:(-1,1,0) 3:(0,0,1) 4:(0,0,-1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_inner {
  float g[5];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void inner(
    const int x, const int y, const int z, __PSCtx_inner &__ctx, float w) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4];
  (__ctx.g2_v = (v * w), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_inner(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, float w, physis_hip::RunShape sh, float *__restrict__ __red) {
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_inner ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
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
          float g_r0[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r2);
          float g_r3[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r4);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[1] = g_r1[i + 0];
              ctx.g[2] = g_r2[i + 0];
              ctx.g[3] = g_r3[i + 0];
              ctx.g[4] = g_r4[i + 0];
              ctx.g2_e = false;
              inner(x, yrow, z, ctx, w);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_inner(const struct __PSStencil_inner &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_inner<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_inner(const struct __PSStencil_inner &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_inner<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_inner<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_inner(const struct __PSStencil_inner &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_inner<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_inner<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_inner<1>(s).blocks;
}

static int __PSRun_inner(const struct __PSStencil_inner &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_inner<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_inner<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_inner<1>(s, stream, red);
}

// Two-sweep run kernel of inner over a domain strictly inside
// the grid: one pass over src computes u' = inner(src) on the
// tile and a one-point halo (bg's own values outside the domain) and
// u'' = inner(u') two planes behind; dst <- u'', and bg <- u'
// when store_mid.  red1 / red2: per-block partials of the two sweeps.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, int RED, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_inner(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, __PSGrid3DFloat_dev bg, int store_mid, float w, physis_hip::RunShape sh, float *__restrict__ red1, float *__restrict__ red2) {
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
    SA st[PD], pro[3];
    const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Load(aw, src.p, src.dim, ra, zb - 2 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      st[k].Load(aw, src.p, src.dim, ra, zb + 1 + k);
    float bg_c1[4][VX];
    // loads of plane z for u': the lane's VX points on mid rows, its halo
    // point in wave 0; emitted-grid values only where a point lies
    // outside the domain
    auto load1 = [&](int z, int slot) {
      if (wave == 0) {
        const int o = hlane ? hx + hy * nx + z * nxy : physis_hip::kDrop;
        const int ob = hlane && !(hin && zin(z)) ? o : physis_hip::kDrop;
        bw.template Load<1>(ob, *reinterpret_cast<float (*)[1]>(&bg_c1[slot][0]));
      } else {
        const int o = mid_row ? xs + yrow * nx + z * nxy : physis_hip::kDrop;
        const int ob = mid_row && !(yin && xin_all && zin(z)) ? o : physis_hip::kDrop;
        bw.template Load<VX>(ob, bg_c1[slot]);
      }
    };
    load1(zb - 1, 0);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Store(a_lds + k * SA::kPlane, wave, lane, ra);
    __syncthreads();
    __PSCtx_inner ctx;
    ctx.g_p = src.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
    ctx.g2_p = dst.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
    for (int sc = zb - 1; sc <= ze + 1; sc += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = sc + k;
        const int abase = k, bbase = k;
        const int cur = k, nxt = (k + 1) & 3;
        if (s > ze + 1) break;  // uniform over the block
        load1(s + 1, nxt);
        if (mid_row && s <= ze) {
          float a_r0[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 0, lane, a_r0);
          float a_r1[VX + 0];
          SA::template ReadRow<1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + -1, lane, a_r1);
          float a_r2[VX + 0];
          SA::template ReadRow<-1, -1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 1, lane, a_r2);
          float a_r3[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 0, lane, a_r3);
          float a_r4[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 0, lane, a_r4);
          float uo[VX];
          unsigned m = 0;
          const bool own = out_row && s >= zb && s < ze;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = a_r0[i + 0];
            ctx.g[1] = a_r1[i + 0];
            ctx.g[2] = a_r2[i + 0];
            ctx.g[3] = a_r3[i + 0];
            ctx.g[4] = a_r4[i + 0];
            ctx.g2_e = false;
            const bool in = yin && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0] && zin(s);
            inner(xs + i, yrow, s, ctx, w);
            uo[i] = in ? ctx.g2_v : bg_c1[cur][i];
            m |= in ? 1u << i : 0u;
          }
          float *brow = b_lds + physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + wave * SB::kRow + SB::kPad + lane * VX;
#pragma unroll
          for (int i = 0; i < VX; ++i) brow[i] = uo[i];
          if (store_mid && own)
            physis_hip::StoreMasked<float, VX>(mw, xs + yrow * nx + s * nxy, uo, m);
        }
        if (hlane && s <= ze) {
          ctx.g[0] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[1] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[2] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[3] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[4] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g2_e = false;
          inner(hx, hy, s, ctx, w);
          b_lds[physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + hr * SB::kRow + SB::kPad + px] = hin && zin(s) ? ctx.g2_v : bg_c1[cur][0];
        }
        if (out_row && s - 2 >= zb) {
          float b_r0[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 0, lane, b_r0);
          float b_r1[VX + 0];
          SB::template ReadRow<1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + -1, lane, b_r1);
          float b_r2[VX + 0];
          SB::template ReadRow<-1, -1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 1, lane, b_r2);
          float b_r3[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 0, lane, b_r3);
          float b_r4[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 0, lane, b_r4);
          float uu[VX];
          unsigned m = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = b_r0[i + 0];
            ctx.g[1] = b_r1[i + 0];
            ctx.g[2] = b_r2[i + 0];
            ctx.g[3] = b_r3[i + 0];
            ctx.g[4] = b_r4[i + 0];
            ctx.g2_e = false;
            const bool in = xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
            inner(xs + i, yrow, s - 2, ctx, w);
            uu[i] = ctx.g2_v;
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

static constexpr int __PS2VX_inner = 4, __PS2BY_inner = 16;
template <int VX, int BY>
static physis_hip::RunShape __PSShape2_inner(const struct __PSStencil_inner &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_inner<VX, BY, -1, false>, 64 * BY);
  return physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g, s.g2}, 3));
}

static int __PSBlocks2_inner(const struct __PSStencil_inner &s) {
  return __PSShape2_inner<__PS2VX_inner, __PS2BY_inner>(s).blocks;
}

template <bool RAGGED>
static void __PSLaunch2R_inner(const struct __PSStencil_inner &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  constexpr int VX = __PS2VX_inner, BY = __PS2BY_inner;
  const physis_hip::RunShape sh = __PSShape2_inner<VX, BY>(s);
  if (sh.blocks == 0) return;
  const dim3 grid(sh.blocks), block(64 * BY);
  {
      hipLaunchKernelGGL((__PSStencilRun2_inner<VX, BY, -1, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, s.w, sh, (float *)red1, (float *)red2);
  }
}

static void __PSLaunch2_inner(const struct __PSStencil_inner &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  if (s.g->dim[0] % __PS2VX_inner == 0)
    __PSLaunch2R_inner<false>(s, src, dst, store_mid, stream, red1, red2);
  else
    __PSLaunch2R_inner<__PS2VX_inner != 1>(s, src, dst, store_mid, stream, red1, red2);
}

// The pair (s0, s1) is inner(a -> b), inner(b -> a) over one domain strictly
// inside the grids, with the same centre-only grids (neither a nor b) and
// scalars: it may run as two-sweep passes.
static bool __PSFusable2_inner(const struct __PSStencil_inner &s0, const struct __PSStencil_inner &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != s1.dom.local_min[d] ||
        s0.dom.local_max[d] != s1.dom.local_max[d]) return false;
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  }
  if (__builtin_memcmp(&s0.w, &s1.w, sizeof(s0.w))) return false;
  if (!physis_hip::DomainPassesPay(s0.dom, a->dim[0], a->num_elms, true)) return false;
  return physis_hip::WindowsFit({a, b}, 3);
}

// Resident-tile pass of inner: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_inner(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, float w, int tiles_x, int tiles_y, physis_hip::TileReds red) {
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
  float bg_c[K][1];
  bool in[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const physis_hip::TilePoint &p = pt[k];
    in[k] = p.at >= 0 && p.x >= dom.local_min[0] && p.x < dom.local_max[0] &&
            p.y >= dom.local_min[1] && p.y < dom.local_max[1] &&
            p.z >= dom.local_min[2] && p.z < dom.local_max[2];
    const bool grid = p.at >= 0 && p.x >= 0 && p.x < nx && p.y >= 0 &&
                      p.y < src.dim[1] && p.z >= 0 && p.z < src.dim[2];
    const int off = p.x + nx * p.y + nxy * p.z;
    bw.template Load<1>(grid && !in[k] ? off : physis_hip::kDrop, bg_c[k]);
  }
  physis_hip::LoadTile<TILE, false>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  __PSCtx_inner ctx;
  ctx.g_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
#pragma unroll
  for (int t = 1; t <= TILE::T; ++t) {
    const float *const cur = lds[(t - 1) & 1];
    float *const nxt = lds[t & 1];
#pragma unroll
    for (int k = 0; k < TILE::Count(t); ++k) {
      const physis_hip::TilePoint &p = pt[k];
      if (p.at < 0) continue;
      ctx.g[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g[1] = cur[p.at + 1 + RX * (-1 + RY * (0))];
      ctx.g[2] = cur[p.at + -1 + RX * (1 + RY * (0))];
      ctx.g[3] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g[4] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g2_e = false;
      inner(p.x, p.y, p.z, ctx, w);
      const int off = p.x + nx * p.y + nxy * p.z;
      const bool keep = in[k];
      const float v[1] = {ctx.g2_v};
      if (t < TILE::T) {
        if (keep)
          nxt[p.at] = v[0];
        else if (t == 1)
          nxt[p.at] = bg_c[k][0];
      }
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
static void __PSLaunchTile_inner(const struct __PSStencil_inner &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_inner<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.w, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_inner(const struct __PSStencil_inner &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_inner<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_inner<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil settle
struct __PSStencil_settle {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  __PSGrid *c;
  int __c_index;
  float w;
  float *__reduce_out;  // PSStencilMapReduce target
  int __reduce_op;
};

static struct __PSStencil_settle __PSStencilMap_settle(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, __PSGrid *c, float w) {
  struct __PSStencil_settle __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), c, __PSGridGetID(c), w, NULL, 0};
  return __s;
}

static struct __PSStencil_settle __PSStencilMapReduce_settle(
    float *__v, int __op, __PSDomain __dom, __PSGrid *g, __PSGrid *g2, __PSGrid *c, float w) {
  struct __PSStencil_settle __s = __PSStencilMap_settle(__dom, g, g2, c, w);
  __s.__reduce_out = __v;
  __s.__reduce_op = __op;
  return __s;
}

// Stencil analysis of settle (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,-1,0) 2:(-1,1,0) 3:(0,0,1) 4:(0,0,-1)
//   g2  not read, emitted
//   c  direct (centre only)
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_settle {
  float g[5];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
  float c_c;
  const float *c_p;
  int c_dim[3];
};

__device__ __forceinline__ float settle(
    const int x, const int y, const int z, __PSCtx_settle &__ctx, float w) {
  float u = __ctx.g[0];
  float v = u + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4];
  v = v * w + __ctx.c_c;
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return v - u;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_settle(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, __PSGrid3DFloat_dev c, float w, physis_hip::RunShape sh, float *__restrict__ __red) {
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
    const int c_nx = c.dim[0], c_nxy = c.dim[0] * c.dim[1];
    const physis_hip::BufWin<float> c_w = physis_hip::BufWin<float>::Make(c.p, c_nxy * c.dim[2], (long)zb * c_nxy, (long)ze * c_nxy);
    float c_dv[2][VX];
    c_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c_nx + zb * c_nxy, c_dv[0]);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_settle ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    ctx.c_p = c.p;
    for (int d = 0; d < 3; ++d) ctx.c_dim[d] = c.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
      __builtin_assume((ctx.c_dim[0] & 3) == 0);
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
        c_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * c_nx + (z + 1) * c_nxy, c_dv[nxt]);
        if (computes && z < ze) {
          float g_r0[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r2);
          float g_r3[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r4);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[1] = g_r1[i + 0];
              ctx.g[2] = g_r2[i + 0];
              ctx.g[3] = g_r3[i + 0];
              ctx.g[4] = g_r4[i + 0];
              ctx.g2_e = false;
              ctx.c_c = c_dv[cur][i];
              const float __r = settle(x, yrow, z, ctx, w);
              if constexpr (RED >= 0) __racc = __in ? physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(__racc, __r) : __racc;
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<4>(g_base, 3) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 2 + PD);
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
static physis_hip::RunShape __PSShape_settle(const struct __PSStencil_settle &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_settle<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2, s.c}, 2));
}

template <int VX>
static int __PSLaunch_settle(const struct __PSStencil_settle &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_settle<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  switch (red ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRun_settle<VX, 16, PS_MAX>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRun_settle<VX, 16, PS_MIN>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRun_settle<VX, 16, PS_SUM>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRun_settle<VX, 16, PS_PROD>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRun_settle<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_settle(const struct __PSStencil_settle &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0 && s.c->dim[0] % 4 == 0) ? __PSShape_settle<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_settle<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_settle<1>(s).blocks;
}

static int __PSRun_settle(const struct __PSStencil_settle &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckGrid3D(s.c, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0 && s.c->dim[0] % 4 == 0) ? __PSLaunch_settle<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_settle<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_settle<1>(s, stream, red);
}

// Two-sweep run kernel of settle over a domain strictly inside
// the grid: one pass over src computes u' = settle(src) on the
// tile and a one-point halo (bg's own values outside the domain) and
// u'' = settle(u') two planes behind; dst <- u'', and bg <- u'
// when store_mid.  red1 / red2: per-block partials of the two sweeps.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, int RED, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_settle(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, __PSGrid3DFloat_dev bg, int store_mid, __PSGrid3DFloat_dev c, float w, physis_hip::RunShape sh, float *__restrict__ red1, float *__restrict__ red2) {
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
    const physis_hip::BufWin<float> c_w = physis_hip::BufWin<float>::Make(c.p, n, (long)(zb - 1) * nxy, (long)(ze + 1) * nxy);
    SA st[PD], pro[3];
    const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Load(aw, src.p, src.dim, ra, zb - 2 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      st[k].Load(aw, src.p, src.dim, ra, zb + 1 + k);
    float c_c1[4][VX];
    float bg_c1[4][VX];
    // loads of plane z for u': the lane's VX points on mid rows, its halo
    // point in wave 0; emitted-grid values only where a point lies
    // outside the domain
    auto load1 = [&](int z, int slot) {
      if (wave == 0) {
        const int o = hlane ? hx + hy * nx + z * nxy : physis_hip::kDrop;
        const int ob = hlane && !(hin && zin(z)) ? o : physis_hip::kDrop;
        c_w.template Load<1>(o, *reinterpret_cast<float (*)[1]>(&c_c1[slot][0]));
        bw.template Load<1>(ob, *reinterpret_cast<float (*)[1]>(&bg_c1[slot][0]));
      } else {
        const int o = mid_row ? xs + yrow * nx + z * nxy : physis_hip::kDrop;
        const int ob = mid_row && !(yin && xin_all && zin(z)) ? o : physis_hip::kDrop;
        c_w.template Load<VX>(o, c_c1[slot]);
        bw.template Load<VX>(ob, bg_c1[slot]);
      }
    };
    load1(zb - 1, 0);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Store(a_lds + k * SA::kPlane, wave, lane, ra);
    __syncthreads();
    __PSCtx_settle ctx;
    ctx.g_p = src.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
    ctx.g2_p = dst.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
    ctx.c_p = c.p;
    for (int d = 0; d < 3; ++d) ctx.c_dim[d] = c.dim[d];
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
          float a_r0[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 0, lane, a_r0);
          float a_r1[VX + 0];
          SA::template ReadRow<1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + -1, lane, a_r1);
          float a_r2[VX + 0];
          SA::template ReadRow<-1, -1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 1, lane, a_r2);
          float a_r3[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 0, lane, a_r3);
          float a_r4[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 0, lane, a_r4);
          float uo[VX];
          unsigned m = 0;
          const bool own = out_row && s >= zb && s < ze;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = a_r0[i + 0];
            ctx.g[1] = a_r1[i + 0];
            ctx.g[2] = a_r2[i + 0];
            ctx.g[3] = a_r3[i + 0];
            ctx.g[4] = a_r4[i + 0];
            ctx.c_c = c_c1[cur][i];
            ctx.g2_e = false;
            const bool in = yin && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0] && zin(s);
            const float r = settle(xs + i, yrow, s, ctx, w);
            if constexpr (RED >= 0) acc1 = in && own ? physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(acc1, r) : acc1;
            uo[i] = in ? ctx.g2_v : bg_c1[cur][i];
            m |= in ? 1u << i : 0u;
          }
          float *brow = b_lds + physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + wave * SB::kRow + SB::kPad + lane * VX;
#pragma unroll
          for (int i = 0; i < VX; ++i) brow[i] = uo[i];
          if (store_mid && own)
            physis_hip::StoreMasked<float, VX>(mw, xs + yrow * nx + s * nxy, uo, m);
        }
        if (hlane && s <= ze) {
          ctx.g[0] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[1] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[2] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[3] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[4] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.c_c = c_c1[cur][0];
          ctx.g2_e = false;
          (void)settle(hx, hy, s, ctx, w);
          b_lds[physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + hr * SB::kRow + SB::kPad + px] = hin && zin(s) ? ctx.g2_v : bg_c1[cur][0];
        }
        if (out_row && s - 2 >= zb) {
          float b_r0[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 0, lane, b_r0);
          float b_r1[VX + 0];
          SB::template ReadRow<1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + -1, lane, b_r1);
          float b_r2[VX + 0];
          SB::template ReadRow<-1, -1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 1, lane, b_r2);
          float b_r3[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 0, lane, b_r3);
          float b_r4[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 0, lane, b_r4);
          float uu[VX];
          unsigned m = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = b_r0[i + 0];
            ctx.g[1] = b_r1[i + 0];
            ctx.g[2] = b_r2[i + 0];
            ctx.g[3] = b_r3[i + 0];
            ctx.g[4] = b_r4[i + 0];
            ctx.c_c = c_c1[old][i];
            ctx.g2_e = false;
            const bool in = xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
            const float r = settle(xs + i, yrow, s - 2, ctx, w);
            if constexpr (RED >= 0) acc2 = in ? physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(acc2, r) : acc2;
            uu[i] = ctx.g2_v;
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

static constexpr int __PS2VX_settle = 4, __PS2BY_settle = 8;
template <int VX, int BY>
static physis_hip::RunShape __PSShape2_settle(const struct __PSStencil_settle &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_settle<VX, BY, -1, false>, 64 * BY);
  return physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g, s.g2, s.c}, 3));
}

static int __PSBlocks2_settle(const struct __PSStencil_settle &s) {
  return __PSShape2_settle<__PS2VX_settle, __PS2BY_settle>(s).blocks;
}

template <bool RAGGED>
static void __PSLaunch2R_settle(const struct __PSStencil_settle &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  constexpr int VX = __PS2VX_settle, BY = __PS2BY_settle;
  const physis_hip::RunShape sh = __PSShape2_settle<VX, BY>(s);
  if (sh.blocks == 0) return;
  const dim3 grid(sh.blocks), block(64 * BY);
  switch (red1 || red2 ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRun2_settle<VX, BY, PS_MAX, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red1, (float *)red2);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRun2_settle<VX, BY, PS_MIN, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red1, (float *)red2);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRun2_settle<VX, BY, PS_SUM, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red1, (float *)red2);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRun2_settle<VX, BY, PS_PROD, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red1, (float *)red2);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRun2_settle<VX, BY, -1, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, sh, (float *)red1, (float *)red2);
  }
}

static void __PSLaunch2_settle(const struct __PSStencil_settle &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  if (s.g->dim[0] % __PS2VX_settle == 0)
    __PSLaunch2R_settle<false>(s, src, dst, store_mid, stream, red1, red2);
  else
    __PSLaunch2R_settle<__PS2VX_settle != 1>(s, src, dst, store_mid, stream, red1, red2);
}

// The pair (s0, s1) is settle(a -> b), settle(b -> a) over one domain strictly
// inside the grids, with the same centre-only grids (neither a nor b) and
// scalars: it may run as two-sweep passes.
static bool __PSFusable2_settle(const struct __PSStencil_settle &s0, const struct __PSStencil_settle &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != s1.dom.local_min[d] ||
        s0.dom.local_max[d] != s1.dom.local_max[d]) return false;
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  }
  if (s0.c != s1.c || !s0.c || s0.c == a || s0.c == b || s0.c->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d)
    if (s0.c->dim[d] != a->dim[d]) return false;
  if (__builtin_memcmp(&s0.w, &s1.w, sizeof(s0.w))) return false;
  if ((s0.__reduce_out == NULL) != (s1.__reduce_out == NULL) ||
      (s0.__reduce_out && s0.__reduce_op != s1.__reduce_op)) return false;
  if (!physis_hip::DomainPassesPay(s0.dom, a->dim[0], a->num_elms, true)) return false;
  return physis_hip::WindowsFit({a, b, s0.c}, 3);
}

// Resident-tile pass of settle: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_settle(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, __PSGrid3DFloat_dev c, float w, int tiles_x, int tiles_y, physis_hip::TileReds red) {
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
  const physis_hip::BufWin<float> c_w = physis_hip::BufWin<float>::Make(c.p, n, 0, n);
  float c_c[K][1];
  float bg_c[K][1];
  bool in[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const physis_hip::TilePoint &p = pt[k];
    in[k] = p.at >= 0 && p.x >= dom.local_min[0] && p.x < dom.local_max[0] &&
            p.y >= dom.local_min[1] && p.y < dom.local_max[1] &&
            p.z >= dom.local_min[2] && p.z < dom.local_max[2];
    const bool grid = p.at >= 0 && p.x >= 0 && p.x < nx && p.y >= 0 &&
                      p.y < src.dim[1] && p.z >= 0 && p.z < src.dim[2];
    const int off = p.x + nx * p.y + nxy * p.z;
    bw.template Load<1>(grid && !in[k] ? off : physis_hip::kDrop, bg_c[k]);
    c_w.template Load<1>(in[k] ? off : physis_hip::kDrop, c_c[k]);
  }
  physis_hip::LoadTile<TILE, false>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  float acc[TILE::T];
#pragma unroll
  for (int t = 0; t < TILE::T; ++t) {
    acc[t] = 0;
    if constexpr (RED >= 0) acc[t] = physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::identity();
  }
  __PSCtx_settle ctx;
  ctx.g_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
  ctx.c_p = c.p;
  for (int d = 0; d < 3; ++d) ctx.c_dim[d] = c.dim[d];
#pragma unroll
  for (int t = 1; t <= TILE::T; ++t) {
    const float *const cur = lds[(t - 1) & 1];
    float *const nxt = lds[t & 1];
#pragma unroll
    for (int k = 0; k < TILE::Count(t); ++k) {
      const physis_hip::TilePoint &p = pt[k];
      if (p.at < 0) continue;
      ctx.g[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g[1] = cur[p.at + 1 + RX * (-1 + RY * (0))];
      ctx.g[2] = cur[p.at + -1 + RX * (1 + RY * (0))];
      ctx.g[3] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g[4] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.c_c = c_c[k][0];
      ctx.g2_e = false;
      const float r = settle(p.x, p.y, p.z, ctx, w);
      if constexpr (RED >= 0)
        if (k < TILE::Owned(0) && in[k]) acc[t - 1] = physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(acc[t - 1], r);
      const int off = p.x + nx * p.y + nxy * p.z;
      const bool keep = in[k];
      const float v[1] = {ctx.g2_v};
      if (t < TILE::T) {
        if (keep)
          nxt[p.at] = v[0];
        else if (t == 1)
          nxt[p.at] = bg_c[k][0];
      }
      if (k < TILE::Owned(0)) {
        if (t == TILE::T)
          dw.template Store<1>(keep ? off : physis_hip::kDrop, v);
        if (t == TILE::T - 1 && store_mid)
          bw.template Store<1>(keep ? off : physis_hip::kDrop, v);
      }
    }
    if (t < TILE::T) __syncthreads();
  }
  if constexpr (RED >= 0) {
    __shared__ float lds_red[TILE::T][TILE::NT / 64];
#pragma unroll
    for (int t = 0; t < TILE::T; ++t) {
      const float r = physis_hip::BlockReduce<float, RED < 0 ? 0 : RED, TILE::NT>(acc[t], lds_red[t]);
      if (threadIdx.x == 0) ((float *)red.p[t])[blockIdx.x] = r;
    }
  }
}

static int __PSBlocksT_settle(const struct __PSStencil_settle &s) {
  return physis_hip::TileBlocks(s.dom);
}

template <typename TILE>
static void __PSLaunchTile_settle(const struct __PSStencil_settle &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  switch (red.p[0] ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRunT_settle<TILE, PS_MAX>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, g.tiles_x, g.tiles_y, red);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRunT_settle<TILE, PS_MIN>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, g.tiles_x, g.tiles_y, red);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRunT_settle<TILE, PS_SUM>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, g.tiles_x, g.tiles_y, red);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRunT_settle<TILE, PS_PROD>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, g.tiles_x, g.tiles_y, red);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRunT_settle<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, physis_hip::DevView<__PSGrid3DFloat_dev>(s.c), s.w, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_settle(const struct __PSStencil_settle &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_settle<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_settle<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil settle_square
struct __PSStencil_settle_square {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  float w;
  double *__reduce_out;  // PSStencilMapReduce target
  int __reduce_op;
};

static struct __PSStencil_settle_square __PSStencilMap_settle_square(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float w) {
  struct __PSStencil_settle_square __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), w, NULL, 0};
  return __s;
}

static struct __PSStencil_settle_square __PSStencilMapReduce_settle_square(
    double *__v, int __op, __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float w) {
  struct __PSStencil_settle_square __s = __PSStencilMap_settle_square(__dom, g, g2, w);
  __s.__reduce_out = __v;
  __s.__reduce_op = __op;
  return __s;
}

// Stencil analysis of settle_square (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,-1,0) 2:(-1,1,0) 3:(0,0,1) 4:(0,0,-1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_settle_square {
  float g[5];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ double settle_square(
    const int x, const int y, const int z, __PSCtx_settle_square &__ctx, float w) {
  float u = __ctx.g[0];
  float v = u + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4];
  v = v * w;
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  double d = v - u;
  return d * d;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_settle_square(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, float w, physis_hip::RunShape sh, double *__restrict__ __red) {
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
  double __racc = 0;
  if constexpr (RED >= 0) __racc = physis_hip::ReduceOp<double, RED < 0 ? 0 : RED>::identity();
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_settle_square ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
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
          float g_r0[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<-1, -1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r2);
          float g_r3[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r4);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[1] = g_r1[i + 0];
              ctx.g[2] = g_r2[i + 0];
              ctx.g[3] = g_r3[i + 0];
              ctx.g[4] = g_r4[i + 0];
              ctx.g2_e = false;
              const double __r = settle_square(x, yrow, z, ctx, w);
              if constexpr (RED >= 0) __racc = __in ? physis_hip::ReduceOp<double, RED < 0 ? 0 : RED>::apply(__racc, __r) : __racc;
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<4>(g_base, 3) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 2 + PD);
      }
    }
  }
  if constexpr (RED >= 0) {
    __shared__ double __lds_red[BY];
    const double __r = physis_hip::BlockReduce<double, RED < 0 ? 0 : RED, 64 * BY>(__racc, __lds_red);
    if (threadIdx.x == 0) __red[blockIdx.x] = __r;
  }
}

template <int VX>
static physis_hip::RunShape __PSShape_settle_square(const struct __PSStencil_settle_square &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_settle_square<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_settle_square(const struct __PSStencil_settle_square &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_settle_square<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  switch (red ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRun_settle_square<VX, 16, PS_MAX>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (double *)red);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRun_settle_square<VX, 16, PS_MIN>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (double *)red);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRun_settle_square<VX, 16, PS_SUM>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (double *)red);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRun_settle_square<VX, 16, PS_PROD>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (double *)red);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRun_settle_square<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (double *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_settle_square(const struct __PSStencil_settle_square &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_settle_square<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_settle_square<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_settle_square<1>(s).blocks;
}

static int __PSRun_settle_square(const struct __PSStencil_settle_square &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_settle_square<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_settle_square<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_settle_square<1>(s, stream, red);
}

// Two-sweep run kernel of settle_square over a domain strictly inside
// the grid: one pass over src computes u' = settle_square(src) on the
// tile and a one-point halo (bg's own values outside the domain) and
// u'' = settle_square(u') two planes behind; dst <- u'', and bg <- u'
// when store_mid.  red1 / red2: per-block partials of the two sweeps.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, int RED, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_settle_square(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, __PSGrid3DFloat_dev bg, int store_mid, float w, physis_hip::RunShape sh, double *__restrict__ red1, double *__restrict__ red2) {
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
  double acc1 = 0, acc2 = 0;
  if constexpr (RED >= 0) acc1 = acc2 = physis_hip::ReduceOp<double, RED < 0 ? 0 : RED>::identity();
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
    SA st[PD], pro[3];
    const typename SA::Addr ra = SA::Prepare(src.dim, x0, yrow, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Load(aw, src.p, src.dim, ra, zb - 2 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      st[k].Load(aw, src.p, src.dim, ra, zb + 1 + k);
    float bg_c1[4][VX];
    // loads of plane z for u': the lane's VX points on mid rows, its halo
    // point in wave 0; emitted-grid values only where a point lies
    // outside the domain
    auto load1 = [&](int z, int slot) {
      if (wave == 0) {
        const int o = hlane ? hx + hy * nx + z * nxy : physis_hip::kDrop;
        const int ob = hlane && !(hin && zin(z)) ? o : physis_hip::kDrop;
        bw.template Load<1>(ob, *reinterpret_cast<float (*)[1]>(&bg_c1[slot][0]));
      } else {
        const int o = mid_row ? xs + yrow * nx + z * nxy : physis_hip::kDrop;
        const int ob = mid_row && !(yin && xin_all && zin(z)) ? o : physis_hip::kDrop;
        bw.template Load<VX>(ob, bg_c1[slot]);
      }
    };
    load1(zb - 1, 0);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      pro[k].Store(a_lds + k * SA::kPlane, wave, lane, ra);
    __syncthreads();
    __PSCtx_settle_square ctx;
    ctx.g_p = src.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
    ctx.g2_p = dst.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
    for (int sc = zb - 1; sc <= ze + 1; sc += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = sc + k;
        const int abase = k, bbase = k;
        const int cur = k, nxt = (k + 1) & 3;
        if (s > ze + 1) break;  // uniform over the block
        load1(s + 1, nxt);
        if (mid_row && s <= ze) {
          float a_r0[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 0, lane, a_r0);
          float a_r1[VX + 0];
          SA::template ReadRow<1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + -1, lane, a_r1);
          float a_r2[VX + 0];
          SA::template ReadRow<-1, -1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 1, lane, a_r2);
          float a_r3[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 0, lane, a_r3);
          float a_r4[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 0, lane, a_r4);
          float uo[VX];
          unsigned m = 0;
          const bool own = out_row && s >= zb && s < ze;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = a_r0[i + 0];
            ctx.g[1] = a_r1[i + 0];
            ctx.g[2] = a_r2[i + 0];
            ctx.g[3] = a_r3[i + 0];
            ctx.g[4] = a_r4[i + 0];
            ctx.g2_e = false;
            const bool in = yin && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0] && zin(s);
            const double r = settle_square(xs + i, yrow, s, ctx, w);
            if constexpr (RED >= 0) acc1 = in && own ? physis_hip::ReduceOp<double, RED < 0 ? 0 : RED>::apply(acc1, r) : acc1;
            uo[i] = in ? ctx.g2_v : bg_c1[cur][i];
            m |= in ? 1u << i : 0u;
          }
          float *brow = b_lds + physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + wave * SB::kRow + SB::kPad + lane * VX;
#pragma unroll
          for (int i = 0; i < VX; ++i) brow[i] = uo[i];
          if (store_mid && own)
            physis_hip::StoreMasked<float, VX>(mw, xs + yrow * nx + s * nxy, uo, m);
        }
        if (hlane && s <= ze) {
          ctx.g[0] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[1] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[2] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[3] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[4] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g2_e = false;
          (void)settle_square(hx, hy, s, ctx, w);
          b_lds[physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + hr * SB::kRow + SB::kPad + px] = hin && zin(s) ? ctx.g2_v : bg_c1[cur][0];
        }
        if (out_row && s - 2 >= zb) {
          float b_r0[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 0, lane, b_r0);
          float b_r1[VX + 0];
          SB::template ReadRow<1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + -1, lane, b_r1);
          float b_r2[VX + 0];
          SB::template ReadRow<-1, -1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 1, lane, b_r2);
          float b_r3[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 0, lane, b_r3);
          float b_r4[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 0, lane, b_r4);
          float uu[VX];
          unsigned m = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = b_r0[i + 0];
            ctx.g[1] = b_r1[i + 0];
            ctx.g[2] = b_r2[i + 0];
            ctx.g[3] = b_r3[i + 0];
            ctx.g[4] = b_r4[i + 0];
            ctx.g2_e = false;
            const bool in = xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
            const double r = settle_square(xs + i, yrow, s - 2, ctx, w);
            if constexpr (RED >= 0) acc2 = in ? physis_hip::ReduceOp<double, RED < 0 ? 0 : RED>::apply(acc2, r) : acc2;
            uu[i] = ctx.g2_v;
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
    __shared__ double lds_r1[BY], lds_r2[BY];
    const double r1 = physis_hip::BlockReduce<double, RED < 0 ? 0 : RED, 64 * BY>(acc1, lds_r1);
    const double r2 = physis_hip::BlockReduce<double, RED < 0 ? 0 : RED, 64 * BY>(acc2, lds_r2);
    if (threadIdx.x == 0) {
      if (red1) red1[blockIdx.x] = r1;
      if (red2) red2[blockIdx.x] = r2;
    }
  } else {
    (void)acc1; (void)acc2; (void)red1; (void)red2;
  }
}

static constexpr int __PS2VX_settle_square = 4, __PS2BY_settle_square = 16;
template <int VX, int BY>
static physis_hip::RunShape __PSShape2_settle_square(const struct __PSStencil_settle_square &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_settle_square<VX, BY, -1, false>, 64 * BY);
  return physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g, s.g2}, 3));
}

static int __PSBlocks2_settle_square(const struct __PSStencil_settle_square &s) {
  return __PSShape2_settle_square<__PS2VX_settle_square, __PS2BY_settle_square>(s).blocks;
}

template <bool RAGGED>
static void __PSLaunch2R_settle_square(const struct __PSStencil_settle_square &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  constexpr int VX = __PS2VX_settle_square, BY = __PS2BY_settle_square;
  const physis_hip::RunShape sh = __PSShape2_settle_square<VX, BY>(s);
  if (sh.blocks == 0) return;
  const dim3 grid(sh.blocks), block(64 * BY);
  switch (red1 || red2 ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRun2_settle_square<VX, BY, PS_MAX, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, s.w, sh, (double *)red1, (double *)red2);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRun2_settle_square<VX, BY, PS_MIN, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, s.w, sh, (double *)red1, (double *)red2);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRun2_settle_square<VX, BY, PS_SUM, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, s.w, sh, (double *)red1, (double *)red2);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRun2_settle_square<VX, BY, PS_PROD, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, s.w, sh, (double *)red1, (double *)red2);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRun2_settle_square<VX, BY, -1, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, s.w, sh, (double *)red1, (double *)red2);
  }
}

static void __PSLaunch2_settle_square(const struct __PSStencil_settle_square &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  if (s.g->dim[0] % __PS2VX_settle_square == 0)
    __PSLaunch2R_settle_square<false>(s, src, dst, store_mid, stream, red1, red2);
  else
    __PSLaunch2R_settle_square<__PS2VX_settle_square != 1>(s, src, dst, store_mid, stream, red1, red2);
}

// The pair (s0, s1) is settle_square(a -> b), settle_square(b -> a) over one domain strictly
// inside the grids, with the same centre-only grids (neither a nor b) and
// scalars: it may run as two-sweep passes.
static bool __PSFusable2_settle_square(const struct __PSStencil_settle_square &s0, const struct __PSStencil_settle_square &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != s1.dom.local_min[d] ||
        s0.dom.local_max[d] != s1.dom.local_max[d]) return false;
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  }
  if (__builtin_memcmp(&s0.w, &s1.w, sizeof(s0.w))) return false;
  if ((s0.__reduce_out == NULL) != (s1.__reduce_out == NULL) ||
      (s0.__reduce_out && s0.__reduce_op != s1.__reduce_op)) return false;
  if (!physis_hip::DomainPassesPay(s0.dom, a->dim[0], a->num_elms, true)) return false;
  return physis_hip::WindowsFit({a, b}, 3);
}

// Resident-tile pass of settle_square: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_settle_square(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, float w, int tiles_x, int tiles_y, physis_hip::TileReds red) {
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
  float bg_c[K][1];
  bool in[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const physis_hip::TilePoint &p = pt[k];
    in[k] = p.at >= 0 && p.x >= dom.local_min[0] && p.x < dom.local_max[0] &&
            p.y >= dom.local_min[1] && p.y < dom.local_max[1] &&
            p.z >= dom.local_min[2] && p.z < dom.local_max[2];
    const bool grid = p.at >= 0 && p.x >= 0 && p.x < nx && p.y >= 0 &&
                      p.y < src.dim[1] && p.z >= 0 && p.z < src.dim[2];
    const int off = p.x + nx * p.y + nxy * p.z;
    bw.template Load<1>(grid && !in[k] ? off : physis_hip::kDrop, bg_c[k]);
  }
  physis_hip::LoadTile<TILE, false>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  double acc[TILE::T];
#pragma unroll
  for (int t = 0; t < TILE::T; ++t) {
    acc[t] = 0;
    if constexpr (RED >= 0) acc[t] = physis_hip::ReduceOp<double, RED < 0 ? 0 : RED>::identity();
  }
  __PSCtx_settle_square ctx;
  ctx.g_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = dst.dim[d];
#pragma unroll
  for (int t = 1; t <= TILE::T; ++t) {
    const float *const cur = lds[(t - 1) & 1];
    float *const nxt = lds[t & 1];
#pragma unroll
    for (int k = 0; k < TILE::Count(t); ++k) {
      const physis_hip::TilePoint &p = pt[k];
      if (p.at < 0) continue;
      ctx.g[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g[1] = cur[p.at + 1 + RX * (-1 + RY * (0))];
      ctx.g[2] = cur[p.at + -1 + RX * (1 + RY * (0))];
      ctx.g[3] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g[4] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g2_e = false;
      const double r = settle_square(p.x, p.y, p.z, ctx, w);
      if constexpr (RED >= 0)
        if (k < TILE::Owned(0) && in[k]) acc[t - 1] = physis_hip::ReduceOp<double, RED < 0 ? 0 : RED>::apply(acc[t - 1], r);
      const int off = p.x + nx * p.y + nxy * p.z;
      const bool keep = in[k];
      const float v[1] = {ctx.g2_v};
      if (t < TILE::T) {
        if (keep)
          nxt[p.at] = v[0];
        else if (t == 1)
          nxt[p.at] = bg_c[k][0];
      }
      if (k < TILE::Owned(0)) {
        if (t == TILE::T)
          dw.template Store<1>(keep ? off : physis_hip::kDrop, v);
        if (t == TILE::T - 1 && store_mid)
          bw.template Store<1>(keep ? off : physis_hip::kDrop, v);
      }
    }
    if (t < TILE::T) __syncthreads();
  }
  if constexpr (RED >= 0) {
    __shared__ double lds_red[TILE::T][TILE::NT / 64];
#pragma unroll
    for (int t = 0; t < TILE::T; ++t) {
      const double r = physis_hip::BlockReduce<double, RED < 0 ? 0 : RED, TILE::NT>(acc[t], lds_red[t]);
      if (threadIdx.x == 0) ((double *)red.p[t])[blockIdx.x] = r;
    }
  }
}

static int __PSBlocksT_settle_square(const struct __PSStencil_settle_square &s) {
  return physis_hip::TileBlocks(s.dom);
}

template <typename TILE>
static void __PSLaunchTile_settle_square(const struct __PSStencil_settle_square &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  switch (red.p[0] ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRunT_settle_square<TILE, PS_MAX>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.w, g.tiles_x, g.tiles_y, red);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRunT_settle_square<TILE, PS_MIN>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.w, g.tiles_x, g.tiles_y, red);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRunT_settle_square<TILE, PS_SUM>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.w, g.tiles_x, g.tiles_y, red);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRunT_settle_square<TILE, PS_PROD>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.w, g.tiles_x, g.tiles_y, red);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRunT_settle_square<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, s.w, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_settle_square(const struct __PSStencil_settle_square &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_settle_square<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_settle_square<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil inner2d
struct __PSStencil_inner2d {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  float w;
};

static struct __PSStencil_inner2d __PSStencilMap_inner2d(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float w) {
  struct __PSStencil_inner2d __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), w};
  return __s;
}

// Stencil analysis of inner2d (2.5D run kernel over the rows view nx x 1 x ny of its 2-D grids, y marched as z):
//   g  staged x[-1,1] y[-0,0] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,0,-1) 2:(-1,0,1) 3:(-1,0,0) 4:(1,0,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_inner2d {
  float g[5];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void inner2d(
    const int x, const int y, __PSCtx_inner2d &__ctx, float w) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4];
  (__ctx.g2_v = (v * w), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_inner2d(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, float w, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 0;
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_inner2d ctx;
    ctx.g_p = g.p;
    ctx.g_dim[0] = g.dim[0];
    ctx.g_dim[1] = g.dim[2];
    ctx.g_dim[2] = 1;
    ctx.g2_p = g2.p;
    ctx.g2_dim[0] = g2.dim[0];
    ctx.g2_dim[1] = g2.dim[2];
    ctx.g2_dim[2] = 1;
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2_dim[0] & 3) == 0);
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
          float g_r0[VX + 1];
          S_g::template ReadRow<-1, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r1);
          float g_r2[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r2);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r1[i + 0];
              ctx.g[2] = g_r2[i + 0];
              ctx.g[3] = g_r0[i + 0];
              ctx.g[4] = g_r2[i + 2];
              ctx.g2_e = false;
              inner2d(x, z, ctx, w);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_inner2d(const struct __PSStencil_inner2d &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_inner2d<VX, 1, -1>, 64 * 1);
  return physis_hip::PlanRun(physis_hip::RowDomain(s.dom), 64 * physis_hip::FormVX(VX), 1 - 2 * 0, per_cu, physis_hip::WindowChunkLimitRows({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_inner2d(const struct __PSStencil_inner2d &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_inner2d<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 1);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_inner2d<VX, 1, -1>), grid, block, 0, stream, physis_hip::RowDomain(s.dom), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_inner2d(const struct __PSStencil_inner2d &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_inner2d<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSShape_inner2d<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_inner2d<1>(s).blocks;
}

static int __PSRun_inner2d(const struct __PSStencil_inner2d &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_inner2d<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSLaunch_inner2d<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_inner2d<1>(s, stream, red);
}

// Rows pass of inner2d: T sweeps of src into dst, the one before the
// last into bg when store_mid.
template <int T>
__global__ __launch_bounds__(64) void __PSStencilRunR_inner2d(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, float w, physis_hip::RunShape sh) {
  constexpr int PD = 3;
  const int lane = threadIdx.x;
  const physis_hip::TileCoord tc = physis_hip::TileOf(sh.tiles_x, 1);
  const int xs = (sh.x_first_tile + tc.bx) * physis_hip::kRowsTX -
                 physis_hip::kRowsHalo + lane * 4;
  const int zb = dom.local_min[2] + tc.bz * sh.zchunk;
  const int ze = min(zb + sh.zchunk, dom.local_max[2]);
  if (zb >= ze) return;
  const int nx = src.dim[0], n = nx * src.dim[2];
  const physis_hip::BufWin<float> aw = physis_hip::BufWin<float>::Make(src.p, n, (long)(zb - T - 1) * nx, (long)(ze + T + 1) * nx);
  const physis_hip::BufWin<float> bw = physis_hip::BufWin<float>::Make(bg, n, (long)(zb - T - 1) * nx, (long)(ze + T + 1) * nx);
  const physis_hip::BufWin<float> dw = physis_hip::BufWin<float>::Make(dst.p, n, (long)zb * nx, (long)ze * nx);
  const physis_hip::BufWin<float> mw = physis_hip::BufWin<float>::Make(bg, n, (long)zb * nx, (long)ze * nx);
  unsigned xm = 0;  // the lane's points inside the domain's columns
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (xs + i >= dom.local_min[0] && xs + i < dom.local_max[0]) xm |= 1u << i;
  const bool xin = __all(xm == 15u);
  const unsigned om = lane >= 1 && lane <= 62 ? xm : 0u;
  const auto zin = [&](int z) { return z >= dom.local_min[2] && z < dom.local_max[2]; };
  float ld[PD][4], lb[PD][4];
  // row z of src, and of b one row behind where the domain leaves points out
  const auto load = [&](int z, int k) {
    aw.template Load<4>(xs + z * nx, ld[k]);
    bw.template Load<4>(xm == 15u && zin(z - 1) ? physis_hip::kDrop
                                                : xs + (z - 1) * nx, lb[k]);
  };
  physis_hip::RowRegs q[T][3];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int i = 0; i < 6; ++i) q[t][k].v[i] = 0.0f;
  __PSCtx_inner2d ctx;
  ctx.g_p = src.p;
  ctx.g_dim[0] = nx;
  ctx.g_dim[1] = src.dim[2];
  ctx.g_dim[2] = 1;
  ctx.g2_p = dst.p;
  ctx.g2_dim[0] = nx;
  ctx.g2_dim[1] = src.dim[2];
  ctx.g2_dim[2] = 1;
#pragma unroll
  for (int k = 0; k < PD; ++k) load(zb - T + k, k);
  for (int sc = zb - T; sc < ze + T; sc += 3) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int s = sc + k;
      q[0][k].Set(ld[k]);
      float b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = lb[k][i];
      load(s + PD, k);
#pragma unroll
      for (int t = 1; t <= T; ++t) {
        const int z = s - t;
        float v[4];
        const auto pts = [&](auto inside) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            ctx.g[0] = q[t - 1][(k + 2) % 3].v[1 + i + 0];
            ctx.g[1] = q[t - 1][(k + 1) % 3].v[1 + i + 1];
            ctx.g[2] = q[t - 1][(k + 0) % 3].v[1 + i + -1];
            ctx.g[3] = q[t - 1][(k + 2) % 3].v[1 + i + -1];
            ctx.g[4] = q[t - 1][(k + 0) % 3].v[1 + i + 1];
            ctx.g2_e = false;
            inner2d(xs + i, z, ctx, w);
            v[i] = ctx.g2_v;
            if constexpr (!decltype(inside)::value)
              if (!((xm >> i) & 1u && zin(z)))
                v[i] = t == 1 ? b[i] : q[t == 1 ? 0 : t - 2][(k + 1) % 3].v[1 + i];
          }
        };
        if (xin && zin(z))
          pts(physis_hip::Flag<true>{});
        else
          pts(physis_hip::Flag<false>{});
        if (t < T) q[t == T ? 0 : t][k].Set(v);
        if (om && z >= zb && z < ze) {
          if (t == T)
            physis_hip::StoreMasked<float, 4>(dw, xs + z * nx, v, om);
          else if (t == T - 1 && store_mid)
            physis_hip::StoreMasked<float, 4>(mw, xs + z * nx, v, om);
        }
      }
    }
  }
}

template <int T>
static void __PSLaunchR_inner2d(const struct __PSStencil_inner2d &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream) {
  const __PSDomain d = physis_hip::RowDomain(s.dom);
  static int per_cu = physis_hip::BlocksPerCU((const void *)__PSStencilRunR_inner2d<T>, 64);
  const physis_hip::RunShape sh = physis_hip::PlanRun(d, physis_hip::kRowsTX, 1, per_cu,
      physis_hip::WindowChunkLimitRows({s.g, s.g2}, T + 1), 2 * T + 3);
  if (sh.blocks == 0) return;
  hipLaunchKernelGGL(__PSStencilRunR_inner2d<T>, dim3(sh.blocks), dim3(64), 0, stream, d, src, dst, bg, store_mid, s.w, sh);
}

// The pair (s0, s1) is inner2d(a -> b), inner2d(b -> a) over one domain strictly
// inside the grids, with the same scalars: it may run as rows passes.
static bool __PSFusable2_inner2d(const struct __PSStencil_inner2d &s0, const struct __PSStencil_inner2d &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 2 || b->num_dims != 2) return false;
  for (int d = 0; d < 2; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != s1.dom.local_min[d] ||
        s0.dom.local_max[d] != s1.dom.local_max[d]) return false;
    if (s0.dom.local_min[d] < 1 || s0.dom.local_max[d] > a->dim[d] - 1 ||
        s0.dom.local_min[d] >= s0.dom.local_max[d]) return false;
  }
  if (__builtin_memcmp(&s0.w, &s1.w, sizeof(s0.w))) return false;
  return physis_hip::WindowsFit({a, b}, 5, true);
}

// ---------------------------------------------- stencil relax_double
struct __PSStencil_relax_double {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  int __rb;  // -1 all points, 0 red, 1 black, 2 red then black
};

static struct __PSStencil_relax_double __PSStencilMap_relax_double(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_relax_double __s = {__dom, g, __PSGridGetID(g), -1};
  return __s;
}

static struct __PSStencil_relax_double __PSStencilMapRed_relax_double(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_relax_double __s = __PSStencilMap_relax_double(__dom, g);
  __s.__rb = 0;
  return __s;
}

static struct __PSStencil_relax_double __PSStencilMapBlack_relax_double(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_relax_double __s = __PSStencilMap_relax_double(__dom, g);
  __s.__rb = 1;
  return __s;
}

static struct __PSStencil_relax_double __PSStencilMapRedBlack_relax_double(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_relax_double __s = __PSStencilMap_relax_double(__dom, g);
  __s.__rb = 2;
  return __s;
}

// Stencil analysis of relax_double (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic, emitted
//     offsets 0:(0,0,0) 1:(1,0,0) 2:(-1,0,0) 3:(0,1,0) 4:(0,-1,0) 5:(0,0,1) 6:(0,0,-1)
//   red-black: in-place colour sweep reads only the other colour
//   two-sweep fusion of map pairs: no (not a float grid)
struct __PSCtx_relax_double {
  double g[7];
  double g_v;
  bool g_e;
  const double *g_p;
  int g_dim[3];
};

__device__ __forceinline__ void relax_double(
    const int x, const int y, const int z, __PSCtx_relax_double &__ctx) {
  double v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6];
  (__ctx.g_v = (v * 0.125), __ctx.g_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_relax_double(
    __PSDomain dom, __PSGrid3DDouble_dev g, physis_hip::RunShape sh, float *__restrict__ __red, int __rb) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<double, VX, BY, 1, HY, 4, false, double, RAGGED> S_g;
  __shared__ __attribute__((aligned(16))) double g_lds[S_g::kLdsElems];
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
    const physis_hip::BufWin<double> g_w = physis_hip::BufWin<double>::Make(g.p, g_nxy * g.dim[2], (long)(zb + -2) * g_nxy, (long)(ze + 2) * g_nxy);
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
    const physis_hip::BufWin<double> g_ew = physis_hip::BufWin<double>::Make(g.p, g_enxy * g.dim[2], (long)zb * g_enxy, (long)ze * g_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_relax_double ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g_dim[0] & 3) == 0);
    }
    constexpr int U = 2;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        if (computes && z < ze) {
          double g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          double g_r1[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r1);
          double g_r2[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r2);
          double g_r3[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r3);
          double g_r4[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r4);
          double g_out[VX];
          unsigned g_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0] &&
                (__rb < 0 || ((x + yrow + z + __rb) & 1) == 0);
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g[5] = g_r3[i + 0];
              ctx.g[6] = g_r4[i + 0];
              ctx.g_e = false;
              relax_double(x, yrow, z, ctx);
              g_out[i] = ctx.g_v;
              g_mask |= (__in && ctx.g_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<double, VX>(g_ew, xs + yrow * g_enx + z * g_enxy, g_out, g_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<4>(g_base, 3) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 2 + PD);
        g_base = physis_hip::RingSlot<4>(g_base, 1);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_relax_double(const struct __PSStencil_relax_double &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_relax_double<VX, 8, -1>, 64 * 8);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 8 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g}, 2));
}

template <int VX>
static int __PSLaunch_relax_double(const struct __PSStencil_relax_double &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_relax_double<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 8);
  for (int __c = s.__rb == 2 ? 0 : s.__rb; __c <= (s.__rb == 2 ? 1 : s.__rb); ++__c) {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_relax_double<VX, 8, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DDouble_dev>(s.g), sh, (float *)NULL, __c);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_relax_double(const struct __PSStencil_relax_double &s) {
  return (s.g->dim[0] % 4 == 0) ? __PSShape_relax_double<4>(s).blocks
         : __PSShape_relax_double<1>(s).blocks;
}

static int __PSRun_relax_double(const struct __PSStencil_relax_double &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_DOUBLE);
  physis_hip::CheckEmitDomain(s.dom, s.g);
  return (s.g->dim[0] % 4 == 0) ? __PSLaunch_relax_double<4>(s, stream, red)
         : __PSLaunch_relax_double<1>(s, stream, red);
}

extern "C" {

static PSDomain3D whole(PSGrid3DFloat g) {
  return PSDomain3DNew(0, PSGridDim(g, 0), 0, PSGridDim(g, 1), 0, PSGridDim(g, 2));
}

}  // extern "C"

static void __PSStencilRun_0(int iter, struct __PSStencil_corners s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("corners");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_corners(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_corners(PSGrid3DFloat g, PSGrid3DFloat g2) {
  __PSStencilRun_0(1, __PSStencilMap_corners(whole(g2), g, g2));
}

}  // extern "C"

static void __PSStencilRun_1(int iter, struct __PSStencil_corners_double s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("corners_double");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_corners_double(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_corners_double(PSGrid3DDouble g, PSGrid3DDouble g2) {
  PSDomain3D d = PSDomain3DNew(0, PSGridDim(g, 0), 0, PSGridDim(g, 1), 0, PSGridDim(g, 2));
  __PSStencilRun_1(1, __PSStencilMap_corners_double(d, g, g2));
}

}  // extern "C"

static void __PSStencilRun_2(int iter, struct __PSStencil_corners2d s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("corners2d");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_corners2d(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_corners2d(PSGrid2DFloat g, PSGrid2DFloat g2) {
  PSDomain2D d = PSDomain2DNew(0, PSGridDim(g, 0), 0, PSGridDim(g, 1));
  __PSStencilRun_2(1, __PSStencilMap_corners2d(d, g, g2));
}

}  // extern "C"

static void __PSStencilRun_3(int iter, struct __PSStencil_wrap2 s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("wrap2");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_wrap2(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_wrap2(PSGrid3DFloat g, PSGrid3DFloat g2) {
  __PSStencilRun_3(1, __PSStencilMap_wrap2(whole(g), g, g2));
}

}  // extern "C"

static void __PSStencilRun_4(int iter, struct __PSStencil_inner s0, struct __PSStencil_inner s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("inner, inner");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_inner(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.g->num_elms * sizeof(float), (!physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2) % 2 != 0);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.g, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.g2, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g2);
    const size_t bytes = (size_t)s0.g->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const bool __small = physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms);
    const int passes = !physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2;
    __PSGrid3DFloat_dev vt2 = va;
    physis_hip::CopyShell(vt.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    if (passes % 2) {
      vt2.p = (float *)__PSHipScratch(9, bytes);
      physis_hip::CopyShell(vt2.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    }
    __PSGrid3DFloat_dev src = va;
    for (int j = 0; j < passes; ++j) {
      __PSGrid3DFloat_dev dst = (j % 2 == (passes % 2 ? 0 : 1)) ? va : vt;
      if (passes % 2 && j < 2) dst = j == 0 ? vt : vt2;
      const int pairs = __small && iter > 2 && (j || iter % 2 == 0) ? 2 : 1;
      if (__small && pairs == 2)
        __PSLaunchT_inner<4>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else if (__small)
        __PSLaunchT_inner<2>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else
        __PSLaunch2_inner(s0, src, dst, (j == passes - 1), stream, NULL, NULL);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_inner(s0, stream, NULL);
    __PSRun_inner(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_inner(PSGrid3DFloat g, PSGrid3DFloat g2, int count, float w) {
  PSDomain3D d = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1, 1, PSGridDim(g, 2) - 1);
  __PSStencilRun_4(count, __PSStencilMap_inner(d, g, g2, w), __PSStencilMap_inner(d, g2, g, w));
}

}  // extern "C"

static void __PSStencilRun_5(int iter, struct __PSStencil_settle s0, struct __PSStencil_settle s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("settle, settle");
  physis_hip::RunTimer timer(stream);
  physis_hip::ReduceSlots __slots;
  const bool __fuse = iter >= 2 && __PSFusable2_settle(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.g->num_elms * sizeof(float), (!physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2) % 2 != 0);
  physis_hip::MapReducer red0(s0.__reduce_out, s0.__reduce_op, PS_FLOAT,
      s0.__reduce_out ? (!__fuse ? __PSBlocks_settle(s0) : physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? __PSBlocksT_settle(s0) : __PSBlocks2_settle(s0)) : 0, iter, __slots);
  physis_hip::MapReducer red1(s1.__reduce_out, s1.__reduce_op, PS_FLOAT,
      s1.__reduce_out ? (!__fuse ? __PSBlocks_settle(s1) : physis_hip::TilesBeatDomainPairs(s1.dom, s1.g->num_elms) ? __PSBlocksT_settle(s1) : __PSBlocks2_settle(s1)) : 0, iter, __slots);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.g, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.g2, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g2);
    const size_t bytes = (size_t)s0.g->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const bool __small = physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms);
    const int passes = !physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2;
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
      const int pairs = __small && iter > 2 && (j || iter % 2 == 0) ? 2 : 1;
      if (__small && pairs == 2)
        __PSLaunchT_settle<4>(s0, src, dst, vb.p, (j == passes - 1), stream, {red0.Slot(i), red1.Slot(i), red0.Slot(i + 1), red1.Slot(i + 1)});
      else if (__small)
        __PSLaunchT_settle<2>(s0, src, dst, vb.p, (j == passes - 1), stream, {red0.Slot(i), red1.Slot(i)});
      else
        __PSLaunch2_settle(s0, src, dst, (j == passes - 1), stream, red0.Slot(i), red1.Slot(i));
      i += pairs;
      red0.After(i - 1);
      red1.After(i - 1);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_settle(s0, stream, red0.Slot(i));
    __PSRun_settle(s1, stream, red1.Slot(i));
    red0.After(i);
    red1.After(i);
  }
  red0.Finish(stream);
  red1.Finish(stream);
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_settle(PSGrid3DFloat g, PSGrid3DFloat g2, PSGrid3DFloat c, int x0, int x1, int y0, int y1, int z0, int z1, int count, float w, float * more, float * back) {
  PSDomain3D d = PSDomain3DNew(x0, x1, y0, y1, z0, z1);
  __PSStencilRun_5(count, __PSStencilMapReduce_settle(more, PS_MAX, d, g, g2, c, w), __PSStencilMapReduce_settle(back, PS_MAX, d, g2, g, c, w));
}

}  // extern "C"

static void __PSStencilRun_6(int iter, struct __PSStencil_settle_square s0, struct __PSStencil_settle_square s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("settle_square, settle_square");
  physis_hip::RunTimer timer(stream);
  physis_hip::ReduceSlots __slots;
  const bool __fuse = iter >= 2 && __PSFusable2_settle_square(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.g->num_elms * sizeof(float), (!physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2) % 2 != 0);
  physis_hip::MapReducer red0(s0.__reduce_out, s0.__reduce_op, PS_DOUBLE,
      s0.__reduce_out ? (!__fuse ? __PSBlocks_settle_square(s0) : physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? __PSBlocksT_settle_square(s0) : __PSBlocks2_settle_square(s0)) : 0, iter, __slots);
  physis_hip::MapReducer red1(s1.__reduce_out, s1.__reduce_op, PS_DOUBLE,
      s1.__reduce_out ? (!__fuse ? __PSBlocks_settle_square(s1) : physis_hip::TilesBeatDomainPairs(s1.dom, s1.g->num_elms) ? __PSBlocksT_settle_square(s1) : __PSBlocks2_settle_square(s1)) : 0, iter, __slots);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.g, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.g2, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g2);
    const size_t bytes = (size_t)s0.g->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const bool __small = physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms);
    const int passes = !physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2;
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
      const int pairs = __small && iter > 2 && (j || iter % 2 == 0) ? 2 : 1;
      if (__small && pairs == 2)
        __PSLaunchT_settle_square<4>(s0, src, dst, vb.p, (j == passes - 1), stream, {red0.Slot(i), red1.Slot(i), red0.Slot(i + 1), red1.Slot(i + 1)});
      else if (__small)
        __PSLaunchT_settle_square<2>(s0, src, dst, vb.p, (j == passes - 1), stream, {red0.Slot(i), red1.Slot(i)});
      else
        __PSLaunch2_settle_square(s0, src, dst, (j == passes - 1), stream, red0.Slot(i), red1.Slot(i));
      i += pairs;
      red0.After(i - 1);
      red1.After(i - 1);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_settle_square(s0, stream, red0.Slot(i));
    __PSRun_settle_square(s1, stream, red1.Slot(i));
    red0.After(i);
    red1.After(i);
  }
  red0.Finish(stream);
  red1.Finish(stream);
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_settle_square(PSGrid3DFloat g, PSGrid3DFloat g2, int x0, int x1, int y0, int y1, int z0, int z1, int count, float w, double * more, double * back) {
  PSDomain3D d = PSDomain3DNew(x0, x1, y0, y1, z0, z1);
  __PSStencilRun_6(count, __PSStencilMapReduce_settle_square(more, PS_SUM, d, g, g2, w), __PSStencilMapReduce_settle_square(back, PS_SUM, d, g2, g, w));
}

}  // extern "C"

static void __PSStencilRun_7(int iter, struct __PSStencil_inner s0, struct __PSStencil_inner s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("inner, inner");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_inner(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.g->num_elms * sizeof(float), (!physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2) % 2 != 0);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.g, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.g2, PS_FLOAT);
    __PSGrid3DFloat_dev va = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g);
    __PSGrid3DFloat_dev vb = physis_hip::DevView<__PSGrid3DFloat_dev>(s0.g2);
    const size_t bytes = (size_t)s0.g->num_elms * sizeof(float);
    __PSGrid3DFloat_dev vt = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const bool __small = physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms);
    const int passes = !physis_hip::TilesBeatDomainPairs(s0.dom, s0.g->num_elms) ? iter : iter == 2 ? 2 : (iter + 1) / 2;
    __PSGrid3DFloat_dev vt2 = va;
    physis_hip::CopyShell(vt.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    if (passes % 2) {
      vt2.p = (float *)__PSHipScratch(9, bytes);
      physis_hip::CopyShell(vt2.p, va.p, va.dim[0], va.dim[1], va.dim[2], s0.dom, stream);
    }
    __PSGrid3DFloat_dev src = va;
    for (int j = 0; j < passes; ++j) {
      __PSGrid3DFloat_dev dst = (j % 2 == (passes % 2 ? 0 : 1)) ? va : vt;
      if (passes % 2 && j < 2) dst = j == 0 ? vt : vt2;
      const int pairs = __small && iter > 2 && (j || iter % 2 == 0) ? 2 : 1;
      if (__small && pairs == 2)
        __PSLaunchT_inner<4>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else if (__small)
        __PSLaunchT_inner<2>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else
        __PSLaunch2_inner(s0, src, dst, (j == passes - 1), stream, NULL, NULL);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_inner(s0, stream, NULL);
    __PSRun_inner(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_box(PSGrid3DFloat g, PSGrid3DFloat g2, int x0, int x1, int y0, int y1, int z0, int z1, int count, float w) {
  PSDomain3D d = PSDomain3DNew(x0, x1, y0, y1, z0, z1);
  __PSStencilRun_7(count, __PSStencilMap_inner(d, g, g2, w), __PSStencilMap_inner(d, g2, g, w));
}

}  // extern "C"

static void __PSStencilRun_8(int iter, struct __PSStencil_inner2d s0, struct __PSStencil_inner2d s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("inner2d, inner2d");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_inner2d(s0, s1) &&
      physis_hip::HaveScratch((size_t)s0.g->num_elms * sizeof(float), (iter == 2 ? 2 : (iter + 1) / 2) % 2 != 0);
  int i0 = 0;
  if (__fuse) {
    physis_hip::CheckGrid3D(s0.g, PS_FLOAT);
    physis_hip::CheckGrid3D(s0.g2, PS_FLOAT);
    const __PSGrid3DFloat_dev va = physis_hip::RowView<__PSGrid3DFloat_dev>(s0.g);
    float *const b = physis_hip::RowView<__PSGrid3DFloat_dev>(s0.g2).p;
    const size_t bytes = (size_t)s0.g->num_elms * sizeof(float);
    const int passes = iter == 2 ? 2 : (iter + 1) / 2;
    __PSGrid3DFloat_dev vt = va, vt2 = va;
    vt.p = (float *)__PSHipScratch(8, bytes);
    const __PSDomain d = physis_hip::RowDomain(s0.dom);
    physis_hip::CopyShell(vt.p, va.p, va.dim[0], 1, va.dim[2], d, stream);
    if (passes % 2) {
      vt2.p = (float *)__PSHipScratch(9, bytes);
      physis_hip::CopyShell(vt2.p, va.p, va.dim[0], 1, va.dim[2], d, stream);
    }
    __PSGrid3DFloat_dev src = va;
    for (int j = 0; j < passes; ++j) {
      __PSGrid3DFloat_dev dst = (j % 2 == (passes % 2 ? 0 : 1)) ? va : vt;
      if (passes % 2 && j < 2) dst = j == 0 ? vt : vt2;
      if (iter > 2 && (j || iter % 2 == 0))
        __PSLaunchR_inner2d<4>(s0, src, dst, b, j == passes - 1, stream);
      else
        __PSLaunchR_inner2d<2>(s0, src, dst, b, j == passes - 1, stream);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_inner2d(s0, stream, NULL);
    __PSRun_inner2d(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_box2d(PSGrid2DFloat g, PSGrid2DFloat g2, int x0, int x1, int y0, int y1, int count, float w) {
  PSDomain2D d = PSDomain2DNew(x0, x1, y0, y1);
  __PSStencilRun_8(count, __PSStencilMap_inner2d(d, g, g2, w), __PSStencilMap_inner2d(d, g2, g, w));
}

}  // extern "C"

static void __PSStencilRun_9(int iter, struct __PSStencil_relax_double s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("relax_double");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_relax_double(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void ragged_relax_double(PSGrid3DDouble g, int count) {
  PSDomain3D d = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1, 1, PSGridDim(g, 2) - 1);
  __PSStencilRun_9(count, __PSStencilMapRedBlack_relax_double(d, g));
}

}  // extern "C"

