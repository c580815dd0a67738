// Generated by physisc-hip from systests.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

// ---------------------------------------------- stencil k7
struct __PSStencil_k7 {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k7 __PSStencilMap_k7(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_k7 __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k7 (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,0,0) 2:(-1,0,0) 3:(0,1,0) 4:(0,-1,0) 5:(0,0,-1) 6:(0,0,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_k7 {
  float g[7];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k7(
    const int x, const int y, const int z, __PSCtx_k7 &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_k7(
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
    __PSCtx_k7 ctx;
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
          float g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r2);
          float g_r3[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r4);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g[5] = g_r3[i + 0];
              ctx.g[6] = g_r4[i + 0];
              ctx.g2_e = false;
              k7(x, yrow, z, ctx);
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
static physis_hip::RunShape __PSShape_k7(const struct __PSStencil_k7 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_k7<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_k7(const struct __PSStencil_k7 &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_k7<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_k7<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_k7(const struct __PSStencil_k7 &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_k7<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_k7<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_k7<1>(s).blocks;
}

static int __PSRun_k7(const struct __PSStencil_k7 &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_k7<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_k7<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_k7<1>(s, stream, red);
}

// Two-sweep run kernel of k7 over a domain strictly inside
// the grid: one pass over src computes u' = k7(src) on the
// tile and a one-point halo (bg's own values outside the domain) and
// u'' = k7(u') two planes behind; dst <- u'', and bg <- u'
// when store_mid.  red1 / red2: per-block partials of the two sweeps.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, int RED, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_k7(
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
    __PSCtx_k7 ctx;
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
          float a_r0[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 0, lane, a_r0);
          float a_r1[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 1, lane, a_r1);
          float a_r2[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + -1, lane, a_r2);
          float a_r3[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 0, lane, a_r3);
          float a_r4[VX + 0];
          SA::template ReadRow<0, 0>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 0, lane, a_r4);
          float uo[VX];
          unsigned m = 0;
          const bool own = out_row && s >= zb && s < ze;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = a_r0[i + 1];
            ctx.g[1] = a_r0[i + 2];
            ctx.g[2] = a_r0[i + 0];
            ctx.g[3] = a_r1[i + 0];
            ctx.g[4] = a_r2[i + 0];
            ctx.g[5] = a_r3[i + 0];
            ctx.g[6] = a_r4[i + 0];
            ctx.g2_e = false;
            const bool in = yin && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0] && zin(s);
            k7(xs + i, yrow, s, ctx);
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
          ctx.g[2] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
          ctx.g[3] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[4] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[5] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[6] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g2_e = false;
          k7(hx, hy, s, ctx);
          b_lds[physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + hr * SB::kRow + SB::kPad + px] = hin && zin(s) ? ctx.g2_v : bg_c1[cur][0];
        }
        if (out_row && s - 2 >= zb) {
          float b_r0[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 0, lane, b_r0);
          float b_r1[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 1, lane, b_r1);
          float b_r2[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + -1, lane, b_r2);
          float b_r3[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 0, lane, b_r3);
          float b_r4[VX + 0];
          SB::template ReadRow<0, 0>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 0, lane, b_r4);
          float uu[VX];
          unsigned m = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = b_r0[i + 1];
            ctx.g[1] = b_r0[i + 2];
            ctx.g[2] = b_r0[i + 0];
            ctx.g[3] = b_r1[i + 0];
            ctx.g[4] = b_r2[i + 0];
            ctx.g[5] = b_r3[i + 0];
            ctx.g[6] = b_r4[i + 0];
            ctx.g2_e = false;
            const bool in = xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
            k7(xs + i, yrow, s - 2, ctx);
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

static constexpr int __PS2VX_k7 = 4, __PS2BY_k7 = 16;
template <int VX, int BY>
static physis_hip::RunShape __PSShape2_k7(const struct __PSStencil_k7 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_k7<VX, BY, -1, false>, 64 * BY);
  return physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g, s.g2}, 3));
}

static int __PSBlocks2_k7(const struct __PSStencil_k7 &s) {
  return __PSShape2_k7<__PS2VX_k7, __PS2BY_k7>(s).blocks;
}

template <bool RAGGED>
static void __PSLaunch2R_k7(const struct __PSStencil_k7 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  constexpr int VX = __PS2VX_k7, BY = __PS2BY_k7;
  const physis_hip::RunShape sh = __PSShape2_k7<VX, BY>(s);
  if (sh.blocks == 0) return;
  const dim3 grid(sh.blocks), block(64 * BY);
  {
      hipLaunchKernelGGL((__PSStencilRun2_k7<VX, BY, -1, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, sh, (float *)red1, (float *)red2);
  }
}

static void __PSLaunch2_k7(const struct __PSStencil_k7 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  if (s.g->dim[0] % __PS2VX_k7 == 0)
    __PSLaunch2R_k7<false>(s, src, dst, store_mid, stream, red1, red2);
  else
    __PSLaunch2R_k7<__PS2VX_k7 != 1>(s, src, dst, store_mid, stream, red1, red2);
}

// The pair (s0, s1) is k7(a -> b), k7(b -> a) over one domain strictly
// inside the grids, with the same centre-only grids (neither a nor b) and
// scalars: it may run as two-sweep passes.
static bool __PSFusable2_k7(const struct __PSStencil_k7 &s0, const struct __PSStencil_k7 &s1) {
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

// Resident-tile pass of k7: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_k7(
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
  __PSCtx_k7 ctx;
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
      ctx.g[2] = cur[p.at + -1 + RX * (0 + RY * (0))];
      ctx.g[3] = cur[p.at + 0 + RX * (1 + RY * (0))];
      ctx.g[4] = cur[p.at + 0 + RX * (-1 + RY * (0))];
      ctx.g[5] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g[6] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g2_e = false;
      k7(p.x, p.y, p.z, ctx);
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
static void __PSLaunchTile_k7(const struct __PSStencil_k7 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_k7<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_k7(const struct __PSStencil_k7 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_k7<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_k7<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil k7p
struct __PSStencil_k7p {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k7p __PSStencilMap_k7p(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_k7p __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k7p (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] periodic
//     offsets 0:(0,0,0)p 1:(1,0,0)p 2:(-1,0,0)p 3:(0,1,0)p 4:(0,-1,0)p 5:(0,0,1)p 6:(0,0,-1)p
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes
struct __PSCtx_k7p {
  float g[7];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k7p(
    const int x, const int y, const int z, __PSCtx_k7p &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_k7p(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, true, float, RAGGED> S_g;
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
    __PSCtx_k7p ctx;
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
          float g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r2);
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
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g[5] = g_r3[i + 0];
              ctx.g[6] = g_r4[i + 0];
              ctx.g2_e = false;
              k7p(x, yrow, z, ctx);
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
static physis_hip::RunShape __PSShape_k7p(const struct __PSStencil_k7p &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_k7p<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_k7p(const struct __PSStencil_k7p &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_k7p<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_k7p<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_k7p(const struct __PSStencil_k7p &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_k7p<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSShape_k7p<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_k7p<1>(s).blocks;
}

static int __PSRun_k7p(const struct __PSStencil_k7p &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_k7p<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSLaunch_k7p<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_k7p<1>(s, stream, red);
}

// Two-sweep run kernel of k7p (temporal blocking): one pass over src
// computes u' = k7p(src) on the tile and a one-point halo and
// u'' = k7p(u') three planes behind; dst <- u'', mid <- u' when
// mid is not NULL.  Two planes per barrier: an interval computes u' of
// planes s0 and s0 + 1 and u'' of s0 - 3 and s0 - 2 from rings of six
// slots (source plane p in slot (p - zb + 2) % 6, u'(p) in slot
// (p - zb + 1) % 6), then stores source planes s0 + 3 and s0 + 4.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_k7p(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ mid, physis_hip::RunShape sh) {
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
  __PSCtx_k7p ctx;
  ctx.g_p = src.p;
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) {
    ctx.g_dim[d] = src.dim[d];
    ctx.g2_dim[d] = src.dim[d];
  }
  auto __uprime = [&](const int s, const int sm, const int sc, const int sp, const int bo) {
    if (mid_row && s <= ze) {
      float a_r0[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sc * SA::kPlane, wave + 0, lane, a_r0);
      float a_r1[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sc * SA::kPlane, wave + 1, lane, a_r1);
      float a_r2[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sc * SA::kPlane, wave + -1, lane, a_r2);
      float a_r3[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sp * SA::kPlane, wave + 0, lane, a_r3);
      float a_r4[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sm * SA::kPlane, wave + 0, lane, a_r4);
      float uo[VX];
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g[0] = a_r0[i + 1];
        ctx.g[1] = a_r0[i + 2];
        ctx.g[2] = a_r0[i + 0];
        ctx.g[3] = a_r1[i + 0];
        ctx.g[4] = a_r2[i + 0];
        ctx.g[5] = a_r3[i + 0];
        ctx.g[6] = a_r4[i + 0];
        ctx.g2_e = false;
        k7p(xs + i, yrow, s, ctx);
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
      ctx.g[0] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[1] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g[2] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g[3] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[4] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[5] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[6] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g2_e = false;
      k7p(x0 + px, y0 - 2 + hr, s, ctx);
      b_lds[bo * SB::kPlane + hr * SB::kRow + SB::kPad + px] = ctx.g2_v;
    }
  };
  auto __udouble = [&](const int z, const int sm, const int sc, const int sp) {
    if (out_row && z >= zb && z < ze) {
      float b_r0[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sc * SB::kPlane, wave + 0, lane, b_r0);
      float b_r1[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sc * SB::kPlane, wave + 1, lane, b_r1);
      float b_r2[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sc * SB::kPlane, wave + -1, lane, b_r2);
      float b_r3[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sp * SB::kPlane, wave + 0, lane, b_r3);
      float b_r4[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sm * SB::kPlane, wave + 0, lane, b_r4);
      float uu[VX];
      unsigned m = 0;
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g[0] = b_r0[i + 1];
        ctx.g[1] = b_r0[i + 2];
        ctx.g[2] = b_r0[i + 0];
        ctx.g[3] = b_r1[i + 0];
        ctx.g[4] = b_r2[i + 0];
        ctx.g[5] = b_r3[i + 0];
        ctx.g[6] = b_r4[i + 0];
        ctx.g2_e = false;
        k7p(xs + i, yrow, z, ctx);
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
static void __PSLaunch2V_k7p(const struct __PSStencil_k7p &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  constexpr int BY = 12;
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_k7p<VX, BY, false>, 64 * BY);
  const physis_hip::RunShape sh = physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g}, 3), 4);
  if (sh.blocks == 0) return;
  if (s.g->dim[0] % VX == 0)
    hipLaunchKernelGGL((__PSStencilRun2_k7p<VX, BY, false>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, sh);
  else
    hipLaunchKernelGGL((__PSStencilRun2_k7p<VX, BY, true>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, sh);
}

static void __PSLaunch2_k7p(const struct __PSStencil_k7p &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  if (physis_hip::PairVX(s.g->dim, true, false) == 4)
    __PSLaunch2V_k7p<4>(s, src, dst, mid, stream);
  else
    __PSLaunch2V_k7p<2>(s, src, dst, mid, stream);
}

// The pair (s0, s1) is k7p(a -> b), k7p(b -> a) over the whole grid with the
// same scalars: it may run as two-sweep passes.
static bool __PSFusable2_k7p(const struct __PSStencil_k7p &s0, const struct __PSStencil_k7p &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != 0 || s0.dom.local_max[d] != a->dim[d]) return false;
    if (s1.dom.local_min[d] != 0 || s1.dom.local_max[d] != a->dim[d]) return false;
  }
  if (!physis_hip::PassesPay(a->dim, true, false, true)) return false;
  return physis_hip::WindowsFit({a}, 3);
}

// Resident-tile pass of k7p: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_k7p(
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
  physis_hip::LoadTile<TILE, true>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  __PSCtx_k7p ctx;
  ctx.g_p = src.p;
  for (int d = 0; d < 3; ++d) ctx.g_dim[d] = src.dim[d];
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
      ctx.g[0] = cur[p.at + 0 + RX * (0 + RY * (0))];
      ctx.g[1] = cur[p.at + 1 + RX * (0 + RY * (0))];
      ctx.g[2] = cur[p.at + -1 + RX * (0 + RY * (0))];
      ctx.g[3] = cur[p.at + 0 + RX * (1 + RY * (0))];
      ctx.g[4] = cur[p.at + 0 + RX * (-1 + RY * (0))];
      ctx.g[5] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g[6] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g2_e = false;
      k7p(p.x, p.y, p.z, ctx);
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
static void __PSLaunchTile_k7p(const struct __PSStencil_k7p &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_k7p<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_k7p(const struct __PSStencil_k7p &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_k7p<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_k7p<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil k7n
struct __PSStencil_k7n {
  __PSDomain dom;
  __PSGrid *g1;
  int __g1_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k7n __PSStencilMap_k7n(
    __PSDomain __dom, __PSGrid *g1, __PSGrid *g2) {
  struct __PSStencil_k7n __s = {__dom, g1, __PSGridGetID(g1), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k7n (2.5D run kernel):
//   g1  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,-1,0) 4:(0,1,0) 5:(0,0,-1) 6:(0,0,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes
struct __PSCtx_k7n {
  float g1[7];
  const float *g1_p;
  int g1_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k7n(
    const int x, const int y, const int z, __PSCtx_k7n &__ctx) {
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
  (__ctx.g2_v = (c + w + e + s + n + b + t), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_k7n(
    __PSDomain dom, __PSGrid3DFloat_dev g1, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
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
    __PSCtx_k7n ctx;
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
              k7n(x, yrow, z, ctx);
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
static physis_hip::RunShape __PSShape_k7n(const struct __PSStencil_k7n &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_k7n<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g1, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_k7n(const struct __PSStencil_k7n &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_k7n<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_k7n<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g1), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_k7n(const struct __PSStencil_k7n &s) {
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_k7n<4>(s).blocks
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_k7n<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_k7n<1>(s).blocks;
}

static int __PSRun_k7n(const struct __PSStencil_k7n &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g1, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_k7n<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_k7n<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_k7n<1>(s, stream, red);
}

// Two-sweep run kernel of k7n (temporal blocking): one pass over src
// computes u' = k7n(src) on the tile and a one-point halo and
// u'' = k7n(u') three planes behind; dst <- u'', mid <- u' when
// mid is not NULL.  Two planes per barrier: an interval computes u' of
// planes s0 and s0 + 1 and u'' of s0 - 3 and s0 - 2 from rings of six
// slots (source plane p in slot (p - zb + 2) % 6, u'(p) in slot
// (p - zb + 1) % 6), then stores source planes s0 + 3 and s0 + 4.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_k7n(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ mid, physis_hip::RunShape sh) {
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
  __PSCtx_k7n ctx;
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
        k7n(xs + i, yrow, s, ctx);
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
      k7n(x0 + px, y0 - 2 + hr, s, ctx);
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
        k7n(xs + i, yrow, z, ctx);
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
static void __PSLaunch2V_k7n(const struct __PSStencil_k7n &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  constexpr int BY = 12;
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_k7n<VX, BY, false>, 64 * BY);
  const physis_hip::RunShape sh = physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g1}, 3), 4);
  if (sh.blocks == 0) return;
  if (s.g1->dim[0] % VX == 0)
    hipLaunchKernelGGL((__PSStencilRun2_k7n<VX, BY, false>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, sh);
  else
    hipLaunchKernelGGL((__PSStencilRun2_k7n<VX, BY, true>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, sh);
}

static void __PSLaunch2_k7n(const struct __PSStencil_k7n &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  if (physis_hip::PairVX(s.g1->dim, false, false) == 4)
    __PSLaunch2V_k7n<4>(s, src, dst, mid, stream);
  else
    __PSLaunch2V_k7n<2>(s, src, dst, mid, stream);
}

// The pair (s0, s1) is k7n(a -> b), k7n(b -> a) over the whole grid with the
// same scalars: it may run as two-sweep passes.
static bool __PSFusable2_k7n(const struct __PSStencil_k7n &s0, const struct __PSStencil_k7n &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g1, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g1 != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != 0 || s0.dom.local_max[d] != a->dim[d]) return false;
    if (s1.dom.local_min[d] != 0 || s1.dom.local_max[d] != a->dim[d]) return false;
  }
  if (!physis_hip::PassesPay(a->dim, false, false, true)) return false;
  return physis_hip::WindowsFit({a}, 3);
}

// Resident-tile pass of k7n: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_k7n(
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
  physis_hip::LoadTile<TILE, false>(lds[0], src.p, src.dim, x0, y0, z0);
  __syncthreads();
  __PSCtx_k7n ctx;
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
      k7n(p.x, p.y, p.z, ctx);
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
static void __PSLaunchTile_k7n(const struct __PSStencil_k7n &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = s.dom;
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_k7n<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, src, dst, bg, store_mid, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_k7n(const struct __PSStencil_k7n &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(s.dom))
    __PSLaunchTile_k7n<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_k7n<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil kasym
struct __PSStencil_kasym {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_kasym __PSStencilMap_kasym(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_kasym __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of kasym (2.5D run kernel):
//   g  staged x[-2,2] y[-2,2] z[-2,1] non-periodic
//     offsets 0:(0,0,0) 1:(1,1,1) 2:(-2,-2,-2)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (halo wider than one point)
struct __PSCtx_kasym {
  float g[3];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void kasym(
    const int x, const int y, const int z, __PSCtx_kasym &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 2 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kasym(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 2;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 2, HY, 5, false, float, RAGGED> S_g;
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
    const physis_hip::BufWin<float> g_w = physis_hip::BufWin<float>::Make(g.p, g_nxy * g.dim[2], (long)(zb + -3) * g_nxy, (long)(ze + 2) * g_nxy);
    S_g g_st[PD];
    const typename S_g::Addr g_ra = S_g::Prepare(g.dim, x0, yrow, lane);
    S_g g_pro[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      g_pro[k].Load(g_w, g.p, g.dim, g_ra, zb + -2 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g_st[k].Load(g_w, g.p, g.dim, g_ra, zb + 2 + k);
    int g_base = 0;
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_kasym ctx;
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
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        if (computes && z < ze) {
          float g_r0[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<5>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<1, 1>(g_lds + physis_hip::RingSlot<5>(g_base, 3) * S_g::kPlane, wave + 1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<-2, -2>(g_lds + physis_hip::RingSlot<5>(g_base, 0) * S_g::kPlane, wave + -2, lane, g_r2);
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
              ctx.g2_e = false;
              kasym(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<5>(g_base, 4) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 2 + PD);
        g_base = physis_hip::RingSlot<5>(g_base, 1);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_kasym(const struct __PSStencil_kasym &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kasym<VX, 8, -1>, 64 * 8);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 8 - 2 * 2, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 3));
}

template <int VX>
static int __PSLaunch_kasym(const struct __PSStencil_kasym &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kasym<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 8);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_kasym<VX, 8, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kasym(const struct __PSStencil_kasym &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kasym<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_kasym<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_kasym<1>(s).blocks;
}

static int __PSRun_kasym(const struct __PSStencil_kasym &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kasym<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_kasym<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_kasym<1>(s, stream, red);
}

// ---------------------------------------------- stencil kasymp
struct __PSStencil_kasymp {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_kasymp __PSStencilMap_kasymp(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_kasymp __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of kasymp (2.5D run kernel):
//   g  staged x[-2,2] y[-0,0] z[0,0] periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(2,0,0)p
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (halo wider than one point)
struct __PSCtx_kasymp {
  float g[3];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void kasymp(
    const int x, const int y, const int z, __PSCtx_kasymp &__ctx) {
  float v = __ctx.g[0] + physis_hip::GetLinear<float>(__ctx.g_p, __ctx.g_dim, 3, x - 1, y, z) + __ctx.g[2];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kasymp(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 0;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 2, HY, 2, true, float, RAGGED> S_g;
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
    const physis_hip::BufWin<float> g_w = physis_hip::BufWin<float>::Make(g.p, g_nxy * g.dim[2], (long)(zb + -1) * g_nxy, (long)(ze + 1) * g_nxy);
    S_g g_st[PD];
    const typename S_g::Addr g_ra = S_g::Prepare(g.dim, x0, yrow, lane);
    S_g g_pro[1];
#pragma unroll
    for (int k = 0; k < 1; ++k)
      g_pro[k].Load(g_w, g.p, g.dim, g_ra, zb + 0 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g_st[k].Load(g_w, g.p, g.dim, g_ra, zb + 1 + k);
    int g_base = 0;
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 1; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_kasymp ctx;
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
        const int g_base = k % 2;
        if (computes && z < ze) {
          float g_r0[VX + 2];
          S_g::template ReadRow<0, 2>(g_lds + physis_hip::RingSlot<2>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r0);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 0];
              ctx.g[2] = g_r0[i + 2];
              ctx.g2_e = false;
              kasymp(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<2>(g_base, 1) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 1 + PD);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_kasymp(const struct __PSStencil_kasymp &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kasymp<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 0, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 1));
}

template <int VX>
static int __PSLaunch_kasymp(const struct __PSStencil_kasymp &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kasymp<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_kasymp<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kasymp(const struct __PSStencil_kasymp &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kasymp<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSShape_kasymp<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_kasymp<1>(s).blocks;
}

static int __PSRun_kasymp(const struct __PSStencil_kasymp &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kasymp<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSLaunch_kasymp<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_kasymp<1>(s, stream, red);
}

// ---------------------------------------------- stencil k27
struct __PSStencil_k27 {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k27 __PSStencilMap_k27(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_k27 __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k27 (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,-1) 1:(1,0,-1) 2:(-1,0,-1) 3:(0,1,-1) 4:(1,1,-1) 5:(-1,1,-1) 6:(0,-1,-1) 7:(1,-1,-1) 8:(-1,-1,-1) 9:(0,0,0) 10:(1,0,0) 11:(-1,0,0) 12:(0,1,0) 13:(1,1,0) 14:(-1,1,0) 15:(0,-1,0) 16:(1,-1,0) 17:(-1,-1,0) 18:(0,0,1) 19:(1,0,1) 20:(-1,0,1) 21:(0,1,1) 22:(1,1,1) 23:(-1,1,1) 24:(0,-1,1) 25:(1,-1,1) 26:(-1,-1,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_k27 {
  float g[27];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k27(
    const int x, const int y, const int z, __PSCtx_k27 &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6] + __ctx.g[7] + __ctx.g[8] + __ctx.g[9] + __ctx.g[10] + __ctx.g[11] + __ctx.g[12] + __ctx.g[13] + __ctx.g[14] + __ctx.g[15] + __ctx.g[16] + __ctx.g[17] + __ctx.g[18] + __ctx.g[19] + __ctx.g[20] + __ctx.g[21] + __ctx.g[22] + __ctx.g[23] + __ctx.g[24] + __ctx.g[25] + __ctx.g[26];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_k27(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
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
    __PSCtx_k27 ctx;
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
          float g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 1, lane, g_r1);
          float g_r2[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + -1, lane, g_r2);
          float g_r3[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r4);
          float g_r5[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r5);
          float g_r6[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r6);
          float g_r7[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 1, lane, g_r7);
          float g_r8[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + -1, lane, g_r8);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 1];
              ctx.g[4] = g_r1[i + 2];
              ctx.g[5] = g_r1[i + 0];
              ctx.g[6] = g_r2[i + 1];
              ctx.g[7] = g_r2[i + 2];
              ctx.g[8] = g_r2[i + 0];
              ctx.g[9] = g_r3[i + 1];
              ctx.g[10] = g_r3[i + 2];
              ctx.g[11] = g_r3[i + 0];
              ctx.g[12] = g_r4[i + 1];
              ctx.g[13] = g_r4[i + 2];
              ctx.g[14] = g_r4[i + 0];
              ctx.g[15] = g_r5[i + 1];
              ctx.g[16] = g_r5[i + 2];
              ctx.g[17] = g_r5[i + 0];
              ctx.g[18] = g_r6[i + 1];
              ctx.g[19] = g_r6[i + 2];
              ctx.g[20] = g_r6[i + 0];
              ctx.g[21] = g_r7[i + 1];
              ctx.g[22] = g_r7[i + 2];
              ctx.g[23] = g_r7[i + 0];
              ctx.g[24] = g_r8[i + 1];
              ctx.g[25] = g_r8[i + 2];
              ctx.g[26] = g_r8[i + 0];
              ctx.g2_e = false;
              k27(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_k27(const struct __PSStencil_k27 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_k27<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_k27(const struct __PSStencil_k27 &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_k27<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_k27<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_k27(const struct __PSStencil_k27 &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_k27<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_k27<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_k27<1>(s).blocks;
}

static int __PSRun_k27(const struct __PSStencil_k27 &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_k27<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_k27<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_k27<1>(s, stream, red);
}

// Two-sweep run kernel of k27 over a domain strictly inside
// the grid: one pass over src computes u' = k27(src) on the
// tile and a one-point halo (bg's own values outside the domain) and
// u'' = k27(u') two planes behind; dst <- u'', and bg <- u'
// when store_mid.  red1 / red2: per-block partials of the two sweeps.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, int RED, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_k27(
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
    __PSCtx_k27 ctx;
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
          float a_r0[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 0, lane, a_r0);
          float a_r1[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + 1, lane, a_r1);
          float a_r2[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 0) * SA::kPlane, wave + -1, lane, a_r2);
          float a_r3[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 0, lane, a_r3);
          float a_r4[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + 1, lane, a_r4);
          float a_r5[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 1) * SA::kPlane, wave + -1, lane, a_r5);
          float a_r6[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 0, lane, a_r6);
          float a_r7[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + 1, lane, a_r7);
          float a_r8[VX + 2];
          SA::template ReadRow<-1, 1>(a_lds + physis_hip::RingSlot<4>(abase, 2) * SA::kPlane, wave + -1, lane, a_r8);
          float uo[VX];
          unsigned m = 0;
          const bool own = out_row && s >= zb && s < ze;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = a_r0[i + 1];
            ctx.g[1] = a_r0[i + 2];
            ctx.g[2] = a_r0[i + 0];
            ctx.g[3] = a_r1[i + 1];
            ctx.g[4] = a_r1[i + 2];
            ctx.g[5] = a_r1[i + 0];
            ctx.g[6] = a_r2[i + 1];
            ctx.g[7] = a_r2[i + 2];
            ctx.g[8] = a_r2[i + 0];
            ctx.g[9] = a_r3[i + 1];
            ctx.g[10] = a_r3[i + 2];
            ctx.g[11] = a_r3[i + 0];
            ctx.g[12] = a_r4[i + 1];
            ctx.g[13] = a_r4[i + 2];
            ctx.g[14] = a_r4[i + 0];
            ctx.g[15] = a_r5[i + 1];
            ctx.g[16] = a_r5[i + 2];
            ctx.g[17] = a_r5[i + 0];
            ctx.g[18] = a_r6[i + 1];
            ctx.g[19] = a_r6[i + 2];
            ctx.g[20] = a_r6[i + 0];
            ctx.g[21] = a_r7[i + 1];
            ctx.g[22] = a_r7[i + 2];
            ctx.g[23] = a_r7[i + 0];
            ctx.g[24] = a_r8[i + 1];
            ctx.g[25] = a_r8[i + 2];
            ctx.g[26] = a_r8[i + 0];
            ctx.g2_e = false;
            const bool in = yin && xs + i >= dom.local_min[0] && xs + i < dom.local_max[0] && zin(s);
            k27(xs + i, yrow, s, ctx);
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
          ctx.g[0] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[1] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.g[2] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
          ctx.g[3] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[4] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[5] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[6] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[7] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[8] = a_lds[physis_hip::RingSlot<4>(abase, 0) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[9] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[10] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.g[11] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
          ctx.g[12] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[13] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[14] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[15] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[16] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[17] = a_lds[physis_hip::RingSlot<4>(abase, 1) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[18] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
          ctx.g[19] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
          ctx.g[20] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
          ctx.g[21] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[22] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[23] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
          ctx.g[24] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
          ctx.g[25] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
          ctx.g[26] = a_lds[physis_hip::RingSlot<4>(abase, 2) * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
          ctx.g2_e = false;
          k27(hx, hy, s, ctx);
          b_lds[physis_hip::RingSlot<4>(bbase, 3) * SB::kPlane + hr * SB::kRow + SB::kPad + px] = hin && zin(s) ? ctx.g2_v : bg_c1[cur][0];
        }
        if (out_row && s - 2 >= zb) {
          float b_r0[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 0, lane, b_r0);
          float b_r1[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + 1, lane, b_r1);
          float b_r2[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 0) * SB::kPlane, wave + -1, lane, b_r2);
          float b_r3[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 0, lane, b_r3);
          float b_r4[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + 1, lane, b_r4);
          float b_r5[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 1) * SB::kPlane, wave + -1, lane, b_r5);
          float b_r6[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 0, lane, b_r6);
          float b_r7[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + 1, lane, b_r7);
          float b_r8[VX + 2];
          SB::template ReadRow<-1, 1>(b_lds + physis_hip::RingSlot<4>(bbase, 2) * SB::kPlane, wave + -1, lane, b_r8);
          float uu[VX];
          unsigned m = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            ctx.g[0] = b_r0[i + 1];
            ctx.g[1] = b_r0[i + 2];
            ctx.g[2] = b_r0[i + 0];
            ctx.g[3] = b_r1[i + 1];
            ctx.g[4] = b_r1[i + 2];
            ctx.g[5] = b_r1[i + 0];
            ctx.g[6] = b_r2[i + 1];
            ctx.g[7] = b_r2[i + 2];
            ctx.g[8] = b_r2[i + 0];
            ctx.g[9] = b_r3[i + 1];
            ctx.g[10] = b_r3[i + 2];
            ctx.g[11] = b_r3[i + 0];
            ctx.g[12] = b_r4[i + 1];
            ctx.g[13] = b_r4[i + 2];
            ctx.g[14] = b_r4[i + 0];
            ctx.g[15] = b_r5[i + 1];
            ctx.g[16] = b_r5[i + 2];
            ctx.g[17] = b_r5[i + 0];
            ctx.g[18] = b_r6[i + 1];
            ctx.g[19] = b_r6[i + 2];
            ctx.g[20] = b_r6[i + 0];
            ctx.g[21] = b_r7[i + 1];
            ctx.g[22] = b_r7[i + 2];
            ctx.g[23] = b_r7[i + 0];
            ctx.g[24] = b_r8[i + 1];
            ctx.g[25] = b_r8[i + 2];
            ctx.g[26] = b_r8[i + 0];
            ctx.g2_e = false;
            const bool in = xs + i >= dom.local_min[0] && xs + i < dom.local_max[0];
            k27(xs + i, yrow, s - 2, ctx);
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

static constexpr int __PS2VX_k27 = 4, __PS2BY_k27 = 16;
template <int VX, int BY>
static physis_hip::RunShape __PSShape2_k27(const struct __PSStencil_k27 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_k27<VX, BY, -1, false>, 64 * BY);
  return physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g, s.g2}, 3));
}

static int __PSBlocks2_k27(const struct __PSStencil_k27 &s) {
  return __PSShape2_k27<__PS2VX_k27, __PS2BY_k27>(s).blocks;
}

template <bool RAGGED>
static void __PSLaunch2R_k27(const struct __PSStencil_k27 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  constexpr int VX = __PS2VX_k27, BY = __PS2BY_k27;
  const physis_hip::RunShape sh = __PSShape2_k27<VX, BY>(s);
  if (sh.blocks == 0) return;
  const dim3 grid(sh.blocks), block(64 * BY);
  {
      hipLaunchKernelGGL((__PSStencilRun2_k27<VX, BY, -1, RAGGED>), grid, block, 0, stream, s.dom, src, dst, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), store_mid, sh, (float *)red1, (float *)red2);
  }
}

static void __PSLaunch2_k27(const struct __PSStencil_k27 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, int store_mid, hipStream_t stream, void *red1, void *red2) {
  if (s.g->dim[0] % __PS2VX_k27 == 0)
    __PSLaunch2R_k27<false>(s, src, dst, store_mid, stream, red1, red2);
  else
    __PSLaunch2R_k27<__PS2VX_k27 != 1>(s, src, dst, store_mid, stream, red1, red2);
}

// The pair (s0, s1) is k27(a -> b), k27(b -> a) over one domain strictly
// inside the grids, with the same centre-only grids (neither a nor b) and
// scalars: it may run as two-sweep passes.
static bool __PSFusable2_k27(const struct __PSStencil_k27 &s0, const struct __PSStencil_k27 &s1) {
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
  if (!physis_hip::DomainPassesPay(s0.dom, a->dim[0], a->num_elms, false)) return false;
  return physis_hip::WindowsFit({a, b}, 3);
}

// ---------------------------------------------- stencil k27p
struct __PSStencil_k27p {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k27p __PSStencilMap_k27p(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_k27p __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k27p (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] periodic
//     offsets 0:(0,0,-1)p 1:(1,0,-1)p 2:(-1,0,-1)p 3:(0,1,-1)p 4:(1,1,-1)p 5:(-1,1,-1)p 6:(0,-1,-1)p 7:(1,-1,-1)p 8:(-1,-1,-1)p 9:(0,0,0)p 10:(1,0,0)p 11:(-1,0,0)p 12:(0,1,0)p 13:(1,1,0)p 14:(-1,1,0)p 15:(0,-1,0)p 16:(1,-1,0)p 17:(-1,-1,0)p 18:(0,0,1)p 19:(1,0,1)p 20:(-1,0,1)p 21:(0,1,1)p 22:(1,1,1)p 23:(-1,1,1)p 24:(0,-1,1)p 25:(1,-1,1)p 26:(-1,-1,1)p
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes
struct __PSCtx_k27p {
  float g[27];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k27p(
    const int x, const int y, const int z, __PSCtx_k27p &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6] + __ctx.g[7] + __ctx.g[8] + __ctx.g[9] + __ctx.g[10] + __ctx.g[11] + __ctx.g[12] + __ctx.g[13] + __ctx.g[14] + __ctx.g[15] + __ctx.g[16] + __ctx.g[17] + __ctx.g[18] + __ctx.g[19] + __ctx.g[20] + __ctx.g[21] + __ctx.g[22] + __ctx.g[23] + __ctx.g[24] + __ctx.g[25] + __ctx.g[26];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_k27p(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, true, float, RAGGED> S_g;
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
    __PSCtx_k27p ctx;
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
          float g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 1, lane, g_r1);
          float g_r2[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + -1, lane, g_r2);
          float g_r3[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r3);
          float g_r4[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r4);
          float g_r5[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r5);
          float g_r6[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r6);
          float g_r7[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 1, lane, g_r7);
          float g_r8[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + -1, lane, g_r8);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 1];
              ctx.g[4] = g_r1[i + 2];
              ctx.g[5] = g_r1[i + 0];
              ctx.g[6] = g_r2[i + 1];
              ctx.g[7] = g_r2[i + 2];
              ctx.g[8] = g_r2[i + 0];
              ctx.g[9] = g_r3[i + 1];
              ctx.g[10] = g_r3[i + 2];
              ctx.g[11] = g_r3[i + 0];
              ctx.g[12] = g_r4[i + 1];
              ctx.g[13] = g_r4[i + 2];
              ctx.g[14] = g_r4[i + 0];
              ctx.g[15] = g_r5[i + 1];
              ctx.g[16] = g_r5[i + 2];
              ctx.g[17] = g_r5[i + 0];
              ctx.g[18] = g_r6[i + 1];
              ctx.g[19] = g_r6[i + 2];
              ctx.g[20] = g_r6[i + 0];
              ctx.g[21] = g_r7[i + 1];
              ctx.g[22] = g_r7[i + 2];
              ctx.g[23] = g_r7[i + 0];
              ctx.g[24] = g_r8[i + 1];
              ctx.g[25] = g_r8[i + 2];
              ctx.g[26] = g_r8[i + 0];
              ctx.g2_e = false;
              k27p(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_k27p(const struct __PSStencil_k27p &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_k27p<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_k27p(const struct __PSStencil_k27p &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_k27p<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_k27p<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_k27p(const struct __PSStencil_k27p &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_k27p<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_k27p<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_k27p<1>(s).blocks;
}

static int __PSRun_k27p(const struct __PSStencil_k27p &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_k27p<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_k27p<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_k27p<1>(s, stream, red);
}

// Two-sweep run kernel of k27p (temporal blocking): one pass over src
// computes u' = k27p(src) on the tile and a one-point halo and
// u'' = k27p(u') three planes behind; dst <- u'', mid <- u' when
// mid is not NULL.  Two planes per barrier: an interval computes u' of
// planes s0 and s0 + 1 and u'' of s0 - 3 and s0 - 2 from rings of six
// slots (source plane p in slot (p - zb + 2) % 6, u'(p) in slot
// (p - zb + 1) % 6), then stores source planes s0 + 3 and s0 + 4.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_k27p(
    __PSDomain dom, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ mid, physis_hip::RunShape sh) {
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
  __PSCtx_k27p ctx;
  ctx.g_p = src.p;
  ctx.g2_p = dst.p;
  for (int d = 0; d < 3; ++d) {
    ctx.g_dim[d] = src.dim[d];
    ctx.g2_dim[d] = src.dim[d];
  }
  auto __uprime = [&](const int s, const int sm, const int sc, const int sp, const int bo) {
    if (mid_row && s <= ze) {
      float a_r0[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sm * SA::kPlane, wave + 0, lane, a_r0);
      float a_r1[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sm * SA::kPlane, wave + 1, lane, a_r1);
      float a_r2[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sm * SA::kPlane, wave + -1, lane, a_r2);
      float a_r3[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sc * SA::kPlane, wave + 0, lane, a_r3);
      float a_r4[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sc * SA::kPlane, wave + 1, lane, a_r4);
      float a_r5[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sc * SA::kPlane, wave + -1, lane, a_r5);
      float a_r6[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sp * SA::kPlane, wave + 0, lane, a_r6);
      float a_r7[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sp * SA::kPlane, wave + 1, lane, a_r7);
      float a_r8[VX + 2];
      SA::template ReadRow<-1, 1>(a_lds + sp * SA::kPlane, wave + -1, lane, a_r8);
      float uo[VX];
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g[0] = a_r0[i + 1];
        ctx.g[1] = a_r0[i + 2];
        ctx.g[2] = a_r0[i + 0];
        ctx.g[3] = a_r1[i + 1];
        ctx.g[4] = a_r1[i + 2];
        ctx.g[5] = a_r1[i + 0];
        ctx.g[6] = a_r2[i + 1];
        ctx.g[7] = a_r2[i + 2];
        ctx.g[8] = a_r2[i + 0];
        ctx.g[9] = a_r3[i + 1];
        ctx.g[10] = a_r3[i + 2];
        ctx.g[11] = a_r3[i + 0];
        ctx.g[12] = a_r4[i + 1];
        ctx.g[13] = a_r4[i + 2];
        ctx.g[14] = a_r4[i + 0];
        ctx.g[15] = a_r5[i + 1];
        ctx.g[16] = a_r5[i + 2];
        ctx.g[17] = a_r5[i + 0];
        ctx.g[18] = a_r6[i + 1];
        ctx.g[19] = a_r6[i + 2];
        ctx.g[20] = a_r6[i + 0];
        ctx.g[21] = a_r7[i + 1];
        ctx.g[22] = a_r7[i + 2];
        ctx.g[23] = a_r7[i + 0];
        ctx.g[24] = a_r8[i + 1];
        ctx.g[25] = a_r8[i + 2];
        ctx.g[26] = a_r8[i + 0];
        ctx.g2_e = false;
        k27p(xs + i, yrow, s, ctx);
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
      ctx.g[0] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[1] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g[2] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g[3] = a_lds[sm * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[4] = a_lds[sm * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
      ctx.g[5] = a_lds[sm * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
      ctx.g[6] = a_lds[sm * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[7] = a_lds[sm * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
      ctx.g[8] = a_lds[sm * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
      ctx.g[9] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[10] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g[11] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g[12] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[13] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
      ctx.g[14] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
      ctx.g[15] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[16] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
      ctx.g[17] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
      ctx.g[18] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[19] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g[20] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g[21] = a_lds[sp * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[22] = a_lds[sp * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 1];
      ctx.g[23] = a_lds[sp * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + -1];
      ctx.g[24] = a_lds[sp * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[25] = a_lds[sp * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 1];
      ctx.g[26] = a_lds[sp * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + -1];
      ctx.g2_e = false;
      k27p(x0 + px, y0 - 2 + hr, s, ctx);
      b_lds[bo * SB::kPlane + hr * SB::kRow + SB::kPad + px] = ctx.g2_v;
    }
  };
  auto __udouble = [&](const int z, const int sm, const int sc, const int sp) {
    if (out_row && z >= zb && z < ze) {
      float b_r0[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sm * SB::kPlane, wave + 0, lane, b_r0);
      float b_r1[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sm * SB::kPlane, wave + 1, lane, b_r1);
      float b_r2[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sm * SB::kPlane, wave + -1, lane, b_r2);
      float b_r3[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sc * SB::kPlane, wave + 0, lane, b_r3);
      float b_r4[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sc * SB::kPlane, wave + 1, lane, b_r4);
      float b_r5[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sc * SB::kPlane, wave + -1, lane, b_r5);
      float b_r6[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sp * SB::kPlane, wave + 0, lane, b_r6);
      float b_r7[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sp * SB::kPlane, wave + 1, lane, b_r7);
      float b_r8[VX + 2];
      SB::template ReadRow<-1, 1>(b_lds + sp * SB::kPlane, wave + -1, lane, b_r8);
      float uu[VX];
      unsigned m = 0;
#pragma unroll
      for (int i = 0; i < VX; ++i) {
        ctx.g[0] = b_r0[i + 1];
        ctx.g[1] = b_r0[i + 2];
        ctx.g[2] = b_r0[i + 0];
        ctx.g[3] = b_r1[i + 1];
        ctx.g[4] = b_r1[i + 2];
        ctx.g[5] = b_r1[i + 0];
        ctx.g[6] = b_r2[i + 1];
        ctx.g[7] = b_r2[i + 2];
        ctx.g[8] = b_r2[i + 0];
        ctx.g[9] = b_r3[i + 1];
        ctx.g[10] = b_r3[i + 2];
        ctx.g[11] = b_r3[i + 0];
        ctx.g[12] = b_r4[i + 1];
        ctx.g[13] = b_r4[i + 2];
        ctx.g[14] = b_r4[i + 0];
        ctx.g[15] = b_r5[i + 1];
        ctx.g[16] = b_r5[i + 2];
        ctx.g[17] = b_r5[i + 0];
        ctx.g[18] = b_r6[i + 1];
        ctx.g[19] = b_r6[i + 2];
        ctx.g[20] = b_r6[i + 0];
        ctx.g[21] = b_r7[i + 1];
        ctx.g[22] = b_r7[i + 2];
        ctx.g[23] = b_r7[i + 0];
        ctx.g[24] = b_r8[i + 1];
        ctx.g[25] = b_r8[i + 2];
        ctx.g[26] = b_r8[i + 0];
        ctx.g2_e = false;
        k27p(xs + i, yrow, z, ctx);
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
static void __PSLaunch2V_k27p(const struct __PSStencil_k27p &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  constexpr int BY = 12;
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_k27p<VX, BY, false>, 64 * BY);
  const physis_hip::RunShape sh = physis_hip::PlanRun(s.dom, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g}, 3), 4);
  if (sh.blocks == 0) return;
  if (s.g->dim[0] % VX == 0)
    hipLaunchKernelGGL((__PSStencilRun2_k27p<VX, BY, false>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, sh);
  else
    hipLaunchKernelGGL((__PSStencilRun2_k27p<VX, BY, true>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, src, dst, mid, sh);
}

static void __PSLaunch2_k27p(const struct __PSStencil_k27p &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  if (physis_hip::PairVX(s.g->dim, true, false) == 4)
    __PSLaunch2V_k27p<4>(s, src, dst, mid, stream);
  else
    __PSLaunch2V_k27p<2>(s, src, dst, mid, stream);
}

// The pair (s0, s1) is k27p(a -> b), k27p(b -> a) over the whole grid with the
// same scalars: it may run as two-sweep passes.
static bool __PSFusable2_k27p(const struct __PSStencil_k27p &s0, const struct __PSStencil_k27p &s1) {
  static const bool off = getenv("PHYSIS_HIP_NO_FUSE") != NULL;
  const __PSGrid *a = s0.g, *b = s0.g2;
  if (off || !a || !b || a == b || s1.g != b || s1.g2 != a) return false;
  if (a->num_dims != 3 || b->num_dims != 3) return false;
  for (int d = 0; d < 3; ++d) {
    if (a->dim[d] != b->dim[d]) return false;
    if (s0.dom.local_min[d] != 0 || s0.dom.local_max[d] != a->dim[d]) return false;
    if (s1.dom.local_min[d] != 0 || s1.dom.local_max[d] != a->dim[d]) return false;
  }
  if (!physis_hip::PassesPay(a->dim, true, false, false)) return false;
  return physis_hip::WindowsFit({a}, 3);
}

// ---------------------------------------------- stencil k27i
struct __PSStencil_k27i {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k27i __PSStencilMap_k27i(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_k27i __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k27i (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,-1) 1:(1,0,-1) 2:(-1,0,-1) 3:(0,1,-1) 4:(1,1,-1) 5:(-1,1,-1) 6:(0,-1,-1) 7:(1,-1,-1) 8:(-1,-1,-1) 9:(0,0,0) 10:(1,0,0) 11:(-1,0,0) 12:(0,1,0) 13:(1,1,0) 14:(-1,1,0) 15:(0,-1,0) 16:(1,-1,0) 17:(-1,-1,0) 18:(0,0,1) 19:(1,0,1) 20:(-1,0,1) 21:(0,1,1) 22:(1,1,1) 23:(-1,1,1) 24:(0,-1,1) 25:(1,-1,1) 26:(-1,-1,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (not float grids)
struct __PSCtx_k27i {
  int g[27];
  const int *g_p;
  int g_dim[3];
  int g2_v;
  bool g2_e;
  const int *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k27i(
    const int x, const int y, const int z, __PSCtx_k27i &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6] + __ctx.g[7] + __ctx.g[8] + __ctx.g[9] + __ctx.g[10] + __ctx.g[11] + __ctx.g[12] + __ctx.g[13] + __ctx.g[14] + __ctx.g[15] + __ctx.g[16] + __ctx.g[17] + __ctx.g[18] + __ctx.g[19] + __ctx.g[20] + __ctx.g[21] + __ctx.g[22] + __ctx.g[23] + __ctx.g[24] + __ctx.g[25] + __ctx.g[26];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_k27i(
    __PSDomain dom, __PSGrid3DInt_dev g, __PSGrid3DInt_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<int, VX, BY, 1, HY, 4, false, int, RAGGED> S_g;
  __shared__ __attribute__((aligned(16))) int g_lds[S_g::kLdsElems];
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
    const physis_hip::BufWin<int> g_w = physis_hip::BufWin<int>::Make(g.p, g_nxy * g.dim[2], (long)(zb + -2) * g_nxy, (long)(ze + 2) * g_nxy);
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
    const physis_hip::BufWin<int> g2_ew = physis_hip::BufWin<int>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_k27i ctx;
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
          int g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r0);
          int g_r1[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 1, lane, g_r1);
          int g_r2[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + -1, lane, g_r2);
          int g_r3[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r3);
          int g_r4[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r4);
          int g_r5[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r5);
          int g_r6[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r6);
          int g_r7[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 1, lane, g_r7);
          int g_r8[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + -1, lane, g_r8);
          int g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 1];
              ctx.g[4] = g_r1[i + 2];
              ctx.g[5] = g_r1[i + 0];
              ctx.g[6] = g_r2[i + 1];
              ctx.g[7] = g_r2[i + 2];
              ctx.g[8] = g_r2[i + 0];
              ctx.g[9] = g_r3[i + 1];
              ctx.g[10] = g_r3[i + 2];
              ctx.g[11] = g_r3[i + 0];
              ctx.g[12] = g_r4[i + 1];
              ctx.g[13] = g_r4[i + 2];
              ctx.g[14] = g_r4[i + 0];
              ctx.g[15] = g_r5[i + 1];
              ctx.g[16] = g_r5[i + 2];
              ctx.g[17] = g_r5[i + 0];
              ctx.g[18] = g_r6[i + 1];
              ctx.g[19] = g_r6[i + 2];
              ctx.g[20] = g_r6[i + 0];
              ctx.g[21] = g_r7[i + 1];
              ctx.g[22] = g_r7[i + 2];
              ctx.g[23] = g_r7[i + 0];
              ctx.g[24] = g_r8[i + 1];
              ctx.g[25] = g_r8[i + 2];
              ctx.g[26] = g_r8[i + 0];
              ctx.g2_e = false;
              k27i(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<int, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
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
static physis_hip::RunShape __PSShape_k27i(const struct __PSStencil_k27i &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_k27i<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_k27i(const struct __PSStencil_k27i &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_k27i<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_k27i<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DInt_dev>(s.g), physis_hip::DevView<__PSGrid3DInt_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_k27i(const struct __PSStencil_k27i &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_k27i<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_k27i<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_k27i<1>(s).blocks;
}

static int __PSRun_k27i(const struct __PSStencil_k27i &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_INT);
  physis_hip::CheckGrid3D(s.g2, PS_INT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_k27i<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_k27i<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_k27i<1>(s, stream, red);
}

static void __PSStencilRun_0(int iter, struct __PSStencil_k7 s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k7");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k7(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_1(int iter, struct __PSStencil_k7p s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k7p");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k7p(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_2(int iter, struct __PSStencil_kasym s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kasym");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kasym(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_3(int iter, struct __PSStencil_kasymp s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kasymp");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kasymp(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_4(int iter, struct __PSStencil_k27 s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k27");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k27(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_5(int iter, struct __PSStencil_k27p s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k27p");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k27p(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

static void run_one(int which, int n, int lo, int hi, float * out) {
  PSGrid3DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, n, n, n);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, n, n, n);
  PSDomain3D d = PSDomain3DNew(lo, hi, lo, hi, lo, hi);
  size_t nelms = n * n * n;
  float *indata = (float*)malloc(sizeof(float) * nelms);
  size_t i;
  for (i = 0; i < nelms; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  if (which == 0)
    __PSStencilRun_0(1, __PSStencilMap_k7(d, g1, g2));
  if (which == 1)
    __PSStencilRun_1(1, __PSStencilMap_k7p(d, g1, g2));
  if (which == 2)
    __PSStencilRun_2(1, __PSStencilMap_kasym(d, g1, g2));
  if (which == 3)
    __PSStencilRun_3(1, __PSStencilMap_kasymp(d, g1, g2));
  if (which == 4)
    __PSStencilRun_4(1, __PSStencilMap_k27(d, g1, g2));
  if (which == 5)
    __PSStencilRun_5(1, __PSStencilMap_k27p(d, g1, g2));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

void systest_7pt(float * out) {
  run_one(0, 32, 1, 32 - 1, out);
}

void systest_7pt_periodic(float * out) {
  run_one(1, 32, 0, 32, out);
}

void systest_asymmetric(float * out) {
  run_one(2, 32, 2, 32 - 2, out);
}

void systest_asymmetric_periodic(float * out) {
  run_one(3, 32, 2, 32 - 2, out);
}

void systest_27pt(float * out) {
  run_one(4, 32, 1, 32 - 1, out);
}

void systest_27pt_periodic(float * out) {
  run_one(5, 32, 0, 32, out);
}

}  // extern "C"

static void __PSStencilRun_6(int iter, struct __PSStencil_k7n s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k7n");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k7n(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_7pt_neumann(float * out) {
  int n = 8;
  PSGrid3DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, n, n, n);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, n, n, n);
  PSDomain3D d = PSDomain3DNew(0, n, 0, n, 0, n);
  float *indata = (float*)malloc(sizeof(float) * n * n * n);
  int i;
  for (i = 0; i < n * n * n; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSStencilRun_6(1, __PSStencilMap_k7n(d, g1, g2));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

}  // extern "C"

static void __PSStencilRun_7(int iter, struct __PSStencil_k7 s0, struct __PSStencil_k7 s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k7, k7");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_k7(s0, s1) &&
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
        __PSLaunchT_k7<4>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else if (__small)
        __PSLaunchT_k7<2>(s0, src, dst, vb.p, (j == passes - 1), stream, {});
      else
        __PSLaunch2_k7(s0, src, dst, (j == passes - 1), stream, NULL, NULL);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_k7(s0, stream, NULL);
    __PSRun_k7(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_7pt_multi_iterations(float * out) {
  PSGrid3DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 32, 32, 32);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 32, 32, 32);
  PSDomain3D d = PSDomain3DNew(1, 32 - 1, 1, 32 - 1, 1, 32 - 1);
  float *indata = (float*)malloc(sizeof(float) * 32 * 32 * 32);
  int i;
  for (i = 0; i < 32 * 32 * 32; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  __PSStencilRun_7(5, __PSStencilMap_k7(d, g1, g2), __PSStencilMap_k7(d, g2, g1));
  __PSGridCopyout(g1, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

}  // extern "C"

static void __PSStencilRun_8(int iter, struct __PSStencil_k27i s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k27i");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k27i(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_9(int iter, struct __PSStencil_k27i s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k27i");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k27i(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_27pt_reduction(int * v1, int * v2) {
  int n = 16;
  PSGrid3DInt g1 = physis_hip::NewGrid(PS_INT, sizeof(int), 3, n, n, n);
  PSGrid3DInt g2 = physis_hip::NewGrid(PS_INT, sizeof(int), 3, n, n, n);
  PSDomain3D d = PSDomain3DNew(1, n - 1, 1, n - 1, 1, n - 1);
  int *indata = (int*)malloc(sizeof(int) * n * n * n);
  int i;
  for (i = 0; i < n * n * n; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  __PSStencilRun_8(1, __PSStencilMap_k27i(d, g1, g2));
  __PSReduceGridInt(v1, (enum PSReduceOp)(PS_SUM), g2);
  __PSStencilRun_9(1, __PSStencilMap_k27i(d, g2, g1));
  __PSReduceGridInt(v2, (enum PSReduceOp)(PS_SUM), g1);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

void systest_reduction_3d_sum(float * v) {
  int n = 16;
  PSGrid3DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, n, n, n);
  float *indata = (float*)malloc(sizeof(float) * n * n * n);
  int i;
  for (i = 0; i < n * n * n; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSReduceGridFloat(v, (enum PSReduceOp)(PS_SUM), g1);
  __PSGridFree(g1, NULL);
  free(indata);
}

}  // extern "C"

// ---------------------------------------------- stencil krb
struct __PSStencil_krb {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  int __rb;  // -1 all points, 0 red, 1 black, 2 red then black
};

static struct __PSStencil_krb __PSStencilMap_krb(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krb __s = {__dom, g, __PSGridGetID(g), -1};
  return __s;
}

static struct __PSStencil_krb __PSStencilMapRed_krb(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krb __s = __PSStencilMap_krb(__dom, g);
  __s.__rb = 0;
  return __s;
}

static struct __PSStencil_krb __PSStencilMapBlack_krb(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krb __s = __PSStencilMap_krb(__dom, g);
  __s.__rb = 1;
  return __s;
}

static struct __PSStencil_krb __PSStencilMapRedBlack_krb(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krb __s = __PSStencilMap_krb(__dom, g);
  __s.__rb = 2;
  return __s;
}

// Stencil analysis of krb (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic, emitted
//     offsets 0:(0,0,0) 1:(1,0,0) 2:(-1,0,0) 3:(0,1,0) 4:(0,-1,0) 5:(0,0,-1) 6:(0,0,1)
//   red-black: in-place colour sweep reads only the other colour
//   two-sweep fusion of map pairs: red-black: one pass per iteration (red, then black) over a domain inside the grid
struct __PSCtx_krb {
  float g[7];
  float g_v;
  bool g_e;
  const float *g_p;
  int g_dim[3];
};

__device__ __forceinline__ void krb(
    const int x, const int y, const int z, __PSCtx_krb &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6];
  (__ctx.g_v = (v), __ctx.g_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_krb(
    __PSDomain dom, __PSGrid3DFloat_dev g, physis_hip::RunShape sh, float *__restrict__ __red, int __rb) {
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
    __PSCtx_krb ctx;
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
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r2);
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
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g[5] = g_r3[i + 0];
              ctx.g[6] = g_r4[i + 0];
              ctx.g_e = false;
              krb(x, yrow, z, ctx);
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
static physis_hip::RunShape __PSShape_krb(const struct __PSStencil_krb &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_krb<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g}, 2));
}

template <int VX>
static int __PSLaunch_krb(const struct __PSStencil_krb &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_krb<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  for (int __c = s.__rb == 2 ? 0 : s.__rb; __c <= (s.__rb == 2 ? 1 : s.__rb); ++__c) {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_krb<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), sh, (float *)NULL, __c);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_krb(const struct __PSStencil_krb &s) {
  return (s.g->dim[0] % 4 == 0) ? __PSShape_krb<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, true)) ? __PSShape_krb<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_krb<1>(s).blocks;
}

static int __PSRun_krb(const struct __PSStencil_krb &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g);
  return (s.g->dim[0] % 4 == 0) ? __PSLaunch_krb<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, true)) ? __PSLaunch_krb<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_krb<1>(s, stream, red);
}

// Two-sweep run kernel of krb (temporal blocking): one pass over src
// computes u' = krb(src) on the tile and a one-point halo and
// u'' = krb(u') three planes behind; dst <- u'', mid <- u' when
// mid is not NULL.  Two planes per barrier: an interval computes u' of
// planes s0 and s0 + 1 and u'' of s0 - 3 and s0 - 2 from rings of six
// slots (source plane p in slot (p - zb + 2) % 6, u'(p) in slot
// (p - zb + 1) % 6), then stores source planes s0 + 3 and s0 + 4.
// Red-black: one pass is one iteration (red sweep u', black sweep
// u''); dom is the map's domain, gd the whole grid the pass tiles.
// RAGGED: x extents that are not multiples of VX.
template <int VX, int BY, bool RAGGED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun2_krb(
    __PSDomain dom, __PSDomain gd, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ mid, physis_hip::RunShape sh) {
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
  __PSCtx_krb ctx;
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
      SA::template ReadRow<0, 0>(a_lds + sc * SA::kPlane, wave + 1, lane, a_r1);
      float a_r2[VX + 0];
      SA::template ReadRow<0, 0>(a_lds + sc * SA::kPlane, wave + -1, lane, a_r2);
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
        ctx.g[1] = a_r0[i + 2];
        ctx.g[2] = a_r0[i + 0];
        ctx.g[3] = a_r1[i + 0];
        ctx.g[4] = a_r2[i + 0];
        ctx.g[5] = a_r3[i + 0];
        ctx.g[6] = a_r4[i + 0];
        ctx.g_e = false;
        krb(xs + i, yrow, s, ctx);
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
      ctx.g[1] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 1];
      ctx.g[2] = a_lds[sc * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + -1];
      ctx.g[3] = a_lds[sc * SA::kPlane + (hr + 1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[4] = a_lds[sc * SA::kPlane + (hr + -1) * SA::kRow + SA::kPad + px + 0];
      ctx.g[5] = a_lds[sm * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g[6] = a_lds[sp * SA::kPlane + (hr + 0) * SA::kRow + SA::kPad + px + 0];
      ctx.g_e = false;
      krb(x0 + px, y0 - 2 + hr, s, ctx);
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
      SB::template ReadRow<0, 0>(b_lds + sc * SB::kPlane, wave + 1, lane, b_r1);
      float b_r2[VX + 0];
      SB::template ReadRow<0, 0>(b_lds + sc * SB::kPlane, wave + -1, lane, b_r2);
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
        ctx.g[1] = b_r0[i + 2];
        ctx.g[2] = b_r0[i + 0];
        ctx.g[3] = b_r1[i + 0];
        ctx.g[4] = b_r2[i + 0];
        ctx.g[5] = b_r3[i + 0];
        ctx.g[6] = b_r4[i + 0];
        ctx.g_e = false;
        krb(xs + i, yrow, z, ctx);
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
static void __PSLaunch2V_krb(const struct __PSStencil_krb &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  constexpr int BY = 12;
  const __PSDomain gd = physis_hip::WholeDomain(s.g);
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun2_krb<VX, BY, false>, 64 * BY);
  const physis_hip::RunShape sh = physis_hip::PlanRun(gd, 64 * VX, BY - 4, per_cu,
      physis_hip::WindowChunkLimit({s.g}, 3), 4);
  if (sh.blocks == 0) return;
  if (s.g->dim[0] % VX == 0)
    hipLaunchKernelGGL((__PSStencilRun2_krb<VX, BY, false>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, gd, src, dst, mid, sh);
  else
    hipLaunchKernelGGL((__PSStencilRun2_krb<VX, BY, true>), dim3(sh.blocks), dim3(64 * BY), 0, stream, s.dom, gd, src, dst, mid, sh);
}

static void __PSLaunch2_krb(const struct __PSStencil_krb &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *mid, hipStream_t stream) {
  if (physis_hip::PairVX(s.g->dim, false, true) == 4)
    __PSLaunch2V_krb<4>(s, src, dst, mid, stream);
  else
    __PSLaunch2V_krb<2>(s, src, dst, mid, stream);
}

// The red-black map s0 may run as one pass per iteration: both colours, a domain
// strictly inside the grid.
static bool __PSFusableRB_krb(const struct __PSStencil_krb &s0) {
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

// Resident-tile pass of krb: TILE::T sweeps of src per launch into dst,
// the one before the last into bg when store_mid.  red: per-block partials of
// each sweep.
template <typename TILE, int RED>
__global__ __launch_bounds__(TILE::NT) void __PSStencilRunT_krb(
    __PSDomain dom, __PSDomain gd, __PSGrid3DFloat_dev src, __PSGrid3DFloat_dev dst, float *__restrict__ bg, int store_mid, int tiles_x, int tiles_y, physis_hip::TileReds red) {
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
  __PSCtx_krb ctx;
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
      ctx.g[1] = cur[p.at + 1 + RX * (0 + RY * (0))];
      ctx.g[2] = cur[p.at + -1 + RX * (0 + RY * (0))];
      ctx.g[3] = cur[p.at + 0 + RX * (1 + RY * (0))];
      ctx.g[4] = cur[p.at + 0 + RX * (-1 + RY * (0))];
      ctx.g[5] = cur[p.at + 0 + RX * (0 + RY * (-1))];
      ctx.g[6] = cur[p.at + 0 + RX * (0 + RY * (1))];
      ctx.g_e = false;
      krb(p.x, p.y, p.z, ctx);
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
static void __PSLaunchTile_krb(const struct __PSStencil_krb &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  const __PSDomain d = physis_hip::WholeDomain(s.g);
  const physis_hip::TileShape g = physis_hip::TileGrid<TILE>(d);
  if (g.blocks == 0) return;
  {
      hipLaunchKernelGGL((__PSStencilRunT_krb<TILE, -1>), dim3(g.blocks), dim3(TILE::NT), 0, stream, s.dom, d, src, dst, bg, store_mid, g.tiles_x, g.tiles_y, red);
  }
}

template <int T>
static void __PSLaunchT_krb(const struct __PSStencil_krb &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream, const physis_hip::TileReds &red) {
  if (physis_hip::InSmallTiles(physis_hip::WholeDomain(s.g)))
    __PSLaunchTile_krb<physis_hip::SmallTile<T>>(s, src, dst, bg, store_mid, stream, red);
  else
    __PSLaunchTile_krb<physis_hip::MidTile<T>>(s, src, dst, bg, store_mid, stream, red);
}

// ---------------------------------------------- stencil krbp
struct __PSStencil_krbp {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  int __rb;  // -1 all points, 0 red, 1 black, 2 red then black
};

static struct __PSStencil_krbp __PSStencilMap_krbp(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krbp __s = {__dom, g, __PSGridGetID(g), -1};
  return __s;
}

static struct __PSStencil_krbp __PSStencilMapRed_krbp(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krbp __s = __PSStencilMap_krbp(__dom, g);
  __s.__rb = 0;
  return __s;
}

static struct __PSStencil_krbp __PSStencilMapBlack_krbp(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krbp __s = __PSStencilMap_krbp(__dom, g);
  __s.__rb = 1;
  return __s;
}

static struct __PSStencil_krbp __PSStencilMapRedBlack_krbp(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_krbp __s = __PSStencilMap_krbp(__dom, g);
  __s.__rb = 2;
  return __s;
}

// Stencil analysis of krbp (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] periodic, emitted
//     offsets 0:(0,0,0)p 1:(1,0,0)p 2:(-1,0,0)p 3:(0,1,0)p 4:(0,-1,0)p 5:(0,0,-1)p 6:(0,0,1)p
//   red-black: in-place colour sweep reads only the other colour
//   two-sweep fusion of map pairs: no (a red-black map reading other grids or periodic gets)
struct __PSCtx_krbp {
  float g[7];
  float g_v;
  bool g_e;
  const float *g_p;
  int g_dim[3];
};

__device__ __forceinline__ void krbp(
    const int x, const int y, const int z, __PSCtx_krbp &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6];
  (__ctx.g_v = (v), __ctx.g_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_krbp(
    __PSDomain dom, __PSGrid3DFloat_dev g, physis_hip::RunShape sh, float *__restrict__ __red, int __rb) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, true, float, RAGGED> S_g;
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
    __PSCtx_krbp ctx;
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
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 1, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + -1, lane, g_r2);
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
              ctx.g[1] = g_r0[i + 2];
              ctx.g[2] = g_r0[i + 0];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g[5] = g_r3[i + 0];
              ctx.g[6] = g_r4[i + 0];
              ctx.g_e = false;
              krbp(x, yrow, z, ctx);
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
static physis_hip::RunShape __PSShape_krbp(const struct __PSStencil_krbp &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_krbp<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g}, 2));
}

template <int VX>
static int __PSLaunch_krbp(const struct __PSStencil_krbp &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_krbp<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  for (int __c = s.__rb == 2 ? 0 : s.__rb; __c <= (s.__rb == 2 ? 1 : s.__rb); ++__c) {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_krbp<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), sh, (float *)NULL, __c);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_krbp(const struct __PSStencil_krbp &s) {
  return (s.g->dim[0] % 4 == 0) ? __PSShape_krbp<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, true)) ? __PSShape_krbp<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_krbp<1>(s).blocks;
}

static int __PSRun_krbp(const struct __PSStencil_krbp &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  if (s.g->dim[0] % 2 || s.g->dim[1] % 2 || s.g->dim[2] % 2) {
    static bool __warned = false;
    if (!__warned) std::fprintf(stderr, "[physis-hip] warning: krbp: a periodic neighbour across an odd extent has the point's own colour; colours are updated in parallel, not in the REFERENCE order\n");
    __warned = true;
  }
  physis_hip::CheckEmitDomain(s.dom, s.g);
  return (s.g->dim[0] % 4 == 0) ? __PSLaunch_krbp<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, true, true)) ? __PSLaunch_krbp<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_krbp<1>(s, stream, red);
}

static void __PSStencilRun_10(int iter, struct __PSStencil_krb s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("krb");
  physis_hip::RunTimer timer(stream);
  int i0 = 0;
  if (iter >= 1 && __PSFusableRB_krb(s0)) {
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
        __PSLaunch2_krb(s0, src, dst, NULL, stream);
      else if (its == 2)
        __PSLaunchT_krb<4>(s0, src, dst, NULL, 0, stream, {});
      else
        __PSLaunchT_krb<2>(s0, src, dst, NULL, 0, stream, {});
      src = dst;
      i += its;
    }
    if (iter % 2) physis_hip::CopyDevice(va.p, vt.p, bytes, stream);
    i0 = iter;
    iter += last;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_krb(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_11(int iter, struct __PSStencil_krb s0, struct __PSStencil_krb s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("krb, krb");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_krb(s0, stream, NULL);
    __PSRun_krb(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_12(int iter, struct __PSStencil_krbp s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("krbp");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_krbp(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

static void run_redblack(int mode, float * out) {
  PSGrid3DFloat g = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 32, 32, 32);
  PSDomain3D d = PSDomain3DNew(1, 32 - 1, 1, 32 - 1, 1, 32 - 1);
  PSDomain3D dall = PSDomain3DNew(0, 32, 0, 32, 0, 32);
  float *indata = (float*)malloc(sizeof(float) * 32 * 32 * 32);
  int i;
  for (i = 0; i < 32 * 32 * 32; i++) 
    indata[i] = i;
  __PSGridCopyin(g, indata, NULL);
  if (mode == 0)
    __PSStencilRun_10(1, __PSStencilMapRedBlack_krb(d, g));
  if (mode == 1)
    __PSStencilRun_11(1, __PSStencilMapRed_krb(d, g), __PSStencilMapBlack_krb(d, g));
  if (mode == 2)
    __PSStencilRun_12(1, __PSStencilMapRedBlack_krbp(dall, g));
  __PSGridCopyout(g, out, NULL);
  __PSGridFree(g, NULL);
  free(indata);
}

void systest_redblack(float * out) {
  run_redblack(0, out);
}

void systest_redblack_separated(float * out) {
  run_redblack(1, out);
}

void systest_redblack_periodic(float * out) {
  run_redblack(2, out);
}

}  // extern "C"

// ---------------------------------------------- stencil k3
struct __PSStencil_k3 {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k3 __PSStencilMap_k3(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_k3 __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k3 (generic run kernel: not a 2-D or 3-D stencil):
//   g  read from memory
//   g2  not read, emitted
struct __PSCtx_k3 {
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k3(
    const int x, __PSCtx_k3 &__ctx) {
  float v = physis_hip::GetLinear<float>(__ctx.g_p, __ctx.g_dim, 1, x - 1) + physis_hip::GetLinear<float>(__ctx.g_p, __ctx.g_dim, 1, x) + physis_hip::GetLinear<float>(__ctx.g_p, __ctx.g_dim, 1, x + 1);
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Generic run kernel (one thread per (x, y) column marching z, all
// gets read from memory): not a 2-D or 3-D stencil.
template <int RED>
__global__ __launch_bounds__(256) void __PSStencilRunGeneric_k3(
    __PSDomain dom, __PSGrid1DFloat_dev g, __PSGrid1DFloat_dev g2, float *__restrict__ __red) {
  const int x = dom.local_min[0] + blockIdx.x * 256 + threadIdx.x;
  if (x < dom.local_max[0]) {
    __PSCtx_k3 ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = d < 1 ? g.dim[d] : 1;
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = d < 1 ? g2.dim[d] : 1;
    do {
      ctx.g2_e = false;
      k3(x, ctx);
      if (ctx.g2_e) g2.p[x] = ctx.g2_v;
    } while (0);
  }
  (void)__red;
}

static dim3 __PSGridDim_k3(const struct __PSStencil_k3 &s) {
  const int nx = s.dom.local_max[0] - s.dom.local_min[0];
  const int ny = 1;
  if (nx <= 0 || ny <= 0) return dim3(0, 0, 1);
  return dim3((nx + 255) / 256, 1, 1);
}

static int __PSBlocks_k3(const struct __PSStencil_k3 &s) {
  const dim3 g = __PSGridDim_k3(s);
  return g.x * g.y;
}

static int __PSRun_k3(const struct __PSStencil_k3 &s, hipStream_t stream, void *red) {
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  const dim3 grid = __PSGridDim_k3(s);
  if (grid.x == 0) return 0;
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRunGeneric_k3<-1>), grid, dim3(256), 0, stream, s.dom, physis_hip::DevView<__PSGrid1DFloat_dev>(s.g), physis_hip::DevView<__PSGrid1DFloat_dev>(s.g2), (float *)NULL);
  }
  }
  return grid.x * grid.y;
}

// ---------------------------------------------- stencil k5
struct __PSStencil_k5 {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_k5 __PSStencilMap_k5(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_k5 __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of k5 (2.5D run kernel over the rows view nx x 1 x ny of its 2-D grids, y marched as z):
//   g  staged x[-1,1] y[-0,0] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,0,-1) 4:(0,0,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_k5 {
  float g[5];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void k5(
    const int x, const int y, __PSCtx_k5 &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_k5(
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
    __PSCtx_k5 ctx;
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
          float g_r0[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 1) * S_g::kPlane, wave + 0, lane, g_r0);
          float g_r1[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r1);
          float g_r2[VX + 0];
          S_g::template ReadRow<0, 0>(g_lds + physis_hip::RingSlot<4>(g_base, 2) * S_g::kPlane, wave + 0, lane, g_r2);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 0];
              ctx.g[2] = g_r0[i + 2];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g2_e = false;
              k5(x, z, ctx);
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
static physis_hip::RunShape __PSShape_k5(const struct __PSStencil_k5 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_k5<VX, 1, -1>, 64 * 1);
  return physis_hip::PlanRun(physis_hip::RowDomain(s.dom), 64 * physis_hip::FormVX(VX), 1 - 2 * 0, per_cu, physis_hip::WindowChunkLimitRows({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_k5(const struct __PSStencil_k5 &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_k5<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 1);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_k5<VX, 1, -1>), grid, block, 0, stream, physis_hip::RowDomain(s.dom), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_k5(const struct __PSStencil_k5 &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_k5<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSShape_k5<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_k5<1>(s).blocks;
}

static int __PSRun_k5(const struct __PSStencil_k5 &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_k5<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSLaunch_k5<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_k5<1>(s, stream, red);
}

// Rows pass of k5: T sweeps of src into dst, the one before the
// last into bg when store_mid.
template <int T>
__global__ __launch_bounds__(64) void __PSStencilRunR_k5(
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
  __PSCtx_k5 ctx;
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
            ctx.g[1] = q[t - 1][(k + 2) % 3].v[1 + i + -1];
            ctx.g[2] = q[t - 1][(k + 2) % 3].v[1 + i + 1];
            ctx.g[3] = q[t - 1][(k + 1) % 3].v[1 + i + 0];
            ctx.g[4] = q[t - 1][(k + 0) % 3].v[1 + i + 0];
            ctx.g2_e = false;
            k5(xs + i, z, ctx);
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
static void __PSLaunchR_k5(const struct __PSStencil_k5 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream) {
  const __PSDomain d = physis_hip::RowDomain(s.dom);
  static int per_cu = physis_hip::BlocksPerCU((const void *)__PSStencilRunR_k5<T>, 64);
  const physis_hip::RunShape sh = physis_hip::PlanRun(d, physis_hip::kRowsTX, 1, per_cu,
      physis_hip::WindowChunkLimitRows({s.g, s.g2}, T + 1), 2 * T + 3);
  if (sh.blocks == 0) return;
  hipLaunchKernelGGL(__PSStencilRunR_k5<T>, dim3(sh.blocks), dim3(64), 0, stream, d, src, dst, bg, store_mid, sh);
}

// The pair (s0, s1) is k5(a -> b), k5(b -> a) over one domain strictly
// inside the grids, with the same scalars: it may run as rows passes.
static bool __PSFusable2_k5(const struct __PSStencil_k5 &s0, const struct __PSStencil_k5 &s1) {
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

static void __PSStencilRun_13(int iter, struct __PSStencil_k3 s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k3");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k3(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_3pt_1d(float * out) {
  int n = 1024, i;
  PSGrid1DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 1, n);
  PSGrid1DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 1, n);
  PSDomain1D d = PSDomain1DNew(1, n - 1);
  float *indata = (float*)malloc(sizeof(float) * n);
  for (i = 0; i < n; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  __PSStencilRun_13(1, __PSStencilMap_k3(d, g1, g2));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

}  // extern "C"

static void __PSStencilRun_14(int iter, struct __PSStencil_k5 s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("k5");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_k5(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_5pt_2d(float * out) {
  int i;
  PSGrid2DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 2, 32, 32);
  PSGrid2DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 2, 32, 32);
  PSDomain2D d = PSDomain2DNew(1, 32 - 1, 1, 32 - 1);
  float *indata = (float*)malloc(sizeof(float) * 32 * 32);
  for (i = 0; i < 32 * 32; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  __PSStencilRun_14(1, __PSStencilMap_k5(d, g1, g2));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

}  // extern "C"

// ---------------------------------------------- stencil kmix
struct __PSStencil_kmix {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  __PSGrid *i;
  int __i_index;
  __PSGrid *j;
  int __j_index;
};

static struct __PSStencil_kmix __PSStencilMap_kmix(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, __PSGrid *i, __PSGrid *j) {
  struct __PSStencil_kmix __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), i, __PSGridGetID(i), j, __PSGridGetID(j)};
  return __s;
}

// Stencil analysis of kmix (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,-1,0) 4:(0,1,0) 5:(0,0,-1) 6:(0,0,1)
//   g2  not read, emitted
//   i  read from memory, irregular gets
//   j  read from memory, irregular gets
//   two-sweep fusion of map pairs: no (grid i is read irregularly)
struct __PSCtx_kmix {
  float g[7];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
  const float *i_p;
  int i_dim[3];
  const float *j_p;
  int j_dim[3];
};

__device__ __forceinline__ void kmix(
    const int x, const int y, const int z, __PSCtx_kmix &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] * physis_hip::GetLinear<float>(__ctx.i_p, __ctx.i_dim, 1, x - 1) + __ctx.g[2] * physis_hip::GetLinear<float>(__ctx.i_p, __ctx.i_dim, 1, x + 1) + __ctx.g[3] * physis_hip::GetLinear<float>(__ctx.j_p, __ctx.j_dim, 2, y - 1, z) + __ctx.g[4] * physis_hip::GetLinear<float>(__ctx.j_p, __ctx.j_dim, 2, y + 1, z) + __ctx.g[5] * physis_hip::GetLinear<float>(__ctx.j_p, __ctx.j_dim, 2, y, z - 1) + __ctx.g[6] * physis_hip::GetLinear<float>(__ctx.j_p, __ctx.j_dim, 2, y, z + 1);
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kmix(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, __PSGrid1DFloat_dev i, __PSGrid2DFloat_dev j, physis_hip::RunShape sh, float *__restrict__ __red) {
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
    __PSCtx_kmix ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    ctx.i_p = i.p;
    for (int d = 0; d < 3; ++d) ctx.i_dim[d] = d < 1 ? i.dim[d] : 1;
    ctx.j_p = j.p;
    for (int d = 0; d < 3; ++d) ctx.j_dim[d] = d < 2 ? j.dim[d] : 1;
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
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 1];
              ctx.g[1] = g_r0[i + 0];
              ctx.g[2] = g_r0[i + 2];
              ctx.g[3] = g_r1[i + 0];
              ctx.g[4] = g_r2[i + 0];
              ctx.g[5] = g_r3[i + 0];
              ctx.g[6] = g_r4[i + 0];
              ctx.g2_e = false;
              kmix(x, yrow, z, ctx);
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
static physis_hip::RunShape __PSShape_kmix(const struct __PSStencil_kmix &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kmix<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_kmix(const struct __PSStencil_kmix &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kmix<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_kmix<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), physis_hip::DevView<__PSGrid1DFloat_dev>(s.i), physis_hip::DevView<__PSGrid2DFloat_dev>(s.j), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kmix(const struct __PSStencil_kmix &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kmix<4>(s).blocks
         : __PSShape_kmix<1>(s).blocks;
}

static int __PSRun_kmix(const struct __PSStencil_kmix &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckGrid3D(s.i, PS_FLOAT);
  physis_hip::CheckGrid3D(s.j, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kmix<4>(s, stream, red)
         : __PSLaunch_kmix<1>(s, stream, red);
}

static void __PSStencilRun_15(int iter, struct __PSStencil_kmix s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kmix");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kmix(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_mixed_dim3(float * out) {
  int ny = 32 + 2, i;
  size_t nelms = (size_t)32 * ny * 32;
  PSGrid3DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 32, ny, 32);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 32, ny, 32);
  PSGrid1DFloat cx = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 1, 32);
  PSGrid2DFloat cy = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 2, ny, 32);
  PSDomain3D d = PSDomain3DNew(1, 32 - 1, 1, ny - 1, 1, 32 - 1);
  float *indata = (float*)malloc(sizeof(float) * nelms);
  for (i = 0; i < (int)nelms; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  for (i = 0; i < 32; i++) 
    indata[i] = 1 + (i % 2);
  __PSGridCopyin(cx, indata, NULL);
  for (i = 0; i < ny * 32; i++) 
    indata[i] = 1 + (i % 2);
  __PSGridCopyin(cy, indata, NULL);
  __PSStencilRun_15(1, __PSStencilMap_kmix(d, g1, g2, cx, cy));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  __PSGridFree(cx, NULL);
  __PSGridFree(cy, NULL);
  free(indata);
}

}  // extern "C"

// ---------------------------------------------- stencil khole
struct __PSStencil_khole {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_khole __PSStencilMap_khole(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_khole __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of khole (2.5D run kernel):
//   g  staged x[-2,2] y[-0,0] z[0,0] non-periodic
//     offsets 0:(0,0,0) 1:(2,0,0) 2:(-2,0,0)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (halo wider than one point)
struct __PSCtx_khole {
  float g[3];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void khole(
    const int x, const int y, const int z, __PSCtx_khole &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2];
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_khole(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 0;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 2, HY, 2, false, float, RAGGED> S_g;
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
    const physis_hip::BufWin<float> g_w = physis_hip::BufWin<float>::Make(g.p, g_nxy * g.dim[2], (long)(zb + -1) * g_nxy, (long)(ze + 1) * g_nxy);
    S_g g_st[PD];
    const typename S_g::Addr g_ra = S_g::Prepare(g.dim, x0, yrow, lane);
    S_g g_pro[1];
#pragma unroll
    for (int k = 0; k < 1; ++k)
      g_pro[k].Load(g_w, g.p, g.dim, g_ra, zb + 0 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g_st[k].Load(g_w, g.p, g.dim, g_ra, zb + 1 + k);
    int g_base = 0;
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
#pragma unroll
    for (int k = 0; k < 1; ++k)
      g_pro[k].Store(g_lds + k * S_g::kPlane, wave, lane, g_ra);
    __syncthreads();
    __PSCtx_khole ctx;
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
        const int g_base = k % 2;
        if (computes && z < ze) {
          float g_r0[VX + 4];
          S_g::template ReadRow<-2, 2>(g_lds + physis_hip::RingSlot<2>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r0);
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g[0] = g_r0[i + 2];
              ctx.g[1] = g_r0[i + 4];
              ctx.g[2] = g_r0[i + 0];
              ctx.g2_e = false;
              khole(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        g_st[k % PD].Store(g_lds + physis_hip::RingSlot<2>(g_base, 1) * S_g::kPlane, wave, lane, g_ra);
        __syncthreads();
        g_st[k % PD].Load(g_w, g.p, g.dim, g_ra, z + 1 + PD);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_khole(const struct __PSStencil_khole &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_khole<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 0, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 1));
}

template <int VX>
static int __PSLaunch_khole(const struct __PSStencil_khole &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_khole<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_khole<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_khole(const struct __PSStencil_khole &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_khole<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_khole<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_khole<1>(s).blocks;
}

static int __PSRun_khole(const struct __PSStencil_khole &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_khole<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_khole<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_khole<1>(s, stream, red);
}

static void __PSStencilRun_16(int iter, struct __PSStencil_khole s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("khole");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_khole(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_stencil_hole(float * out) {
  int i;
  PSGrid3DFloat g1 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 32, 32, 32);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 32, 32, 32);
  PSDomain3D d = PSDomain3DNew(2, 32 - 2, 2, 32 - 2, 2, 32 - 2);
  float *indata = (float*)malloc(sizeof(float) * 32 * 32 * 32);
  for (i = 0; i < 32 * 32 * 32; i++) 
    indata[i] = i;
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  __PSStencilRun_16(1, __PSStencilMap_khole(d, g1, g2));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

struct Vec3 { float x; float y; float z; };

DeclareGrid3D(Vec3, struct Vec3);

}  // extern "C"

// ---------------------------------------------- point type Vec3 (struct Vec3)
// Type info of the reference's REF target (reference_runtime_builder.cc:
// 959-1065): one entry per member, scalar size, array rank and extents.
static __PSGridTypeMemberInfo __PSTypeMembers_Vec3[] = {
  {PS_FLOAT, sizeof(float), 0, {0}},
  {PS_FLOAT, sizeof(float), 0, {0}},
  {PS_FLOAT, sizeof(float), 0, {0}},
};
static __PSGridTypeInfo __PSTypeInfo_Vec3 = {PS_USER, sizeof(struct Vec3), 3, __PSTypeMembers_Vec3};

// Device view: the first component plane of each member (component c
// of an array member, row-major, c * n elements further).
struct __PSUdtView_Vec3 {
  float *m_x;
  float *m_y;
  float *m_z;
  long n;
  int dim[3];
};

static inline __PSUdtView_Vec3 __PSUdtViewOf_Vec3(__PSGrid *g) {
  __PSUdtView_Vec3 v;
  v.m_x = (float *)__PSGridUserMember(g, 0);
  v.m_y = (float *)__PSGridUserMember(g, 1);
  v.m_z = (float *)__PSGridUserMember(g, 2);
  v.n = (long)g->num_elms;
  for (int d = 0; d < 3; ++d) v.dim[d] = g->dim[d];
  return v;
}

__device__ __forceinline__ struct Vec3 __PSUdtLoad_Vec3(const __PSUdtView_Vec3 &v, long off) {
  struct Vec3 r{};
  if (off < 0) return r;
  r.x = v.m_x[off];
  r.y = v.m_y[off];
  r.z = v.m_z[off];
  return r;
}

__device__ __forceinline__ void __PSUdtStore_Vec3(const __PSUdtView_Vec3 &v, long off, const struct Vec3 &r) {
  v.m_x[off] = r.x;
  v.m_y[off] = r.y;
  v.m_z[off] = r.z;
}

__device__ __forceinline__ struct Vec3 __PSUdtMake_Vec3(float m0, float m1, float m2) {
  struct Vec3 r;
  r.x = m0;
  r.y = m1;
  r.z = m2;
  return r;
}

// ---------------------------------------------- stencil kvec3
struct __PSStencil_kvec3 {
  __PSDomain dom;
  __PSGrid *g1;
  int __g1_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_kvec3 __PSStencilMap_kvec3(
    __PSDomain __dom, __PSGrid *g1, __PSGrid *g2) {
  struct __PSStencil_kvec3 __s = {__dom, g1, __PSGridGetID(g1), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of kvec3 (2.5D run kernel):
//   g1  split into one grid per member it uses
//   g2  split into one grid per member it uses
//   g1__x  staged x[-1,1] y[-0,0] z[0,0] non-periodic
//     offsets 0:(0,0,0) 1:(1,0,0) 2:(-1,0,0)
//   g1__y  staged x[-0,0] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(0,1,0) 2:(0,-1,0) 3:(0,0,1) 4:(0,0,-1)
//   g1__z  staged x[-0,0] y[-0,0] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(0,0,1) 2:(0,0,-1)
//   g2__x  not read, emitted
//   g2__y  not read, emitted
//   g2__z  not read, emitted
//   two-sweep fusion of map pairs: no (a grid of user-defined points)
struct __PSCtx_kvec3 {
  float g1__x[3];
  const float *g1__x_p;
  int g1__x_dim[3];
  float g1__y[5];
  const float *g1__y_p;
  int g1__y_dim[3];
  float g1__z[3];
  const float *g1__z_p;
  int g1__z_dim[3];
  float g2__x_v;
  bool g2__x_e;
  const float *g2__x_p;
  int g2__x_dim[3];
  float g2__y_v;
  bool g2__y_e;
  const float *g2__y_p;
  int g2__y_dim[3];
  float g2__z_v;
  bool g2__z_e;
  const float *g2__z_p;
  int g2__z_dim[3];
};

__device__ __forceinline__ void kvec3(
    const int x, const int y, const int z, __PSCtx_kvec3 &__ctx) {
  float p = (__ctx.g1__x[0] + __ctx.g1__x[1] + __ctx.g1__x[2]) / 3.3f;
  float q = (__ctx.g1__y[0] + __ctx.g1__y[1] + __ctx.g1__y[2] + __ctx.g1__y[3] + __ctx.g1__y[4]) / 5.5f;
  float r = (__ctx.g1__z[0] + __ctx.g1__z[1] + __ctx.g1__z[2]) / 3.3f;
  struct Vec3 v = {p, q, r};
  ((__ctx.g2__x_v = ((v).x), __ctx.g2__x_e = true), (__ctx.g2__y_v = ((v).y), __ctx.g2__y_e = true), (__ctx.g2__z_v = ((v).z), __ctx.g2__z_e = true));
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kvec3(
    __PSDomain dom, __PSGrid3DFloat_dev g1__x, __PSGrid3DFloat_dev g1__y, __PSGrid3DFloat_dev g1__z, __PSGrid3DFloat_dev g2__x, __PSGrid3DFloat_dev g2__y, __PSGrid3DFloat_dev g2__z, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 2, false, float, RAGGED> S_g1__x;
  __shared__ __attribute__((aligned(16))) float g1__x_lds[S_g1__x::kLdsElems];
  typedef physis_hip::Stage<float, VX, BY, 0, HY, 4, false, float, RAGGED> S_g1__y;
  __shared__ __attribute__((aligned(16))) float g1__y_lds[S_g1__y::kLdsElems];
  typedef physis_hip::Stage<float, VX, BY, 0, HY, 4, false, float, RAGGED> S_g1__z;
  __shared__ __attribute__((aligned(16))) float g1__z_lds[S_g1__z::kLdsElems];
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
    const int g1__x_nxy = g1__x.dim[0] * g1__x.dim[1];
    const physis_hip::BufWin<float> g1__x_w = physis_hip::BufWin<float>::Make(g1__x.p, g1__x_nxy * g1__x.dim[2], (long)(zb + -1) * g1__x_nxy, (long)(ze + 1) * g1__x_nxy);
    S_g1__x g1__x_st[PD];
    const typename S_g1__x::Addr g1__x_ra = S_g1__x::Prepare(g1__x.dim, x0, yrow, lane);
    S_g1__x g1__x_pro[1];
#pragma unroll
    for (int k = 0; k < 1; ++k)
      g1__x_pro[k].Load(g1__x_w, g1__x.p, g1__x.dim, g1__x_ra, zb + 0 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g1__x_st[k].Load(g1__x_w, g1__x.p, g1__x.dim, g1__x_ra, zb + 1 + k);
    int g1__x_base = 0;
    const int g1__y_nxy = g1__y.dim[0] * g1__y.dim[1];
    const physis_hip::BufWin<float> g1__y_w = physis_hip::BufWin<float>::Make(g1__y.p, g1__y_nxy * g1__y.dim[2], (long)(zb + -2) * g1__y_nxy, (long)(ze + 2) * g1__y_nxy);
    S_g1__y g1__y_st[PD];
    const typename S_g1__y::Addr g1__y_ra = S_g1__y::Prepare(g1__y.dim, x0, yrow, lane);
    S_g1__y g1__y_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__y_pro[k].Load(g1__y_w, g1__y.p, g1__y.dim, g1__y_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g1__y_st[k].Load(g1__y_w, g1__y.p, g1__y.dim, g1__y_ra, zb + 2 + k);
    int g1__y_base = 0;
    const int g1__z_nxy = g1__z.dim[0] * g1__z.dim[1];
    const physis_hip::BufWin<float> g1__z_w = physis_hip::BufWin<float>::Make(g1__z.p, g1__z_nxy * g1__z.dim[2], (long)(zb + -2) * g1__z_nxy, (long)(ze + 2) * g1__z_nxy);
    S_g1__z g1__z_st[PD];
    const typename S_g1__z::Addr g1__z_ra = S_g1__z::Prepare(g1__z.dim, x0, yrow, lane);
    S_g1__z g1__z_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__z_pro[k].Load(g1__z_w, g1__z.p, g1__z.dim, g1__z_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g1__z_st[k].Load(g1__z_w, g1__z.p, g1__z.dim, g1__z_ra, zb + 2 + k);
    int g1__z_base = 0;
    const int g2__x_enx = g2__x.dim[0], g2__x_enxy = g2__x.dim[0] * g2__x.dim[1];
    const physis_hip::BufWin<float> g2__x_ew = physis_hip::BufWin<float>::Make(g2__x.p, g2__x_enxy * g2__x.dim[2], (long)zb * g2__x_enxy, (long)ze * g2__x_enxy);
    const int g2__y_enx = g2__y.dim[0], g2__y_enxy = g2__y.dim[0] * g2__y.dim[1];
    const physis_hip::BufWin<float> g2__y_ew = physis_hip::BufWin<float>::Make(g2__y.p, g2__y_enxy * g2__y.dim[2], (long)zb * g2__y_enxy, (long)ze * g2__y_enxy);
    const int g2__z_enx = g2__z.dim[0], g2__z_enxy = g2__z.dim[0] * g2__z.dim[1];
    const physis_hip::BufWin<float> g2__z_ew = physis_hip::BufWin<float>::Make(g2__z.p, g2__z_enxy * g2__z.dim[2], (long)zb * g2__z_enxy, (long)ze * g2__z_enxy);
#pragma unroll
    for (int k = 0; k < 1; ++k)
      g1__x_pro[k].Store(g1__x_lds + k * S_g1__x::kPlane, wave, lane, g1__x_ra);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__y_pro[k].Store(g1__y_lds + k * S_g1__y::kPlane, wave, lane, g1__y_ra);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__z_pro[k].Store(g1__z_lds + k * S_g1__z::kPlane, wave, lane, g1__z_ra);
    __syncthreads();
    __PSCtx_kvec3 ctx;
    ctx.g1__x_p = g1__x.p;
    for (int d = 0; d < 3; ++d) ctx.g1__x_dim[d] = g1__x.dim[d];
    ctx.g1__y_p = g1__y.p;
    for (int d = 0; d < 3; ++d) ctx.g1__y_dim[d] = g1__y.dim[d];
    ctx.g1__z_p = g1__z.p;
    for (int d = 0; d < 3; ++d) ctx.g1__z_dim[d] = g1__z.dim[d];
    ctx.g2__x_p = g2__x.p;
    for (int d = 0; d < 3; ++d) ctx.g2__x_dim[d] = g2__x.dim[d];
    ctx.g2__y_p = g2__y.p;
    for (int d = 0; d < 3; ++d) ctx.g2__y_dim[d] = g2__y.dim[d];
    ctx.g2__z_p = g2__z.p;
    for (int d = 0; d < 3; ++d) ctx.g2__z_dim[d] = g2__z.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g1__x_dim[0] & 3) == 0);
      __builtin_assume((ctx.g1__y_dim[0] & 3) == 0);
      __builtin_assume((ctx.g1__z_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2__x_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2__y_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2__z_dim[0] & 3) == 0);
    }
    constexpr int U = 2;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        if (computes && z < ze) {
          float g1__x_r0[VX + 2];
          S_g1__x::template ReadRow<-1, 1>(g1__x_lds + physis_hip::RingSlot<2>(g1__x_base, 0) * S_g1__x::kPlane, wave + 0, lane, g1__x_r0);
          float g1__y_r0[VX + 0];
          S_g1__y::template ReadRow<0, 0>(g1__y_lds + physis_hip::RingSlot<4>(g1__y_base, 1) * S_g1__y::kPlane, wave + 0, lane, g1__y_r0);
          float g1__y_r1[VX + 0];
          S_g1__y::template ReadRow<0, 0>(g1__y_lds + physis_hip::RingSlot<4>(g1__y_base, 1) * S_g1__y::kPlane, wave + 1, lane, g1__y_r1);
          float g1__y_r2[VX + 0];
          S_g1__y::template ReadRow<0, 0>(g1__y_lds + physis_hip::RingSlot<4>(g1__y_base, 1) * S_g1__y::kPlane, wave + -1, lane, g1__y_r2);
          float g1__y_r3[VX + 0];
          S_g1__y::template ReadRow<0, 0>(g1__y_lds + physis_hip::RingSlot<4>(g1__y_base, 2) * S_g1__y::kPlane, wave + 0, lane, g1__y_r3);
          float g1__y_r4[VX + 0];
          S_g1__y::template ReadRow<0, 0>(g1__y_lds + physis_hip::RingSlot<4>(g1__y_base, 0) * S_g1__y::kPlane, wave + 0, lane, g1__y_r4);
          float g1__z_r0[VX + 0];
          S_g1__z::template ReadRow<0, 0>(g1__z_lds + physis_hip::RingSlot<4>(g1__z_base, 1) * S_g1__z::kPlane, wave + 0, lane, g1__z_r0);
          float g1__z_r1[VX + 0];
          S_g1__z::template ReadRow<0, 0>(g1__z_lds + physis_hip::RingSlot<4>(g1__z_base, 2) * S_g1__z::kPlane, wave + 0, lane, g1__z_r1);
          float g1__z_r2[VX + 0];
          S_g1__z::template ReadRow<0, 0>(g1__z_lds + physis_hip::RingSlot<4>(g1__z_base, 0) * S_g1__z::kPlane, wave + 0, lane, g1__z_r2);
          float g2__x_out[VX];
          unsigned g2__x_mask = 0;
          float g2__y_out[VX];
          unsigned g2__y_mask = 0;
          float g2__z_out[VX];
          unsigned g2__z_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g1__x[0] = g1__x_r0[i + 1];
              ctx.g1__x[1] = g1__x_r0[i + 2];
              ctx.g1__x[2] = g1__x_r0[i + 0];
              ctx.g1__y[0] = g1__y_r0[i + 0];
              ctx.g1__y[1] = g1__y_r1[i + 0];
              ctx.g1__y[2] = g1__y_r2[i + 0];
              ctx.g1__y[3] = g1__y_r3[i + 0];
              ctx.g1__y[4] = g1__y_r4[i + 0];
              ctx.g1__z[0] = g1__z_r0[i + 0];
              ctx.g1__z[1] = g1__z_r1[i + 0];
              ctx.g1__z[2] = g1__z_r2[i + 0];
              ctx.g2__x_e = false;
              ctx.g2__y_e = false;
              ctx.g2__z_e = false;
              kvec3(x, yrow, z, ctx);
              g2__x_out[i] = ctx.g2__x_v;
              g2__x_mask |= (__in && ctx.g2__x_e) ? 1u << i : 0u;
              g2__y_out[i] = ctx.g2__y_v;
              g2__y_mask |= (__in && ctx.g2__y_e) ? 1u << i : 0u;
              g2__z_out[i] = ctx.g2__z_v;
              g2__z_mask |= (__in && ctx.g2__z_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2__x_ew, xs + yrow * g2__x_enx + z * g2__x_enxy, g2__x_out, g2__x_mask);
          physis_hip::StoreMasked<float, VX>(g2__y_ew, xs + yrow * g2__y_enx + z * g2__y_enxy, g2__y_out, g2__y_mask);
          physis_hip::StoreMasked<float, VX>(g2__z_ew, xs + yrow * g2__z_enx + z * g2__z_enxy, g2__z_out, g2__z_mask);
        }
        g1__x_st[k % PD].Store(g1__x_lds + physis_hip::RingSlot<2>(g1__x_base, 1) * S_g1__x::kPlane, wave, lane, g1__x_ra);
        g1__y_st[k % PD].Store(g1__y_lds + physis_hip::RingSlot<4>(g1__y_base, 3) * S_g1__y::kPlane, wave, lane, g1__y_ra);
        g1__z_st[k % PD].Store(g1__z_lds + physis_hip::RingSlot<4>(g1__z_base, 3) * S_g1__z::kPlane, wave, lane, g1__z_ra);
        __syncthreads();
        g1__x_st[k % PD].Load(g1__x_w, g1__x.p, g1__x.dim, g1__x_ra, z + 1 + PD);
        g1__x_base = physis_hip::RingSlot<2>(g1__x_base, 1);
        g1__y_st[k % PD].Load(g1__y_w, g1__y.p, g1__y.dim, g1__y_ra, z + 2 + PD);
        g1__y_base = physis_hip::RingSlot<4>(g1__y_base, 1);
        g1__z_st[k % PD].Load(g1__z_w, g1__z.p, g1__z.dim, g1__z_ra, z + 2 + PD);
        g1__z_base = physis_hip::RingSlot<4>(g1__z_base, 1);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_kvec3(const struct __PSStencil_kvec3 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kvec3<VX, 4, -1>, 64 * 4);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 4 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g1, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_kvec3(const struct __PSStencil_kvec3 &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kvec3<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 4);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_kvec3<VX, 4, -1>), grid, block, 0, stream, s.dom, physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g1, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g1, 1, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g1, 2, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g2, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g2, 1, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g2, 2, 0), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kvec3(const struct __PSStencil_kvec3 &s) {
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kvec3<4>(s).blocks
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_kvec3<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_kvec3<1>(s).blocks;
}

static int __PSRun_kvec3(const struct __PSStencil_kvec3 &s, hipStream_t stream, void *red) {
  physis_hip::CheckUserGrid3D(s.g1);
  physis_hip::CheckUserGrid3D(s.g2);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kvec3<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_kvec3<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_kvec3<1>(s, stream, red);
}

static void __PSStencilRun_17(int iter, struct __PSStencil_kvec3 s0, struct __PSStencil_kvec3 s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kvec3, kvec3");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kvec3(s0, stream, NULL);
    __PSRun_kvec3(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_udt_vec3(struct Vec3 * out) {
  size_t nelms = (size_t)32 * 32 * 32, i;
  PSGrid3DVec3 g1 = physis_hip::NewUserGrid(&__PSTypeInfo_Vec3, 3, 32, 32, 32);
  PSGrid3DVec3 g2 = physis_hip::NewUserGrid(&__PSTypeInfo_Vec3, 3, 32, 32, 32);
  PSDomain3D d = PSDomain3DNew(1, 32 - 1, 1, 32 - 1, 1, 32 - 1);
  struct Vec3 *indata = (struct Vec3*)malloc(sizeof(struct Vec3) * nelms);
  for (i = 0; i < nelms; i++) {
    indata[i].x = i;
    indata[i].y = i + 1;
    indata[i].z = i + 2;
  }
  __PSGridCopyin(g1, indata, NULL);
  __PSGridCopyin(g2, indata, NULL);
  __PSStencilRun_17(5, __PSStencilMap_kvec3(d, g1, g2), __PSStencilMap_kvec3(d, g2, g1));
  __PSGridCopyout(g1, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

struct Tensor { float p[3][2]; };

DeclareGrid3D(Tensor, struct Tensor);

}  // extern "C"

// ---------------------------------------------- point type Tensor (struct Tensor)
// Type info of the reference's REF target (reference_runtime_builder.cc:
// 959-1065): one entry per member, scalar size, array rank and extents.
static __PSGridTypeMemberInfo __PSTypeMembers_Tensor[] = {
  {PS_FLOAT, sizeof(float), 2, {3, 2}},
};
static __PSGridTypeInfo __PSTypeInfo_Tensor = {PS_USER, sizeof(struct Tensor), 1, __PSTypeMembers_Tensor};

// Device view: the first component plane of each member (component c
// of an array member, row-major, c * n elements further).
struct __PSUdtView_Tensor {
  float *m_p;
  long n;
  int dim[3];
};

static inline __PSUdtView_Tensor __PSUdtViewOf_Tensor(__PSGrid *g) {
  __PSUdtView_Tensor v;
  v.m_p = (float *)__PSGridUserMember(g, 0);
  v.n = (long)g->num_elms;
  for (int d = 0; d < 3; ++d) v.dim[d] = g->dim[d];
  return v;
}

__device__ __forceinline__ struct Tensor __PSUdtLoad_Tensor(const __PSUdtView_Tensor &v, long off) {
  struct Tensor r{};
  if (off < 0) return r;
  for (int c = 0; c < 6; ++c) (&r.p[0][0])[c] = v.m_p[c * v.n + off];
  return r;
}

__device__ __forceinline__ void __PSUdtStore_Tensor(const __PSUdtView_Tensor &v, long off, const struct Tensor &r) {
  for (int c = 0; c < 6; ++c) v.m_p[c * v.n + off] = (&r.p[0][0])[c];
}

// ---------------------------------------------- stencil ktensor
struct __PSStencil_ktensor {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
};

static struct __PSStencil_ktensor __PSStencilMap_ktensor(
    __PSDomain __dom, __PSGrid *g) {
  struct __PSStencil_ktensor __s = {__dom, g, __PSGridGetID(g)};
  return __s;
}

// Stencil analysis of ktensor (2.5D run kernel):
//   g  split into one grid per member it uses
//   g__p_0_0  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,-1,0) 4:(0,1,0) 5:(0,0,-1) 6:(0,0,1)
//   g__p_2_1  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,-1,0) 4:(0,1,0) 5:(0,0,-1) 6:(0,0,1)
//   g__p_1_0  not read, emitted
//   two-sweep fusion of map pairs: no (a grid of user-defined points)
struct __PSCtx_ktensor {
  float g__p_0_0[7];
  const float *g__p_0_0_p;
  int g__p_0_0_dim[3];
  float g__p_2_1[7];
  const float *g__p_2_1_p;
  int g__p_2_1_dim[3];
  float g__p_1_0_v;
  bool g__p_1_0_e;
  const float *g__p_1_0_p;
  int g__p_1_0_dim[3];
};

__device__ __forceinline__ void ktensor(
    const int x, const int y, const int z, __PSCtx_ktensor &__ctx) {
  float v1 = __ctx.g__p_0_0[0] + __ctx.g__p_0_0[1] + __ctx.g__p_0_0[2] + __ctx.g__p_0_0[3] + __ctx.g__p_0_0[4] + __ctx.g__p_0_0[5] + __ctx.g__p_0_0[6];
  float v2 = __ctx.g__p_2_1[0] + __ctx.g__p_2_1[1] + __ctx.g__p_2_1[2] + __ctx.g__p_2_1[3] + __ctx.g__p_2_1[4] + __ctx.g__p_2_1[5] + __ctx.g__p_2_1[6];
  (__ctx.g__p_1_0_v = (v1 + v2), __ctx.g__p_1_0_e = true);
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_ktensor(
    __PSDomain dom, __PSGrid3DFloat_dev g__p_0_0, __PSGrid3DFloat_dev g__p_2_1, __PSGrid3DFloat_dev g__p_1_0, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, false, float, RAGGED> S_g__p_0_0;
  __shared__ __attribute__((aligned(16))) float g__p_0_0_lds[S_g__p_0_0::kLdsElems];
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, false, float, RAGGED> S_g__p_2_1;
  __shared__ __attribute__((aligned(16))) float g__p_2_1_lds[S_g__p_2_1::kLdsElems];
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
    const int g__p_0_0_nxy = g__p_0_0.dim[0] * g__p_0_0.dim[1];
    const physis_hip::BufWin<float> g__p_0_0_w = physis_hip::BufWin<float>::Make(g__p_0_0.p, g__p_0_0_nxy * g__p_0_0.dim[2], (long)(zb + -2) * g__p_0_0_nxy, (long)(ze + 2) * g__p_0_0_nxy);
    S_g__p_0_0 g__p_0_0_st[PD];
    const typename S_g__p_0_0::Addr g__p_0_0_ra = S_g__p_0_0::Prepare(g__p_0_0.dim, x0, yrow, lane);
    S_g__p_0_0 g__p_0_0_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_0_0_pro[k].Load(g__p_0_0_w, g__p_0_0.p, g__p_0_0.dim, g__p_0_0_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g__p_0_0_st[k].Load(g__p_0_0_w, g__p_0_0.p, g__p_0_0.dim, g__p_0_0_ra, zb + 2 + k);
    int g__p_0_0_base = 0;
    const int g__p_2_1_nxy = g__p_2_1.dim[0] * g__p_2_1.dim[1];
    const physis_hip::BufWin<float> g__p_2_1_w = physis_hip::BufWin<float>::Make(g__p_2_1.p, g__p_2_1_nxy * g__p_2_1.dim[2], (long)(zb + -2) * g__p_2_1_nxy, (long)(ze + 2) * g__p_2_1_nxy);
    S_g__p_2_1 g__p_2_1_st[PD];
    const typename S_g__p_2_1::Addr g__p_2_1_ra = S_g__p_2_1::Prepare(g__p_2_1.dim, x0, yrow, lane);
    S_g__p_2_1 g__p_2_1_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_2_1_pro[k].Load(g__p_2_1_w, g__p_2_1.p, g__p_2_1.dim, g__p_2_1_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g__p_2_1_st[k].Load(g__p_2_1_w, g__p_2_1.p, g__p_2_1.dim, g__p_2_1_ra, zb + 2 + k);
    int g__p_2_1_base = 0;
    const int g__p_1_0_enx = g__p_1_0.dim[0], g__p_1_0_enxy = g__p_1_0.dim[0] * g__p_1_0.dim[1];
    const physis_hip::BufWin<float> g__p_1_0_ew = physis_hip::BufWin<float>::Make(g__p_1_0.p, g__p_1_0_enxy * g__p_1_0.dim[2], (long)zb * g__p_1_0_enxy, (long)ze * g__p_1_0_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_0_0_pro[k].Store(g__p_0_0_lds + k * S_g__p_0_0::kPlane, wave, lane, g__p_0_0_ra);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g__p_2_1_pro[k].Store(g__p_2_1_lds + k * S_g__p_2_1::kPlane, wave, lane, g__p_2_1_ra);
    __syncthreads();
    __PSCtx_ktensor ctx;
    ctx.g__p_0_0_p = g__p_0_0.p;
    for (int d = 0; d < 3; ++d) ctx.g__p_0_0_dim[d] = g__p_0_0.dim[d];
    ctx.g__p_2_1_p = g__p_2_1.p;
    for (int d = 0; d < 3; ++d) ctx.g__p_2_1_dim[d] = g__p_2_1.dim[d];
    ctx.g__p_1_0_p = g__p_1_0.p;
    for (int d = 0; d < 3; ++d) ctx.g__p_1_0_dim[d] = g__p_1_0.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g__p_0_0_dim[0] & 3) == 0);
      __builtin_assume((ctx.g__p_2_1_dim[0] & 3) == 0);
      __builtin_assume((ctx.g__p_1_0_dim[0] & 3) == 0);
    }
    constexpr int U = 2;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        if (computes && z < ze) {
          float g__p_0_0_r0[VX + 2];
          S_g__p_0_0::template ReadRow<-1, 1>(g__p_0_0_lds + physis_hip::RingSlot<4>(g__p_0_0_base, 1) * S_g__p_0_0::kPlane, wave + 0, lane, g__p_0_0_r0);
          float g__p_0_0_r1[VX + 0];
          S_g__p_0_0::template ReadRow<0, 0>(g__p_0_0_lds + physis_hip::RingSlot<4>(g__p_0_0_base, 1) * S_g__p_0_0::kPlane, wave + -1, lane, g__p_0_0_r1);
          float g__p_0_0_r2[VX + 0];
          S_g__p_0_0::template ReadRow<0, 0>(g__p_0_0_lds + physis_hip::RingSlot<4>(g__p_0_0_base, 1) * S_g__p_0_0::kPlane, wave + 1, lane, g__p_0_0_r2);
          float g__p_0_0_r3[VX + 0];
          S_g__p_0_0::template ReadRow<0, 0>(g__p_0_0_lds + physis_hip::RingSlot<4>(g__p_0_0_base, 0) * S_g__p_0_0::kPlane, wave + 0, lane, g__p_0_0_r3);
          float g__p_0_0_r4[VX + 0];
          S_g__p_0_0::template ReadRow<0, 0>(g__p_0_0_lds + physis_hip::RingSlot<4>(g__p_0_0_base, 2) * S_g__p_0_0::kPlane, wave + 0, lane, g__p_0_0_r4);
          float g__p_2_1_r0[VX + 2];
          S_g__p_2_1::template ReadRow<-1, 1>(g__p_2_1_lds + physis_hip::RingSlot<4>(g__p_2_1_base, 1) * S_g__p_2_1::kPlane, wave + 0, lane, g__p_2_1_r0);
          float g__p_2_1_r1[VX + 0];
          S_g__p_2_1::template ReadRow<0, 0>(g__p_2_1_lds + physis_hip::RingSlot<4>(g__p_2_1_base, 1) * S_g__p_2_1::kPlane, wave + -1, lane, g__p_2_1_r1);
          float g__p_2_1_r2[VX + 0];
          S_g__p_2_1::template ReadRow<0, 0>(g__p_2_1_lds + physis_hip::RingSlot<4>(g__p_2_1_base, 1) * S_g__p_2_1::kPlane, wave + 1, lane, g__p_2_1_r2);
          float g__p_2_1_r3[VX + 0];
          S_g__p_2_1::template ReadRow<0, 0>(g__p_2_1_lds + physis_hip::RingSlot<4>(g__p_2_1_base, 0) * S_g__p_2_1::kPlane, wave + 0, lane, g__p_2_1_r3);
          float g__p_2_1_r4[VX + 0];
          S_g__p_2_1::template ReadRow<0, 0>(g__p_2_1_lds + physis_hip::RingSlot<4>(g__p_2_1_base, 2) * S_g__p_2_1::kPlane, wave + 0, lane, g__p_2_1_r4);
          float g__p_1_0_out[VX];
          unsigned g__p_1_0_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g__p_0_0[0] = g__p_0_0_r0[i + 1];
              ctx.g__p_0_0[1] = g__p_0_0_r0[i + 0];
              ctx.g__p_0_0[2] = g__p_0_0_r0[i + 2];
              ctx.g__p_0_0[3] = g__p_0_0_r1[i + 0];
              ctx.g__p_0_0[4] = g__p_0_0_r2[i + 0];
              ctx.g__p_0_0[5] = g__p_0_0_r3[i + 0];
              ctx.g__p_0_0[6] = g__p_0_0_r4[i + 0];
              ctx.g__p_2_1[0] = g__p_2_1_r0[i + 1];
              ctx.g__p_2_1[1] = g__p_2_1_r0[i + 0];
              ctx.g__p_2_1[2] = g__p_2_1_r0[i + 2];
              ctx.g__p_2_1[3] = g__p_2_1_r1[i + 0];
              ctx.g__p_2_1[4] = g__p_2_1_r2[i + 0];
              ctx.g__p_2_1[5] = g__p_2_1_r3[i + 0];
              ctx.g__p_2_1[6] = g__p_2_1_r4[i + 0];
              ctx.g__p_1_0_e = false;
              ktensor(x, yrow, z, ctx);
              g__p_1_0_out[i] = ctx.g__p_1_0_v;
              g__p_1_0_mask |= (__in && ctx.g__p_1_0_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g__p_1_0_ew, xs + yrow * g__p_1_0_enx + z * g__p_1_0_enxy, g__p_1_0_out, g__p_1_0_mask);
        }
        g__p_0_0_st[k % PD].Store(g__p_0_0_lds + physis_hip::RingSlot<4>(g__p_0_0_base, 3) * S_g__p_0_0::kPlane, wave, lane, g__p_0_0_ra);
        g__p_2_1_st[k % PD].Store(g__p_2_1_lds + physis_hip::RingSlot<4>(g__p_2_1_base, 3) * S_g__p_2_1::kPlane, wave, lane, g__p_2_1_ra);
        __syncthreads();
        g__p_0_0_st[k % PD].Load(g__p_0_0_w, g__p_0_0.p, g__p_0_0.dim, g__p_0_0_ra, z + 2 + PD);
        g__p_0_0_base = physis_hip::RingSlot<4>(g__p_0_0_base, 1);
        g__p_2_1_st[k % PD].Load(g__p_2_1_w, g__p_2_1.p, g__p_2_1.dim, g__p_2_1_ra, z + 2 + PD);
        g__p_2_1_base = physis_hip::RingSlot<4>(g__p_2_1_base, 1);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_ktensor(const struct __PSStencil_ktensor &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_ktensor<VX, 8, -1>, 64 * 8);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 8 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g}, 2));
}

template <int VX>
static int __PSLaunch_ktensor(const struct __PSStencil_ktensor &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_ktensor<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 8);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_ktensor<VX, 8, -1>), grid, block, 0, stream, s.dom, physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g, 0, 5), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g, 0, 2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_ktensor(const struct __PSStencil_ktensor &s) {
  return (s.g->dim[0] % 4 == 0) ? __PSShape_ktensor<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_ktensor<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_ktensor<1>(s).blocks;
}

static int __PSRun_ktensor(const struct __PSStencil_ktensor &s, hipStream_t stream, void *red) {
  physis_hip::CheckUserGrid3D(s.g);
  physis_hip::CheckEmitDomain(s.dom, s.g);
  return (s.g->dim[0] % 4 == 0) ? __PSLaunch_ktensor<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_ktensor<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_ktensor<1>(s, stream, red);
}

static void __PSStencilRun_18(int iter, struct __PSStencil_ktensor s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("ktensor");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_ktensor(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_udt_tensor(struct Tensor * out) {
  int nelms = 32 * 32 * 32, i, j, k;
  PSGrid3DTensor g = physis_hip::NewUserGrid(&__PSTypeInfo_Tensor, 3, 32, 32, 32);
  PSDomain3D d = PSDomain3DNew(1, 32 - 1, 1, 32 - 1, 1, 32 - 1);
  struct Tensor *indata = (struct Tensor*)malloc(sizeof(struct Tensor) * nelms);
  for (i = 0; i < nelms; i++) 
    for (j = 0; j < 3; ++j) 
      for (k = 0; k < 2; ++k) 
        indata[i].p[j][k] = i + j + k;
  __PSGridCopyin(g, indata, NULL);
  __PSStencilRun_18(1, __PSStencilMap_ktensor(d, g));
  __PSGridCopyout(g, out, NULL);
  __PSGridFree(g, NULL);
  free(indata);
}

struct Cplx { float r; float i; };

DeclareGrid3D(Cplx, struct Cplx);

}  // extern "C"

// ---------------------------------------------- point type Cplx (struct Cplx)
// Type info of the reference's REF target (reference_runtime_builder.cc:
// 959-1065): one entry per member, scalar size, array rank and extents.
static __PSGridTypeMemberInfo __PSTypeMembers_Cplx[] = {
  {PS_FLOAT, sizeof(float), 0, {0}},
  {PS_FLOAT, sizeof(float), 0, {0}},
};
static __PSGridTypeInfo __PSTypeInfo_Cplx = {PS_USER, sizeof(struct Cplx), 2, __PSTypeMembers_Cplx};

// Device view: the first component plane of each member (component c
// of an array member, row-major, c * n elements further).
struct __PSUdtView_Cplx {
  float *m_r;
  float *m_i;
  long n;
  int dim[3];
};

static inline __PSUdtView_Cplx __PSUdtViewOf_Cplx(__PSGrid *g) {
  __PSUdtView_Cplx v;
  v.m_r = (float *)__PSGridUserMember(g, 0);
  v.m_i = (float *)__PSGridUserMember(g, 1);
  v.n = (long)g->num_elms;
  for (int d = 0; d < 3; ++d) v.dim[d] = g->dim[d];
  return v;
}

__device__ __forceinline__ struct Cplx __PSUdtLoad_Cplx(const __PSUdtView_Cplx &v, long off) {
  struct Cplx r{};
  if (off < 0) return r;
  r.r = v.m_r[off];
  r.i = v.m_i[off];
  return r;
}

__device__ __forceinline__ void __PSUdtStore_Cplx(const __PSUdtView_Cplx &v, long off, const struct Cplx &r) {
  v.m_r[off] = r.r;
  v.m_i[off] = r.i;
}

__device__ __forceinline__ struct Cplx __PSUdtMake_Cplx(float m0, float m1) {
  struct Cplx r;
  r.r = m0;
  r.i = m1;
  return r;
}

// ---------------------------------------------- stencil kcplx
struct __PSStencil_kcplx {
  __PSDomain dom;
  __PSGrid *g1;
  int __g1_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_kcplx __PSStencilMap_kcplx(
    __PSDomain __dom, __PSGrid *g1, __PSGrid *g2) {
  struct __PSStencil_kcplx __s = {__dom, g1, __PSGridGetID(g1), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of kcplx (2.5D run kernel):
//   g1  split into one grid per member it uses
//   g2  split into one grid per member it uses
//   g1__r  staged x[-1,1] y[-1,1] z[-1,1] periodic
//     offsets 0:(0,0,0)p 1:(1,0,0)p 2:(-1,0,0)p 3:(0,1,0)p 4:(0,-1,0)p 5:(0,0,1)p 6:(0,0,-1)p
//   g1__i  staged x[-1,1] y[-1,1] z[-1,1] periodic
//     offsets 0:(0,0,0)p 1:(1,0,0)p 2:(-1,0,0)p 3:(0,1,0)p 4:(0,-1,0)p 5:(0,0,1)p 6:(0,0,-1)p
//   g2__r  not read, emitted
//   g2__i  not read, emitted
//   two-sweep fusion of map pairs: no (a grid of user-defined points)
struct __PSCtx_kcplx {
  float g1__r[7];
  const float *g1__r_p;
  int g1__r_dim[3];
  float g1__i[7];
  const float *g1__i_p;
  int g1__i_dim[3];
  float g2__r_v;
  bool g2__r_e;
  const float *g2__r_p;
  int g2__r_dim[3];
  float g2__i_v;
  bool g2__i_e;
  const float *g2__i_p;
  int g2__i_dim[3];
};

__device__ __forceinline__ void kcplx(
    const int x, const int y, const int z, __PSCtx_kcplx &__ctx) {
  struct Cplx t = __PSUdtMake_Cplx(__ctx.g1__r[0], __ctx.g1__i[0]);
  struct Cplx t1 = __PSUdtMake_Cplx(__ctx.g1__r[1], __ctx.g1__i[1]);
  struct Cplx t2 = __PSUdtMake_Cplx(__ctx.g1__r[2], __ctx.g1__i[2]);
  struct Cplx t3 = __PSUdtMake_Cplx(__ctx.g1__r[3], __ctx.g1__i[3]);
  struct Cplx t4 = __PSUdtMake_Cplx(__ctx.g1__r[4], __ctx.g1__i[4]);
  struct Cplx t5 = __PSUdtMake_Cplx(__ctx.g1__r[5], __ctx.g1__i[5]);
  struct Cplx t6 = __PSUdtMake_Cplx(__ctx.g1__r[6], __ctx.g1__i[6]);
  float r = t.r + t1.r + t2.r + t3.r + t4.r + t5.r + t6.r;
  float i = t.i + t1.i + t2.i + t3.i + t4.i + t5.i + t6.i;
  struct Cplx v = {r, i};
  ((__ctx.g2__r_v = ((v).r), __ctx.g2__r_e = true), (__ctx.g2__i_v = ((v).i), __ctx.g2__i_e = true));
  return;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kcplx(
    __PSDomain dom, __PSGrid3DFloat_dev g1__r, __PSGrid3DFloat_dev g1__i, __PSGrid3DFloat_dev g2__r, __PSGrid3DFloat_dev g2__i, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 2;
  constexpr int HY = 1;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, true, float, RAGGED> S_g1__r;
  __shared__ __attribute__((aligned(16))) float g1__r_lds[S_g1__r::kLdsElems];
  typedef physis_hip::Stage<float, VX, BY, 1, HY, 4, true, float, RAGGED> S_g1__i;
  __shared__ __attribute__((aligned(16))) float g1__i_lds[S_g1__i::kLdsElems];
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
    const int g1__r_nxy = g1__r.dim[0] * g1__r.dim[1];
    const physis_hip::BufWin<float> g1__r_w = physis_hip::BufWin<float>::Make(g1__r.p, g1__r_nxy * g1__r.dim[2], (long)(zb + -2) * g1__r_nxy, (long)(ze + 2) * g1__r_nxy);
    S_g1__r g1__r_st[PD];
    const typename S_g1__r::Addr g1__r_ra = S_g1__r::Prepare(g1__r.dim, x0, yrow, lane);
    S_g1__r g1__r_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__r_pro[k].Load(g1__r_w, g1__r.p, g1__r.dim, g1__r_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g1__r_st[k].Load(g1__r_w, g1__r.p, g1__r.dim, g1__r_ra, zb + 2 + k);
    int g1__r_base = 0;
    const int g1__i_nxy = g1__i.dim[0] * g1__i.dim[1];
    const physis_hip::BufWin<float> g1__i_w = physis_hip::BufWin<float>::Make(g1__i.p, g1__i_nxy * g1__i.dim[2], (long)(zb + -2) * g1__i_nxy, (long)(ze + 2) * g1__i_nxy);
    S_g1__i g1__i_st[PD];
    const typename S_g1__i::Addr g1__i_ra = S_g1__i::Prepare(g1__i.dim, x0, yrow, lane);
    S_g1__i g1__i_pro[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__i_pro[k].Load(g1__i_w, g1__i.p, g1__i.dim, g1__i_ra, zb + -1 + k);
#pragma unroll
    for (int k = 0; k < PD; ++k)
      g1__i_st[k].Load(g1__i_w, g1__i.p, g1__i.dim, g1__i_ra, zb + 2 + k);
    int g1__i_base = 0;
    const int g2__r_enx = g2__r.dim[0], g2__r_enxy = g2__r.dim[0] * g2__r.dim[1];
    const physis_hip::BufWin<float> g2__r_ew = physis_hip::BufWin<float>::Make(g2__r.p, g2__r_enxy * g2__r.dim[2], (long)zb * g2__r_enxy, (long)ze * g2__r_enxy);
    const int g2__i_enx = g2__i.dim[0], g2__i_enxy = g2__i.dim[0] * g2__i.dim[1];
    const physis_hip::BufWin<float> g2__i_ew = physis_hip::BufWin<float>::Make(g2__i.p, g2__i_enxy * g2__i.dim[2], (long)zb * g2__i_enxy, (long)ze * g2__i_enxy);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__r_pro[k].Store(g1__r_lds + k * S_g1__r::kPlane, wave, lane, g1__r_ra);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      g1__i_pro[k].Store(g1__i_lds + k * S_g1__i::kPlane, wave, lane, g1__i_ra);
    __syncthreads();
    __PSCtx_kcplx ctx;
    ctx.g1__r_p = g1__r.p;
    for (int d = 0; d < 3; ++d) ctx.g1__r_dim[d] = g1__r.dim[d];
    ctx.g1__i_p = g1__i.p;
    for (int d = 0; d < 3; ++d) ctx.g1__i_dim[d] = g1__i.dim[d];
    ctx.g2__r_p = g2__r.p;
    for (int d = 0; d < 3; ++d) ctx.g2__r_dim[d] = g2__r.dim[d];
    ctx.g2__i_p = g2__i.p;
    for (int d = 0; d < 3; ++d) ctx.g2__i_dim[d] = g2__i.dim[d];
    if constexpr (VX > 1) __builtin_assume((xs & (VX - 1)) == 0);
    if constexpr (VX > 1 && !RAGGED) {
      __builtin_assume((ctx.g1__r_dim[0] & 3) == 0);
      __builtin_assume((ctx.g1__i_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2__r_dim[0] & 3) == 0);
      __builtin_assume((ctx.g2__i_dim[0] & 3) == 0);
    }
    constexpr int U = 2;
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        if (computes && z < ze) {
          float g1__r_r0[VX + 2];
          S_g1__r::template ReadRow<-1, 1>(g1__r_lds + physis_hip::RingSlot<4>(g1__r_base, 1) * S_g1__r::kPlane, wave + 0, lane, g1__r_r0);
          float g1__r_r1[VX + 0];
          S_g1__r::template ReadRow<0, 0>(g1__r_lds + physis_hip::RingSlot<4>(g1__r_base, 1) * S_g1__r::kPlane, wave + 1, lane, g1__r_r1);
          float g1__r_r2[VX + 0];
          S_g1__r::template ReadRow<0, 0>(g1__r_lds + physis_hip::RingSlot<4>(g1__r_base, 1) * S_g1__r::kPlane, wave + -1, lane, g1__r_r2);
          float g1__r_r3[VX + 0];
          S_g1__r::template ReadRow<0, 0>(g1__r_lds + physis_hip::RingSlot<4>(g1__r_base, 2) * S_g1__r::kPlane, wave + 0, lane, g1__r_r3);
          float g1__r_r4[VX + 0];
          S_g1__r::template ReadRow<0, 0>(g1__r_lds + physis_hip::RingSlot<4>(g1__r_base, 0) * S_g1__r::kPlane, wave + 0, lane, g1__r_r4);
          float g1__i_r0[VX + 2];
          S_g1__i::template ReadRow<-1, 1>(g1__i_lds + physis_hip::RingSlot<4>(g1__i_base, 1) * S_g1__i::kPlane, wave + 0, lane, g1__i_r0);
          float g1__i_r1[VX + 0];
          S_g1__i::template ReadRow<0, 0>(g1__i_lds + physis_hip::RingSlot<4>(g1__i_base, 1) * S_g1__i::kPlane, wave + 1, lane, g1__i_r1);
          float g1__i_r2[VX + 0];
          S_g1__i::template ReadRow<0, 0>(g1__i_lds + physis_hip::RingSlot<4>(g1__i_base, 1) * S_g1__i::kPlane, wave + -1, lane, g1__i_r2);
          float g1__i_r3[VX + 0];
          S_g1__i::template ReadRow<0, 0>(g1__i_lds + physis_hip::RingSlot<4>(g1__i_base, 2) * S_g1__i::kPlane, wave + 0, lane, g1__i_r3);
          float g1__i_r4[VX + 0];
          S_g1__i::template ReadRow<0, 0>(g1__i_lds + physis_hip::RingSlot<4>(g1__i_base, 0) * S_g1__i::kPlane, wave + 0, lane, g1__i_r4);
          float g2__r_out[VX];
          unsigned g2__r_mask = 0;
          float g2__i_out[VX];
          unsigned g2__i_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g1__r[0] = g1__r_r0[i + 1];
              ctx.g1__r[1] = g1__r_r0[i + 2];
              ctx.g1__r[2] = g1__r_r0[i + 0];
              ctx.g1__r[3] = g1__r_r1[i + 0];
              ctx.g1__r[4] = g1__r_r2[i + 0];
              ctx.g1__r[5] = g1__r_r3[i + 0];
              ctx.g1__r[6] = g1__r_r4[i + 0];
              ctx.g1__i[0] = g1__i_r0[i + 1];
              ctx.g1__i[1] = g1__i_r0[i + 2];
              ctx.g1__i[2] = g1__i_r0[i + 0];
              ctx.g1__i[3] = g1__i_r1[i + 0];
              ctx.g1__i[4] = g1__i_r2[i + 0];
              ctx.g1__i[5] = g1__i_r3[i + 0];
              ctx.g1__i[6] = g1__i_r4[i + 0];
              ctx.g2__r_e = false;
              ctx.g2__i_e = false;
              kcplx(x, yrow, z, ctx);
              g2__r_out[i] = ctx.g2__r_v;
              g2__r_mask |= (__in && ctx.g2__r_e) ? 1u << i : 0u;
              g2__i_out[i] = ctx.g2__i_v;
              g2__i_mask |= (__in && ctx.g2__i_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2__r_ew, xs + yrow * g2__r_enx + z * g2__r_enxy, g2__r_out, g2__r_mask);
          physis_hip::StoreMasked<float, VX>(g2__i_ew, xs + yrow * g2__i_enx + z * g2__i_enxy, g2__i_out, g2__i_mask);
        }
        g1__r_st[k % PD].Store(g1__r_lds + physis_hip::RingSlot<4>(g1__r_base, 3) * S_g1__r::kPlane, wave, lane, g1__r_ra);
        g1__i_st[k % PD].Store(g1__i_lds + physis_hip::RingSlot<4>(g1__i_base, 3) * S_g1__i::kPlane, wave, lane, g1__i_ra);
        __syncthreads();
        g1__r_st[k % PD].Load(g1__r_w, g1__r.p, g1__r.dim, g1__r_ra, z + 2 + PD);
        g1__r_base = physis_hip::RingSlot<4>(g1__r_base, 1);
        g1__i_st[k % PD].Load(g1__i_w, g1__i.p, g1__i.dim, g1__i_ra, z + 2 + PD);
        g1__i_base = physis_hip::RingSlot<4>(g1__i_base, 1);
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_kcplx(const struct __PSStencil_kcplx &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kcplx<VX, 8, -1>, 64 * 8);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 8 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g1, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_kcplx(const struct __PSStencil_kcplx &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kcplx<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 8);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_kcplx<VX, 8, -1>), grid, block, 0, stream, s.dom, physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g1, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g1, 1, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g2, 0, 0), physis_hip::MemberView<__PSGrid3DFloat_dev>(s.g2, 1, 0), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kcplx(const struct __PSStencil_kcplx &s) {
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kcplx<4>(s).blocks
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSShape_kcplx<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_kcplx<1>(s).blocks;
}

static int __PSRun_kcplx(const struct __PSStencil_kcplx &s, hipStream_t stream, void *red) {
  physis_hip::CheckUserGrid3D(s.g1);
  physis_hip::CheckUserGrid3D(s.g2);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g1->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kcplx<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g1->dim[0] && !physis_hip::OnePointRows(s.dom, true, false)) ? __PSLaunch_kcplx<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_kcplx<1>(s, stream, red);
}

static void __PSStencilRun_19(int iter, struct __PSStencil_kcplx s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kcplx");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kcplx(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_udt_complex(struct Cplx * out) {
  size_t nelms = (size_t)32 * 32 * 32, i;
  PSGrid3DCplx g1 = physis_hip::NewUserGrid(&__PSTypeInfo_Cplx, 3, 32, 32, 32);
  PSGrid3DCplx g2 = physis_hip::NewUserGrid(&__PSTypeInfo_Cplx, 3, 32, 32, 32);
  PSDomain3D d = PSDomain3DNew(0, 32, 0, 32, 0, 32);
  struct Cplx *indata = (struct Cplx*)malloc(sizeof(struct Cplx) * nelms);
  for (i = 0; i < nelms; i++) {
    indata[i].r = i;
    indata[i].i = i + 1;
  }
  __PSGridCopyin(g1, indata, NULL);
  __PSStencilRun_19(1, __PSStencilMap_kcplx(d, g1, g2));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g1, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

}  // extern "C"

// ---------------------------------------------- stencil kdouble
struct __PSStencil_kdouble {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_kdouble __PSStencilMap_kdouble(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_kdouble __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of kdouble (2.5D run kernel):
//   g  direct (centre only)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (not one read grid and one emitted grid)
struct __PSCtx_kdouble {
  float g_c;
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void kdouble(
    const int x, const int y, const int z, __PSCtx_kdouble &__ctx) {
  (__ctx.g2_v = (__ctx.g_c * 2.0f), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kdouble(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 0;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
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
    // centre-only grids are read at the nearest compute row, so halo
    // waves repeat their neighbours' addresses and every wave issues
    // the same loads
    const int drow = wave < HY ? y0 : (wave >= BY - HY ? y0 + TY - 1 : yrow);
    const int g_nx = g.dim[0], g_nxy = g.dim[0] * g.dim[1];
    const physis_hip::BufWin<float> g_w = physis_hip::BufWin<float>::Make(g.p, g_nxy * g.dim[2], (long)zb * g_nxy, (long)ze * g_nxy);
    float g_dv[2][VX];
    g_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * g_nx + zb * g_nxy, g_dv[0]);
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
    __syncthreads();
    __PSCtx_kdouble ctx;
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
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        g_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * g_nx + (z + 1) * g_nxy, g_dv[nxt]);
        if (computes && z < ze) {
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g_c = g_dv[cur][i];
              ctx.g2_e = false;
              kdouble(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        __syncthreads();
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_kdouble(const struct __PSStencil_kdouble &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kdouble<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 0, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 0));
}

template <int VX>
static int __PSLaunch_kdouble(const struct __PSStencil_kdouble &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kdouble<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_kdouble<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kdouble(const struct __PSStencil_kdouble &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kdouble<4>(s).blocks
         : (!physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_kdouble<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_kdouble<1>(s).blocks;
}

static int __PSRun_kdouble(const struct __PSStencil_kdouble &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kdouble<4>(s, stream, red)
         : (!physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_kdouble<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_kdouble<1>(s, stream, red);
}

static void __PSStencilRun_20(int iter, struct __PSStencil_kdouble s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kdouble");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kdouble(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

float systest_host_get(int x, int y, int z) {
  int i, j, k;
  float v = 0;
  PSGrid3DFloat g = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 4, 3, 2);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, 4, 3, 2);
  PSDomain3D d = PSDomain3DNew(0, 4, 0, 3, 0, 2);
  for (k = 0; k < 2; ++k) 
    for (j = 0; j < 3; ++j) 
      for (i = 0; i < 4; ++i) {
        physis_hip::SetElem<float>(g, v, i, j, k);
        v += 1;
      }
  __PSStencilRun_20(1, __PSStencilMap_kdouble(d, g, g2));
  v = physis_hip::GetElem<float>(g2, x, y, z);
  __PSGridFree(g, NULL);
  __PSGridFree(g2, NULL);
  return v;
}

}  // extern "C"

// ---------------------------------------------- stencil kshadow
struct __PSStencil_kshadow {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
};

static struct __PSStencil_kshadow __PSStencilMap_kshadow(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2) {
  struct __PSStencil_kshadow __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2)};
  return __s;
}

// Stencil analysis of kshadow (2.5D run kernel):
//   g  read from memory, irregular gets
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (an index parameter is rebound)
struct __PSCtx_kshadow {
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void kshadow(
    const int x, const int y, const int z, __PSCtx_kshadow &__ctx) {
  float v;
  int xx = x;
{
    int x = xx + 2;
    v = physis_hip::GetLinear<float>(__ctx.g_p, __ctx.g_dim, 3, x - 1, y, z);
  }
  (__ctx.g2_v = (v), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kshadow(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 0;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
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
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
    __syncthreads();
    __PSCtx_kshadow ctx;
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
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        if (computes && z < ze) {
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g2_e = false;
              kshadow(x, yrow, z, ctx);
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        __syncthreads();
      }
    }
  }
  (void)__red;
}

template <int VX>
static physis_hip::RunShape __PSShape_kshadow(const struct __PSStencil_kshadow &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kshadow<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 0, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 0));
}

template <int VX>
static int __PSLaunch_kshadow(const struct __PSStencil_kshadow &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kshadow<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_kshadow<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kshadow(const struct __PSStencil_kshadow &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kshadow<4>(s).blocks
         : __PSShape_kshadow<1>(s).blocks;
}

static int __PSRun_kshadow(const struct __PSStencil_kshadow &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kshadow<4>(s, stream, red)
         : __PSLaunch_kshadow<1>(s, stream, red);
}

static void __PSStencilRun_21(int iter, struct __PSStencil_kshadow s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kshadow");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kshadow(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_shadowed_index(const float * in, float * out, int nx, int ny, int nz) {
  PSGrid3DFloat g = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, nx, ny, nz);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, nx, ny, nz);
  PSDomain3D d = PSDomain3DNew(0, nx, 0, ny, 0, nz);
  __PSGridCopyin(g, in, NULL);
  __PSStencilRun_21(1, __PSStencilMap_kshadow(d, g, g2));
  __PSGridCopyout(g2, out, NULL);
  __PSGridFree(g, NULL);
  __PSGridFree(g2, NULL);
}

}  // extern "C"

// ---------------------------------------------- stencil kscaled
struct __PSStencil_kscaled {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  float s;
  float *__reduce_out;  // PSStencilMapReduce target
  int __reduce_op;
};

static struct __PSStencil_kscaled __PSStencilMap_kscaled(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float s) {
  struct __PSStencil_kscaled __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), s, NULL, 0};
  return __s;
}

static struct __PSStencil_kscaled __PSStencilMapReduce_kscaled(
    float *__v, int __op, __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float s) {
  struct __PSStencil_kscaled __s = __PSStencilMap_kscaled(__dom, g, g2, s);
  __s.__reduce_out = __v;
  __s.__reduce_op = __op;
  return __s;
}

// Stencil analysis of kscaled (2.5D run kernel):
//   g  direct (centre only)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: no (not one read grid and one emitted grid)
struct __PSCtx_kscaled {
  float g_c;
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ float kscaled(
    const int x, const int y, const int z, __PSCtx_kscaled &__ctx, float s) {
  float v = __ctx.g_c * s;
  (__ctx.g2_v = (v), __ctx.g2_e = true);
  return v;
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_kscaled(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, float s, physis_hip::RunShape sh, float *__restrict__ __red) {
  constexpr int VX = physis_hip::FormVX(FORM);
  constexpr bool RAGGED = physis_hip::FormRagged(FORM);
  constexpr int PD = 4;
  constexpr int HY = 0;
  constexpr int TX = 64 * VX, TY = BY - 2 * HY;
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
    const int g_nx = g.dim[0], g_nxy = g.dim[0] * g.dim[1];
    const physis_hip::BufWin<float> g_w = physis_hip::BufWin<float>::Make(g.p, g_nxy * g.dim[2], (long)zb * g_nxy, (long)ze * g_nxy);
    float g_dv[2][VX];
    g_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * g_nx + zb * g_nxy, g_dv[0]);
    const int g2_enx = g2.dim[0], g2_enxy = g2.dim[0] * g2.dim[1];
    const physis_hip::BufWin<float> g2_ew = physis_hip::BufWin<float>::Make(g2.p, g2_enxy * g2.dim[2], (long)zb * g2_enxy, (long)ze * g2_enxy);
    __syncthreads();
    __PSCtx_kscaled ctx;
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
    for (int zc = zb; zc < ze; zc += U) {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int z = zc + k;
        const int cur = k & 1, nxt = cur ^ 1;
        (void)cur; (void)nxt;
        g_w.template Load<VX, physis_hip::kStreamLoad>(xs + drow * g_nx + (z + 1) * g_nxy, g_dv[nxt]);
        if (computes && z < ze) {
          float g2_out[VX];
          unsigned g2_mask = 0;
#pragma unroll
          for (int i = 0; i < VX; ++i) {
            const int x = xs + i;
            const bool __in = x >= dom.local_min[0] && x < dom.local_max[0];
            {
              ctx.g_c = g_dv[cur][i];
              ctx.g2_e = false;
              const float __r = kscaled(x, yrow, z, ctx, s);
              if constexpr (RED >= 0) __racc = __in ? physis_hip::ReduceOp<float, RED < 0 ? 0 : RED>::apply(__racc, __r) : __racc;
              g2_out[i] = ctx.g2_v;
              g2_mask |= (__in && ctx.g2_e) ? 1u << i : 0u;
            }
          }
          physis_hip::StoreMasked<float, VX>(g2_ew, xs + yrow * g2_enx + z * g2_enxy, g2_out, g2_mask);
        }
        __syncthreads();
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
static physis_hip::RunShape __PSShape_kscaled(const struct __PSStencil_kscaled &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_kscaled<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 0, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 0));
}

template <int VX>
static int __PSLaunch_kscaled(const struct __PSStencil_kscaled &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_kscaled<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  switch (red ? s.__reduce_op : -1) {
    case PS_MAX:
      hipLaunchKernelGGL((__PSStencilRun_kscaled<VX, 16, PS_MAX>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.s, sh, (float *)red);
      break;
    case PS_MIN:
      hipLaunchKernelGGL((__PSStencilRun_kscaled<VX, 16, PS_MIN>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.s, sh, (float *)red);
      break;
    case PS_SUM:
      hipLaunchKernelGGL((__PSStencilRun_kscaled<VX, 16, PS_SUM>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.s, sh, (float *)red);
      break;
    case PS_PROD:
      hipLaunchKernelGGL((__PSStencilRun_kscaled<VX, 16, PS_PROD>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.s, sh, (float *)red);
      break;
    default:
      hipLaunchKernelGGL((__PSStencilRun_kscaled<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), s.s, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_kscaled(const struct __PSStencil_kscaled &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_kscaled<4>(s).blocks
         : (!physis_hip::OnePointRows(s.dom, false, false)) ? __PSShape_kscaled<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_kscaled<1>(s).blocks;
}

static int __PSRun_kscaled(const struct __PSStencil_kscaled &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_kscaled<4>(s, stream, red)
         : (!physis_hip::OnePointRows(s.dom, false, false)) ? __PSLaunch_kscaled<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_kscaled<1>(s, stream, red);
}

static void __PSStencilRun_22(int iter, struct __PSStencil_kscaled s0, struct __PSStencil_kscaled s1, struct __PSStencil_kscaled s2, struct __PSStencil_kscaled s3, struct __PSStencil_kscaled s4, struct __PSStencil_kscaled s5, struct __PSStencil_kscaled s6) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("kscaled, kscaled, kscaled, kscaled, kscaled, kscaled, kscaled");
  physis_hip::RunTimer timer(stream);
  physis_hip::ReduceSlots __slots;
  physis_hip::MapReducer red0(s0.__reduce_out, s0.__reduce_op, PS_FLOAT,
      s0.__reduce_out ? __PSBlocks_kscaled(s0) : 0, iter, __slots);
  physis_hip::MapReducer red1(s1.__reduce_out, s1.__reduce_op, PS_FLOAT,
      s1.__reduce_out ? __PSBlocks_kscaled(s1) : 0, iter, __slots);
  physis_hip::MapReducer red2(s2.__reduce_out, s2.__reduce_op, PS_FLOAT,
      s2.__reduce_out ? __PSBlocks_kscaled(s2) : 0, iter, __slots);
  physis_hip::MapReducer red3(s3.__reduce_out, s3.__reduce_op, PS_FLOAT,
      s3.__reduce_out ? __PSBlocks_kscaled(s3) : 0, iter, __slots);
  physis_hip::MapReducer red4(s4.__reduce_out, s4.__reduce_op, PS_FLOAT,
      s4.__reduce_out ? __PSBlocks_kscaled(s4) : 0, iter, __slots);
  physis_hip::MapReducer red5(s5.__reduce_out, s5.__reduce_op, PS_FLOAT,
      s5.__reduce_out ? __PSBlocks_kscaled(s5) : 0, iter, __slots);
  physis_hip::MapReducer red6(s6.__reduce_out, s6.__reduce_op, PS_FLOAT,
      s6.__reduce_out ? __PSBlocks_kscaled(s6) : 0, iter, __slots);
  for (int i = 0; i < iter; ++i) {
    __PSRun_kscaled(s0, stream, red0.Slot(i));
    __PSRun_kscaled(s1, stream, red1.Slot(i));
    __PSRun_kscaled(s2, stream, red2.Slot(i));
    __PSRun_kscaled(s3, stream, red3.Slot(i));
    __PSRun_kscaled(s4, stream, red4.Slot(i));
    __PSRun_kscaled(s5, stream, red5.Slot(i));
    __PSRun_kscaled(s6, stream, red6.Slot(i));
    red0.After(i);
    red1.After(i);
    red2.After(i);
    red3.After(i);
    red4.After(i);
    red5.After(i);
    red6.After(i);
  }
  red0.Finish(stream);
  red1.Finish(stream);
  red2.Finish(stream);
  red3.Finish(stream);
  red4.Finish(stream);
  red5.Finish(stream);
  red6.Finish(stream);
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void systest_seven_reductions(float * sums) {
  int n = 16, i;
  PSGrid3DFloat g = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, n, n, n);
  PSGrid3DFloat g2 = physis_hip::NewGrid(PS_FLOAT, sizeof(float), 3, n, n, n);
  float *indata = (float*)malloc(sizeof(float) * n * n * n);
  for (i = 0; i < n * n * n; i++) 
    indata[i] = (float)(i % 7);
  __PSGridCopyin(g, indata, NULL);
  PSDomain3D d0 = PSDomain3DNew(0, n, 0, n, 0, n);
  PSDomain3D d1 = PSDomain3DNew(0, n, 0, n, 0, n / 2);
  __PSStencilRun_22(1, __PSStencilMapReduce_kscaled(&sums[0], PS_SUM, d0, g, g2, 1.0f), __PSStencilMapReduce_kscaled(&sums[1], PS_SUM, d1, g, g2, 2.0f), __PSStencilMapReduce_kscaled(&sums[2], PS_SUM, d0, g, g2, 3.0f), __PSStencilMapReduce_kscaled(&sums[3], PS_SUM, d1, g, g2, 4.0f), __PSStencilMapReduce_kscaled(&sums[4], PS_SUM, d0, g, g2, 5.0f), __PSStencilMapReduce_kscaled(&sums[5], PS_SUM, d1, g, g2, 6.0f), __PSStencilMapReduce_kscaled(&sums[6], PS_SUM, d0, g, g2, 7.0f));
  __PSGridFree(g, NULL);
  __PSGridFree(g2, NULL);
  free(indata);
}

}  // extern "C"

