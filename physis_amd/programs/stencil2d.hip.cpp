// Generated by physisc-hip from stencil2d.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

// ---------------------------------------------- stencil s2d5
struct __PSStencil_s2d5 {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  float w;
};

static struct __PSStencil_s2d5 __PSStencilMap_s2d5(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float w) {
  struct __PSStencil_s2d5 __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), w};
  return __s;
}

// Stencil analysis of s2d5 (2.5D run kernel over the rows view nx x 1 x ny of its 2-D grids, y marched as z):
//   g  staged x[-1,1] y[-0,0] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,0,-1) 4:(0,0,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_s2d5 {
  float g[5];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void s2d5(
    const int x, const int y, __PSCtx_s2d5 &__ctx, float w) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4];
  (__ctx.g2_v = (v * w), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_s2d5(
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
    __PSCtx_s2d5 ctx;
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
              s2d5(x, z, ctx, w);
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
static physis_hip::RunShape __PSShape_s2d5(const struct __PSStencil_s2d5 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_s2d5<VX, 1, -1>, 64 * 1);
  return physis_hip::PlanRun(physis_hip::RowDomain(s.dom), 64 * physis_hip::FormVX(VX), 1 - 2 * 0, per_cu, physis_hip::WindowChunkLimitRows({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_s2d5(const struct __PSStencil_s2d5 &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_s2d5<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 1);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_s2d5<VX, 1, -1>), grid, block, 0, stream, physis_hip::RowDomain(s.dom), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_s2d5(const struct __PSStencil_s2d5 &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_s2d5<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSShape_s2d5<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_s2d5<1>(s).blocks;
}

static int __PSRun_s2d5(const struct __PSStencil_s2d5 &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_s2d5<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSLaunch_s2d5<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_s2d5<1>(s, stream, red);
}

// Rows pass of s2d5: T sweeps of src into dst, the one before the
// last into bg when store_mid.
template <int T>
__global__ __launch_bounds__(64) void __PSStencilRunR_s2d5(
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
  __PSCtx_s2d5 ctx;
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
            s2d5(xs + i, z, ctx, w);
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
static void __PSLaunchR_s2d5(const struct __PSStencil_s2d5 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream) {
  const __PSDomain d = physis_hip::RowDomain(s.dom);
  static int per_cu = physis_hip::BlocksPerCU((const void *)__PSStencilRunR_s2d5<T>, 64);
  const physis_hip::RunShape sh = physis_hip::PlanRun(d, physis_hip::kRowsTX, 1, per_cu,
      physis_hip::WindowChunkLimitRows({s.g, s.g2}, T + 1), 2 * T + 3);
  if (sh.blocks == 0) return;
  hipLaunchKernelGGL(__PSStencilRunR_s2d5<T>, dim3(sh.blocks), dim3(64), 0, stream, d, src, dst, bg, store_mid, s.w, sh);
}

// The pair (s0, s1) is s2d5(a -> b), s2d5(b -> a) over one domain strictly
// inside the grids, with the same scalars: it may run as rows passes.
static bool __PSFusable2_s2d5(const struct __PSStencil_s2d5 &s0, const struct __PSStencil_s2d5 &s1) {
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

// ---------------------------------------------- stencil s2d9
struct __PSStencil_s2d9 {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  float w;
};

static struct __PSStencil_s2d9 __PSStencilMap_s2d9(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, float w) {
  struct __PSStencil_s2d9 __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), w};
  return __s;
}

// Stencil analysis of s2d9 (2.5D run kernel over the rows view nx x 1 x ny of its 2-D grids, y marched as z):
//   g  staged x[-1,1] y[-0,0] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,0,-1) 4:(0,0,1) 5:(-1,0,-1) 6:(1,0,-1) 7:(-1,0,1) 8:(1,0,1)
//   g2  not read, emitted
//   two-sweep fusion of map pairs: yes, over a domain inside the grid
struct __PSCtx_s2d9 {
  float g[9];
  const float *g_p;
  int g_dim[3];
  float g2_v;
  bool g2_e;
  const float *g2_p;
  int g2_dim[3];
};

__device__ __forceinline__ void s2d9(
    const int x, const int y, __PSCtx_s2d9 &__ctx, float w) {
  float v = __ctx.g[0] + __ctx.g[1] + __ctx.g[2] + __ctx.g[3] + __ctx.g[4] + __ctx.g[5] + __ctx.g[6] + __ctx.g[7] + __ctx.g[8];
  (__ctx.g2_v = (v * w), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 0 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_s2d9(
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
    __PSCtx_s2d9 ctx;
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
          float g_r1[VX + 2];
          S_g::template ReadRow<-1, 1>(g_lds + physis_hip::RingSlot<4>(g_base, 0) * S_g::kPlane, wave + 0, lane, g_r1);
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
              ctx.g[1] = g_r0[i + 0];
              ctx.g[2] = g_r0[i + 2];
              ctx.g[3] = g_r1[i + 1];
              ctx.g[4] = g_r2[i + 1];
              ctx.g[5] = g_r1[i + 0];
              ctx.g[6] = g_r1[i + 2];
              ctx.g[7] = g_r2[i + 0];
              ctx.g[8] = g_r2[i + 2];
              ctx.g2_e = false;
              s2d9(x, z, ctx, w);
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
static physis_hip::RunShape __PSShape_s2d9(const struct __PSStencil_s2d9 &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_s2d9<VX, 1, -1>, 64 * 1);
  return physis_hip::PlanRun(physis_hip::RowDomain(s.dom), 64 * physis_hip::FormVX(VX), 1 - 2 * 0, per_cu, physis_hip::WindowChunkLimitRows({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_s2d9(const struct __PSStencil_s2d9 &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_s2d9<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 1);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_s2d9<VX, 1, -1>), grid, block, 0, stream, physis_hip::RowDomain(s.dom), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g), physis_hip::RowView<__PSGrid3DFloat_dev>(s.g2), s.w, sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_s2d9(const struct __PSStencil_s2d9 &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_s2d9<4>(s).blocks
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSShape_s2d9<4 + physis_hip::kRagged>(s).blocks
         : __PSShape_s2d9<1>(s).blocks;
}

static int __PSRun_s2d9(const struct __PSStencil_s2d9 &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_s2d9<4>(s, stream, red)
         : (s.dom.local_max[0] <= s.g->dim[0] && !physis_hip::OnePointRows(physis_hip::RowDomain(s.dom), false, false)) ? __PSLaunch_s2d9<4 + physis_hip::kRagged>(s, stream, red)
         : __PSLaunch_s2d9<1>(s, stream, red);
}

// Rows pass of s2d9: T sweeps of src into dst, the one before the
// last into bg when store_mid.
template <int T>
__global__ __launch_bounds__(64) void __PSStencilRunR_s2d9(
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
  __PSCtx_s2d9 ctx;
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
            ctx.g[5] = q[t - 1][(k + 1) % 3].v[1 + i + -1];
            ctx.g[6] = q[t - 1][(k + 1) % 3].v[1 + i + 1];
            ctx.g[7] = q[t - 1][(k + 0) % 3].v[1 + i + -1];
            ctx.g[8] = q[t - 1][(k + 0) % 3].v[1 + i + 1];
            ctx.g2_e = false;
            s2d9(xs + i, z, ctx, w);
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
static void __PSLaunchR_s2d9(const struct __PSStencil_s2d9 &s, const __PSGrid3DFloat_dev &src, const __PSGrid3DFloat_dev &dst, float *bg, int store_mid, hipStream_t stream) {
  const __PSDomain d = physis_hip::RowDomain(s.dom);
  static int per_cu = physis_hip::BlocksPerCU((const void *)__PSStencilRunR_s2d9<T>, 64);
  const physis_hip::RunShape sh = physis_hip::PlanRun(d, physis_hip::kRowsTX, 1, per_cu,
      physis_hip::WindowChunkLimitRows({s.g, s.g2}, T + 1), 2 * T + 3);
  if (sh.blocks == 0) return;
  hipLaunchKernelGGL(__PSStencilRunR_s2d9<T>, dim3(sh.blocks), dim3(64), 0, stream, d, src, dst, bg, store_mid, s.w, sh);
}

// The pair (s0, s1) is s2d9(a -> b), s2d9(b -> a) over one domain strictly
// inside the grids, with the same scalars: it may run as rows passes.
static bool __PSFusable2_s2d9(const struct __PSStencil_s2d9 &s0, const struct __PSStencil_s2d9 &s1) {
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

static void __PSStencilRun_0(int iter, struct __PSStencil_s2d5 s0, struct __PSStencil_s2d5 s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("s2d5, s2d5");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_s2d5(s0, s1) &&
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
        __PSLaunchR_s2d5<4>(s0, src, dst, b, j == passes - 1, stream);
      else
        __PSLaunchR_s2d5<2>(s0, src, dst, b, j == passes - 1, stream);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_s2d5(s0, stream, NULL);
    __PSRun_s2d5(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_1(int iter, struct __PSStencil_s2d9 s0, struct __PSStencil_s2d9 s1) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("s2d9, s2d9");
  physis_hip::RunTimer timer(stream);
  const bool __fuse = iter >= 2 && __PSFusable2_s2d9(s0, s1) &&
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
        __PSLaunchR_s2d9<4>(s0, src, dst, b, j == passes - 1, stream);
      else
        __PSLaunchR_s2d9<2>(s0, src, dst, b, j == passes - 1, stream);
      src = dst;
    }
    i0 = iter;
  }
  for (int i = i0; i < iter; ++i) {
    __PSRun_s2d9(s0, stream, NULL);
    __PSRun_s2d9(s1, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void stencil2d_run(PSGrid2DFloat a, PSGrid2DFloat b, int points, int count, float w) {
  PSDomain2D d = PSDomain2DNew(1, PSGridDim(a, 0) - 1, 1, PSGridDim(a, 1) - 1);
  if (points == 5)
    __PSStencilRun_0(count, __PSStencilMap_s2d5(d, a, b, w), __PSStencilMap_s2d5(d, b, a, w));
  else
    __PSStencilRun_1(count, __PSStencilMap_s2d9(d, a, b, w), __PSStencilMap_s2d9(d, b, a, w));
}

}  // extern "C"

static void __PSStencilRun_2(int iter, struct __PSStencil_s2d5 s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("s2d5");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_s2d5(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

static void __PSStencilRun_3(int iter, struct __PSStencil_s2d9 s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("s2d9");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_s2d9(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void stencil2d_sweep(PSGrid2DFloat a, PSGrid2DFloat b, int points, float w) {
  PSDomain2D d = PSDomain2DNew(1, PSGridDim(a, 0) - 1, 1, PSGridDim(a, 1) - 1);
  if (points == 5)
    __PSStencilRun_2(1, __PSStencilMap_s2d5(d, a, b, w));
  else
    __PSStencilRun_3(1, __PSStencilMap_s2d9(d, a, b, w));
}

}  // extern "C"

