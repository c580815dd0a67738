// Generated by physisc-hip from mixed7.c.
#define PHYSIS_HIP
#include "physis/physis.h"
#include "physis/hip/stencil.h"
#include "physis/hip/run.h"
#include "physis/hip/tile.h"


#pragma clang fp contract(off)

// ---------------------------------------------- stencil mixed7_kernel
struct __PSStencil_mixed7_kernel {
  __PSDomain dom;
  __PSGrid *g;
  int __g_index;
  __PSGrid *g2;
  int __g2_index;
  __PSGrid *i;
  int __i_index;
  __PSGrid *j;
  int __j_index;
  __PSGrid *k;
  int __k_index;
};

static struct __PSStencil_mixed7_kernel __PSStencilMap_mixed7_kernel(
    __PSDomain __dom, __PSGrid *g, __PSGrid *g2, __PSGrid *i, __PSGrid *j, __PSGrid *k) {
  struct __PSStencil_mixed7_kernel __s = {__dom, g, __PSGridGetID(g), g2, __PSGridGetID(g2), i, __PSGridGetID(i), j, __PSGridGetID(j), k, __PSGridGetID(k)};
  return __s;
}

// Stencil analysis of mixed7_kernel (2.5D run kernel):
//   g  staged x[-1,1] y[-1,1] z[-1,1] non-periodic
//     offsets 0:(0,0,0) 1:(-1,0,0) 2:(1,0,0) 3:(0,-1,0) 4:(0,1,0) 5:(0,0,-1) 6:(0,0,1)
//   g2  not read, emitted
//   i  read from memory, irregular gets
//   j  read from memory, irregular gets
//   k  read from memory, irregular gets
//   two-sweep fusion of map pairs: no (grid i is read irregularly)
struct __PSCtx_mixed7_kernel {
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
  const float *k_p;
  int k_dim[3];
};

__device__ __forceinline__ void mixed7_kernel(
    const int x, const int y, const int z, __PSCtx_mixed7_kernel &__ctx) {
  float v = __ctx.g[0] + __ctx.g[1] * physis_hip::GetLinear<float>(__ctx.i_p, __ctx.i_dim, 1, x - 1) + __ctx.g[2] * physis_hip::GetLinear<float>(__ctx.i_p, __ctx.i_dim, 1, x + 1) + __ctx.g[3] * physis_hip::GetLinear<float>(__ctx.j_p, __ctx.j_dim, 1, y - 1) + __ctx.g[4] * physis_hip::GetLinear<float>(__ctx.j_p, __ctx.j_dim, 1, y + 1) + __ctx.g[5] * physis_hip::GetLinear<float>(__ctx.k_p, __ctx.k_dim, 1, z - 1) + __ctx.g[6] * physis_hip::GetLinear<float>(__ctx.k_p, __ctx.k_dim, 1, z + 1);
  (__ctx.g2_v = (v), __ctx.g2_e = true);
}

// Run kernel: VX points per lane, BY waves per block (the first and
// last 1 load halo rows), staged planes PD steps ahead,
// centre-only grids one step ahead.  RED: reduction operator of a
// PSStencilMapReduce execution, or -1.
// FORM: VX, plus kRagged for x extents that are not multiples of VX.
template <int FORM, int BY, int RED>
__global__ __launch_bounds__(64 * BY) void __PSStencilRun_mixed7_kernel(
    __PSDomain dom, __PSGrid3DFloat_dev g, __PSGrid3DFloat_dev g2, __PSGrid1DFloat_dev i, __PSGrid1DFloat_dev j, __PSGrid1DFloat_dev k, physis_hip::RunShape sh, float *__restrict__ __red) {
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
    __PSCtx_mixed7_kernel ctx;
    ctx.g_p = g.p;
    for (int d = 0; d < 3; ++d) ctx.g_dim[d] = g.dim[d];
    ctx.g2_p = g2.p;
    for (int d = 0; d < 3; ++d) ctx.g2_dim[d] = g2.dim[d];
    ctx.i_p = i.p;
    for (int d = 0; d < 3; ++d) ctx.i_dim[d] = d < 1 ? i.dim[d] : 1;
    ctx.j_p = j.p;
    for (int d = 0; d < 3; ++d) ctx.j_dim[d] = d < 1 ? j.dim[d] : 1;
    ctx.k_p = k.p;
    for (int d = 0; d < 3; ++d) ctx.k_dim[d] = d < 1 ? k.dim[d] : 1;
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
              mixed7_kernel(x, yrow, z, ctx);
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
static physis_hip::RunShape __PSShape_mixed7_kernel(const struct __PSStencil_mixed7_kernel &s) {
  static int per_cu = physis_hip::BlocksPerCU(
      (const void *)__PSStencilRun_mixed7_kernel<VX, 16, -1>, 64 * 16);
  return physis_hip::PlanRun(s.dom, 64 * physis_hip::FormVX(VX), 16 - 2 * 1, per_cu, physis_hip::WindowChunkLimit({s.g, s.g2}, 2));
}

template <int VX>
static int __PSLaunch_mixed7_kernel(const struct __PSStencil_mixed7_kernel &s, hipStream_t stream, void *red) {
  const physis_hip::RunShape sh = __PSShape_mixed7_kernel<VX>(s);
  if (sh.blocks == 0) return 0;
  const dim3 grid(sh.blocks), block(64 * 16);
  {
  (void)red;
  {
      hipLaunchKernelGGL((__PSStencilRun_mixed7_kernel<VX, 16, -1>), grid, block, 0, stream, s.dom, physis_hip::DevView<__PSGrid3DFloat_dev>(s.g), physis_hip::DevView<__PSGrid3DFloat_dev>(s.g2), physis_hip::DevView<__PSGrid1DFloat_dev>(s.i), physis_hip::DevView<__PSGrid1DFloat_dev>(s.j), physis_hip::DevView<__PSGrid1DFloat_dev>(s.k), sh, (float *)NULL);
  }
  }
  return sh.blocks;
}

static int __PSBlocks_mixed7_kernel(const struct __PSStencil_mixed7_kernel &s) {
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSShape_mixed7_kernel<4>(s).blocks
         : __PSShape_mixed7_kernel<1>(s).blocks;
}

static int __PSRun_mixed7_kernel(const struct __PSStencil_mixed7_kernel &s, hipStream_t stream, void *red) {
  physis_hip::CheckGrid3D(s.g, PS_FLOAT);
  physis_hip::CheckGrid3D(s.g2, PS_FLOAT);
  physis_hip::CheckGrid3D(s.i, PS_FLOAT);
  physis_hip::CheckGrid3D(s.j, PS_FLOAT);
  physis_hip::CheckGrid3D(s.k, PS_FLOAT);
  physis_hip::CheckEmitDomain(s.dom, s.g2);
  return (s.g->dim[0] % 4 == 0 && s.g2->dim[0] % 4 == 0) ? __PSLaunch_mixed7_kernel<4>(s, stream, red)
         : __PSLaunch_mixed7_kernel<1>(s, stream, red);
}

static void __PSStencilRun_0(int iter, struct __PSStencil_mixed7_kernel s0) {
  hipStream_t stream = (hipStream_t)__PSHipStream();
  __PSTraceStencilPre("mixed7_kernel");
  physis_hip::RunTimer timer(stream);
  for (int i = 0; i < iter; ++i) {
    __PSRun_mixed7_kernel(s0, stream, NULL);
  }
  __PSTraceStencilPost(timer.Stop());
}

extern "C" {

void mixed7_run(PSGrid3DFloat g, PSGrid3DFloat g2, PSGrid1DFloat cx, PSGrid1DFloat cy, PSGrid1DFloat cz) {
  PSDomain3D d = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1, 1, PSGridDim(g, 2) - 1);
  __PSStencilRun_0(1, __PSStencilMap_mixed7_kernel(d, g, g2, cx, cy, cz));
}

}  // extern "C"

