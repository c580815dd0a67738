// libphysis_warmstart_hip: the U-Net warm start of the Poisson solve
// (include/physis/physis_warmstart.h), forward, backward and Adam on the GPU.
//
// Tensors are channels-last BF16 ([position][channel], position
// ((n*D + z)*H + y)*W + x, channels a multiple of 8), so the 8 K-values an
// MFMA lane feeds are one 16-byte load.
//
// 3x3x3 convolution as an implicit GEMM on v_mfma_f32_16x16x32_bf16:
//   forward   D[16 cout][16 x] += W[16 cout][32 k] X[32 k][16 x], k = tap *
//             CIN + ci, X read from LDS-staged input planes with zero
//             padding, W the weights stored [cout][k] (K padded to 32);
//   backward  dX = the forward kernel on dZ with the flipped, transposed
//             weights Wf[ci][tap' * COUT + co] = W[co][26 - tap'][ci];
//   filter    dW[co][k] = sum over positions of dZ[p][co] X[p + off(k)][ci]:
//             GEMM with the positions as K, FP32 partials per block summed in
//             a fixed order (deterministic); both operands read transposed
//             from LDS.
// MFMA lane layout (checked on the device against a host product): lane l
// feeds A row l%16 and B column l%16 with k = 8*(l/16) .. +7, and receives
// D rows 4*(l/16) .. +3 of column l%16.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "physis/hip/device.h"
#include "physis/hip/stencil.h"
#include "physis/physis_warmstart.h"
#include "../runtime/runtime_hip.h"

#pragma clang fp contract(off)

namespace physis_unet {

typedef unsigned short u16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

constexpr int kPool = 4;           // pooling / upsampling factor per axis
// Weight fragments (K steps x 16-channel tiles) that the z-marching
// convolution keeps in registers; more are staged in LDS.  21 covers the
// 24 -> 8 layer (6% faster than staging its weights).
constexpr int kRegWeightSteps = 21;

__device__ __forceinline__ float Bf2F(u16 h) {
  return __uint_as_float((unsigned)h << 16);
}
__device__ __forceinline__ u16 F2Bf(float f) {
  return physis_hip::Convert<physis_hip::bf16_t, float>(f).bits;
}
__device__ __forceinline__ bf16x8 Load8(const u16 *p) {
  const uint4 v = *reinterpret_cast<const uint4 *>(p);
  return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ bf16x8 Zero8() {
  return __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
}

// Two floats rounded to BF16 (nearest even) in one word.
__device__ __forceinline__ unsigned Pack2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(
      unsigned, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}
// The halves of v whose activation (the halves of a) is positive.
__device__ __forceinline__ unsigned GateWord(unsigned v, unsigned a) {
  return (__uint_as_float(a << 16) > 0.0f ? v & 0xffffu : 0u) |
         (__uint_as_float(a & 0xffff0000u) > 0.0f ? v & 0xffff0000u : 0u);
}

constexpr int KPad(int cin) { return ((27 * cin + 31) / 32) * 32; }

// ------------------------------------------------------------ convolution
// 3x3x3 convolution marching z (the 2.5D scheme of the stencil run
// kernels).  Block (x tile, y tile, problem n, z chunk) owns XT x TY output
// positions of every plane of its chunk.  An LDS ring holds the input planes
// z-1 .. z+1 over rows y0-1 .. y0+TY and x0-1 .. x0+XT (zero outside the
// grid) and the plane z+2 being staged; the plane after that is loaded into
// registers a step ahead.  Each input plane is thus staged once per tile,
// with one barrier per step.
// The GEMM is D[cout][16 x] = W[cout][32 k] X[32 k][16 x]: the weights are
// the A operand (registers, or LDS when they are many), the staged input the
// B operand (one aligned 16-byte LDS read per lane), and a lane's result is
// four consecutive channels of one position, stored as one 8-byte word.  GATE:
// the results are gated by act > 0 (the ReLU whose input gradient they are); as
// a run-time choice it cost 16 -> 48 at rows of 32 positions its registers (112
// VGPRs -> 256 and 9 spilled).
template <int CIN, int COUT, bool RELU, bool GATE, int XT, int TY>
__global__ __launch_bounds__(64 * TY) void ConvZKernel(
    const u16 *__restrict__ x, const u16 *__restrict__ wt,
    const float *__restrict__ bias, const u16 *__restrict__ act,
    u16 *__restrict__ y, int D, int H, int W, int tz, int zchunk) {
  constexpr int K = 27 * CIN, KB = (K + 31) / 32, KP = KB * 32;
  constexpr int MT = (COUT + 15) / 16;
  constexpr bool kRegW = KB * MT <= kRegWeightSteps;
  constexpr int XS = XT + 2, RS = TY + 2, NV = CIN / 8;
  constexpr int PLANE = RS * XS * CIN;  // u16 elements of a staged plane
  constexpr int SV = RS * XS * NV;      // 16-byte vectors of a staged plane
  constexpr int NTH = 64 * TY;
  constexpr int VPT = (SV + NTH - 1) / NTH;
  constexpr int WL = kRegW ? 1 : MT * 16 * KP;  // weights staged in LDS
  __shared__ __attribute__((aligned(16))) u16 ring[4 * PLANE];
  __shared__ __attribute__((aligned(16))) u16 wlds[WL];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int tiles_x = (W + XT - 1) / XT;
  const int x0 = (blockIdx.x % tiles_x) * XT, y0 = (blockIdx.x / tiles_x) * TY;
  const int n = blockIdx.y / tz;
  const int zb = (blockIdx.y - n * tz) * zchunk;
  const int ze = min(zb + zchunk, D);
  if (zb >= ze) return;  // uniform over the block
  auto fetch = [&](int zz, uint4 (&buf)[VPT]) {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * NTH;
      const int c8 = v % NV, t = v / NV;
      const int xp = t % XS, pr = t / XS;
      const int yy = y0 - 1 + pr, xx = x0 - 1 + xp;
      uint4 u = make_uint4(0, 0, 0, 0);
      if (v < SV && zz >= 0 && zz < D && yy >= 0 && yy < H && xx >= 0 &&
          xx < W)
        u = *reinterpret_cast<const uint4 *>(
            x + ((((long)n * D + zz) * H + yy) * W + xx) * CIN + c8 * 8);
      buf[i] = u;
    }
  };
  auto put = [&](int slot, const uint4 (&buf)[VPT]) {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * NTH;
      if (v < SV)
        *reinterpret_cast<uint4 *>(ring + slot * PLANE + (v / NV) * CIN +
                                   (v % NV) * 8) = buf[i];
    }
  };
  uint4 buf[VPT];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    fetch(zb - 1 + k, buf);
    put(k, buf);
  }
  fetch(zb + 2, buf);
  bf16x8 aw[kRegW ? KB : 1][MT];
  if constexpr (kRegW) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int co = t * 16 + r;
        aw[kb][t] = co < COUT ? Load8(wt + (long)co * KP + kb * 32 + 8 * g)
                              : Zero8();
      }
  } else {
    for (int v = threadIdx.x; v < MT * 16 * KP / 8; v += NTH) {
      const int co = (v * 8) / KP;
      uint4 u = make_uint4(0, 0, 0, 0);
      if (co < COUT) u = *reinterpret_cast<const uint4 *>(wt + (long)v * 8);
      *reinterpret_cast<uint4 *>(wlds + v * 8) = u;
    }
  }
  // With the weights in registers and at most 14 K steps the K loop is
  // unrolled and the B operand's LDS offset of every K step (u16 elements
  // within a staged plane, relative to the lane's row and x) is decoded
  // once, with the tap's plane (0..2) in bits 24 and up; -1 past K.
  // (Measured at level 1: backward data 8 -> 24 392 -> 279 us, forward
  // 8 -> 8 198 -> 187 us; the 21-step 24 -> 8 forward went 617 -> 729 us
  // and keeps the per-step decode.)
  constexpr bool kDecode = kRegW && KB <= 14;
  int boff[kDecode ? KB : 1];
  if constexpr (kDecode) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int k0 = kb * 32 + 8 * g;
      if (k0 < K) {
        const int tap = k0 / CIN, ci0 = k0 - tap * CIN;
        boff[kb] = ((((tap / 3) % 3) * XS + tap % 3) * CIN + ci0) |
                   ((tap / 9) << 24);
      } else {
        boff[kb] = -1;
      }
    }
  }
  // bias of the four channels co = 16 t + 4 g + v this lane receives
  float bb[MT][4];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int co = t * 16 + 4 * g + v;
      bb[t][v] = (bias && co < COUT) ? bias[co] : 0.0f;
    }
  __syncthreads();
  const int yy = y0 + wv;
  for (int z = zb; z < ze; ++z) {
    const int base = z - zb;  // ring slot of plane z - 1 (mod 4)
    if (yy < H) {
      const long row = (((long)n * D + z) * H + yy) * W;
      for (int xs0 = 0; xs0 < XT && x0 + xs0 < W; xs0 += 16) {
        f32x4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int xa = xs0 + r;
        if constexpr (kDecode) {
          const u16 *rb = ring + (wv * XS + xa) * CIN;
          const int so[3] = {(base & 3) * PLANE, ((base + 1) & 3) * PLANE,
                             ((base + 2) & 3) * PLANE};
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) {
            bf16x8 b = Zero8();
            if (boff[kb] >= 0) {
              const int pz = boff[kb] >> 24;
              const int sp = pz == 0 ? so[0] : (pz == 1 ? so[1] : so[2]);
              b = *reinterpret_cast<const bf16x8 *>(rb + sp +
                                                    (boff[kb] & 0xffffff));
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  aw[kb][t], b, acc[t], 0, 0, 0);
          }
        } else {
#pragma unroll 4
          for (int kb = 0; kb < KB; ++kb) {
            const int k0 = kb * 32 + 8 * g;
            bf16x8 b = Zero8();
            if (k0 < K) {
              const int tap = k0 / CIN, ci0 = k0 - tap * CIN;
              const int slot = (base + tap / 9) & 3;
              b = *reinterpret_cast<const bf16x8 *>(
                  ring + slot * PLANE +
                  ((wv + (tap / 3) % 3) * XS + xa + tap % 3) * CIN + ci0);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
              bf16x8 a;
              if constexpr (kRegW)
                a = aw[kb][t];
              else
                a = *reinterpret_cast<const bf16x8 *>(
                    wlds + (t * 16 + r) * KP + kb * 32 + 8 * g);
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[t],
                                                               0, 0, 0);
            }
          }
        }
        const int xo = x0 + xs0 + r;
        if (xo < W) {
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            const int co = t * 16 + 4 * g;
            if (co >= COUT) continue;
            unsigned w2[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              float v0 = acc[t][2 * h] + bb[t][2 * h];
              float v1 = acc[t][2 * h + 1] + bb[t][2 * h + 1];
              if (RELU) {
                v0 = v0 > 0.0f ? v0 : 0.0f;
                v1 = v1 > 0.0f ? v1 : 0.0f;
              }
              w2[h] = (unsigned)F2Bf(v0) | ((unsigned)F2Bf(v1) << 16);
            }
            if constexpr (GATE) {
              const uint2 a = *reinterpret_cast<const uint2 *>(
                  act + (row + xo) * COUT + co);
              w2[0] = GateWord(w2[0], a.x);
              w2[1] = GateWord(w2[1], a.y);
            }
            *reinterpret_cast<uint2 *>(y + (row + xo) * COUT + co) =
                make_uint2(w2[0], w2[1]);
          }
        }
      }
    }
    put((base + 3) & 3, buf);
    __syncthreads();
    fetch(z + 3, buf);
  }
}

// ------------------------------------------------- staging of input planes
// A block's view of one input plane: rows y0-1 .. y0+RS-2 and x0-1 ..
// x0+XS-2 of problem n, CIN channels per position in LDS.  A stream moves
// NCH of them (from channel COFF) between a channels-last tensor and LDS,
// 16 bytes per thread and load; the tensor has the staged resolution, or
// (UP) a quarter of it per axis, read once per fine position: an upsampled
// tensor is never written out.  Positions outside the grid are zero: the
// loads are range-checked buffer loads over the rows of one plane that the
// block reads (none of a plane outside the problem), whose offsets are computed
// once.  The rows and not the plane, so that only their bytes have to stay
// below kReach (CheckRows on the host).
constexpr unsigned kOutside = 0xfffffff0u, kReach = 0xfffffff0u;
// `rows` rows of W positions of `channels` from row y of H on, in bytes.
__device__ __forceinline__ unsigned RowBytes(int y, int rows, int H, int W,
                                             int channels) {
  return (unsigned)min(rows, H - y) * (unsigned)W * (unsigned)(channels * 2);
}

template <int CIN, int NCH, int COFF, bool UP, int RS, int XS, int NTH>
struct PlaneStream {
  static constexpr int NV = NCH / 8, SV = RS * XS * NV;
  static constexpr int VPT = (SV + NTH - 1) / NTH;
  static constexpr int Q = UP ? kPool : 1;
  unsigned off[VPT];  // bytes from row yb, kOutside outside the grid
  unsigned bytes;     // of the rows from yb on
  int yb;
  uint4 buf[VPT];

  __device__ __forceinline__ void Init(int y0, int x0, int H, int W) {
    yb = max(y0 - 1, 0) / Q;
    bytes = RowBytes(yb, RS, H / Q, W / Q, NCH);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * NTH;
      const int c8 = v % NV, t = v / NV;
      const int yy = y0 - 1 + t / XS, xx = x0 - 1 + t % XS;
      const bool in = v < SV && yy >= 0 && yy < H && xx >= 0 && xx < W;
      const unsigned pos = (yy / Q - yb) * (W / Q) + xx / Q;
      off[i] = in ? (pos * NCH + c8 * 8) * 2 : kOutside;
    }
  }
  __device__ __forceinline__ void Fetch(const u16 *p, int n, int z, int D,
                                        int H, int W) {
    const bool in = z >= 0 && z < D;
    const long row = ((long)n * (D / Q) + z / Q) * (H / Q) + yb;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<u16 *>(p) + (in ? row * (W / Q) * NCH : 0), 0,
        in ? bytes : 0, physis_hip::kBufDword3);
#pragma unroll
    for (int i = 0; i < VPT; ++i)
      buf[i] = __builtin_bit_cast(
          uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off[i], 0, 0));
  }
  __device__ __forceinline__ void Put(u16 *plane) const {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * NTH;
      if (v < SV)
        *reinterpret_cast<uint4 *>(plane + (v / NV) * CIN + COFF +
                                   (v % NV) * 8) = buf[i];
    }
  }
};

// Sources of a convolution's input.
struct SrcArgs {
  const void *a, *b;  // tensor; or coarse tensor and skip; or rhs and bnd
  long off;           // first element of rhs and bnd
};
template <int CIN, int RS, int XS, int NTH>
struct PlainSrc {
  PlaneStream<CIN, CIN, 0, false, RS, XS, NTH> s;
  __device__ __forceinline__ void Init(int y0, int x0, int H, int W) {
    s.Init(y0, x0, H, W);
  }
  __device__ __forceinline__ void Fetch(const SrcArgs &p, int n, int z, int D,
                                        int H, int W) {
    s.Fetch((const u16 *)p.a, n, z, D, H, W);
  }
  __device__ __forceinline__ void Put(u16 *plane) const { s.Put(plane); }
};
// Concatenation of an upsampled coarse tensor (two thirds of the channels)
// and a skip tensor.
template <int CIN, int RS, int XS, int NTH>
struct ConcatSrc {
  static constexpr int CA = CIN / 3 * 2, CB = CIN - CA;
  PlaneStream<CIN, CA, 0, true, RS, XS, NTH> up;
  PlaneStream<CIN, CB, CA, false, RS, XS, NTH> skip;
  __device__ __forceinline__ void Init(int y0, int x0, int H, int W) {
    up.Init(y0, x0, H, W);
    skip.Init(y0, x0, H, W);
  }
  __device__ __forceinline__ void Fetch(const SrcArgs &p, int n, int z, int D,
                                        int H, int W) {
    up.Fetch((const u16 *)p.a, n, z, D, H, W);
    skip.Fetch((const u16 *)p.b, n, z, D, H, W);
  }
  __device__ __forceinline__ void Put(u16 *plane) const {
    up.Put(plane);
    skip.Put(plane);
  }
};
// The network input: channels (rhs, bnd) rounded to BF16 from the float
// grids; with CIN = 4 two more per position, which are not written.
template <int CIN, int RS, int XS, int NTH>
struct InputSrc {
  static_assert(CIN == 2 || CIN == 4, "rhs and bnd");
  static constexpr int SV = RS * XS, VPT = (SV + NTH - 1) / NTH;
  unsigned off[VPT];
  float r[VPT], m[VPT];
  __device__ __forceinline__ void Init(int y0, int x0, int H, int W) {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * NTH;
      const int yy = y0 - 1 + v / XS, xx = x0 - 1 + v % XS;
      const bool in = v < SV && yy >= 0 && yy < H && xx >= 0 && xx < W;
      off[i] = in ? (yy * W + xx) * 4 : kOutside;
    }
  }
  __device__ __forceinline__ void Fetch(const SrcArgs &p, int n, int z, int D,
                                        int H, int W) {
    const bool in = z >= 0 && z < D;
    const long first = in ? p.off + ((long)n * D + z) * H * W : 0;
    const int bytes = in ? H * W * 4 : 0;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (float *)const_cast<void *>(p.a) + first, 0, bytes,
        physis_hip::kBufDword3);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        (float *)const_cast<void *>(p.b) + first, 0, bytes,
        physis_hip::kBufDword3);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      r[i] = __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(ra, off[i], 0, 0));
      m[i] = __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(rb, off[i], 0, 0));
    }
  }
  __device__ __forceinline__ void Put(u16 *plane) const {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * NTH;
      if (v < SV)
        *reinterpret_cast<unsigned *>(plane + v * CIN) = Pack2(r[i], m[i]);
    }
  }
};

// What becomes of a convolution's results (COUT 8 or 24 channels).
enum Epi {
  kEpiStore,    // + bias, ReLU when RELU, rounded and stored
  kEpiPool,     // stored, and averaged over the 4x4x4 cells of the coarse grid
                // (8 x 128^3: a pass of its own read the tensor again, 58 us
                // of a prediction's 744; the sums of rounded values here, in
                // another order, are what that pass summed)
  kEpiGate,     // gated by act > 0 (the ReLU whose input gradient this is)
  kEpiPredict,  // + bias, ReLU, rounded, 1x1 head, p = scale out bnd
  kEpiUpSkip    // 24 channels: 16 summed over the 4x4x4 cells of the coarse
                // grid, gated by act and stored there, 8 stored
};
struct EpiArgs {
  const float *bias = nullptr;
  u16 *y = nullptr;            // stored channels (kEpiUpSkip: the last 8)
  const u16 *act = nullptr;    // kEpiGate, kEpiUpSkip
  u16 *coarse = nullptr;       // kEpiPool, kEpiUpSkip
  const float *head = nullptr; // kEpiPredict: 8 weights and the bias
  const float *bnd = nullptr;  // kEpiPredict, from element off, as p
  void *p = nullptr;
  long off = 0;
  float scale = 0.0f;
};

// 3x3x3 convolution marching the input planes: wave w of a block owns output
// rows y0 + 2w and y0 + 2w + 1 over XT positions of every plane of a z chunk
// of one problem.  Step z' stages input plane z' + 1 while the MFMAs
// (D[16 rows][16 x] += A[16][32 k] B[32 k][16 x]) apply plane z' to the three
// output planes it reaches: the B operand of a K step (8 channels of one
// staged position per lane: k = (3 ry + dx) CIN + ci over the four input rows
// ry of the two output rows) is read from LDS once and feeds the three z
// taps, whose sums live in registers and rotate.  (An input that is not finite
// makes NaN of the zero weights of the row beyond a tap's reach: a result then
// depends on one row more than it should.)  A rows: with 8 output
// channels, 8 h + co of output row y + h (zero where ry - h is no tap); with
// 24, sets 0 and 1 hold channels 0 .. 15 of the two rows and set 2 channels
// 16 .. 23 of both.  With 2 staged input channels the B operand's other six
// are zeros, so that the sums are those of the layer's 8 channels to the bit:
// one K step of 4 ry x 3 dx x 2 channels sums in another order, and the BF16
// roundings of ten layers make 6e-4 of a prediction of those last bits (its
// error against 64 bits, 2.8e-3, stays the same).  That costs 34 us of 731 at
// 8 x 128^3; held to four waves per SIMD (130 VGPRs without) 14 less.
// The kernel it replaces held a ring of planes and read every B operand
// three times: LDS reads bounded it (24 -> 8 at 8 x 128^3: 184 us of LDS
// time in 396 us, now 245 with the concatenation read in place, which was
// another 240; 8 -> 8 172 -> 105).  The 8-channel layers run near what their
// bytes take (92 us at the rate of a copy, 140 gated), the 24-channel ones
// are bound by latency at two waves per SIMD (92 us of MFMA).
template <int CIN, int COUT, bool RELU, int XT, int TY,
          template <int, int, int, int> class SRC, int EPI,
          typename PT = double>
__global__ __launch_bounds__(64 * TY, CIN == 2 ? 4 : 1) void ConvMKernel(
    SrcArgs src, const u16 *__restrict__ wt, EpiArgs ep, int D, int H, int W,
    int tz, int zchunk) {
  static_assert(COUT == (EPI == kEpiUpSkip ? 24 : 8), "output channels");
  constexpr int S = COUT == 8 ? 1 : 3;  // A operands per B operand
  constexpr int WC = CIN == 2 ? 8 : CIN;  // channels of the stored weights
  constexpr int KPW = KPad(WC);
  constexpr int KS = 12 * WC / 32;  // K steps per plane
  constexpr int NTH = 64 * TY, ROWS = 2 * TY;
  constexpr int XS = XT + 2, RS = ROWS + 2;
  constexpr int PLANE = RS * XS * CIN;  // u16 elements of a staged plane
  constexpr int SEG = XT / 16;
  // sums over 4x4x4 cells
  constexpr bool kCells = EPI == kEpiPool || EPI == kEpiUpSkip;
  __shared__ __attribute__((aligned(16))) u16 ring[2 * PLANE];
  __shared__ __attribute__((aligned(16))) float cells[kCells ? TY / 2 : 1]
      [kCells ? SEG : 1][kCells ? 64 : 1];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int tiles_x = (W + XT - 1) / XT, tiles_y = (H + ROWS - 1) / ROWS;
  int b = physis_hip::XcdLogicalBlock(blockIdx.x, gridDim.x);
  const int x0 = (b % tiles_x) * XT;
  b /= tiles_x;
  const int y0 = (b % tiles_y) * ROWS;
  b /= tiles_y;
  const int n = b / tz, zb = (b - n * tz) * zchunk;
  const int ze = min(zb + zchunk, D);
  if (zb >= ze) return;  // uniform over the block
  SRC<CIN, RS, XS, NTH> in;
  in.Init(y0, x0, H, W);
  in.Fetch(src, n, zb - 1, D, H, W);
  in.Put(ring);
  in.Fetch(src, n, zb, D, H, W);
  // A operands of (set, z tap, K step), and the LDS offset of each K step's
  // B operand relative to the wave's first row and the lane's x
  bf16x8 aw[S][3][KS];
  int boff[KS];
#pragma unroll
  for (int kb = 0; kb < KS; ++kb) {
    const int k0 = kb * 32 + 8 * g;
    const int cell = k0 / WC, ci0 = k0 - cell * WC;
    const int ry = cell / 3, dx = cell % 3;
    boff[kb] = (ry * XS + dx) * CIN + ci0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int h = COUT == 8 || s == 2 ? r >> 3 : s;
      const int co = COUT == 8 ? r & 7 : (s == 2 ? 16 + (r & 7) : r);
      const int dy = ry - h;
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        aw[s][t][kb] =
            dy >= 0 && dy <= 2
                ? Load8(wt + (long)co * KPW + (9 * t + 3 * dy + dx) * WC + ci0)
                : Zero8();
      }
    }
  }
  float bb[4];  // bias of the lane's four channels of the paired results
#pragma unroll
  for (int v = 0; v < 4; ++v)
    bb[v] = ep.bias ? ep.bias[COUT - 8 + 4 * (g & 1) + v] : 0.0f;
  float hw[4], hb = 0.0f;  // head weights of the lane's four channels
  if constexpr (EPI == kEpiPredict) {
#pragma unroll
    for (int v = 0; v < 4; ++v) hw[v] = ep.head[4 * (g & 1) + v];
    hb = ep.head[8];
  }
  const int yw = y0 + 2 * wv;    // the wave's first output row
  const int yo = yw + (g >> 1);  // row of the lane's paired results
  f32x4 acc[SEG][S][3];
  f32x4 csum[kCells ? SEG : 1];
#pragma unroll
  for (int i = 0; i < SEG; ++i) {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < 3; ++t) acc[i][s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (kCells) csum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
  for (int m0 = 0;; m0 += 3) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int m = m0 + j, zp = zb - 1 + m;  // input plane of this step
      if (zp > ze) return;  // uniform over the block
      const int z = zp - 1;  // output plane this step completes
      const bool done = z >= zb;
      const long row = (((long)n * D + z) * H + yo) * W;
      // what the epilogue reads, ahead of the MFMAs
      uint2 av[EPI == kEpiGate ? SEG : 1];
      // (a pair of segments shares its stores: lanes of odd g take the
      // second, so that no lane is idle)
      constexpr int PSEG = (SEG + 1) / 2;
      float bv[EPI == kEpiPredict ? PSEG : 1], pv[EPI == kEpiPredict ? SEG : 1];
      const int px = SEG > 1 ? 16 * (g & 1) : 0;
#pragma unroll
      for (int i = 0; i < SEG; ++i) {
        const int xo = x0 + 16 * i + r;
        const bool in_row = done && yo < H && xo < W;
        if constexpr (EPI == kEpiGate)
          av[i] = in_row ? *reinterpret_cast<const uint2 *>(
                               ep.act + (row + xo) * 8 + 4 * (g & 1))
                         : make_uint2(0, 0);
        if constexpr (EPI == kEpiPredict) {
          if (i % 2 == 0)
            bv[i / 2] = done && yo < H && xo + px < W
                            ? ep.bnd[ep.off + row + xo + px] : 0.0f;
        }
      }
      const u16 *rb = ring + (m & 1) * PLANE + (2 * wv * XS + r) * CIN;
#pragma unroll
      for (int i = 0; i < SEG; ++i)
#pragma unroll
        for (int kb = 0; kb < KS; ++kb) {
          bf16x8 bo;
          if constexpr (CIN == 2) {
            bo = __builtin_bit_cast(
                bf16x8, make_uint4(*reinterpret_cast<const unsigned *>(
                                       rb + 16 * i * CIN + boff[kb]),
                                   0u, 0u, 0u));
          } else {
            bo = *reinterpret_cast<const bf16x8 *>(rb + 16 * i * CIN + boff[kb]);
          }
          // plane zp is tap t of output plane zp + 1 - t (slot (j - t) mod 3)
#pragma unroll
          for (int s = 0; s < S; ++s)
#pragma unroll
            for (int t = 0; t < 3; ++t)
              acc[i][s][(j + 3 - t) % 3] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                      aw[s][t][kb], bo, acc[i][s][(j + 3 - t) % 3], 0, 0, 0);
        }
#pragma unroll
      for (int i = 0; i < SEG; ++i) {
        const int xo = x0 + 16 * i + r;
        const bool in_row = done && yo < H && xo < W;
        if constexpr (EPI == kEpiUpSkip) {
          if (done) csum[i] += acc[i][0][(j + 1) % 3] + acc[i][1][(j + 1) % 3];
        }
        f32x4 v = acc[i][S - 1][(j + 1) % 3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] += bb[e];
          if (RELU) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
        }
        uint2 w2 = make_uint2(Pack2(v[0], v[1]), Pack2(v[2], v[3]));
        if constexpr (EPI == kEpiGate) {
          w2.x = GateWord(w2.x, av[i].x);
          w2.y = GateWord(w2.y, av[i].y);
        }
        if constexpr (EPI == kEpiPool) {
          if (done)
            csum[i] += f32x4{__uint_as_float(w2.x << 16),
                             __uint_as_float(w2.x & 0xffff0000u),
                             __uint_as_float(w2.y << 16),
                             __uint_as_float(w2.y & 0xffff0000u)};
        }
        if constexpr (EPI == kEpiPredict) {
          // channel by channel: the even lane's four, then the odd lane's
          const auto dot = [&](float s) {
            s += hw[0] * __uint_as_float(w2.x << 16);
            s += hw[1] * __uint_as_float(w2.x & 0xffff0000u);
            s += hw[2] * __uint_as_float(w2.y << 16);
            s += hw[3] * __uint_as_float(w2.y & 0xffff0000u);
            return s;
          };
          const float all = dot(__shfl_xor(dot(0.0f), 16, 64));  // odd lanes'
          const float below = __shfl_xor(all, 16, 64);
          pv[i] = g & 1 ? all : below;
          if (i % 2 == 1 || i == SEG - 1) {  // the pair's stores
            const int xp = x0 + 16 * (i & ~1) + r + px;
            const float q = (g & 1) && i % 2 == 1 ? pv[i] : pv[i & ~1];
            if (done && yo < H && xp < W && (SEG > 1 || !(g & 1)))
              ((PT *)ep.p)[ep.off + row + xp] =
                  (PT)(ep.scale * (q + hb)) * (PT)bv[i / 2];
          }
        } else if (in_row) {
          *reinterpret_cast<uint2 *>(ep.y + (row + xo) * 8 + 4 * (g & 1)) = w2;
        }
#pragma unroll
        for (int s = 0; s < S; ++s)
          acc[i][s][(j + 1) % 3] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      if constexpr (kCells) {
        // the last plane of a row of cells: sums over 4 x (lanes), over a
        // wave's two rows where lanes hold them apart, and over the rows of a
        // pair of waves (LDS), in a fixed order
        if (done && (z & (kPool - 1)) == kPool - 1) {  // uniform
#pragma unroll
          for (int i = 0; i < SEG; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              csum[i][e] += __shfl_xor(csum[i][e], 1, 64);
              csum[i][e] += __shfl_xor(csum[i][e], 2, 64);
              if constexpr (EPI == kEpiPool)
                csum[i][e] += __shfl_xor(csum[i][e], 32, 64);
            }
            if ((wv & 1) && (r & 3) == 0)
              *reinterpret_cast<f32x4 *>(&cells[wv >> 1][i][4 * (4 * g + (r >> 2))]) =
                  csum[i];
          }
          __syncthreads();
          if (!(wv & 1)) {
            const int Wc = W / kPool;
            const long crow = (((long)n * (D / kPool) + z / kPool) *
                                   (H / kPool) + yw / kPool) * Wc;
#pragma unroll
            for (int i = 0; i < SEG; ++i) {
              const int xo = x0 + 16 * i + r;
              if ((r & 3) == 0 && xo < W && yw < H) {
                const f32x4 v = csum[i] + *reinterpret_cast<const f32x4 *>(
                    &cells[wv >> 1][i][4 * (4 * g + (r >> 2))]);
                if constexpr (EPI == kEpiPool) {
                  constexpr float q = 1.0f / (kPool * kPool * kPool);
                  if (g < 2)
                    *reinterpret_cast<uint2 *>(
                        ep.coarse + (crow + xo / kPool) * 8 + 4 * g) =
                        make_uint2(Pack2(q * v[0], q * v[1]),
                                   Pack2(q * v[2], q * v[3]));
                } else {
                  const long o = (crow + xo / kPool) * 16 + 4 * g;
                  const uint2 a = *reinterpret_cast<const uint2 *>(ep.act + o);
                  *reinterpret_cast<uint2 *>(ep.coarse + o) =
                      make_uint2(GateWord(Pack2(v[0], v[1]), a.x),
                                 GateWord(Pack2(v[2], v[3]), a.y));
                }
              }
            }
          }
#pragma unroll
          for (int i = 0; i < SEG; ++i) csum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
      in.Put(ring + ((m + 1) & 1) * PLANE);
      __syncthreads();
      in.Fetch(src, n, zp + 2, D, H, W);
    }
  }
}

// Filter gradient partials marching the input planes: block (x tile, y
// tile, problem, z chunk [zb, ze) of output-gradient planes) sums over its
// XT x ROWS x zchunk positions
//   part[block][co][k] = sum_p dz[p][co] x[p + off(k)][ci],  k = tap CIN + ci
// as a GEMM over positions (K) on v_mfma_f32_16x16x32_bf16.  Step z' uses
// input plane z' (2 slots) for the three taps whose z offset t - 1 maps it
// to output-gradient plane z' + 1 - t (t = 0, 1, 2; planes outside [zb, ze)
// stage as zeros, ring of 4).  Both are staged channels-last, as they lie in
// memory, and the transposing LDS read (ds_read_b64_tr_b16: four positions of
// 16 channels per 16 lanes, each lane's address its own) makes the operands:
// the shift of a tap is an address, and 16 columns may be any four runs of
// four channels.  B columns (3 dy + dx) CIN + ci, then a column of ones (the
// bias gradient); A rows (t, co), q = t COUT + co, so that one B operand
// feeds every t.  CIN is the staged channel count: 4 for the network input
// (2 of them real), whose other weights of WC = 8 get zero gradients.
// Waves split into WT groups over column tiles and NW / WT over the steps of
// 32 positions of a plane; the step groups' sums are added in a fixed order
// at the end (deterministic).  One barrier per step.
// The version it replaces stored both operands transposed, 2 bytes at a time,
// and shifted B by register: at 8 x 128^3 24 -> 8 took 471 us, now 249, and
// 8 -> 8 207, now 122 (92 us of bytes); rows that are not multiples of 32 ran
// on a kernel that gathered its operands 2 bytes at a time.
// An input that is not finite times the zeros of gradient planes outside a chunk
// is NaN: gradients of taps that lead out of the grid are then NaN too (as they
// were for rows of multiples of 32).
__device__ __forceinline__ bf16x8 ReadTr(const u16 *a, const u16 *b) {
  typedef __attribute__((address_space(3))) s16x4 *P;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)a);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)b);
  return __builtin_bit_cast(
      bf16x8, s16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
}

template <int CIN, int WC, int COUT, int XT, int ROWS, int NW, int WT,
          template <int, int, int, int> class SRC>
__global__ __launch_bounds__(64 * NW) void WgradZKernel(
    SrcArgs src, const u16 *__restrict__ dz, float *__restrict__ part,
    float *__restrict__ bpart, int D, int H, int W, int tz, int zchunk) {
  static_assert(XT % 32 == 0, "steps of 32 positions along x");
  static_assert(NW % WT == 0, "wave groups");
  constexpr int K = 27 * WC, NC = 9 * CIN;
  constexpr int NTN = (NC + 16) / 16;       // column tiles (with the ones)
  constexpr int MM = (3 * COUT + 15) / 16;  // MFMAs per B operand
  constexpr int WS = NW / WT;               // step groups
  constexpr int TPW = (NTN + WT - 1) / WT;  // column tiles per wave
  constexpr int NSTEP = ROWS * XT / 32;     // 32-position steps per plane
  static_assert(NSTEP % WS == 0, "steps split evenly");
  constexpr int XR = XT + 2, RS = ROWS + 2, NTH = 64 * NW;
  constexpr int XPL = RS * XR * CIN;        // u16 per staged x plane
  constexpr int DPL = ROWS * XT * COUT;     // u16 per staged dz plane
  constexpr int DV = DPL / 8, DVT = (DV + NTH - 1) / NTH;
  constexpr int LOOP_WORDS = (2 * XPL + 4 * DPL) / 2;
  constexpr int RED_WORDS = (WS - 1) * WT * TPW * MM * 4 * 64;
  constexpr int LDS_WORDS = LOOP_WORDS > RED_WORDS ? LOOP_WORDS : RED_WORDS;
  __shared__ __attribute__((aligned(16))) unsigned lds[LDS_WORDS];
  u16 *const xs = reinterpret_cast<u16 *>(lds);
  u16 *const ds = xs + 2 * XPL;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wt = wv % WT, ws = wv / WT;
  const int g = lane >> 4, r = lane & 15;
  const int tiles_x = (W + XT - 1) / XT, tiles_y = (H + ROWS - 1) / ROWS;
  const long bid = physis_hip::XcdLogicalBlock(blockIdx.x, gridDim.x);
  int b = (int)bid;
  const int x0 = (b % tiles_x) * XT;
  b /= tiles_x;
  const int y0 = (b % tiles_y) * ROWS;
  b /= tiles_y;
  const int n = b / tz, zb = (b - n * tz) * zchunk;
  const int ze = min(zb + zchunk, D);
  // What this lane addresses in a transposing read: position 8g + (r >> 2)
  // (+ 4 in the second half) of the step, and four columns from 4 (r & 3).
  const int pos = 8 * g + (r >> 2), c4 = 4 * (r & 3);
  int lofs[TPW];  // element offset of (step position 0, the lane's columns)
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    int col = (wt + WT * i) * 16 + c4;
    col = col < NC ? col : 0;  // (columns past the last are not used)
    const int o = col / CIN, ci = col - o * CIN;
    lofs[i] = ((o / 3) * XR + o % 3 + pos) * CIN + ci;
  }
  int at[MM], aofs[MM];  // z tap and offset of the lane's A rows
#pragma unroll
  for (int m = 0; m < MM; ++m) {
    const int q = 16 * m + c4;
    at[m] = q < 3 * COUT ? q / COUT : 2;  // (rows past the last: not used)
    aofs[m] = pos * COUT + q % COUT;
  }
  f32x4 acc[TPW][MM];
#pragma unroll
  for (int i = 0; i < TPW; ++i)
#pragma unroll
    for (int m = 0; m < MM; ++m) acc[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (zb < ze) {
    SRC<CIN, RS, XR, NTH> in;
    in.Init(y0, x0, H, W);
    // output-gradient plane zz (zeros outside [zb, ze))
    uint4 bd[DVT];
    unsigned doff[DVT];  // from row y0
    const unsigned dbytes = RowBytes(y0, ROWS, H, W, COUT);
#pragma unroll
    for (int i = 0; i < DVT; ++i) {
      const int v = threadIdx.x + i * NTH, t = v / (COUT / 8);
      const int yy = y0 + t / XT, xx = x0 + t % XT;
      doff[i] = v < DV && yy < H && xx < W
                    ? ((unsigned)(t / XT * W + xx) * COUT + v % (COUT / 8) * 8) * 2
                    : kOutside;
    }
    auto fetchd = [&](int zz) {
      const bool ok = zz >= zb && zz < ze;
      const long row = ((long)n * D + zz) * H + y0;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<u16 *>(dz) + (ok ? row * W * COUT : 0), 0, ok ? dbytes : 0,
          physis_hip::kBufDword3);
#pragma unroll
      for (int i = 0; i < DVT; ++i)
        bd[i] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, doff[i], 0, 0));
    };
    auto putd = [&](int slot) {
#pragma unroll
      for (int i = 0; i < DVT; ++i) {
        const int v = threadIdx.x + i * NTH;
        if (v < DV)
          *reinterpret_cast<uint4 *>(ds + slot * DPL + v * 8) = bd[i];
      }
    };
    // x plane zz in slot (zz - zb + 1) & 1, dz plane zz in (zz - zb + 2) & 3
    in.Fetch(src, n, zb - 1, D, H, W);
    in.Put(xs);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      fetchd(zb - 2 + k);
      putd(k);
    }
    in.Fetch(src, n, zb, D, H, W);
    fetchd(zb + 1);
    __syncthreads();
    for (int zp = zb - 1; zp <= ze; ++zp) {
      const int k = zp - zb + 1;  // dz plane zp + 1 - t in slot (k + 2 - t) & 3
      const u16 *const xp = xs + (k & 1) * XPL;
#pragma unroll
      for (int j = 0; j < NSTEP / WS; ++j) {
        const int st = (ws * (NSTEP / WS) + j) * 32;  // first position
        const int ry = st / XT, rx = st - ry * XT;
        bf16x8 a[MM];
#pragma unroll
        for (int m = 0; m < MM; ++m) {
          const u16 *p =
              ds + ((k + 2 - at[m]) & 3) * DPL + st * COUT + aofs[m];
          a[m] = ReadTr(p, p + 4 * COUT);
        }
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
          if (wt + WT * i >= NTN) break;  // wave-uniform
          const u16 *p = xp + (ry * XR + rx) * CIN + lofs[i];
          bf16x8 o = ReadTr(p, p + 4 * CIN);
          if (wt + WT * i == NC / 16 && r == NC % 16)  // the column of ones
            o = __builtin_bit_cast(
                bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u,
                                   0x3f803f80u));
#pragma unroll
          for (int m = 0; m < MM; ++m)
            acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], o,
                                                                acc[i][m], 0,
                                                                0, 0);
        }
      }
      // x plane zp + 1 and dz plane zp + 2 into the slots no wave reads in
      // this step (x: plane zp - 1, dz: plane zp - 2)
      in.Put(xs + ((k + 1) & 1) * XPL);
      putd((k + 3) & 3);
      __syncthreads();
      in.Fetch(src, n, zp + 2, D, H, W);
      fetchd(zp + 3);
    }
  }
  // step groups 1 .. WS-1 hand their sums to group 0 through LDS
  if constexpr (WS > 1) {
    __syncthreads();  // the staged planes are no longer read
    float *red = reinterpret_cast<float *>(lds);
    constexpr int PER = TPW * MM * 4;  // floats per lane and wave
    if (ws > 0) {
      float *o = red + ((ws - 1) * WT + wt) * PER * 64;
#pragma unroll
      for (int i = 0; i < TPW; ++i)
#pragma unroll
        for (int m = 0; m < MM; ++m)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            o[((i * MM + m) * 4 + v) * 64 + lane] = acc[i][m][v];
    }
    __syncthreads();
    if (ws == 0) {
      for (int u = 1; u < WS; ++u) {
        const float *o = red + ((u - 1) * WT + wt) * PER * 64;
#pragma unroll
        for (int i = 0; i < TPW; ++i)
#pragma unroll
          for (int m = 0; m < MM; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              acc[i][m][v] += o[((i * MM + m) * 4 + v) * 64 + lane];
      }
    }
  }
  if (ws == 0) {
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int col = (wt + WT * i) * 16 + r;
      if (wt + WT * i >= NTN || col > NC) continue;
      const int o = col / CIN, ci = col - o * CIN;
#pragma unroll
      for (int m = 0; m < MM; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int q = 16 * m + 4 * g + v;
          if (q >= 3 * COUT) continue;
          const int t = q / COUT, co = q - t * COUT;
          if (col == NC) {
            if (t == 1) bpart[bid * COUT + co] = acc[i][m][v];
          } else if (CIN == WC) {
            part[(bid * COUT + co) * K + 9 * t * CIN + col] = acc[i][m][v];
          } else {  // 2 real channels of WC
            float *w = part + (bid * COUT + co) * K + (9 * t + o) * WC;
            w[ci < 2 ? ci : ci * 3 - 4] = ci < 2 ? acc[i][m][v] : 0.0f;
            if (ci >= 2) w[ci * 3 - 3] = w[ci * 3 - 2] = 0.0f;
          }
        }
    }
  }
}

// Deterministic sums over blocks: out[i] = sum_b part[b][i] for i < n, and
// out2[i] = sum_b part2[b][i] for i < n2.  A block owns 64 columns; its 16
// waves sum an equal run of the blocks each, in order, then the runs are
// added in order.
constexpr int kSumWaves = 16;
__global__ __launch_bounds__(64 * kSumWaves) void SumPartsKernel(
    const float *__restrict__ part, long n, float *__restrict__ out,
    const float *__restrict__ part2, long n2, float *__restrict__ out2,
    int nparts) {
  __shared__ float red[kSumWaves][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const long nb = (n + 63) / 64;  // blocks of the first sum
  const bool second = (long)blockIdx.x >= nb;
  const float *p = second ? part2 : part;
  const long m = second ? n2 : n;
  const long i = ((long)blockIdx.x - (second ? nb : 0)) * 64 + lane;
  const int run = (nparts + kSumWaves - 1) / kSumWaves;
  const int b0 = wv * run, b1 = b0 + run < nparts ? b0 + run : nparts;
  float s = 0.0f;
  if (i < m) {
#pragma unroll 8
    for (int b = b0; b < b1; ++b) s += p[b * m + i];
  }
  red[wv][lane] = s;
  __syncthreads();
  if (wv == 0 && i < m) {
    for (int k = 1; k < kSumWaves; ++k) s += red[k][lane];
    (second ? out2 : out)[i] = s;
  }
}

// ------------------------------------------------------ elementwise layers
// Threads own 8 consecutive channels (one 16-byte vector) of one position;
// positions are decoded with 32-bit arithmetic (< 2^31 positions).
struct V8 {
  float v[8];
};
__device__ __forceinline__ V8 Load8F(const u16 *p) {
  const uint4 u = *reinterpret_cast<const uint4 *>(p);
  const unsigned w[4] = {u.x, u.y, u.z, u.w};
  V8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r.v[2 * i] = __uint_as_float(w[i] << 16);
    r.v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
  return r;
}
__device__ __forceinline__ void Store8F(u16 *p, const V8 &r) {
  unsigned w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w[i] = (unsigned)F2Bf(r.v[2 * i]) | ((unsigned)F2Bf(r.v[2 * i + 1]) << 16);
  *reinterpret_cast<uint4 *>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

struct Pos {
  int n, z, y, x;
};
__device__ __forceinline__ Pos Decode(int p, int D, int H, int W) {
  Pos r;
  r.x = p % W;
  p /= W;
  r.y = p % H;
  p /= H;
  r.z = p % D;
  r.n = p / D;
  return r;
}

// 4x4x4 average pool: out[coarse][c] = (FP32 sum of the 64 inputs) / 64.
__global__ void PoolKernel(const u16 *__restrict__ in, u16 *__restrict__ out,
                           int C, int Dc, int Hc, int Wc, int total) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int G = C / 8;
  if (i >= total) return;
  const int gi = i % G;
  const Pos q = Decode(i / G, Dc, Hc, Wc);
  const int D = Dc * kPool, H = Hc * kPool, W = Wc * kPool;
  V8 s;
#pragma unroll
  for (int k = 0; k < 8; ++k) s.v[k] = 0.0f;
  for (int dz = 0; dz < kPool; ++dz)
    for (int dy = 0; dy < kPool; ++dy)
      for (int dx = 0; dx < kPool; ++dx) {
        const long f = (((long)q.n * D + q.z * kPool + dz) * H + q.y * kPool +
                        dy) * W + q.x * kPool + dx;
        const V8 a = Load8F(in + f * C + gi * 8);
#pragma unroll
        for (int k = 0; k < 8; ++k) s.v[k] += a.v[k];
      }
#pragma unroll
  for (int k = 0; k < 8; ++k) s.v[k] *= (1.0f / 64.0f);
  Store8F(out + (long)i * 8, s);
}

// out[fine p][0:CA] = coarse[p / 4][0:CA]; out[p][CA:CA+CB] = skip[p].
__global__ void UpConcatKernel(const u16 *__restrict__ coarse,
                               const u16 *__restrict__ skip,
                               u16 *__restrict__ out, int CA, int CB, int D,
                               int H, int W, int total) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int G = (CA + CB) / 8, GA = CA / 8;
  if (i >= total) return;
  const int gi = i % G, p = i / G;
  uint4 v;
  if (gi >= GA) {
    v = *reinterpret_cast<const uint4 *>(skip + (long)p * CB + (gi - GA) * 8);
  } else {
    const Pos q = Decode(p, D, H, W);
    const int Dc = D / kPool, Hc = H / kPool, Wc = W / kPool;
    const long c = (((long)q.n * Dc + q.z / kPool) * Hc + q.y / kPool) * Wc +
                   q.x / kPool;
    v = *reinterpret_cast<const uint4 *>(coarse + c * CA + gi * 8);
  }
  *reinterpret_cast<uint4 *>(out + (long)i * 8) = v;
}

// Gradient of the upsampled part of a concatenation: gc[coarse][c] = FP32
// sum over the 64 fine positions of g[fine][c], c < CA of C channels, gated
// by the coarse activation.
__global__ void UpBackKernel(const u16 *__restrict__ g,
                             const u16 *__restrict__ act,
                             u16 *__restrict__ gc, int CA, int C, int Dc,
                             int Hc, int Wc, int total) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int GA = CA / 8;
  if (i >= total) return;
  const int gi = i % GA;
  const Pos q = Decode(i / GA, Dc, Hc, Wc);
  const int D = Dc * kPool, H = Hc * kPool, W = Wc * kPool;
  V8 s;
#pragma unroll
  for (int k = 0; k < 8; ++k) s.v[k] = 0.0f;
  for (int dz = 0; dz < kPool; ++dz)
    for (int dy = 0; dy < kPool; ++dy)
      for (int dx = 0; dx < kPool; ++dx) {
        const long f = (((long)q.n * D + q.z * kPool + dz) * H + q.y * kPool +
                        dy) * W + q.x * kPool + dx;
        const V8 a = Load8F(g + f * C + gi * 8);
#pragma unroll
        for (int k = 0; k < 8; ++k) s.v[k] += a.v[k];
      }
  const V8 a = Load8F(act + (long)i * 8);
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (!(a.v[k] > 0.0f)) s.v[k] = 0.0f;
  Store8F(gc + (long)i * 8, s);
}

// dz[p][c] = (gpool[p/4][c] / 64 + gskip[p][CA + c]) if act[p][c] > 0 else 0:
// the gradient reaching a pooled encoder output through its pool and its
// skip connection (gskip: the concatenation gradient, CA + CB channels),
// gated by its ReLU.  FP32 sum, one rounding.
__global__ void PoolBackSkipGateKernel(const u16 *__restrict__ gpool,
                                       const u16 *__restrict__ gskip,
                                       const u16 *__restrict__ act,
                                       u16 *__restrict__ dz, int CB, int CA,
                                       int D, int H, int W, int total) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int G = CB / 8;
  if (i >= total) return;
  const int gi = i % G, p = i / G;
  const Pos q = Decode(p, D, H, W);
  const int Dc = D / kPool, Hc = H / kPool, Wc = W / kPool;
  const long c = (((long)q.n * Dc + q.z / kPool) * Hc + q.y / kPool) * Wc +
                 q.x / kPool;
  const V8 gp = Load8F(gpool + c * CB + gi * 8);
  const V8 gs = Load8F(gskip + (long)p * (CA + CB) + CA + gi * 8);
  const V8 a = Load8F(act + (long)i * 8);
  V8 o;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    o.v[k] = a.v[k] > 0.0f ? gp.v[k] * (1.0f / 64.0f) + gs.v[k] : 0.0f;
  Store8F(dz + (long)i * 8, o);
}

// 1x1 convolution 8 -> 1: out[p] = sum_c w[c] in[p][c] + b (FP32), for the
// cell means of the smooth loss terms.
__global__ void HeadKernel(const u16 *__restrict__ in,
                           const float *__restrict__ w,
                           float *__restrict__ out, long P) {
  const long p = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (p >= P) return;
  const V8 a = Load8F(in + p * 8);
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < 8; ++c) s += w[c] * a.v[c];
  out[p] = s + w[8];
}

// Smooth-error terms of the loss.  The error d = out - target * inv_scale
// averaged over the 4x4x4 cells of the pooling grid: one wave per cell
// (lane l at offset (l & 3, (l >> 2) & 3, l >> 4)), summed across the wave
// in a fixed order.  e4 has the level-2 layout ((n D2 + Z) H2 + Y) W2 + X.
__global__ __launch_bounds__(256) void SmoothCellKernel(
    const float *__restrict__ out, const float *__restrict__ target,
    long toff, float inv_scale, float *__restrict__ e4, int D1, int H1,
    int W1, long P2) {
  const long c = (blockIdx.x * (long)blockDim.x + threadIdx.x) >> 6;
  const int l = threadIdx.x & 63;
  if (c >= P2) return;  // uniform over the wave
  const int W2 = W1 / kPool, H2 = H1 / kPool, D2 = D1 / kPool;
  const int X = (int)(c % W2), Y = (int)((c / W2) % H2);
  const long nz = c / ((long)W2 * H2);  // n D2 + Z
  const long n = nz / D2, Z = nz - n * D2;
  const long p = ((n * D1 + Z * kPool + (l >> 4)) * H1 + Y * kPool +
                  ((l >> 2) & 3)) * W1 + X * kPool + (l & 3);
  float v = out[p] - target[toff + p] * inv_scale;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  if (l == 0) e4[c] = v * (1.0f / 64.0f);
}

// e16: the means of e4 over 4x4x4 cells of the level-2 grid (the error
// averaged over 16x16x16 cells), one thread per cell, summed z-y-x.
__global__ void SmoothCoarseKernel(const float *__restrict__ e4,
                                   float *__restrict__ e16, int D2, int H2,
                                   int W2, long P3) {
  const long c = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (c >= P3) return;
  const int W3 = W2 / kPool, H3 = H2 / kPool, D3 = D2 / kPool;
  const int X = (int)(c % W3), Y = (int)((c / W3) % H3);
  const long nz = c / ((long)W3 * H3);
  const long n = nz / D3, Z = nz - n * D3;
  float s = 0.0f;
  for (int dz = 0; dz < kPool; ++dz)
    for (int dy = 0; dy < kPool; ++dy)
      for (int dx = 0; dx < kPool; ++dx)
        s += e4[((n * D2 + Z * kPool + dz) * H2 + Y * kPool + dy) * W2 +
                X * kPool + dx];
  e16[c] = s * (1.0f / 64.0f);
}

// Head, loss, and the head's backward in one pass over the last layer's
// activations `in`: out = w . in + b (1x1 convolution 8 -> 1, FP32),
// d = out - target * inv_scale, and with e4 / e16 the means of d over the
// point's 4^3 / 16^3 cell
//   loss = (1/P) sum_p (d^2 + w4 e4^2 + w16 e16^2)
//        = mean d^2 + w4 mean over 4^3 cells e4^2 + w16 mean e16^2,
//   dout = 2 (d + w4 e4 + w16 e16) / P,
// din[p][c] = w[c] dout[p] gated by in (BF16), and per-block partials of the
// loss, dw[c] = sum dout[p] in[p][c] and db = sum dout[p].  SMOOTH false:
// w4 = w16 = 0 (e4, e16 unused).  Bound by its 36 bytes per point (in,
// target, din); as three passes (head, loss, head backward with 2-byte
// loads) it took 364 us at 8 x 128^3.
constexpr int kHeadThreads = 512;
template <bool SMOOTH>
__global__ __launch_bounds__(kHeadThreads) void HeadLossBackKernel(
    const u16 *__restrict__ in, const float *__restrict__ w,
    const float *__restrict__ target, long toff, float inv_scale,
    const float *__restrict__ e4, const float *__restrict__ e16, float w4,
    float w16, int D1, int H1, int W1, u16 *__restrict__ din,
    double *__restrict__ lpart, float *__restrict__ part, long P) {
  __shared__ double lred[kHeadThreads / 64];
  __shared__ float red[9][kHeadThreads / 64];
  float wc[9], acc[9];
#pragma unroll
  for (int c = 0; c < 9; ++c) {
    wc[c] = w[c];
    acc[c] = 0.0f;
  }
  double s = 0.0;
#pragma unroll 2
  for (long p = blockIdx.x * (long)kHeadThreads + threadIdx.x; p < P;
       p += (long)gridDim.x * kHeadThreads) {
    const V8 a = Load8F(in + p * 8);
    float o = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) o += wc[c] * a.v[c];
    o += wc[8];
    const float d = o - target[toff + p] * inv_scale;
    float g;
    if constexpr (SMOOTH) {
      const int x = (int)(p % W1), y = (int)((p / W1) % H1);
      const long nz = p / ((long)W1 * H1);
      const long n = nz / D1, z = nz - n * D1;
      const int W2 = W1 / kPool, H2 = H1 / kPool, D2 = D1 / kPool;
      const long c2 = ((n * D2 + z / kPool) * H2 + y / kPool) * W2 +
                      x / kPool;
      const int W3 = W2 / kPool, H3 = H2 / kPool, D3 = D2 / kPool;
      const long c3 = ((n * D3 + z / (kPool * kPool)) * H3 +
                       y / (kPool * kPool)) * W3 + x / (kPool * kPool);
      const float m4 = e4[c2], m16 = e16[c3];
      g = 2.0f * (d + w4 * m4 + w16 * m16) / (float)P;
      s += (double)d * d + (double)w4 * m4 * m4 + (double)w16 * m16 * m16;
    } else {
      g = 2.0f * d / (float)P;
      s += (double)d * d;
    }
    float v[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      acc[c] += g * a.v[c];
      v[c] = a.v[c] > 0.0f ? wc[c] * g : 0.0f;
    }
    acc[8] += g;
    *reinterpret_cast<uint4 *>(din + p * 8) =
        make_uint4(Pack2(v[0], v[1]), Pack2(v[2], v[3]), Pack2(v[4], v[5]),
                   Pack2(v[6], v[7]));
  }
  s = physis_hip::BlockReduce<double, PS_SUM, kHeadThreads>(s, lred);
  if (threadIdx.x == 0) lpart[blockIdx.x] = s;
#pragma unroll
  for (int c = 0; c < 9; ++c) {
    const float t =
        physis_hip::BlockReduce<float, PS_SUM, kHeadThreads>(acc[c], red[c]);
    if (threadIdx.x == 0) part[blockIdx.x * 9 + c] = t;
  }
}

// Weights: wt[co][k] = bf16(W[co][k]) (zero for k >= 27 cin) and the
// flipped, transposed wf[ci][tap' cout + co] = bf16(W[co][26 - tap'][ci]).
__global__ void PackKernel(const float *__restrict__ w, u16 *__restrict__ wt,
                           u16 *__restrict__ wf, int cin, int cout) {
  const int K = 27 * cin, kp = KPad(cin), kf = KPad(cout);
  const int n1 = cout * kp, n2 = cin * kf;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n1 + n2;
       i += gridDim.x * blockDim.x) {
    if (i < n1) {
      const int co = i / kp, k = i - co * kp;
      wt[i] = k < K ? F2Bf(w[co * K + k]) : (u16)0;
    } else {
      const int j = i - n1, ci = j / kf, k = j - ci * kf;
      u16 v = 0;
      if (k < 27 * cout) {
        const int tp = k / cout, co = k - tp * cout;
        v = F2Bf(w[co * K + (26 - tp) * cin + ci]);
      }
      wf[j] = v;
    }
  }
}

// Reflected copy of whole problems: dst problem q' = dst_first + q holds
// src problem first + q with the axes whose bit is set in `flips` (1 x,
// 2 y, 4 z) reversed inside the problem.
__global__ void ReflectKernel(const float *__restrict__ src,
                              float *__restrict__ dst, int nx, int ny,
                              int nzs, long soff, long doff, int flips,
                              long n) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long m = (long)nx * ny * nzs;
  const long q = i / m;
  long r = i - q * m;
  const int z = (int)(r / ((long)nx * ny));
  r -= (long)z * nx * ny;
  const int y = (int)(r / nx), x = (int)(r - (long)y * nx);
  const int sx = flips & 1 ? nx - 1 - x : x;
  const int sy = flips & 2 ? ny - 1 - y : y;
  const int sz = flips & 4 ? nzs - 1 - z : z;
  dst[doff + i] = src[soff + q * m + ((long)sz * ny + sy) * nx + sx];
}

__global__ void AdamKernel(float *__restrict__ p, const float *__restrict__ g,
                           float *__restrict__ m, float *__restrict__ v,
                           long n, float lr, float c1, float c2) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = 0.9f * m[i] + 0.1f * gi;
  const float vi = 0.999f * v[i] + 0.001f * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}

// ------------------------------------------------------------ dispatch
hipStream_t Stream() { return (hipStream_t)__PSHipStream(); }
void Check() { PS_HIP_CHECK(hipGetLastError()); }
unsigned Blocks(long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

// Blocks per compute unit that the ring convolutions and the filter gradient
// aim for: what their registers and LDS let reside at level 1.
constexpr int kConvZBlocksPerCU = 2;
constexpr int kWgradZBlocksPerCU = 2;

// z chunks of a z-marching launch: enough blocks for per_cu per compute
// unit over `tiles` xy tiles of N problems of D planes.
void ZChunks(long tiles, int N, int D, int per_cu, int *tz, int *zchunk) {
  const long want = (long)per_cu * __PSHipNumCUs();
  long t = (want + tiles * N - 1) / (tiles * N);
  if (t < 1) t = 1;
  if (t > D) t = D;
  *zchunk = (int)((D + t - 1) / t);
  *tz = (D + *zchunk - 1) / *zchunk;
}

// The rows of a plane that a block reads through one buffer descriptor.
void CheckRows(int rows, int H, int W, int channels) {
  const long bytes = (long)std::min(rows, H) * W * channels * 2;
  if (bytes > (long)kReach)
    PS_FATAL("convolution: %d rows of %d positions of %d channels exceed the "
             "reach of a buffer descriptor", std::min(rows, H), W, channels);
}

template <int CIN, int COUT, int XT, int TY>
void ConvZLaunch(const u16 *x, const u16 *wt, const float *b, bool relu,
                 const u16 *act, u16 *y, int N, int D, int H, int W) {
  const int tiles = ((W + XT - 1) / XT) * ((H + TY - 1) / TY);
  int tz, zchunk;
  ZChunks(tiles, N, D, kConvZBlocksPerCU, &tz, &zchunk);
  const dim3 grid(tiles, N * tz), block(64 * TY);
  const auto kernel = relu  ? ConvZKernel<CIN, COUT, true, false, XT, TY>
                      : act ? ConvZKernel<CIN, COUT, false, true, XT, TY>
                            : ConvZKernel<CIN, COUT, false, false, XT, TY>;
  hipLaunchKernelGGL(kernel, grid, block, 0, Stream(), x, wt, b, act, y, D, H,
                     W, tz, zchunk);
  Check();
}

// The input-marching convolution.  Block shapes
// (XT positions by 2 TY rows) measured at 8 x 128^3, us, of 64x8, 32x8, 64x16
// and 32x16: plain 8 -> 8 115 / 102 / 131 / 109; gated 164 / 216 / 177 / 150;
// prediction 202 / 228 / 201 / 143; network input (a whole prediction) 731 /
// 736 / 741 / 736; 24 -> 8 (32x8, 32x16) 234 / 267; 8 -> 24 with cell sums 401
// / 288.  Other sizes take the same shapes unmeasured, but rows of at most 16
// positions XT = 16.
constexpr int kConvMWavesPerCU = 16;
template <int CIN, int COUT, bool RELU, int XT, int TY,
          template <int, int, int, int> class SRC, int EPI, typename PT>
void ConvMLaunchXT(const SrcArgs &src, const u16 *wt, const EpiArgs &ep, int N,
                   int D, int H, int W) {
  static_assert(EPI != kEpiPredict || XT == 16 || XT % 32 == 0, "pairs");
  CheckRows(2 * TY + 2, H, W, CIN);
  const long tiles = (long)((W + XT - 1) / XT) * ((H + 2 * TY - 1) / (2 * TY));
  int tz, zchunk;
  ZChunks(tiles, N, D, kConvMWavesPerCU / TY, &tz, &zchunk);
  if (EPI == kEpiPool || EPI == kEpiUpSkip) {  // whole cells
    zchunk = (zchunk + kPool - 1) / kPool * kPool;
    tz = (D + zchunk - 1) / zchunk;
  }
  hipLaunchKernelGGL((ConvMKernel<CIN, COUT, RELU, XT, TY, SRC, EPI, PT>),
                     dim3((unsigned)(tiles * N * tz)), dim3(64 * TY), 0,
                     Stream(), src, wt, ep, D, H, W, tz, zchunk);
  Check();
}
template <int CIN, int COUT, bool RELU,
          template <int, int, int, int> class SRC, int EPI,
          typename PT = double>
void ConvMLaunch(const SrcArgs &src, const u16 *wt, const EpiArgs &ep, int N,
                 int D, int H, int W) {
  constexpr int XT = CIN == 2 ? 64 : 32;
  constexpr int TY = COUT == 24 || EPI == kEpiGate || EPI == kEpiPredict ? 8 : 4;
  if (W > 16)
    ConvMLaunchXT<CIN, COUT, RELU, XT, TY, SRC, EPI, PT>(src, wt, ep, N, D, H,
                                                         W);
  else
    ConvMLaunchXT<CIN, COUT, RELU, 16, 4, SRC, EPI, PT>(src, wt, ep, N, D, H,
                                                        W);
}

// A convolution of whole tensors; act: gate of the results, or NULL.  8 output
// channels march the input planes (ConvMKernel); more keep the ring of planes:
// x tile of 64 positions below 24 input channels, else 32, 16 for rows of at
// most 16; 8 rows per block below 24 input channels, else 4 (the ring of 4
// staged planes then stays within LDS).
template <int CIN, int COUT>
void ConvT(const u16 *x, const u16 *wt, const float *b, bool relu,
           const u16 *act, u16 *y, int N, int D, int H, int W) {
  if constexpr (COUT == 8) {
    SrcArgs src{x, nullptr, 0};
    EpiArgs ep;
    ep.bias = b;
    ep.act = act;
    ep.y = y;
    if (act)
      ConvMLaunch<CIN, 8, false, PlainSrc, kEpiGate>(src, wt, ep, N, D, H, W);
    else if (relu)
      ConvMLaunch<CIN, 8, true, PlainSrc, kEpiStore>(src, wt, ep, N, D, H, W);
    else
      ConvMLaunch<CIN, 8, false, PlainSrc, kEpiStore>(src, wt, ep, N, D, H, W);
  } else {
    constexpr int TY = CIN < 24 ? 8 : 4;
    if constexpr (CIN < 24) {
      if (W > 32)
        return ConvZLaunch<CIN, COUT, 64, TY>(x, wt, b, relu, act, y, N, D, H,
                                              W);
    }
    if (W > 16)
      ConvZLaunch<CIN, COUT, 32, TY>(x, wt, b, relu, act, y, N, D, H, W);
    else
      ConvZLaunch<CIN, COUT, 16, TY>(x, wt, b, relu, act, y, N, D, H, W);
  }
}

// Launch shape of the filter gradient: x tile 64 when the rows are multiples
// of 64 and the input has at most 24 channels, else 32 (positions past a
// row's end stage as zeros).
// Returns the block count (= partials).
constexpr int WgradZRows(int cin) { return cin <= 8 ? 8 : 4; }
constexpr int kWgradZWaves = 4;
// Wave groups over the column tiles (9 cin / 16 of them): one up to 5
// tiles, two up to 14, else four (the rest of the waves split the steps).
constexpr int WgradZGroups(int cin) {
  return (9 * cin + 16) / 16 <= 5 ? 1 : ((9 * cin + 16) / 16 <= 14 ? 2 : 4);
}
int WgradZXT(int cin, int W) { return (W % 64 == 0 && cin <= 24) ? 64 : 32; }
long WgradZBlocks(int cin, int N, int D, int H, int W, int *tz, int *zchunk) {
  const int xt = WgradZXT(cin, W);
  const long tiles = (long)((W + xt - 1) / xt) *
                     ((H + WgradZRows(cin) - 1) / WgradZRows(cin));
  ZChunks(tiles, N, D, kWgradZBlocksPerCU, tz, zchunk);
  return tiles * N * *tz;
}

// Partials (blocks) of a filter-gradient launch over N problems of
// D x H x W positions with cin input channels: every buffer of partials is
// sized by this.
long WgradBlocks(int cin, int N, int D, int H, int W) {
  int tz, zchunk;
  return WgradZBlocks(cin, N, D, H, W, &tz, &zchunk);
}

// The filter gradient of a layer with CIN input channels (SC staged: 4 for the
// network input) into part / bpart, which hold `capacity` blocks of partials;
// *nparts receives the blocks written.
template <int SC, int CIN, int COUT,
          template <int, int, int, int> class SRC>
void WgradZLaunch(const SrcArgs &src, const u16 *dz, float *part, float *bpart,
                  int N, int D, int H, int W, long capacity, int *nparts) {
  const long P = (long)N * D * H * W;
  if (P >= 1L << 31)
    PS_FATAL("filter gradient: %ld positions exceed 32-bit indexing", P);
  int tz, zchunk;
  const long nb = WgradZBlocks(CIN, N, D, H, W, &tz, &zchunk);
  if (nb > capacity)
    PS_FATAL("filter gradient: %ld partial blocks exceed the %ld allocated",
             nb, capacity);
  constexpr int R = WgradZRows(CIN), NW = kWgradZWaves;
  CheckRows(R + 2, H, W, std::max(CIN, COUT));
  const dim3 grid((unsigned)nb), block(64 * NW);
  if (WgradZXT(CIN, W) == 64) {
    if constexpr (CIN <= 24)
      hipLaunchKernelGGL((WgradZKernel<SC, CIN, COUT, 64, R, NW,
                                       WgradZGroups(SC), SRC>),
                         grid, block, 0, Stream(), src, dz, part, bpart, D, H,
                         W, tz, zchunk);
  } else {
    hipLaunchKernelGGL((WgradZKernel<SC, CIN, COUT, 32, R, NW,
                                     WgradZGroups(SC), SRC>),
                       grid, block, 0, Stream(), src, dz, part, bpart, D, H, W,
                       tz, zchunk);
  }
  Check();
  *nparts = (int)nb;
}

// out = sums of n columns over nparts blocks of part, out2 of n2 columns of
// part2 (n2 = 0: none).
void SumParts(const float *part, long n, float *out, const float *part2,
              long n2, float *out2, int nparts) {
  hipLaunchKernelGGL(SumPartsKernel,
                     dim3((unsigned)((n + 63) / 64 + (n2 + 63) / 64)),
                     dim3(64 * kSumWaves), 0, Stream(), part, n, out, part2,
                     n2, out2, nparts);
  Check();
}

#define PS_UNET_PAIRS(X) \
  X(8, 8) X(8, 16) X(16, 16) X(16, 32) X(32, 32) X(48, 16) X(24, 8) \
  X(16, 8) X(32, 16) X(16, 48) X(8, 24)

void Conv(int cin, int cout, const u16 *x, const u16 *wt, const float *b,
          bool relu, const u16 *act, u16 *y, int N, int D, int H, int W) {
  if (act && (relu || b))
    PS_FATAL("no gated convolution kernel with a bias or a ReLU");
#define PS_CASE(I, O) \
  if (cin == I && cout == O) \
    return ConvT<I, O>(x, wt, b, relu, act, y, N, D, H, W);
  PS_UNET_PAIRS(PS_CASE)
#undef PS_CASE
  PS_FATAL("no convolution kernel for %d -> %d channels", cin, cout);
}

void Wgrad(int cin, int cout, const u16 *x, const u16 *dz, float *part,
           float *bpart, int N, int D, int H, int W, long capacity,
           int *nparts) {
#define PS_CASE(I, O) \
  if (cin == I && cout == O) \
    return WgradZLaunch<I, I, O, PlainSrc>(SrcArgs{x, nullptr, 0}, dz, part, \
                                           bpart, N, D, H, W, capacity, nparts);
  PS_UNET_PAIRS(PS_CASE)
#undef PS_CASE
  PS_FATAL("no filter-gradient kernel for %d -> %d channels", cin, cout);
}

struct Layer {
  int cin, cout;
  size_t w_off, b_off;  // into the flat parameter vector
  u16 *wt = nullptr, *wf = nullptr;
};

void *Alloc(size_t bytes) {
  void *p = nullptr;
  if (bytes == 0) bytes = 16;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}

uint64_t SplitMix(uint64_t &s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

}  // namespace physis_unet

using namespace physis_unet;

struct __PSUNet {
  int nx, ny, nzs, max_batch;
  float out_scale;
  std::vector<Layer> layers;  // 10 convolutions
  size_t head_off, nparams;
  float *params = nullptr, *grad = nullptr, *adam_m = nullptr,
        *adam_v = nullptr;
  long step = 0;
  // activations (BF16) at batch max_batch
  u16 *a[10] = {}, *q1 = nullptr, *q2 = nullptr, *c2 = nullptr;
  float *out = nullptr;  // head outputs, for the smooth loss terms alone
  // gradient scratch
  u16 *g1a = nullptr, *g1b = nullptr, *gc1 = nullptr;  // level 1
  u16 *g2a = nullptr, *g2b = nullptr, *gc2 = nullptr;  // level 2
  u16 *g3a = nullptr, *g3b = nullptr;                  // level 3
  float *part = nullptr, *bpart = nullptr;
  double *lpart = nullptr, *lhost = nullptr;
  size_t part_elems = 0, bpart_elems = 0;
  // smooth-error loss weights and the cell means of the error
  float w4 = 0.0f, w16 = 0.0f;
  float *e4 = nullptr, *e16 = nullptr;
};

namespace {

const int kLayerCh[10][2] = {{8, 8},  {8, 8},   {8, 16},  {16, 16}, {16, 32},
                             {32, 32}, {48, 16}, {16, 16}, {24, 8},  {8, 8}};
constexpr int kHeadBlocks = 1024;  // of HeadLossBackKernel: its partials

void Upload(__PSUNet *net) {  // master weights -> BF16 copies
  for (auto &L : net->layers) {
    hipLaunchKernelGGL(PackKernel, dim3(64), dim3(256), 0, Stream(),
                       net->params + L.w_off, L.wt, L.wf, L.cin, L.cout);
    Check();
  }
}

struct Dims {
  int N, D1, H1, W1, D2, H2, W2, D3, H3, W3;
  long P1, P2, P3;
};

Dims DimsOf(const __PSUNet *net, int count) {
  Dims d;
  d.N = count;
  d.D1 = net->nzs; d.H1 = net->ny; d.W1 = net->nx;
  d.D2 = d.D1 / kPool; d.H2 = d.H1 / kPool; d.W2 = d.W1 / kPool;
  d.D3 = d.D2 / kPool; d.H3 = d.H2 / kPool; d.W3 = d.W2 / kPool;
  d.P1 = (long)count * d.D1 * d.H1 * d.W1;
  d.P2 = (long)count * d.D2 * d.H2 * d.W2;
  d.P3 = (long)count * d.D3 * d.H3 * d.W3;
  return d;
}

void ConvL(const __PSUNet *net, int l, const u16 *in, u16 *out, int N, int D,
           int H, int W) {
  const Layer &L = net->layers[l];
  Conv(L.cin, L.cout, in, L.wt, net->params + L.b_off, true, nullptr, out, N,
       D, H, W);
}

void CheckGrid(const __PSUNet *net, const __PSGrid *g, int first, int count,
               const char *what) {
  if (!g || !g->p || g->num_dims != 3 || g->dim[0] != net->nx ||
      g->dim[1] != net->ny || g->dim[2] % net->nzs != 0)
    PS_FATAL("U-Net: %s is not a 3-D grid of %d x %d x (k * %d)", what,
             net->nx, net->ny, net->nzs);
  const int nb = g->dim[2] / net->nzs;
  if (first < 0 || count < 1 || count > net->max_batch || first + count > nb)
    PS_FATAL("U-Net: problems [%d, %d) outside 0..%d or above the batch %d",
             first, first + count, nb, net->max_batch);
}

// An 8-channel layer on a source of its own (the network input, or an
// upsampled tensor next to a skip connection).
template <int CIN, template <int, int, int, int> class SRC>
void ConvSrc(const __PSUNet *net, int l, const SrcArgs &src, u16 *out, int N,
             int D, int H, int W) {
  const Layer &L = net->layers[l];
  EpiArgs ep;
  ep.bias = net->params + L.b_off;
  ep.y = out;
  ConvMLaunch<CIN, 8, true, SRC, kEpiStore>(src, L.wt, ep, N, D, H, W);
}

// An 8-channel layer and its 4x4x4 average pool (47 us of a prediction of 8 x
// 128^3 less than a pass of its own).
void ConvPool(const __PSUNet *net, int l, const u16 *x, u16 *out, u16 *pool,
              int N, int D, int H, int W) {
  const Layer &L = net->layers[l];
  EpiArgs ep;
  ep.bias = net->params + L.b_off;
  ep.y = out;
  ep.coarse = pool;
  ConvMLaunch<8, 8, true, PlainSrc, kEpiPool>(SrcArgs{x, nullptr, 0}, L.wt, ep,
                                              N, D, H, W);
}

// The last layer, the head and the scaled, masked prediction into p.
template <typename T>
void ConvPredict(const __PSUNet *net, const __PSGrid *bnd, __PSGrid *p,
                 long off, int N, int D, int H, int W) {
  const Layer &L = net->layers[9];
  EpiArgs ep;
  ep.bias = net->params + L.b_off;
  ep.head = net->params + net->head_off;
  ep.bnd = (const float *)bnd->p;
  ep.p = p->p;
  ep.off = off;
  ep.scale = net->out_scale;
  ConvMLaunch<8, 8, true, PlainSrc, kEpiPredict, T>(
      SrcArgs{net->a[8], nullptr, 0}, L.wt, ep, N, D, H, W);
}

// Forward pass of problems [first, first+count): fills the activations; with
// p the last layer's are not kept, the prediction goes to p.
void Forward(__PSUNet *net, const __PSGrid *rhs, const __PSGrid *bnd,
             int first, int count, __PSGrid *p) {
  CheckGrid(net, rhs, first, count, "rhs");
  CheckGrid(net, bnd, first, count, "bnd");
  if (rhs->type != PS_FLOAT || bnd->type != PS_FLOAT)
    PS_FATAL("U-Net: rhs and bnd must be float grids");
  const Dims d = DimsOf(net, count);
  const long off = (long)first * net->nx * net->ny * net->nzs;
  ConvSrc<2, InputSrc>(net, 0, SrcArgs{rhs->p, bnd->p, off}, net->a[0], d.N,
                       d.D1, d.H1, d.W1);
  ConvPool(net, 1, net->a[0], net->a[1], net->q1, d.N, d.D1, d.H1, d.W1);
  ConvL(net, 2, net->q1, net->a[2], d.N, d.D2, d.H2, d.W2);
  ConvL(net, 3, net->a[2], net->a[3], d.N, d.D2, d.H2, d.W2);
  hipLaunchKernelGGL(PoolKernel, dim3(Blocks(d.P3 * 2)), dim3(256), 0,
                     Stream(), net->a[3], net->q2, 16, d.D3, d.H3, d.W3,
                     (int)(d.P3 * 2));
  Check();
  ConvL(net, 4, net->q2, net->a[4], d.N, d.D3, d.H3, d.W3);
  ConvL(net, 5, net->a[4], net->a[5], d.N, d.D3, d.H3, d.W3);
  hipLaunchKernelGGL(UpConcatKernel, dim3(Blocks(d.P2 * 6)), dim3(256), 0,
                     Stream(), net->a[5], net->a[3], net->c2, 32, 16, d.D2,
                     d.H2, d.W2, (int)(d.P2 * 6));
  Check();
  ConvL(net, 6, net->c2, net->a[6], d.N, d.D2, d.H2, d.W2);
  ConvL(net, 7, net->a[6], net->a[7], d.N, d.D2, d.H2, d.W2);
  ConvSrc<24, ConcatSrc>(net, 8, SrcArgs{net->a[7], net->a[1], 0}, net->a[8],
                         d.N, d.D1, d.H1, d.W1);
  if (!p)
    ConvL(net, 9, net->a[8], net->a[9], d.N, d.D1, d.H1, d.W1);
  else if (p->type == PS_DOUBLE)
    ConvPredict<double>(net, bnd, p, off, d.N, d.D1, d.H1, d.W1);
  else
    ConvPredict<float>(net, bnd, p, off, d.N, d.D1, d.H1, d.W1);
}

// Blocks of partials that layer l may write.
long WgradCapacity(const __PSUNet *net, const Layer &L) {
  return std::min<long>((long)net->part_elems / ((long)L.cout * 27 * L.cin),
                        (long)net->bpart_elems / L.cout);
}
void SumLayer(__PSUNet *net, const Layer &L, int np) {
  SumParts(net->part, (long)L.cout * 27 * L.cin, net->grad + L.w_off,
           net->bpart, L.cout, net->grad + L.b_off, np);
}

// Filter gradient of layer l from input `in` and gated output gradient dz.
void LayerWgrad(__PSUNet *net, int l, const u16 *in, const u16 *dz, int N,
                int D, int H, int W) {
  const Layer &L = net->layers[l];
  int np = 0;
  Wgrad(L.cin, L.cout, in, dz, net->part, net->bpart, N, D, H, W,
        WgradCapacity(net, L), &np);
  SumLayer(net, L, np);
}

// The same from a source of its own.
template <int SC, int CIN, template <int, int, int, int> class SRC>
void SrcWgrad(__PSUNet *net, int l, const SrcArgs &src, const u16 *dz, int N,
              int D, int H, int W) {
  const Layer &L = net->layers[l];
  int np = 0;
  WgradZLaunch<SC, CIN, 8, SRC>(src, dz, net->part, net->bpart, N, D, H, W,
                                WgradCapacity(net, L), &np);
  SumLayer(net, L, np);
}

// Data gradient of layer l: dx = conv(dz, flipped W), no bias, no ReLU,
// gated by the activation act when not NULL (the ReLU of the layer before).
void LayerDgrad(__PSUNet *net, int l, const u16 *dz, const u16 *act, u16 *dx,
                int N, int D, int H, int W) {
  const Layer &L = net->layers[l];
  Conv(L.cout, L.cin, dz, L.wf, nullptr, false, act, dx, N, D, H, W);
}

// Loss of the current forward pass against target, and the full gradient
// into net->grad.
double Backward(__PSUNet *net, const __PSGrid *rhs, const __PSGrid *bnd,
                const __PSGrid *target, int first, int count) {
  CheckGrid(net, target, first, count, "target");
  if (target->type != PS_FLOAT) PS_FATAL("U-Net: target must be a float grid");
  const Dims d = DimsOf(net, count);
  const long off = (long)first * net->nx * net->ny * net->nzs;
  const float inv_scale = 1.0f / net->out_scale;
  // head and loss: g1a = gated dD1 (layer 9's dz), partials in part, lpart
  const bool smooth = net->w4 != 0.0f || net->w16 != 0.0f;
  if (smooth) {
    hipLaunchKernelGGL(HeadKernel, dim3(Blocks(d.P1)), dim3(256), 0, Stream(),
                       net->a[9], net->params + net->head_off, net->out, d.P1);
    Check();
    hipLaunchKernelGGL(SmoothCellKernel, dim3(Blocks(d.P2 * 64)), dim3(256),
                       0, Stream(), net->out, (const float *)target->p, off,
                       inv_scale, net->e4, d.D1, d.H1, d.W1, d.P2);
    Check();
    hipLaunchKernelGGL(SmoothCoarseKernel, dim3(Blocks(d.P3)), dim3(256), 0,
                       Stream(), net->e4, net->e16, d.D2, d.H2, d.W2, d.P3);
    Check();
  }
  const auto head = smooth ? HeadLossBackKernel<true> : HeadLossBackKernel<false>;
  hipLaunchKernelGGL(head, dim3(kHeadBlocks), dim3(kHeadThreads), 0, Stream(),
                     net->a[9], net->params + net->head_off,
                     (const float *)target->p, off, inv_scale, net->e4,
                     net->e16, net->w4, net->w16, d.D1, d.H1, d.W1, net->g1a,
                     net->lpart, net->part, d.P1);
  Check();
  SumParts(net->part, 9, net->grad + net->head_off, nullptr, 0, nullptr,
           kHeadBlocks);
  // level 1 decoder
  LayerWgrad(net, 9, net->a[8], net->g1a, d.N, d.D1, d.H1, d.W1);
  LayerDgrad(net, 9, net->g1a, net->a[8], net->g1b, d.N, d.D1, d.H1, d.W1);
  SrcWgrad<24, 24, ConcatSrc>(net, 8, SrcArgs{net->a[7], net->a[1], 0},
                              net->g1b, d.N, d.D1, d.H1, d.W1);
  // 24 channels: 16 to the level-2 decoder (summed over the upsampled cells
  // and gated: g2a), 8 to the skip connection (gc1)
  {
    const Layer &L = net->layers[8];
    EpiArgs ep;
    ep.y = net->gc1;
    ep.act = net->a[7];
    ep.coarse = net->g2a;
    ConvMLaunch<8, 24, false, PlainSrc, kEpiUpSkip>(
        SrcArgs{net->g1b, nullptr, 0}, L.wf, ep, d.N, d.D1, d.H1, d.W1);
  }
  // level 2 decoder
  LayerWgrad(net, 7, net->a[6], net->g2a, d.N, d.D2, d.H2, d.W2);
  LayerDgrad(net, 7, net->g2a, net->a[6], net->g2b, d.N, d.D2, d.H2, d.W2);
  LayerWgrad(net, 6, net->c2, net->g2b, d.N, d.D2, d.H2, d.W2);
  LayerDgrad(net, 6, net->g2b, nullptr, net->gc2, d.N, d.D2, d.H2, d.W2);
  hipLaunchKernelGGL(UpBackKernel, dim3(Blocks(d.P3 * 4)), dim3(256), 0,
                     Stream(), net->gc2, net->a[5], net->g3a, 32, 48, d.D3,
                     d.H3, d.W3, (int)(d.P3 * 4));
  Check();
  // level 3
  LayerWgrad(net, 5, net->a[4], net->g3a, d.N, d.D3, d.H3, d.W3);
  LayerDgrad(net, 5, net->g3a, net->a[4], net->g3b, d.N, d.D3, d.H3, d.W3);
  LayerWgrad(net, 4, net->q2, net->g3b, d.N, d.D3, d.H3, d.W3);
  LayerDgrad(net, 4, net->g3b, nullptr, net->g3a, d.N, d.D3, d.H3, d.W3);
  // level 2 encoder: E2 receives the pool gradient and the skip gradient
  hipLaunchKernelGGL(PoolBackSkipGateKernel, dim3(Blocks(d.P2 * 2)),
                     dim3(256), 0, Stream(), net->g3a, net->gc2, net->a[3],
                     net->g2a, 16, 32, d.D2, d.H2, d.W2, (int)(d.P2 * 2));
  Check();
  LayerWgrad(net, 3, net->a[2], net->g2a, d.N, d.D2, d.H2, d.W2);
  LayerDgrad(net, 3, net->g2a, net->a[2], net->g2b, d.N, d.D2, d.H2, d.W2);
  LayerWgrad(net, 2, net->q1, net->g2b, d.N, d.D2, d.H2, d.W2);
  LayerDgrad(net, 2, net->g2b, nullptr, net->g2a, d.N, d.D2, d.H2, d.W2);
  // level 1 encoder
  hipLaunchKernelGGL(PoolBackSkipGateKernel, dim3(Blocks(d.P1)), dim3(256),
                     0, Stream(), net->g2a, net->gc1, net->a[1], net->g1a, 8,
                     0, d.D1, d.H1, d.W1, (int)d.P1);
  Check();
  LayerWgrad(net, 1, net->a[0], net->g1a, d.N, d.D1, d.H1, d.W1);
  LayerDgrad(net, 1, net->g1a, net->a[0], net->g1b, d.N, d.D1, d.H1, d.W1);
  SrcWgrad<4, 8, InputSrc>(net, 0, SrcArgs{rhs->p, bnd->p, off}, net->g1b,
                           d.N, d.D1, d.H1, d.W1);
  PS_HIP_CHECK(hipMemcpyAsync(net->lhost, net->lpart,
                              sizeof(double) * kHeadBlocks,
                              hipMemcpyDeviceToHost, Stream()));
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
  double loss = 0.0;
  for (int b = 0; b < kHeadBlocks; ++b) loss += net->lhost[b];
  return loss / (double)d.P1;
}

void FreeNet(__PSUNet *net) {
  (void)hipStreamSynchronize(Stream());
  std::vector<void *> ptrs = {net->params, net->grad, net->adam_m,
                              net->adam_v, net->q1, net->q2,
                              net->c2, net->out, net->g1a,
                              net->g1b, net->gc1, net->g2a, net->g2b,
                              net->gc2, net->g3a, net->g3b, net->part,
                              net->bpart, net->lpart, net->e4,
                              net->e16};
  for (int i = 0; i < 10; ++i) ptrs.push_back(net->a[i]);
  for (auto &L : net->layers) {
    ptrs.push_back(L.wt);
    ptrs.push_back(L.wf);
  }
  for (void *p : ptrs)
    if (p) PS_HIP_CHECK(hipFree(p));
  if (net->lhost) PS_HIP_CHECK(hipHostFree(net->lhost));
  delete net;
}

// Host-side device buffer for the single-layer entry points.
struct DevBuf {
  void *p = nullptr;
  explicit DevBuf(size_t bytes) {
    p = Alloc(bytes);
    if (!p) PS_FATAL("out of device memory");
  }
  ~DevBuf() { (void)hipFree(p); }
};

void CheckLayerArgs(int n, int d, int h, int w, int cin, int cout) {
  if (n < 1 || d < 1 || h < 1 || w < 1 || cin % 8 || cout < 1)
    PS_FATAL("convolution: bad sizes n=%d d=%d h=%d w=%d cin=%d cout=%d", n,
             d, h, w, cin, cout);
}

}  // namespace

extern "C" {

__PSUNet *PSUNetNew(int nx, int ny, int nzs, int max_batch, float out_scale,
                    uint64_t seed) {
  if (nx % 16 || ny % 16 || nzs % 16 || nx < 16 || ny < 16 || nzs < 16 ||
      max_batch < 1 || !(out_scale > 0.0f)) {
    std::fprintf(stderr,
                 "[physis-hip] PSUNetNew: sizes must be positive multiples "
                 "of 16, batch >= 1, scale > 0\n");
    return nullptr;
  }
  __PSUNet *net = new __PSUNet();
  net->nx = nx;
  net->ny = ny;
  net->nzs = nzs;
  net->max_batch = max_batch;
  net->out_scale = out_scale;
  size_t off = 0;
  for (int l = 0; l < 10; ++l) {
    Layer L;
    L.cin = kLayerCh[l][0];
    L.cout = kLayerCh[l][1];
    L.w_off = off;
    off += (size_t)L.cout * 27 * L.cin;
    L.b_off = off;
    off += L.cout;
    net->layers.push_back(L);
  }
  net->head_off = off;
  off += 9;
  net->nparams = off;
  // He-normal weights (std sqrt(2 / fan_in)), zero biases; head std 1/sqrt(8)
  std::vector<float> h(off, 0.0f);
  uint64_t s = seed;
  auto normal = [&]() {
    const double u1 = ((SplitMix(s) >> 11) + 1.0) * (1.0 / 9007199254740993.0);
    const double u2 = (SplitMix(s) >> 11) * (1.0 / 9007199254740992.0);
    return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
  };
  for (auto &L : net->layers) {
    const double sd = std::sqrt(2.0 / (27.0 * L.cin));
    for (size_t i = 0; i < (size_t)L.cout * 27 * L.cin; ++i)
      h[L.w_off + i] = (float)(sd * normal());
  }
  for (int c = 0; c < 8; ++c) h[net->head_off + c] = (float)(normal() / std::sqrt(8.0));
  const Dims d = DimsOf(net, max_batch);
  bool ok = true;
  auto A16 = [&](long elems) {
    u16 *p = (u16 *)Alloc(sizeof(u16) * (size_t)elems);
    ok = ok && p;
    return p;
  };
  auto A32 = [&](long elems) {
    float *p = (float *)Alloc(sizeof(float) * (size_t)elems);
    ok = ok && p;
    return p;
  };
  net->params = A32(off);
  net->grad = A32(off);
  net->adam_m = A32(off);
  net->adam_v = A32(off);
  for (auto &L : net->layers) {
    L.wt = A16((long)L.cout * KPad(L.cin));
    L.wf = A16((long)L.cin * KPad(L.cout));
  }
  const long act[10] = {d.P1 * 8,  d.P1 * 8,  d.P2 * 16, d.P2 * 16, d.P3 * 32,
                        d.P3 * 32, d.P2 * 16, d.P2 * 16, d.P1 * 8,  d.P1 * 8};
  for (int l = 0; l < 10; ++l) net->a[l] = A16(act[l]);
  net->q1 = A16(d.P2 * 8);
  net->q2 = A16(d.P3 * 16);
  net->c2 = A16(d.P2 * 48);
  net->out = A32(d.P1);
  net->g1a = A16(d.P1 * 8);
  net->g1b = A16(d.P1 * 8);
  net->gc1 = A16(d.P1 * 8);
  net->g2a = A16(d.P2 * 16);
  net->g2b = A16(d.P2 * 16);
  net->gc2 = A16(d.P2 * 48);
  net->g3a = A16(d.P3 * 32);
  net->g3b = A16(d.P3 * 32);
  size_t pe = (size_t)kHeadBlocks * 9, be = 0;
  for (int l = 0; l < 10; ++l) {
    const int lv = l < 2 || l > 7 ? 1 : (l < 4 || l > 5 ? 2 : 3);
    const int W = lv == 1 ? d.W1 : (lv == 2 ? d.W2 : d.W3);
    const int H = lv == 1 ? d.H1 : (lv == 2 ? d.H2 : d.H3);
    const int D = lv == 1 ? d.D1 : (lv == 2 ? d.D2 : d.D3);
    // the block count depends on the batch: the largest over every batch a
    // call may use
    size_t nb = 0;
    for (int nbat = 1; nbat <= max_batch; ++nbat)
      nb = std::max<size_t>(
          nb, (size_t)WgradBlocks(net->layers[l].cin, nbat, D, H, W));
    const size_t nw = (size_t)net->layers[l].cout * 27 * net->layers[l].cin;
    pe = std::max(pe, nb * nw);
    be = std::max(be, nb * net->layers[l].cout);
  }
  net->part_elems = pe;
  net->bpart_elems = be;
  net->part = A32((long)pe);
  net->bpart = A32((long)be);
  net->e4 = A32(d.P2);
  net->e16 = A32(d.P3);
  net->lpart = (double *)Alloc(sizeof(double) * kHeadBlocks);
  ok = ok && net->lpart;
  if (ok && hipHostMalloc((void **)&net->lhost, sizeof(double) * kHeadBlocks) !=
                hipSuccess) {
    (void)hipGetLastError();
    ok = false;
  }
  if (!ok) {
    std::fprintf(stderr, "[physis-hip] PSUNetNew: out of device memory\n");
    FreeNet(net);
    return nullptr;
  }
  PS_HIP_CHECK(hipMemcpy(net->params, h.data(), sizeof(float) * off,
                         hipMemcpyHostToDevice));
  PS_HIP_CHECK(hipMemset(net->adam_m, 0, sizeof(float) * off));
  PS_HIP_CHECK(hipMemset(net->adam_v, 0, sizeof(float) * off));
  PS_HIP_CHECK(hipMemset(net->grad, 0, sizeof(float) * off));
  Upload(net);
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
  return net;
}

void PSUNetFree(__PSUNet *net) {
  if (net) FreeNet(net);
}

size_t PSUNetNumParams(const __PSUNet *net) { return net->nparams; }

void PSUNetGetParams(const __PSUNet *net, float *host) {
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
  PS_HIP_CHECK(hipMemcpy(host, net->params, sizeof(float) * net->nparams,
                         hipMemcpyDeviceToHost));
}

void PSUNetSetParams(__PSUNet *net, const float *host) {
  PS_HIP_CHECK(hipMemcpy(net->params, host, sizeof(float) * net->nparams,
                         hipMemcpyHostToDevice));
  Upload(net);
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
}

void PSUNetPredict(__PSUNet *net, const __PSGrid *rhs, const __PSGrid *bnd,
                   int first, int count, __PSGrid *p) {
  CheckGrid(net, p, first, count, "p");
  if (p->type != PS_FLOAT && p->type != PS_DOUBLE)
    PS_FATAL("U-Net: p must be a float or double grid");
  Forward(net, rhs, bnd, first, count, p);
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
}

void PSUNetReflect(const __PSGrid *src, int first, int count, __PSGrid *dst,
                   int dst_first, int nx, int ny, int nzs, int flips) {
  if (!src || !dst || src->type != PS_FLOAT || dst->type != PS_FLOAT ||
      src->num_dims != 3 || dst->num_dims != 3 || src->dim[0] != nx ||
      dst->dim[0] != nx || src->dim[1] != ny || dst->dim[1] != ny ||
      nzs < 1 || src->dim[2] % nzs || dst->dim[2] % nzs || first < 0 ||
      dst_first < 0 || count < 0 || flips < 0 || flips > 7 ||
      (long)(first + count) * nzs > src->dim[2] ||
      (long)(dst_first + count) * nzs > dst->dim[2] ||
      (src->p == dst->p && count > 0))
    PS_FATAL("PSUNetReflect: bad grids or problem range");
  const long m = (long)nx * ny * nzs, n = m * count;
  if (n == 0) return;
  hipLaunchKernelGGL(ReflectKernel, dim3((unsigned)((n + 255) / 256)),
                     dim3(256), 0, Stream(), (const float *)src->p,
                     (float *)dst->p, nx, ny, nzs, m * first, m * dst_first,
                     flips, n);
  Check();
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
}

double PSUNetLossGrad(__PSUNet *net, const __PSGrid *rhs, const __PSGrid *bnd,
                      const __PSGrid *target, int first, int count,
                      float *grad_host) {
  Forward(net, rhs, bnd, first, count, nullptr);
  const double loss = Backward(net, rhs, bnd, target, first, count);
  if (grad_host)
    PS_HIP_CHECK(hipMemcpy(grad_host, net->grad, sizeof(float) * net->nparams,
                           hipMemcpyDeviceToHost));
  return loss;
}

void PSUNetSetLossWeights(__PSUNet *net, float w4, float w16) {
  if (!(w4 >= 0.0f) || !(w16 >= 0.0f))
    PS_FATAL("U-Net: loss weights must be >= 0 (got %g, %g)", w4, w16);
  net->w4 = w4;
  net->w16 = w16;
}

double PSUNetTrainStep(__PSUNet *net, const __PSGrid *rhs,
                       const __PSGrid *bnd, const __PSGrid *target, int first,
                       int count, float lr) {
  Forward(net, rhs, bnd, first, count, nullptr);
  const double loss = Backward(net, rhs, bnd, target, first, count);
  net->step += 1;
  const float c1 = 1.0f - std::pow(0.9f, (float)net->step);
  const float c2 = 1.0f - std::pow(0.999f, (float)net->step);
  hipLaunchKernelGGL(AdamKernel, dim3(Blocks((long)net->nparams)), dim3(256),
                     0, Stream(), net->params, net->grad, net->adam_m,
                     net->adam_v, (long)net->nparams, lr, c1, c2);
  Check();
  Upload(net);
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
  return loss;
}

void PSConv3dForwardHost(const uint16_t *x, const uint16_t *w,
                         const float *bias, int relu, int n, int d, int h,
                         int wd, int cin, int cout, uint16_t *y) {
  CheckLayerArgs(n, d, h, wd, cin, cout);
  const long P = (long)n * d * h * wd;
  const size_t nw = (size_t)cout * 27 * cin;
  DevBuf dx(P * cin * 2), dw32(nw * 4), dwt((size_t)cout * KPad(cin) * 2),
      dwf((size_t)cin * KPad(cout) * 2), db(cout * 4), dy(P * cout * 2);
  std::vector<float> wf(nw);
  for (size_t i = 0; i < nw; ++i) {
    const uint32_t u = (uint32_t)w[i] << 16;
    std::memcpy(&wf[i], &u, 4);
  }
  PS_HIP_CHECK(hipMemcpy(dx.p, x, P * cin * 2, hipMemcpyHostToDevice));
  PS_HIP_CHECK(hipMemcpy(dw32.p, wf.data(), nw * 4, hipMemcpyHostToDevice));
  PS_HIP_CHECK(hipMemcpy(db.p, bias, cout * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(PackKernel, dim3(64), dim3(256), 0, Stream(),
                     (const float *)dw32.p, (u16 *)dwt.p, (u16 *)dwf.p, cin,
                     cout);
  Check();
  Conv(cin, cout, (const u16 *)dx.p, (const u16 *)dwt.p, (const float *)db.p,
       relu != 0, nullptr, (u16 *)dy.p, n, d, h, wd);
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
  PS_HIP_CHECK(hipMemcpy(y, dy.p, P * cout * 2, hipMemcpyDeviceToHost));
}

void PSConv3dBackwardDataHost(const uint16_t *dy, const uint16_t *w, int n,
                              int d, int h, int wd, int cin, int cout,
                              uint16_t *dx) {
  CheckLayerArgs(n, d, h, wd, cin, cout);
  if (cout % 8) PS_FATAL("convolution: cout must be a multiple of 8");
  const long P = (long)n * d * h * wd;
  const size_t nw = (size_t)cout * 27 * cin;
  DevBuf ddy(P * cout * 2), dw32(nw * 4), dwt((size_t)cout * KPad(cin) * 2),
      dwf((size_t)cin * KPad(cout) * 2), ddx(P * cin * 2);
  std::vector<float> wf(nw);
  for (size_t i = 0; i < nw; ++i) {
    const uint32_t u = (uint32_t)w[i] << 16;
    std::memcpy(&wf[i], &u, 4);
  }
  PS_HIP_CHECK(hipMemcpy(ddy.p, dy, P * cout * 2, hipMemcpyHostToDevice));
  PS_HIP_CHECK(hipMemcpy(dw32.p, wf.data(), nw * 4, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(PackKernel, dim3(64), dim3(256), 0, Stream(),
                     (const float *)dw32.p, (u16 *)dwt.p, (u16 *)dwf.p, cin,
                     cout);
  Check();
  Conv(cout, cin, (const u16 *)ddy.p, (const u16 *)dwf.p, nullptr, false,
       nullptr, (u16 *)ddx.p, n, d, h, wd);
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
  PS_HIP_CHECK(hipMemcpy(dx, ddx.p, P * cin * 2, hipMemcpyDeviceToHost));
}

void PSConv3dBackwardFilterHost(const uint16_t *x, const uint16_t *dy, int n,
                                int d, int h, int wd, int cin, int cout,
                                float *dw, float *db) {
  CheckLayerArgs(n, d, h, wd, cin, cout);
  const long P = (long)n * d * h * wd;
  const long nb = WgradBlocks(cin, n, d, h, wd);
  const size_t nw = (size_t)cout * 27 * cin;
  DevBuf ddx(P * cin * 2), ddy(P * cout * 2), part(nb * nw * 4),
      bpart(nb * cout * 4), dw_d(nw * 4), db_d(cout * 4);
  PS_HIP_CHECK(hipMemcpy(ddx.p, x, P * cin * 2, hipMemcpyHostToDevice));
  PS_HIP_CHECK(hipMemcpy(ddy.p, dy, P * cout * 2, hipMemcpyHostToDevice));
  int np = 0;
  Wgrad(cin, cout, (const u16 *)ddx.p, (const u16 *)ddy.p, (float *)part.p,
        (float *)bpart.p, n, d, h, wd, nb, &np);
  SumParts((const float *)part.p, (long)nw, (float *)dw_d.p,
           (const float *)bpart.p, cout, (float *)db_d.p, np);
  PS_HIP_CHECK(hipStreamSynchronize(Stream()));
  PS_HIP_CHECK(hipMemcpy(dw, dw_d.p, nw * 4, hipMemcpyDeviceToHost));
  PS_HIP_CHECK(hipMemcpy(db, db_d.p, cout * 4, hipMemcpyDeviceToHost));
}

}  // extern "C"
