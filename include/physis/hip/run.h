// Host-side helpers of the run functions that physisc-hip generates: launch
// planning for 2.5D run kernels, argument checks and the run timer that backs
// --physis-trace (reference: translator/reference_runtime_builder.cc:896-940
// emits the equivalent stopwatch code inline).
#ifndef PHYSIS_HIP_RUN_H_
#define PHYSIS_HIP_RUN_H_

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

#include "physis/physis_hip.h"
#include "physis/hip/stencil.h"

namespace physis_hip {

// ------------------------------------------------ host intrinsic helpers
// PSGrid<N>D<T>New(d0, d1, d2): the type-info block the reference emits
// inline (reference_runtime_builder.cc:959-1065) folded into one call.
inline __PSGrid *NewGrid(int type, int size, int num_dims, int d0, int d1 = 1,
                         int d2 = 1) {
  __PSGridTypeInfo ti = {type, size, 0, nullptr};
  PSVectorInt dim = {d0, d1, d2};
  return __PSGridNew(&ti, num_dims, dim, nullptr);
}

// PSGrid<n>D<Name>New for a user-defined point type: ti describes its members.
inline __PSGrid *NewUserGrid(__PSGridTypeInfo *ti, int num_dims, int d0,
                             int d1 = 1, int d2 = 1) {
  PSVectorInt dim = {d0, d1, d2};
  return __PSGridNew(ti, num_dims, dim, nullptr);
}

// PSGridGet(g, i...) in host code: one element copied back (synchronous).
template <typename T>
inline T GetElem(__PSGrid *g, PSIndex i0, PSIndex i1 = 0, PSIndex i2 = 0) {
  T v;
  __PSGridGet(g, &v, i0, i1, i2);
  return v;
}

// PSGridSet(g, i..., v) with v converted to the element type.
template <typename T>
inline void SetElem(__PSGrid *g, T v, PSIndex i0, PSIndex i1 = 0,
                    PSIndex i2 = 0) {
  __PSGridSet(g, &v, i0, i1, i2);
}

// Resident blocks of `kernel` per compute unit at `threads` per block.
inline int BlocksPerCU(const void *kernel, int threads) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) !=
          hipSuccess ||
      n < 1) {
    (void)hipGetLastError();
    n = 1;
  }
  return n;
}

// Buffer windows (stencil.h: BufWin) address at most 2^31 - 1 bytes, the
// reach of a 32-bit buffer range.  The largest z chunk for which a window of
// grid g over the chunk plus `margin` planes on each side stays within that
// reach; a grid of which not even one such window fits is rejected (the
// reference's 32-bit PSIndex, include/physis/physis_common.h:33-55, bounds
// elements, not bytes).
inline int64_t WindowPlanes(const __PSGrid *g, int margin) {
  if (!g) return INT32_MAX;
  int64_t plane = (int64_t)g->elm_size;
  for (int d = 0; d < g->num_dims && d < 2; ++d) plane *= g->dim[d];
  if (plane <= 0) return INT32_MAX;
  return (int64_t)INT32_MAX / plane - 2 * (int64_t)margin;
}
inline int WindowChunkLimit(const __PSGrid *g, int margin) {
  const int64_t planes = WindowPlanes(g, margin);
  if (planes < 1) {
    int64_t plane = (int64_t)g->elm_size;
    for (int d = 0; d < g->num_dims && d < 2; ++d) plane *= g->dim[d];
    std::fprintf(stderr,
                 "[physis-hip] a %lld-byte plane (with %d halo planes per "
                 "side) exceeds the 2 GiB reach of a buffer window\n",
                 (long long)plane, margin);
    std::exit(EXIT_FAILURE);
  }
  return planes > INT32_MAX ? INT32_MAX : (int)planes;
}
// Whether a pass with `margin` planes (rows of a 2-D grid in the rows view) per
// side has a window at all: passes of several sweeps reach further than single
// sweeps, which serve the grids whose planes are too large for them.
inline bool WindowsFit(std::initializer_list<const __PSGrid *> grids,
                       int margin, bool rows = false) {
  for (const __PSGrid *g : grids) {
    if (!g) continue;
    __PSGrid w = *g;
    if (rows) w.num_dims = 1;
    if (WindowPlanes(&w, margin) < 1) return false;
  }
  return true;
}
inline int WindowChunkLimit(std::initializer_list<const __PSGrid *> grids,
                            int margin) {
  int m = INT32_MAX;
  for (const __PSGrid *g : grids) {
    const int c = WindowChunkLimit(g, margin);
    m = c < m ? c : m;
  }
  return m;
}

// The same reach for a 2-D grid in the rows view (nx x 1 x ny): z chunks
// are chunks of rows.
inline int WindowChunkLimitRows(std::initializer_list<const __PSGrid *> grids,
                                int margin) {
  int m = INT32_MAX;
  for (const __PSGrid *g : grids) {
    if (!g) continue;
    __PSGrid row = *g;
    row.num_dims = 1;  // one row of dim[0] elements per "plane"
    const int c = WindowChunkLimit(&row, margin);
    m = c < m ? c : m;
  }
  return m;
}

// Tiles a domain into TX x TY column tiles and picks the number of z chunks.
// Each block costs (chunk + extra) plane steps (prologue planes), blocks run
// in waves of `resident` blocks; the chunk count minimising
// waves * (chunk + extra) is chosen so that the last wave is not left mostly
// idle.  Chunks never exceed max_chunk planes (the window reach).
inline RunShape PlanRunFor(const __PSDomain &dom, int tx, int ty,
                           long resident, int max_chunk = INT32_MAX,
                           int extra = 2) {
  RunShape s = {0, 0, 0, 0, 0, 0};
  const int nx = dom.local_max[0] - dom.local_min[0];
  const int ny = dom.local_max[1] - dom.local_min[1];
  const int nz = dom.local_max[2] - dom.local_min[2];
  if (nx <= 0 || ny <= 0 || nz <= 0) return s;
  if (max_chunk < 1) max_chunk = 1;
  if (resident < 1) resident = 1;
  // x tiles are anchored at x = 0 so that vector loads stay aligned.
  const int xf = dom.local_min[0] >= 0 ? dom.local_min[0] / tx
                                       : -((-dom.local_min[0] + tx - 1) / tx);
  const int xl = (dom.local_max[0] - 1) >= 0
                     ? (dom.local_max[0] - 1) / tx
                     : -((-(dom.local_max[0] - 1) + tx - 1) / tx);
  s.x_first_tile = xf;
  s.tiles_x = xl - xf + 1;
  s.tiles_y = (ny + ty - 1) / ty;
  const long xy = (long)s.tiles_x * s.tiles_y;
  long best_cost = -1;
  int best_tz = 0;
  for (int tz = (nz + max_chunk - 1) / max_chunk; tz <= nz; ++tz) {
    const int chunk = (nz + tz - 1) / tz;
    if (chunk > max_chunk) continue;
    if ((long)(tz - 1) * chunk >= nz) continue;  // same chunk, fewer blocks
    const long blocks = xy * tz;
    if (blocks > (1L << 30)) break;
    const long waves = (blocks + resident - 1) / resident;
    const long cost = waves * (chunk + extra);
    if (best_cost < 0 || cost < best_cost) {
      best_cost = cost;
      best_tz = tz;
    }
  }
  if (best_tz == 0) {
    std::fprintf(stderr, "[physis-hip] no launch shape fits a domain of "
                 "%d x %d x %d points\n", nx, ny, nz);
    std::exit(EXIT_FAILURE);
  }
  s.tiles_z = best_tz;
  s.zchunk = (nz + best_tz - 1) / best_tz;
  s.blocks = (int)(xy * best_tz);
  return s;
}

inline RunShape PlanRun(const __PSDomain &dom, int tx, int ty, int per_cu,
                        int max_chunk = INT32_MAX, int extra = 2) {
  return PlanRunFor(dom, tx, ty, (long)__PSHipNumCUs() * per_cu, max_chunk,
                    extra);
}

// Whether a single sweep over rows whose extents are not multiples of 4 runs
// at one point per lane (tiles of 64 points) and not in the ragged form at four
// (tiles of 256): it does where it covers the domain with so many fewer lanes
// that the work shared by a lane's four points does not count.  Periodic planes
// are loaded through a window of their own each, four times as often per point,
// but small grids still gain from the blocks (77x60x60 12.1 and 13, 222x60x60 12.9
// and 13.4).
// us at one point and ragged, rows of 63, 127, 191, 255 and 290 points by
// 256 x 200: 7-point clamped diffusion 11.1 and 16.9, 19.2 and 20.3, 27.1 and
// 23.3, 33 and 27, 36 and 37; periodic 15.3 and 18.9, 23 and 20, 33 and 24;
// 7-point over user points 58 and 92, 81 and 94, 117 and 99, 136 and 110, 150
// and 170; 19-point 49 and 103, 104 and 119, 151 and 139, 208 and 171, 245 and
// 242; 7 gets at corners 10 and 17, 13 and 17, 18 and 18, 22 and 20, 25 and 33.
// (8-byte grids always do: 14 and 49, 24 and 50, 30 and 50, 42 and 51, 45 and
// 98; four of their points are two 16-byte vectors, and LDS holds half as many
// blocks.)
// A colour sweep leaves every other point of a lane's four as it is: large ones
// run at one point per lane (255^3 63 and 70 an iteration, 383x200x150 48 and 51;
// 150^3 26 and 23).
inline bool OnePointRows(const __PSDomain &d, bool periodic, bool colour) {
  const auto tiles = [&](int t) {
    return (d.local_max[0] + t - 1) / t - d.local_min[0] / t;
  };
  double points = 1;
  for (int i = 0; i < 3; ++i) points *= d.local_max[i] - d.local_min[i];
  if (periodic) return tiles(64) <= tiles(256) || points < 1.5e6;
  return 2 * tiles(64) <= 5 * tiles(256) || (colour && points >= 8e6);
}

// Points per lane (4 or 2) of a whole-grid two-sweep pass over rows of nx
// points: tiles of 256 points, or of 128 where those pad the rows so much
// less that they win although a point costs more in them (its row's loads,
// addresses and masks are shared by half as many points; periodic planes are
// loaded through a window of their own each), and more the fewer planes a block
// has.  us a sweep at 4 and 2 points, clamped 7-point map: 128x100x100 6.4 and
// 5.9, 128x256x256 19.0 and 13.5; 384x60x60 5.7 and 6.1, 368x200x150 18.0 and
// 18.9, 301x256x256 34.3 and 32.7, 384^3 74 and 67.  Periodic: 128x100x100 7.1 and
// 7.6, 100x128x128 7.7 and 7.4, 128x256x256 19.8 and 15.1, 321x190x157 20.9 and
// 21.4.  Red-black iteration: 128x164x65 11.4 and 11.8, 100x128x128 13.0 and 12.2,
// 128x256x256 35 and 26; 384x60x60 10.0 and 12.1, 368x200x200 43 and 45,
// 301x256x256 63 and 64, 375x256x256 65 and 67, 257x218x400 86 and 79,
// 301x218x400 92 and 82, 384^3 147 and 130.
inline int PairVX(const int *dim, bool periodic, bool colours) {
  const long wide = (dim[0] + 255) / 256 * 256L, narrow = (dim[0] + 127) / 128 * 128L;
  const double n = (double)dim[0] * dim[1] * dim[2];
  if (narrow * 2 == wide)
    return n >= (periodic || colours ? 1.5e6 : 0.0) ? 2 : 4;
  if (periodic || narrow * 5 >= wide * 4) return 4;
  return n >= (colours ? 2e7 : 1.6e7) ? 2 : 4;
}

// A 3-D grid argument must be live, of the stencil's element type, and small
// enough for 32-bit PSIndex offsets (the reference's default index type).
inline void CheckGrid3D(const __PSGrid *g, int type) {
  if (!g || !g->p) {
    std::fprintf(stderr, "[physis-hip] stencil map on a freed or NULL grid\n");
    std::exit(EXIT_FAILURE);
  }
  if (g->type != type) {
    std::fprintf(stderr,
                 "[physis-hip] grid element type %d does not match the "
                 "stencil's type %d\n", g->type, type);
    std::exit(EXIT_FAILURE);
  }
  if (g->num_elms >= (int64_t)PSINDEX_MAX) {
    std::fprintf(stderr,
                 "[physis-hip] grid of %lld elements exceeds 32-bit PSIndex\n",
                 (long long)g->num_elms);
    std::exit(EXIT_FAILURE);
  }
}

// Device-to-device copy of `bytes` on `stream`; aborts on an error.
inline void CopyDevice(void *dst, const void *src, size_t bytes,
                       hipStream_t stream) {
  const hipError_t e =
      hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, stream);
  if (e != hipSuccess) {
    std::fprintf(stderr, "[physis-hip] device copy failed: %s\n",
                 hipGetErrorString(e));
    std::exit(EXIT_FAILURE);
  }
}

// Copies the points of an nx x ny x nz grid view that lie outside a domain and
// at most one point from it: one thread per row of the domain copies the point
// beyond either end, then one thread per point the rows of the shell.
template <typename T>
__global__ __launch_bounds__(256) void CopyShellKernel(
    T *__restrict__ dst, const T *__restrict__ src, int nx, int ny,
    __PSDomain d, __PSDomain box, int row_blocks, int outer) {
  const int x0 = d.local_min[0], x1 = d.local_max[0];
  const int y0 = d.local_min[1], dy = d.local_max[1] - y0;
  const int z0 = d.local_min[2], dz = d.local_max[2] - z0;
  if ((int)blockIdx.x < row_blocks) {
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= dy * dz) return;
    const long row = ((long)(z0 + r / dy) * ny + y0 + r % dy) * nx;
    if (x0 > box.local_min[0]) dst[row + x0 - 1] = src[row + x0 - 1];
    if (x1 < box.local_max[0]) dst[row + x1] = src[row + x1];
    return;
  }
  const int bx = box.local_max[0] - box.local_min[0];
  const int by = box.local_max[1] - box.local_min[1];
  const int bz = box.local_max[2] - box.local_min[2];
  const int i = (blockIdx.x - row_blocks) * 256 + threadIdx.x;
  if (i >= outer) return;
  int r = i / bx, y, z;  // row of the shell
  if (r < (bz - dz) * by) {  // in a plane before or behind the domain's
    z = r / by;
    y = box.local_min[1] + r - z * by;
    z = box.local_min[2] + z;
    if (z >= z0) z += dz;
  } else {
    r -= (bz - dz) * by;
    z = r / (by - dy);
    y = box.local_min[1] + r - z * (by - dy);
    if (y >= y0) y += dy;
    z += z0;
  }
  const long at = ((long)z * ny + y) * nx + box.local_min[0] + i % bx;
  dst[at] = src[at];
}

// Grid view src's points around domain d into dst: what the passes over a
// domain need of a scratch grid they write (stores stay inside the domain, and
// a point reads no further than one beyond it).  The rest of the scratch grid
// stays as it is: copying whole grids took 34 us of the 10 sweeps of a 4096^2
// map, and copying every point outside the domain 3.6 ms of two pairs over 100 x
// 100 points of 16384^2 (15 us now) and 354 us of two over 64^3 points of 512^3
// (30 now).
template <typename T>
inline void CopyShell(T *dst, const T *src, int nx, int ny, int nz,
                      const __PSDomain &d, hipStream_t stream) {
  const int n[3] = {nx, ny, nz};
  __PSDomain box = d;
  int e[3], b[3];
  for (int i = 0; i < 3; ++i) {
    if (box.local_min[i] > 0) --box.local_min[i];
    if (box.local_max[i] < n[i]) ++box.local_max[i];
    e[i] = d.local_max[i] - d.local_min[i];
    b[i] = box.local_max[i] - box.local_min[i];
  }
  const int row_blocks = (e[1] * e[2] + 255) / 256;
  const int outer = ((b[2] - e[2]) * b[1] + e[2] * (b[1] - e[1])) * b[0];
  hipLaunchKernelGGL(CopyShellKernel<T>, dim3(row_blocks + (outer + 255) / 256),
                     dim3(256), 0, stream, dst, src, nx, ny, d, box, row_blocks,
                     outer);
}

// The domain of a map must lie inside every grid the map emits to; the run
// kernel stores at every domain point.
// The device view of a runtime grid as a run kernel takes it.  The runtime
// keeps one form per grid, {int dim[3]; void *p}; the 1-D and 2-D views are
// {int dim[N]; T *p}, whose pointer sits at another offset, so views are
// built field by field rather than by reinterpreting that form.
template <typename View>
inline View DevView(const __PSGrid *g) {
  View v;
  constexpr int nd = (int)(sizeof(v.dim) / sizeof(v.dim[0]));
  if (!g || !g->dev || g->num_dims != nd) {
    std::fprintf(stderr, "[physis-hip] stencil map on a %s grid where a "
                 "%d-D grid is expected\n", g ? "mismatched" : "NULL", nd);
    std::exit(EXIT_FAILURE);
  }
  for (int i = 0; i < nd; ++i) v.dim[i] = g->dev->dim[i];
  v.p = static_cast<decltype(v.p)>(g->dev->p);
  return v;
}

// The domain of a whole 3-D grid (the tiling of a red-black pass, which
// writes every point of its output).
inline __PSDomain WholeDomain(const __PSGrid *g) {
  __PSDomain d;
  for (int i = 0; i < 3; ++i) {
    d.min[i] = d.local_min[i] = 0;
    d.max[i] = d.local_max[i] = g->dim[i];
  }
  return d;
}

// The rows view of a 2-D grid: the 3-D view nx x 1 x ny of the same
// memory (equal linear offsets), in which a 2-D stencil runs on the 2.5D
// path, marching y as z.
template <typename View>
inline View RowView(const __PSGrid *g) {
  View v;
  static_assert(sizeof(v.dim) / sizeof(v.dim[0]) == 3, "a 3-D view");
  if (!g || !g->dev || g->num_dims != 2) {
    std::fprintf(stderr, "[physis-hip] stencil map on a %s grid where a "
                 "2-D grid is expected\n", g ? "mismatched" : "NULL");
    std::exit(EXIT_FAILURE);
  }
  v.dim[0] = g->dev->dim[0];
  v.dim[1] = 1;
  v.dim[2] = g->dev->dim[1];
  v.p = static_cast<decltype(v.p)>(g->dev->p);
  return v;
}
// The domain of a 2-D map in the rows view: [x0, x1) x [0, 1) x [y0, y1).
inline __PSDomain RowDomain(const __PSDomain &d) {
  __PSDomain r = d;
  r.min[2] = d.min[1];
  r.max[2] = d.max[1];
  r.local_min[2] = d.local_min[1];
  r.local_max[2] = d.local_max[1];
  r.min[1] = r.local_min[1] = 0;
  r.max[1] = r.local_max[1] = 1;
  return r;
}

// The device view of one plane of a grid of user-defined points as a grid of
// its own: component `comp` (row-major; 0 for a scalar member) of member
// `member` (the runtime stores the points member by member, the components
// of an array member one after another), with the grid's extents.
template <typename View>
inline View MemberView(__PSGrid *g, int member, int comp) {
  View v;
  constexpr int nd = (int)(sizeof(v.dim) / sizeof(v.dim[0]));
  if (!g || !g->user || g->num_dims != nd) {
    std::fprintf(stderr, "[physis-hip] stencil map on a %s grid where a "
                 "%d-D grid of user-defined points is expected\n",
                 g ? "mismatched" : "NULL", nd);
    std::exit(EXIT_FAILURE);
  }
  for (int i = 0; i < nd; ++i) v.dim[i] = g->dim[i];
  v.p = static_cast<decltype(v.p)>(__PSGridUserMember(g, member)) +
        (long)comp * (long)g->num_elms;
  return v;
}

// Checks a grid of user-defined points whose member planes a 2.5D run
// kernel reads or writes as grids: 3-D, allocated, and within 32-bit
// indexing.
inline void CheckUserGrid3D(const __PSGrid *g) {
  if (!g || !g->p || !g->user || g->num_dims != 3) {
    std::fprintf(stderr, "[physis-hip] stencil map on a freed, NULL or "
                 "mismatched grid where a 3-D grid of user-defined points is "
                 "expected\n");
    std::exit(EXIT_FAILURE);
  }
  if (g->num_elms >= (int64_t)PSINDEX_MAX) {
    std::fprintf(stderr,
                 "[physis-hip] grid of %lld elements exceeds 32-bit PSIndex\n",
                 (long long)g->num_elms);
    std::exit(EXIT_FAILURE);
  }
}

inline void CheckEmitDomain(const __PSDomain &dom, const __PSGrid *g) {
  for (int d = 0; d < g->num_dims; ++d) {
    if (dom.local_max[d] <= dom.local_min[d]) return;  // empty domain
  }
  for (int d = 0; d < g->num_dims; ++d) {
    if (dom.local_min[d] < 0 || dom.local_max[d] > g->dim[d]) {
      std::fprintf(stderr,
                   "[physis-hip] domain [%d,%d) on axis %d exceeds the "
                   "emitted grid's extent %d\n",
                   dom.local_min[d], dom.local_max[d], d, g->dim[d]);
      std::exit(EXIT_FAILURE);
    }
  }
}

// Brackets a run function.  Launches stay asynchronous, as in the
// reference's run functions (cuda_runtime_builder.cc:1465-1507: they wait
// for the device only under CUDA_KERNEL_ERROR_CHECK, which the translator's
// kernel_error_check option mirrors with __PSCheckHipError); launch errors
// are checked here, faults inside a kernel surface at the next synchronising
// call (copy-out, reduction, free).  With tracing on (--physis-trace) the
// run is timed with HIP events, which waits for it.
class RunTimer {
 public:
  explicit RunTimer(hipStream_t stream) : stream_(stream) {
    if (__ps_trace) {
      (void)hipEventCreate(&start_);
      (void)hipEventCreate(&stop_);
      (void)hipEventRecord(start_, stream_);
    }
  }
  float Stop() {
    float ms = 0.0f;
    hipError_t e = hipGetLastError();
    if (__ps_trace) {
      (void)hipEventRecord(stop_, stream_);
      if (e == hipSuccess) e = hipStreamSynchronize(stream_);
    }
    if (e != hipSuccess) {
      std::fprintf(stderr, "[physis-hip] stencil run failed: %s\n",
                   hipGetErrorString(e));
      std::exit(EXIT_FAILURE);
    }
    if (__ps_trace) {
      (void)hipEventElapsedTime(&ms, start_, stop_);
      (void)hipEventDestroy(start_);
      (void)hipEventDestroy(stop_);
    }
    return ms;
  }

 private:
  hipStream_t stream_;
  hipEvent_t start_ = nullptr, stop_ = nullptr;
};

// Whether the device holds the scratch grids (slot 8, and 9 when `second`) of
// passes of several sweeps.  Where it does not, a run takes single sweeps,
// which need none.
inline bool HaveScratch(size_t bytes, bool second) {
  return __PSHipTryScratch(8, bytes) &&
         (!second || __PSHipTryScratch(9, bytes));
}

// Scratch slots of the reducing maps of one run function: runtime scratch
// areas 1..7 (__PSHipScratch), one per map that reduces, in map order, so
// no two maps of a run share partials.
class ReduceSlots {
 public:
  int Next() {
    if (next_ > kLast) {
      std::fprintf(stderr,
                   "[physis-hip] a PSStencilRun holds more than %d "
                   "PSStencilMapReduce maps\n", kLast);
      std::exit(EXIT_FAILURE);
    }
    return next_++;
  }

 private:
  static constexpr int kLast = 7;
  int next_ = 1;
};

// Partial results of a PSStencilMapReduce map inside one run function.  A
// launch of executions i, i + 1 (a pass of several pairs; else i alone) writes
// one partial per block into Slot(i), Slot(i + 1); After(last of them) queues
// the fold of the executions so far into pinned memory once they are a batch
// (one slot is to spare for the launch that goes past it), and Finish() waits
// and hands the results to the user's array (out[i] = reduction of execution
// i).  A NULL out makes it a no-op.  (A wait and a copy per map and batch cost
// 50 us each.)
class MapReducer {
 public:
  MapReducer(void *out, int op, int type, int nblocks, int iter,
             ReduceSlots &slots)
      : out_((char *)out), op_(op), type_(type), nblocks_(nblocks),
        iter_(iter) {
    if (!out_ || iter <= 0 || nblocks <= 0) {
      out_ = nullptr;
      return;
    }
    elm_ = (type == PS_DOUBLE || type == PS_LONG) ? 8 : 4;
    const int slot = slots.Next();
    const int held = iter <= kBatch ? iter : kBatch + 1;
    base_ = (char *)__PSHipScratch(slot, (size_t)held * nblocks_ * elm_);
    pinned_ = (char *)__PSHipPinned(slot, (size_t)iter * elm_);
  }
  void *Slot(int i) const {
    if (!out_) return nullptr;
    return base_ + (size_t)(i - first_) * nblocks_ * elm_;
  }
  void After(int i) {
    if (!out_) return;
    const int count = i + 1 - first_;
    if (count < kBatch && i + 1 != iter_) return;
    __PSHipReduceFoldAsync(type_, op_, base_, nblocks_, count,
                           pinned_ + (size_t)first_ * elm_);
    first_ = i + 1;
  }
  void Finish(hipStream_t stream) {
    if (!out_) return;
    const hipError_t e = hipStreamSynchronize(stream);
    if (e != hipSuccess) {
      std::fprintf(stderr, "[physis-hip] stencil run failed: %s\n",
                   hipGetErrorString(e));
      std::exit(EXIT_FAILURE);
    }
    std::memcpy(out_, pinned_, (size_t)iter_ * elm_);
  }

 private:
  static constexpr int kBatch = 256;
  char *out_;
  int op_, type_, nblocks_, iter_;
  int elm_ = 4, first_ = 0;  // first execution not folded yet
  char *base_ = nullptr, *pinned_ = nullptr;
};

}  // namespace physis_hip

#endif  // PHYSIS_HIP_RUN_H_
