/* HIP target ABI of Physis: what code generated by physisc-hip includes and
 * what libphysis_rt_hip exports.
 *
 * Every extern "C" entry point below replaces the CUDA target's counterpart
 * one for one (reference: include/physis/physis_cuda.h:131-282 and
 * runtime/libphysis_rt_cuda.cc:25-189); argument meaning, ownership and error
 * behaviour follow the reference unless a comment says otherwise.
 *
 * Error contract (reference runtime/runtime_common_cuda.h:16-27): a failing
 * HIP call prints file:line and the HIP error string to stderr and exits with
 * EXIT_FAILURE.  The only soft failure is allocation: __PSGridNew returns
 * INVALID_GRID (NULL) when device memory cannot be obtained.
 *
 * Threading: one host thread, one process-global runtime, every launch and
 * copy on the runtime stream (the HIP null stream).  Launches are
 * asynchronous; copy-out, reductions and grid set/get are synchronous. */
#ifndef PHYSIS_PHYSIS_HIP_H_
#define PHYSIS_PHYSIS_HIP_H_

#include "physis/physis_common.h"

#ifdef __cplusplus
extern "C" {
#endif

/* ---- device views: passed by value to run kernels (physis_cuda.h:18-94) */
#define __PS_DECLARE_DEV_VIEW(nd, name, type) \
  typedef struct { int dim[nd]; type *p; } __PSGrid##nd##D##name##_dev;
__PS_DECLARE_DEV_VIEW(1, Float, float)
__PS_DECLARE_DEV_VIEW(1, Double, double)
__PS_DECLARE_DEV_VIEW(1, Int, int)
__PS_DECLARE_DEV_VIEW(1, Long, long)
__PS_DECLARE_DEV_VIEW(2, Float, float)
__PS_DECLARE_DEV_VIEW(2, Double, double)
__PS_DECLARE_DEV_VIEW(2, Int, int)
__PS_DECLARE_DEV_VIEW(2, Long, long)
__PS_DECLARE_DEV_VIEW(3, Float, float)
__PS_DECLARE_DEV_VIEW(3, Double, double)
__PS_DECLARE_DEV_VIEW(3, Int, int)
__PS_DECLARE_DEV_VIEW(3, Long, long)
#undef __PS_DECLARE_DEV_VIEW

typedef struct { int dim[3]; void *p; } __PSGrid_dev;

/* Host handle of a grid (physis_cuda.h:96-103).  p is the device buffer,
 * dense and x-fastest: offset = x + y*dim[0] + z*dim[0]*dim[1]. */
typedef struct {
  void *p;
  PSVectorInt dim;
  int elm_size;
  int num_dims;
  int64_t num_elms;
  __PSGrid_dev *dev;
  int type; /* PSPrimitiveType of the elements (HIP target addition) */
  /* Grids of user-defined points (type PS_USER): the runtime's member
   * layout (HIP target addition; NULL for primitive element types). */
  void *user;
} __PSGrid;

#ifndef PHYSIS_USER
typedef __PSGrid *PSGrid1DFloat;
typedef __PSGrid *PSGrid2DFloat;
typedef __PSGrid *PSGrid3DFloat;
typedef __PSGrid *PSGrid1DDouble;
typedef __PSGrid *PSGrid2DDouble;
typedef __PSGrid *PSGrid3DDouble;
typedef __PSGrid *PSGrid1DInt;
typedef __PSGrid *PSGrid2DInt;
typedef __PSGrid *PSGrid3DInt;
typedef __PSGrid *PSGrid1DLong;
typedef __PSGrid *PSGrid2DLong;
typedef __PSGrid *PSGrid3DLong;
#define DeclareGrid1D(name, type) typedef __PSGrid *PSGrid1D##name;
#define DeclareGrid2D(name, type) typedef __PSGrid *PSGrid2D##name;
#define DeclareGrid3D(name, type) typedef __PSGrid *PSGrid3D##name;
#define PSGridDim(p, d) ((p)->dim[(d)])
#define __PSGridDimDev(p, d) ((p)->dim[d])
#endif

/* ---- lifecycle (physis_common.h:78-79; libphysis_rt_cuda.cc:25-41).
 * PSInit parses --physis-trace and selects device 0 (or $PHYSIS_HIP_DEVICE).
 * PSFinalize synchronises and releases runtime-owned buffers; it does not
 * reset the device, so a host process may keep other HIP state alive. */
extern void PSInit(int *argc, char ***argv, int grid_num_dims, ...);
extern void PSFinalize(void);

/* ---- grids (physis_cuda.h:131-145; libphysis_rt_cuda.cc:48-177) */
typedef void *(*__PSGrid_devNewFunc)(int num_dims, PSVectorInt dim);
typedef void (*__PSGrid_devFreeFunc)(void *);
typedef void (*__PSGrid_devCopyinFunc)(void *g, const void *src,
                                       size_t num_elms);
typedef void (*__PSGrid_devCopyoutFunc)(void *g, void *dst, size_t num_elms);

/* Allocates a zero-filled device grid; INVALID_GRID on allocation failure.
 * func is the user-type allocator hook; NULL for primitive element types.
 * A type_info with members (user-defined point types, type PS_USER,
 * reference_runtime_builder.cc:959-1065) makes a grid stored member by
 * member, one dense plane per scalar component (the CUDA target's layout,
 * cuda_runtime_builder.cc:262-345); copy-in and copy-out then convert from
 * and to the host's array of structs. */
extern __PSGrid *__PSGridNew(__PSGridTypeInfo *type_info, int num_dims,
                             PSVectorInt dim, __PSGrid_devNewFunc func);
/* Releases the device buffer and the handle itself (the reference leaks the
 * handle, libphysis_rt_cuda.cc:101-112). */
extern void __PSGridFree(void *g, __PSGrid_devFreeFunc func);
/* Whole-grid synchronous host->device / device->host copies of
 * num_elms*elm_size bytes (libphysis_rt_cuda.cc:114-137). */
extern void __PSGridCopyin(void *g, const void *src_array,
                           __PSGrid_devCopyinFunc func);
extern void __PSGridCopyout(void *g, void *dst_array,
                            __PSGrid_devCopyoutFunc func);
/* Kept for generated code that calls it after each launch; does nothing
 * (libphysis_rt_cuda.cc:139-140). */
extern void __PSGridSwap(__PSGrid *g);
extern int __PSGridGetID(__PSGrid *g);
/* Writes / reads one element; indices follow buf as num_dims PSIndex
 * varargs (libphysis_rt_cuda.cc:162-177; REF physis_ref.h:46). */
extern void __PSGridSet(__PSGrid *g, void *buf, ...);
extern void __PSGridGet(__PSGrid *g, void *buf, ...);

/* Sub-grid transfers: the box [offset, offset+size) of a grid to or from a
 * dense host array of prod(size) elements, x fastest.  Non-contiguous boxes
 * are packed on the device (reference runtime/buffer_cuda.cu:88-311, used
 * there for MPI halo staging; BufferCUDADev::Copyin/Copyout). */
extern void __PSGridCopyoutSubgrid(__PSGrid *g, void *dst,
                                   const PSIndex *offset, const PSIndex *size);
extern void __PSGridCopyinSubgrid(__PSGrid *g, const void *src,
                                  const PSIndex *offset, const PSIndex *size);

/* Check-and-abort after launches when HIP_KERNEL_ERROR_CHECK is set in the
 * translator configuration (analogue of __PSCheckCudaError,
 * physis_cuda.h:150). */
extern void __PSCheckHipError(const char *message);

/* ---- reductions over all num_elms elements (physis_cuda.h:272-282;
 * runtime/reduce_cuda.h:19-40).  The result is written to *buf in the grid
 * element type; the call returns after the value is on the host. */
extern void __PSReduceGridFloat(void *buf, enum PSReduceOp op, __PSGrid *g);
extern void __PSReduceGridDouble(void *buf, enum PSReduceOp op, __PSGrid *g);
extern void __PSReduceGridInt(void *buf, enum PSReduceOp op, __PSGrid *g);
extern void __PSReduceGridLong(void *buf, enum PSReduceOp op, __PSGrid *g);

/* ---- reduction that allocates nothing.  No counterpart in the reference:
 * for callers that cannot allocate device or pinned memory (code under HIP
 * graph capture, tight serving loops, harnesses that forbid hipMalloc).
 * Same result as __PSReduceGrid{Float,Double,Int,Long} for `type` PS_FLOAT,
 * PS_DOUBLE, PS_INT, PS_LONG (bit-identical: the same kernels and block
 * count).  The per-block partials and the result live in a fixed 32 KiB
 * device array of the library (up to 4096 partials of 8 bytes, enough for
 * any grid: the stage-1 block count is capped at that), one per GPU, whose
 * address is looked up when the runtime is set up; PSInit must have been
 * called.  The result is copied into *buf (host memory) and the call
 * returns after it is there.  Calls that overlap on one GPU (several host
 * threads, or streams of other libraries using the array) race on it. */
extern void __PSReduceGridNoAlloc(void *buf, enum PSReduceOp op, __PSGrid *g,
                                  PSType type);

/* ---- HIP target additions (no reference counterpart) */
/* Device address of the first component plane of member `member` of a grid
 * of user-defined points; component c of an array member (row-major over its
 * extents) is c * num_elms elements further. */
extern void *__PSGridUserMember(__PSGrid *g, int member);
/* Stream all runtime work and generated launches are issued on, as a
 * hipStream_t stored in a void*. */
extern void *__PSHipStream(void);
/* Number of compute units of the selected device (sizes launches). */
extern int __PSHipNumCUs(void);
/* Device scratch area number `slot` (0 <= slot < 10) of at least `bytes`,
 * kept and grown across calls; generated run functions keep the per-block
 * partials of fused reductions in slots 1..7 and the ping-pong grids of
 * two-sweep (temporally blocked) runs in slots 8 and 9; slot 0 is
 * PSReduce's own. */
extern void *__PSHipScratch(int slot, size_t bytes);
/* The same, or NULL when the device memory is out. */
extern void *__PSHipTryScratch(int slot, size_t bytes);
/* Folds the per-block partial results of a PSStencilMapReduce map: row r of
 * the device array partials (count rows of nparts elements of `type`) is
 * reduced with op into host_out[r]; float sums accumulate in double.
 * Synchronous. */
extern void __PSHipReduceFold(int type, int op, const void *partials,
                              int nparts, int count, void *host_out);
/* Pinned host area number `slot` (0 <= slot < 10) of at least `bytes`, kept
 * and grown across calls: kernels write it, the host reads it after a wait
 * on the runtime stream.  Generated run functions keep the results of fused
 * reductions in slots 1..7; slot 0 is __PSHipReduceFold's own (the waiting form,
 * for callers of their own: generated run functions use the one below). */
extern void *__PSHipPinned(int slot, size_t bytes);
/* __PSHipReduceFold without the wait: the results are in `out` (pinned or
 * device memory) once the runtime stream has drained. */
extern void __PSHipReduceFoldAsync(int type, int op, const void *partials,
                                   int nparts, int count, void *out);

/* ---- offset helpers (physis_cuda.h:196-269): host and device versions. */
#if defined(__HIPCC__)
#define __PS_HD __host__ __device__
#else
#define __PS_HD
#endif

static inline __PS_HD PSIndex __PSGridGetOffset1D(const __PSGrid *g,
                                                  PSIndex i1) {
  (void)g;
  return i1;
}
static inline __PS_HD PSIndex __PSGridGetOffset2D(const __PSGrid *g,
                                                  PSIndex i1, PSIndex i2) {
  return i1 + i2 * g->dim[0];
}
static inline __PS_HD PSIndex __PSGridGetOffset3D(const __PSGrid *g,
                                                  PSIndex i1, PSIndex i2,
                                                  PSIndex i3) {
  return i1 + i2 * g->dim[0] + i3 * g->dim[0] * g->dim[1];
}
static inline __PS_HD PSIndex __PSGridGetOffsetPeriodic1D(const __PSGrid *g,
                                                          PSIndex i1) {
  return (i1 + g->dim[0]) % g->dim[0];
}
static inline __PS_HD PSIndex __PSGridGetOffsetPeriodic2D(const __PSGrid *g,
                                                          PSIndex i1,
                                                          PSIndex i2) {
  return __PSGridGetOffsetPeriodic1D(g, i1) +
         (i2 + g->dim[1]) % g->dim[1] * g->dim[0];
}
static inline __PS_HD PSIndex __PSGridGetOffsetPeriodic3D(const __PSGrid *g,
                                                          PSIndex i1,
                                                          PSIndex i2,
                                                          PSIndex i3) {
  return __PSGridGetOffsetPeriodic2D(g, i1, i2) +
         (i3 + g->dim[2]) % g->dim[2] * g->dim[0] * g->dim[1];
}

/* Device-view forms; g points at any __PSGrid<N>D<T>_dev (dim first). */
static inline __PS_HD PSIndex __PSGridGetOffset1DDev(const void *g,
                                                     PSIndex i1) {
  (void)g;
  return i1;
}
static inline __PS_HD PSIndex __PSGridGetOffset2DDev(const void *g,
                                                     PSIndex i1, PSIndex i2) {
  const int *d = (const int *)g;
  return i1 + i2 * d[0];
}
static inline __PS_HD PSIndex __PSGridGetOffset3DDev(const void *g,
                                                     PSIndex i1, PSIndex i2,
                                                     PSIndex i3) {
  const int *d = (const int *)g;
  return i1 + i2 * d[0] + i3 * d[0] * d[1];
}
static inline __PS_HD PSIndex __PSGridGetOffsetPeriodic1DDev(const void *g,
                                                             PSIndex i1) {
  const int *d = (const int *)g;
  return (i1 + d[0]) % d[0];
}
static inline __PS_HD PSIndex __PSGridGetOffsetPeriodic2DDev(const void *g,
                                                             PSIndex i1,
                                                             PSIndex i2) {
  const int *d = (const int *)g;
  return (i1 + d[0]) % d[0] + (i2 + d[1]) % d[1] * d[0];
}
static inline __PS_HD PSIndex __PSGridGetOffsetPeriodic3DDev(const void *g,
                                                             PSIndex i1,
                                                             PSIndex i2,
                                                             PSIndex i3) {
  const int *d = (const int *)g;
  return (i1 + d[0]) % d[0] + (i2 + d[1]) % d[1] * d[0] +
         (i3 + d[2]) % d[2] * d[0] * d[1];
}
#undef __PS_HD

#ifdef __cplusplus
}
#endif

#endif /* PHYSIS_PHYSIS_HIP_H_ */
