/* Maps that read past the ends of rows whose extents are multiples of
 * nothing: non-periodic gets over the whole grid (an index past the end of a
 * row names the next row's points, one outside the grid 0), periodic gets
 * two points away, a map pair over the interior, pairs over a box of the
 * grid whose kernels return the change of each point, and a red-black map of
 * an 8-byte grid. */
#include "physis/physis.h"

static void corners(const int x, const int y, const int z, PSGrid3DFloat g,
                    PSGrid3DFloat g2) {
  float v = 0.5f * PSGridGet(g, x, y, z) + PSGridGet(g, x+1, y, z) +
            2.0f * PSGridGet(g, x+1, y-1, z) +
            3.0f * PSGridGet(g, x-1, y+1, z) +
            4.0f * PSGridGet(g, x+1, y+1, z+1) +
            5.0f * PSGridGet(g, x-1, y-1, z-1) +
            6.0f * PSGridGet(g, x+1, y, z-1);
  PSGridEmit(g2, v);
}

static void corners_double(const int x, const int y, const int z,
                           PSGrid3DDouble g, PSGrid3DDouble g2) {
  double v = 0.5 * PSGridGet(g, x, y, z) + PSGridGet(g, x+1, y, z) +
             2.0 * PSGridGet(g, x+1, y-1, z) +
             3.0 * PSGridGet(g, x-1, y+1, z) +
             4.0 * PSGridGet(g, x+1, y+1, z+1) +
             5.0 * PSGridGet(g, x-1, y-1, z-1) +
             6.0 * PSGridGet(g, x+1, y, z-1);
  PSGridEmit(g2, v);
}

static void corners2d(const int x, const int y, PSGrid2DFloat g,
                      PSGrid2DFloat g2) {
  float v = 0.5f * PSGridGet(g, x, y) + 2.0f * PSGridGet(g, x+1, y-1) +
            3.0f * PSGridGet(g, x-1, y+1) + 4.0f * PSGridGet(g, x+1, y);
  PSGridEmit(g2, v);
}

static void wrap2(const int x, const int y, const int z, PSGrid3DFloat g,
                  PSGrid3DFloat g2) {
  float v = 0.5f * PSGridGet(g, x, y, z) +
            2.0f * PSGridGetPeriodic(g, x+2, y-1, z) +
            3.0f * PSGridGetPeriodic(g, x-2, y+1, z) +
            4.0f * PSGridGetPeriodic(g, x+1, y, z+1) +
            5.0f * PSGridGetPeriodic(g, x-1, y, z-1);
  PSGridEmit(g2, v);
}

static void inner(const int x, const int y, const int z, PSGrid3DFloat g,
                  PSGrid3DFloat g2, float w) {
  float v = PSGridGet(g, x, y, z) + PSGridGet(g, x+1, y-1, z) +
            PSGridGet(g, x-1, y+1, z) + PSGridGet(g, x, y, z+1) +
            PSGridGet(g, x, y, z-1);
  PSGridEmit(g2, v * w);
}

static float settle(const int x, const int y, const int z, PSGrid3DFloat g,
                    PSGrid3DFloat g2, PSGrid3DFloat c, float w) {
  float u = PSGridGet(g, x, y, z);
  float v = u + PSGridGet(g, x+1, y-1, z) + PSGridGet(g, x-1, y+1, z) +
            PSGridGet(g, x, y, z+1) + PSGridGet(g, x, y, z-1);
  v = v * w + PSGridGet(c, x, y, z);
  PSGridEmit(g2, v);
  return v - u;
}

static double settle_square(const int x, const int y, const int z,
                            PSGrid3DFloat g, PSGrid3DFloat g2, float w) {
  float u = PSGridGet(g, x, y, z);
  float v = u + PSGridGet(g, x+1, y-1, z) + PSGridGet(g, x-1, y+1, z) +
            PSGridGet(g, x, y, z+1) + PSGridGet(g, x, y, z-1);
  v = v * w;
  PSGridEmit(g2, v);
  double d = v - u;
  return d * d;
}

static void inner2d(const int x, const int y, PSGrid2DFloat g,
                    PSGrid2DFloat g2, float w) {
  float v = PSGridGet(g, x, y) + PSGridGet(g, x+1, y-1) +
            PSGridGet(g, x-1, y+1) + PSGridGet(g, x-1, y) +
            PSGridGet(g, x+1, y+1);
  PSGridEmit(g2, v * w);
}

static void relax_double(const int x, const int y, const int z,
                         PSGrid3DDouble g) {
  double v = PSGridGet(g, x, y, z) + PSGridGet(g, x+1, y, z) +
             PSGridGet(g, x-1, y, z) + PSGridGet(g, x, y+1, z) +
             PSGridGet(g, x, y-1, z) + PSGridGet(g, x, y, z+1) +
             PSGridGet(g, x, y, z-1);
  PSGridEmit(g, v * 0.125);
}

static PSDomain3D whole(PSGrid3DFloat g) {
  return PSDomain3DNew(0, PSGridDim(g, 0), 0, PSGridDim(g, 1), 0,
                       PSGridDim(g, 2));
}

/* One sweep g -> g2 over the whole of g2 (which may be larger than g). */
void ragged_corners(PSGrid3DFloat g, PSGrid3DFloat g2) {
  PSStencilRun(PSStencilMap(corners, whole(g2), g, g2));
}

void ragged_corners_double(PSGrid3DDouble g, PSGrid3DDouble g2) {
  PSDomain3D d = PSDomain3DNew(0, PSGridDim(g, 0), 0, PSGridDim(g, 1), 0,
                               PSGridDim(g, 2));
  PSStencilRun(PSStencilMap(corners_double, d, g, g2));
}

void ragged_corners2d(PSGrid2DFloat g, PSGrid2DFloat g2) {
  PSDomain2D d = PSDomain2DNew(0, PSGridDim(g, 0), 0, PSGridDim(g, 1));
  PSStencilRun(PSStencilMap(corners2d, d, g, g2));
}

void ragged_wrap2(PSGrid3DFloat g, PSGrid3DFloat g2) {
  PSStencilRun(PSStencilMap(wrap2, whole(g), g, g2));
}

/* count pairs of sweeps g -> g2 -> g over the interior. */
void ragged_inner(PSGrid3DFloat g, PSGrid3DFloat g2, int count, float w) {
  PSDomain3D d = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1,
                               1, PSGridDim(g, 2) - 1);
  PSStencilRun(PSStencilMap(inner, d, g, g2, w), PSStencilMap(inner, d, g2, g, w),
               count);
}

/* count pairs over the box; more[i] and back[i]: the largest change of the
 * sweeps of pair i. */
void ragged_settle(PSGrid3DFloat g, PSGrid3DFloat g2, PSGrid3DFloat c, int x0,
                   int x1, int y0, int y1, int z0, int z1, int count, float w,
                   float *more, float *back) {
  PSDomain3D d = PSDomain3DNew(x0, x1, y0, y1, z0, z1);
  PSStencilRun(PSStencilMapReduce(more, PS_MAX, settle, d, g, g2, c, w),
               PSStencilMapReduce(back, PS_MAX, settle, d, g2, g, c, w),
               count);
}

/* The same without the third grid; the sums of the squared changes. */
void ragged_settle_square(PSGrid3DFloat g, PSGrid3DFloat g2, int x0, int x1,
                          int y0, int y1, int z0, int z1, int count, float w,
                          double *more, double *back) {
  PSDomain3D d = PSDomain3DNew(x0, x1, y0, y1, z0, z1);
  PSStencilRun(PSStencilMapReduce(more, PS_SUM, settle_square, d, g, g2, w),
               PSStencilMapReduce(back, PS_SUM, settle_square, d, g2, g, w),
               count);
}

/* count pairs of sweeps over a box, without results. */
void ragged_box(PSGrid3DFloat g, PSGrid3DFloat g2, int x0, int x1, int y0,
                int y1, int z0, int z1, int count, float w) {
  PSDomain3D d = PSDomain3DNew(x0, x1, y0, y1, z0, z1);
  PSStencilRun(PSStencilMap(inner, d, g, g2, w), PSStencilMap(inner, d, g2, g, w),
               count);
}

void ragged_box2d(PSGrid2DFloat g, PSGrid2DFloat g2, int x0, int x1, int y0,
                  int y1, int count, float w) {
  PSDomain2D d = PSDomain2DNew(x0, x1, y0, y1);
  PSStencilRun(PSStencilMap(inner2d, d, g, g2, w),
               PSStencilMap(inner2d, d, g2, g, w), count);
}

void ragged_relax_double(PSGrid3DDouble g, int count) {
  PSDomain3D d = PSDomain3DNew(1, PSGridDim(g, 0) - 1, 1, PSGridDim(g, 1) - 1,
                               1, PSGridDim(g, 2) - 1);
  PSStencilRun(PSStencilMapRedBlack(relax_double, d, g), count);
}
