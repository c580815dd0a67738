// Building blocks of the resident-tile passes that physisc-hip emits for
// fusable maps on small grids.
//
// A small grid's z-marching pass is a chain of latencies: a launch, then a
// barrier and a load per few planes, on blocks that own a handful of points.
// A resident-tile pass does T sweeps of a map pair per launch on tiles that
// stay in LDS: a block loads its tile with a T-point halo once, then computes
// sweep after sweep between two LDS buffers, each on a box one point smaller,
// and stores the last (one barrier per sweep).  The price is the halo's
// arithmetic (a tile of 16x8x8 computes 2.4 times its points over 4 sweeps),
// which is cheap as long as the grid leaves most of the chip idle.
#ifndef PHYSIS_HIP_TILE_H_
#define PHYSIS_HIP_TILE_H_

#include <cstdint>

#include "physis/hip/run.h"
#include "physis/hip/stencil.h"
#include "physis/physis_hip.h"

namespace physis_hip {

// Shape of a resident tile of TX x TY x TZ points for T sweeps by NT
// threads.  The points are numbered by shells: shell s is the points s
// points outside the tile (shell 0 the tile itself); sweep t (1 .. T)
// computes shells 0 .. T - t.  Thread i owns points i, i + NT, ... of each
// shell, so that a sweep's loop ends with its shells.
template <int T_, int TX_, int TY_, int TZ_, int NT_>
struct Tile {
  static constexpr int T = T_, TX = TX_, TY = TY_, TZ = TZ_, NT = NT_;
  // the staged box: halo T, row pitch RX
  static constexpr int RX = TX + 2 * T, RY = TY + 2 * T, RZ = TZ + 2 * T;
  static constexpr int kElems = RX * RY * RZ;
  static constexpr int kLoads = (kElems + NT - 1) / NT;
  static constexpr int Box(int s) {  // points of shells 0 .. s
    return (TX + 2 * s) * (TY + 2 * s) * (TZ + 2 * s);
  }
  static constexpr int Shell(int s) { return s == 0 ? Box(0) : Box(s) - Box(s - 1); }
  // owned points per thread in shells 0 .. s
  static constexpr int Owned(int s) {
    int k = 0;
    for (int i = 0; i <= s; ++i) k += (Shell(i) + NT - 1) / NT;
    return k;
  }
  static constexpr int K = Owned(T - 1);
  // Points of the sweep t's loop: k < Count(t)
  static constexpr int Count(int t) { return Owned(T - t); }

  // LDS offsets (x + RX (y + RY z)) of the owned points: entry k * NT + i is
  // thread i's k-th point, -1 where a shell has none left.
  struct Table {
    short at[K * NT];
  };
  static constexpr Table Make() {
    Table t{};
    int k0 = 0;
    for (int s = 0; s < T; ++s) {
      const int x0 = T - s, y0 = T - s, z0 = T - s;
      const int x1 = T + TX + s, y1 = T + TY + s, z1 = T + TZ + s;
      int n = k0 * NT;
      for (int z = z0; z < z1; ++z)
        for (int y = y0; y < y1; ++y) {
          const bool rim = s == 0 || z == z0 || z == z1 - 1 || y == y0 ||
                           y == y1 - 1;
          // a row of the shell: whole on its rim, else its two ends
          for (int x = x0; x < x1; x += rim ? 1 : x1 - 1 - x0)
            t.at[n++] = (short)(x + RX * (y + RY * z));
        }
      k0 += (Shell(s) + NT - 1) / NT;
      for (; n < k0 * NT; ++n) t.at[n] = -1;
    }
    return t;
  }
};

template <typename TILE>
struct TileTable {
  static __device__ const typename TILE::Table value;
};
template <typename TILE>
__device__ const typename TILE::Table TileTable<TILE>::value = TILE::Make();

// One owned point: its LDS offset and its coordinates in the grid.
struct TilePoint {
  int at, x, y, z;
};
template <typename TILE>
__device__ __forceinline__ TilePoint OwnedPoint(int k, int x0, int y0, int z0) {
  TilePoint p;
  p.at = TileTable<TILE>::value.at[k * TILE::NT + threadIdx.x];
  const int a = p.at < 0 ? 0 : p.at;
  const int r = a / TILE::RX, z = r / TILE::RY;
  p.x = x0 - TILE::T + a - r * TILE::RX;
  p.y = y0 - TILE::T + r - z * TILE::RY;
  p.z = z0 - TILE::T + z;
  return p;
}

// Loads the tile at (x0, y0, z0) with its halo; a periodic grid wraps, other
// points outside the grid have no value that a map reads.
template <typename TILE, bool PERIODIC, typename E>
__device__ __forceinline__ void LoadTile(E *lds, const E *p, const int *dim,
                                         int x0, int y0, int z0) {
  const int n = dim[0] * dim[1] * dim[2];
  const BufWin<E> w = BufWin<E>::Make(p, n, 0, n);
  E v[TILE::kLoads][1];
#pragma unroll
  for (int k = 0; k < TILE::kLoads; ++k) {
    const int e = k * TILE::NT + threadIdx.x;
    const int r = e / TILE::RX, zz = r / TILE::RY;
    int x = x0 - TILE::T + e - r * TILE::RX;
    int y = y0 - TILE::T + r - zz * TILE::RY;
    int z = z0 - TILE::T + zz;
    bool in = e < TILE::kElems;
    if (PERIODIC) {
      x = WrapNear(x, dim[0]);
      y = WrapNear(y, dim[1]);
      z = WrapNear(z, dim[2]);
    } else {
      in = in && x >= 0 && x < dim[0] && y >= 0 && y < dim[1] && z >= 0 &&
           z < dim[2];
    }
    w.template Load<1>(in ? x + dim[0] * (y + dim[1] * z) : kDrop, v[k]);
  }
#pragma unroll
  for (int k = 0; k < TILE::kLoads; ++k) {
    const int e = k * TILE::NT + threadIdx.x;
    if (e < TILE::kElems) lds[e] = v[k][0];
  }
}

// ------------------------------------------------------ launch arithmetic
// Tiles of one small grid per compute unit, and those of larger ones, whose
// halo costs less.  Measured for T = 4 (us per sweep of the clamped 7-point
// diffusion, small tile / mid tile): 64^3 1.94 / 2.51, 80^3 2.75 / 2.63, 96^3
// 4.53 / 3.85, 128^3 7.97 / 6.49.  A kernel with the 12 centre-only
// grids of the 19-point Jacobi sweep gains nothing (its tiles read the halo's
// values of every one of them: 96^3 14.4 against 10.1), nor does one of 27 points
// (their halo's arithmetic: 256x60x60 9.5 against 8.4).
template <int T> using SmallTile = Tile<T, 16, 8, 8, 1024>;
template <int T> using MidTile = Tile<T, 16, 16, 8, 1024>;
// Whether a pass over a whole grid runs in tiles, from what a sweep costs in
// either kind of pass (us): 1.5 + 1.2 per round of mid tiles (a block per CU; 23
// to 24 for 18 rounds), and for z-marching pairs the lines below by the million
// points of their padded tiles, fitted to 130 grids where the kinds lie close:
// the rule's choice is 0.5 % slower than the better one in the mean, and 11 % at
// most (red-black 112x230x33; clamped 180x191x27 7 %).  Tiles and pairs, clamped
// 7-point map: 112^3 5.2 and 6.3, 128^3 6.4 and 6.0, 150^3 11.3 and 9.3, 250x80x80
// 6.5 and 5.7, 250x64x64 4.0 and 4.9, 64x256x256 11.4 and 11.9, 80x137x356 11.3
// and 10.7, 16x400x400 8.1 and 22.7, 48x300x300 12.5 and 15.3, 100x68x124 5.0 and
// 5.7, 180x110x96 6.6 and 6.0, 148x124x87 6.5 and 6.2 (periodic 6.4 and 6.8,
// red-black 6.4 and 5.6).  Past 16 million points (a grid of 64 MB) nothing was
// measured, and the tiles' halos no longer come from the cache.
inline bool TilesBeatPairs(const int *dim, bool periodic, bool colours) {
  constexpr long kCUs = 256;
  const auto in = [](long n, long t) { return (n + t - 1) / t; };
  const long blocks = in(dim[0], 16) * in(dim[1], 16) * in(dim[2], 8);
  if (blocks > 16000000 / 2048) return false;
  const bool narrow = PairVX(dim, periodic, colours) == 2;
  const int tx = narrow ? 128 : 256;
  const double points = 1e-6 * in(dim[0], tx) * tx * in(dim[1], 8) * 8 * dim[2];
  const double pair = colours    ? narrow ? 4.5 + 0.9 * points : 3.6 + 0.7 * points
                      : periodic ? narrow ? 5.4 + 1.1 * points : 4.6 + 0.9 * points
                      : narrow   ? 4.3 + 0.95 * points : 3.8 + 0.8 * points;
  return 1.5 + 1.2 * in(blocks, kCUs) < pair;
}

// Padded points (millions) of an extent box in tiles of tx x ty x tz.
inline double PaddedMega(long ex, long ey, long ez, int tx, int ty, int tz) {
  const auto up = [](long n, int t) { return (double)((n + t - 1) / t * t); };
  return up(ex, tx) * up(ey, ty) * up(ez, tz) * 1e-6;
}
// Whether passes of several sweeps over a whole grid beat single sweeps.  Rows
// that are no multiples of 4 and fit a 64-point tile run their single sweeps at
// one point per lane there, half the lanes of the narrowest z-marching pass, and
// those sweeps cost less than it (us a sweep, single and pair, clamped 7-point:
// 41x700x700 47 and 73, 41x1000x1000 87 and 133; red-black iteration 54x292x284
// 27 and 30); tiles beat them as long as the sweeps' latency counts (1.4 + 2.5
// per million padded points against 6 + 1.5: 41x300x300 13 and 15, 33x500x500
// 31 and 29).  Colour sweeps do without the last column and its tile: they also
// win over large grids whose rows end just past a tile of the pass (us an
// iteration, sweeps and pass: 129x249x249 34 and 35, 129x422x422 84 and 95,
// 129x622x623 160 and 193, 257x299x299 80 and 87, 131x617x618 171 and 193,
// 135x608x609 176 and 181; but 131x247x247 42 and 34, 141x403x404 89 and 79,
// 257x200x200 43 and 40, 258x440x440 194 and 167, 513x312x312 165 and 141); a lane
// of a 128-point tile counts 1.2 times.  A kernel of many gets (`tiles` false) has
// no tiles and pays for every lane: its passes have to cover the rows with no more
// of them.
inline bool PassesPay(const int *dim, bool periodic, bool colours, bool tiles) {
  if (dim[0] % 4 == 0) return true;
  const int wide = PairVX(dim, periodic, colours) == 2 ? 128 : 256;
  if (!tiles) return (dim[0] + wide - 1) / wide * wide <= (dim[0] + 63) / 64 * 64;
  if (dim[0] > 64) {
    const long lanes = (dim[0] + wide - 1) / wide * wide;
    const long sweep = (dim[0] - 1 + 63) / 64 * 64;
    const double n = (double)dim[0] * dim[1] * dim[2];
    return !colours || TilesBeatPairs(dim, periodic, colours) ||
           !(((wide == 128 ? 1.2 : 1.0) * lanes >= 1.75 * sweep &&
              n >= (lanes == 256 ? 7.5e6 : 2e7)) ||
             (lanes >= 1.85 * dim[0] && n >= 2e7));
  }
  return TilesBeatPairs(dim, periodic, colours) &&
         2.5 * PaddedMega(dim[0], dim[1], dim[2], 16, 16, 8) <
             4.6 + 1.5 * PaddedMega(dim[0], dim[1], dim[2], 64, 1, 1);
}
// Whether the last of an odd number of red-black iterations runs as two colour
// sweeps in place: a pass ends in the scratch grid there and takes a copy.  On
// rows that are no multiples of 4 (us of one iteration, sweeps, pass and copy):
// 129^3 20 and 23, 150^3 23 and 28, 257^3 63 and 81, 54x200x200 21 and 28, but
// 255^3 63 and 59, 65^3 14 and 8, 383x200x150 48 and 50; the estimates fit these (sweeps 5.5 + 0.75 per
// million points + 0.95 per million of the lanes, twice; copies 2.2 + 0.9 per MB
// up to 8.5 + 0.155).  Rows of multiples of 4 take the pass, as measured faster
// from 255^3 on.
inline bool RedBlackLastAsSweeps(const int *dim, int iterations) {
  if (iterations % 2 == 0 || dim[0] % 4 == 0) return false;
  const bool narrow = PairVX(dim, false, true) == 2;
  const double n = PaddedMega(dim[0], dim[1], dim[2], 1, 1, 1), mb = 4 * n;
  const double sweeps = 2 * (5.5 + 0.75 * n + 0.95 * PaddedMega(dim[0], dim[1],
                                                                 dim[2], 64, 1, 1));
  const double pass =
      TilesBeatPairs(dim, false, true)
          ? 2 * (1.4 + 2.5 * PaddedMega(dim[0], dim[1], dim[2], 16, 16, 8))
          : 2 * (4.3 + (narrow ? 1.0 : 0.83) *
                           PaddedMega(dim[0], dim[1], dim[2], narrow ? 128 : 256, 8, 1));
  const double copy = 2.2 + 0.9 * mb < 8.5 + 0.155 * mb ? 2.2 + 0.9 * mb
                                                        : 8.5 + 0.155 * mb;
  return sweeps < 1.08 * (pass + copy);
}

// Whether a pass over a domain inside a grid of `points` points runs in tiles,
// beside EmitFusedDomainKernel's pairs (tiles of 256 x 12 points): us a sweep
// about 1.4 + 2.5 per million points of the padded tiles here and 4.3 + 0.83
// there.  Tiles and pairs, 5-point map over the interior, no results, 80 sweeps:
// 256x60x60 3.8 and 5.3, 512x40x40 3.8 and 5.5, 128x130x130 6.3 and 7.8,
// 24x300x300 8.8 and 21.5, 260x92x90 7.6 and 7.9, 300x100x70 7.8 and 7.7,
// 512x128x32 6.3 and 6.6, 512x66x62 6.4 and 6.0, 256x92x92 7.4 and 5.7,
// 1024x46x46 7.5 and 6.4; with a centre-only grid and a result per sweep both
// cost about 1.4 times as much (256x92x92 9.8 and 8.5).  Past kTileMaxPoints
// nothing was measured; the byte offsets of a grid of kTileMaxGrid 8-byte points
// stay within a buffer window.
constexpr long kTileMaxPoints = 2200000;
constexpr int64_t kTileMaxGrid = 1 << 27;
inline bool TilesBeatDomainPairs(const __PSDomain &d, int64_t points) {
  const auto up = [](int n, int t) { return (double)((n + t - 1) / t * t); };
  long e[3];
  for (int i = 0; i < 3; ++i) e[i] = d.local_max[i] - d.local_min[i];
  if (points > kTileMaxGrid || e[0] * e[1] * e[2] > kTileMaxPoints) return false;
  const double tile = up(e[0], 16) * up(e[1], 16) * up(e[2], 8) * 1e-6;
  const double wide = up(d.local_max[0], 256) - d.local_min[0] / 256 * 256;
  const double pair = wide * up(e[1], 12) * e[2] * 1e-6;
  return 2.5 * tile - 0.83 * pair < 2.9;
}

// Whether passes of a domain pair of 4 points per lane (EmitFusedDomainKernel's
// with few centre-only grids, or tiles) beat single sweeps, on rows of nx points
// that are no multiples of 4: single sweeps run at one point per lane in tiles
// of 64 there.  Us a sweep, single and pair, 5-point map over the interior:
// 41x300x300 12 and 27, 41x1000x1000 80 and 274, 97x300x300 23 and 29,
// 129x400x400 48 and 57, 290x200x200 30 and 30, 257x200x200 and 161x300x300
// faster as pairs; tiles as above.  27 points (`tiles` false), 4 pairs: 191x256x200
// 241 and 263 us, 321x256x200 400 and 471, 222x60x60 61 and 65, 255x256x200
// faster as pairs.
inline bool DomainPassesPay(const __PSDomain &d, int nx, int64_t points,
                            bool use_tiles) {
  if (nx % 4 == 0) return true;
  long e[3];
  for (int i = 0; i < 3; ++i) e[i] = d.local_max[i] - d.local_min[i];
  const auto tiles = [&](int t) {
    return (d.local_max[0] + t - 1) / t - d.local_min[0] / t;
  };
  if (!use_tiles)
    return tiles(256) * 4 <= tiles(64) && e[0] * e[1] * e[2] >= 2000000;
  if (TilesBeatDomainPairs(d, points))
    return 2.5 * PaddedMega(e[0], e[1], e[2], 16, 16, 8) <
           1.6 + 1.5 * tiles(64) * 64e-6 * e[1] * e[2];
  return tiles(256) * 12 <= tiles(64) * 5;
}

// Per-block partials of each sweep of a pass (NULL: none).
struct TileReds {
  void *p[4];
};

struct TileShape {
  int tiles_x, tiles_y, blocks;
};
template <typename TILE>
inline TileShape TileGrid(const __PSDomain &d) {
  TileShape s = {0, 0, 0};
  int n[3];
  const int t[3] = {TILE::TX, TILE::TY, TILE::TZ};
  for (int i = 0; i < 3; ++i) {
    const int e = d.local_max[i] - d.local_min[i];
    if (e <= 0) return s;
    n[i] = (e + t[i] - 1) / t[i];
  }
  s.tiles_x = n[0];
  s.tiles_y = n[1];
  s.blocks = n[0] * n[1] * n[2];
  return s;
}

// Whether a domain runs in small tiles (else in mid ones), and its blocks.
inline bool InSmallTiles(const __PSDomain &d) {
  return TileGrid<SmallTile<2>>(d).blocks <= __PSHipNumCUs();
}
inline int TileBlocks(const __PSDomain &d) {
  return InSmallTiles(d) ? TileGrid<SmallTile<2>>(d).blocks
                         : TileGrid<MidTile<2>>(d).blocks;
}

}  // namespace physis_hip

#endif  // PHYSIS_HIP_TILE_H_
