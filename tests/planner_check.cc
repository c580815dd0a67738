// Host-only check of the run-kernel launch planner (include/physis/hip/run.h):
// prints, for each case, the z chunk and window bytes that PlanRunFor picks;
// "tiles": whether pairs over a domain run in resident tiles
// (include/physis/hip/tile.h); "fits": whether a pass has a window at all; "one":
// whether a single sweep runs at one point per lane; "vx": the points per lane of
// a whole-grid pass, whether it runs in tiles and whether it beats sweeps; "pay":
// whether passes over a whole grid, and over its interior, beat single sweeps, and
// whether the last of one red-black iteration runs as colour sweeps.  Built and
// run by tests/test_planner.py; no device is touched.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "physis/hip/run.h"
#include "physis/hip/tile.h"

namespace {

__PSGrid MakeGrid(int nx, int ny, int nz, int elm) {
  __PSGrid g = {};
  g.num_dims = 3;
  g.dim[0] = nx;
  g.dim[1] = ny;
  g.dim[2] = nz;
  g.elm_size = elm;
  g.num_elms = (int64_t)nx * ny * nz;
  return g;
}

// One launch: tiles of tx x ty, `resident` blocks per wave of the device,
// windows of `margin` planes per side.  Prints
//   nx ny nz elm margin tiles_z zchunk blocks window_bytes
void Case(int nx, int ny, int nz, int elm, int margin, int tx, int ty,
          long resident) {
  __PSGrid g = MakeGrid(nx, ny, nz, elm);
  __PSDomain dom = {};
  for (int d = 0; d < 3; ++d) {
    dom.local_min[d] = dom.local_max[d] = 0;
  }
  dom.local_max[0] = nx;
  dom.local_max[1] = ny;
  dom.local_max[2] = nz;
  const int mc = physis_hip::WindowChunkLimit({&g, &g}, margin);
  const physis_hip::RunShape s =
      physis_hip::PlanRunFor(dom, tx, ty, resident, mc);
  const long long window =
      (long long)(s.zchunk + 2 * margin) * nx * ny * (long long)elm;
  std::printf("%d %d %d %d %d %d %d %d %lld\n", nx, ny, nz, elm, margin,
              s.tiles_z, s.zchunk, s.blocks, window);
}

}  // namespace

int main(int argc, char **argv) {
  if (argc == 9 && std::strcmp(argv[1], "tiles") == 0) {
    __PSDomain dom = {};
    for (int d = 0; d < 3; ++d) {
      dom.local_min[d] = std::atoi(argv[2 + 2 * d]);
      dom.local_max[d] = std::atoi(argv[3 + 2 * d]);
    }
    std::printf("%d\n", physis_hip::TilesBeatDomainPairs(dom, std::atol(argv[8])));
    return 0;
  }
  if (argc == 7 && std::strcmp(argv[1], "one") == 0) {
    __PSDomain dom = {};
    for (int d = 0; d < 3; ++d) dom.local_max[d] = std::atoi(argv[2 + d]);
    std::printf("%d\n", physis_hip::OnePointRows(dom, std::atoi(argv[5]) != 0,
                                                 std::atoi(argv[6]) != 0));
    return 0;
  }
  if (argc == 7 && std::strcmp(argv[1], "vx") == 0) {
    const int dim[3] = {std::atoi(argv[2]), std::atoi(argv[3]),
                        std::atoi(argv[4])};
    const bool periodic = std::atoi(argv[5]) != 0;
    const bool colours = std::atoi(argv[6]) != 0;
    std::printf("%d %d %d\n", physis_hip::PairVX(dim, periodic, colours),
                physis_hip::TilesBeatPairs(dim, periodic, colours),
                physis_hip::PassesPay(dim, periodic, colours, true));
    return 0;
  }
  if (argc == 6 && std::strcmp(argv[1], "pay") == 0) {
    __PSDomain dom = {};
    int dim[3];
    for (int d = 0; d < 3; ++d) {
      dim[d] = std::atoi(argv[2 + d]);
      dom.local_min[d] = 1;
      dom.local_max[d] = dim[d] - 1;
    }
    std::printf("%d %d %d\n", physis_hip::PassesPay(dim, false, false, std::atoi(argv[5]) != 0),
                physis_hip::DomainPassesPay(dom, dim[0],
                                            (int64_t)dim[0] * dim[1] * dim[2],
                                            std::atoi(argv[5]) != 0),
                physis_hip::RedBlackLastAsSweeps(dim, 1));
    return 0;
  }
  if (argc == 8 && std::strcmp(argv[1], "fits") == 0) {
    __PSGrid g = MakeGrid(std::atoi(argv[2]), std::atoi(argv[3]),
                          std::atoi(argv[4]), std::atoi(argv[5]));
    std::printf("%d\n", physis_hip::WindowsFit({&g}, std::atoi(argv[6]),
                                               std::atoi(argv[7]) != 0));
    return 0;
  }
  if (argc > 1) {
    // one case from the command line (the rejection path exits here)
    if (argc != 9) return 2;
    Case(std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]),
         std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6]),
         std::atoi(argv[7]), std::atol(argv[8]));
    return 0;
  }
  // shapes whose single-chunk windows exceed 2 GiB, and ordinary ones
  Case(8192, 8192, 16, 4, 2, 256, 14, 256);
  Case(4096, 4096, 64, 4, 2, 256, 14, 256);
  Case(4096, 4096, 64, 4, 3, 256, 12, 256);
  Case(2048, 2048, 255, 8, 2, 256, 14, 256);
  Case(512, 512, 512, 4, 2, 256, 14, 256);
  Case(512, 256, 256, 4, 2, 256, 6, 256);
  return 0;
}
