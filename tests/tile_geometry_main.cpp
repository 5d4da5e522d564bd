// tile_geometry_main.cpp — CPU check of the tile kernel's geometry (phasefield_amd/csrc/pf_diffuse_tile.h):
// which planes take tiles, and that a geometry's tiles cover a plane and fit a workgroup.
// tests/test_tile_geometry.py builds it with hipcc (host code) and runs it.
#include <cstdio>

#include "../phasefield_amd/csrc/pf_diffuse_tile.h"

using namespace pfamd;

static int bad = 0;

static void expect(int nx, int ny, int nz, bool fp64, bool mixed) {
  for (int m = 0; m < 2; ++m) {
    TileGeom g;
    const bool tiles = m ? mixed : fp64;
    if (tile_geometry(nx, ny, nz, m == 1, 200, nullptr, g) == tiles) continue;
    std::fprintf(stderr, "%d x %d x %d %s: expected %s\n", nx, ny, nz, m ? "mixed" : "FP64",
                 tiles ? "tiles" : "single sub-steps");
    ++bad;
  }
}
static void expect(int nx, int ny, int nz, bool tiles) { expect(nx, ny, nz, tiles, tiles); }

int main() {
  // planes as wide as high, up to the cells that tiles are taken for
  for (int e : {2, 8, 61, 90, 91, 256, 331, 362, 363, 512, 700, 1000, 1024, 1217, 1224}) expect(e, e, 1, true);
  expect(1000, 600, 1, true);
  expect(1250, 1250, 1, false);
  // Rows one cell wide: the halo in y is the row itself, `steps` times over on either side, so the
  // tiles of a wide domain compute many times its cells (1000 x 1 x 600: 18 times, 10.5 ms a step
  // against 1.7 with single sub-steps).
  expect(64, 1, 64, true);
  expect(128, 1, 128, true);
  expect(160, 1, 160, true);
  expect(200, 1, 200, false, true);
  expect(230, 1, 230, false, true);
  expect(260, 1, 260, false);
  expect(300, 1, 300, false);
  expect(1000, 1, 600, false);
  expect(20, 1, 3000, false);
  // narrow planes
  expect(3, 20000, 1, true);
  expect(20000, 3, 1, true);
  expect(2, 700000, 1, false);
  // cover and fit, for every number of sub-steps left
  for (int nx : {1, 2, 5, 40, 64, 131, 400, 1100})
    for (int ny : {1, 2, 3, 37, 64, 333})
      for (int nz : {1, 7}) {
        if (nx * ny == 1) continue;
        for (int left = 1; left <= 60; ++left) {
          TileGeom g;
          if (!tile_geometry(nx, ny, nz, nz > 1, left, nullptr, g)) continue;
          const bool ok = g.steps >= 1 && g.steps <= left && long(g.bx) * g.nbx >= nx &&
                          long(g.by) * g.nby >= ny && g.bx * (g.nbx - 1) < nx && g.by * (g.nby - 1) < ny &&
                          g.nblocks == g.nbx * g.nby * nz &&
                          (g.bx + 2 * g.steps) * (g.by + 2 * g.steps) <= kTileNT * kTileV;
          if (!ok) {
            std::fprintf(stderr, "%d x %d x %d, %d left: bad geometry\n", nx, ny, nz, left);
            ++bad;
          }
        }
      }
  if (bad) return 1;
  std::printf("tile_geometry_main: ok\n");
  return 0;
}
