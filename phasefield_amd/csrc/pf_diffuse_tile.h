// pf_diffuse_tile.h — several diffusion sub-steps per launch on planes (pf_diffuse_tile.hip).
#pragma once
#include <algorithm>

#include "pf_diffuse_common.h"

namespace pfamd {

// One workgroup of 16 wavefronts per tile: with 8 wavefronts of twice the cells each a sub-step took
// 1.59 instead of 1.42 us (256^2 FP64): it is a chain of LDS and FP64 latencies, hidden by wavefronts.
constexpr int kTileNT = 1024;  // threads of a workgroup
constexpr int kTileV = 2;      // cells per thread: a tile and its halo hold at most kTileNT * kTileV

// Geometry of a launch of up to `left` sub-steps on nz planes of nx x ny cells; false when single
// sub-steps are faster.  pin: tile and sub-steps to use instead (pin[2] == 0: none).
struct TileGeom {
  int nx, ny;            // the domain's planes
  int bx, by;            // a tile's cells (the last ones of an axis may hold fewer)
  int nbx, nby, nblocks;
  int steps;             // sub-steps of the launch: the width of the halo
};

// Tile and sub-steps per launch.  Time per sub-step, FP64 (halo computed again against launches):
//   64 x 48:   8 x 8 cells, 8 sub-steps 1.18 us; 16 x 16, 12: 1.38
//   256^2:     16 x 16, 12: 1.42; 16 x 16, 8: 1.52; 32 x 16, 10: 1.6
//   512^2:     32 x 32, 6: 2.30; 24 x 24, 10: 2.97; 20 x 20, 12: 3.75
//   1000 x 600: 32 x 32, 6: 4.89 (single sub-steps: 10.9)
// so tiles grow once they outnumber the compute units.
//
// Tiles are taken as long as what they compute, halo included, is at most 2.2 M cells (mixed 3.5 M) or
// 2.1 times the domain.  A step with single sub-steps / with tiles, three domains in turn (one domain
// alone gains more):
//                                  FP64            mixed
//   1024^2 (2.0 M computed)        1.55 / 1.20     1.40 / 0.83 ms
//   1224^2 (2.9 M)                 1.85 / 1.68     1.50 / 1.17
//   160 x 1 x 160 (1.6 M)          1.19 / 0.80     1.18 / 0.54
//   200 x 1 x 200 (2.6 M)          1.14 / 1.27     1.17 / 0.86
//   230 x 1 x 230 (3.5 M)          1.15 / 1.66     1.13 / 1.13
//   300 x 1 x 300 (5.7 M)          1.44 / 2.74     1.44 / 1.86
//   1000 x 1 x 600 (10.7 M)        1.66 / 10.5     1.57 / 7.40
// (a row one cell wide is its own halo in y, `steps` times over on either side).  Planes above 1.5 M
// cells keep single sub-steps; tiles of 32 x 32 and 6 sub-steps would gain there as well up to about
// 6 M cells (1500^2 FP64 2.57 / 2.42) and lose at 4096^2 (16.3 / 18.3).
inline bool tile_geometry(int nx, int ny, int nz, bool mixed, int left, const int *pin, TileGeom &g) {
  const long n = long(nx) * ny * nz;
  int bx = 32, by = 32, steps = 6;
  if (n <= 8192) bx = by = steps = 8;
  else if (n <= 131072) bx = by = 16, steps = 12;
  if (pin && pin[2] > 0) bx = pin[0], by = pin[1], steps = pin[2];
  else if (n > 1500000) return false;
  auto split = [](int e, int most, int &size, int &count) {
    count = (e + most - 1) / most;
    size = (e + count - 1) / count;
    count = (e + size - 1) / size;
  };
  g.nx = nx;
  g.ny = ny;
  split(nx, bx, g.bx, g.nbx);
  split(ny, by, g.by, g.nby);
  const long nblocks = long(g.nbx) * g.nby * nz;
  if (!(pin && pin[2] > 0) &&
      double(nblocks) * (g.bx + 2 * steps) * (g.by + 2 * steps) > std::max(mixed ? 3.5e6 : 2.2e6, 2.1 * double(n)))
    return false;
  const int launches = (left + steps - 1) / steps;
  g.nblocks = int(nblocks);
  g.steps = (left + launches - 1) / launches;
  return nblocks <= 0x7fffffffL && (g.bx + 2 * steps) * (g.by + 2 * steps) <= kTileNT * kTileV;
}

// SELF_Z: z faces that join each cell to itself (six-face calls on one plane).
template <class F, int P, bool SELF_Z>
__global__ void diffuse_tile_kernel(const typename F::C *__restrict__ cin,
                                    typename F::C *__restrict__ cout,
                                    const typename F::T *__restrict__ pfrac,
                                    const uint8_t *__restrict__ flag,
                                    const DiffConsts<typename F::A> dc, const TileGeom geo,
                                    const long ncell, const uint32_t k0, const int solute);

}  // namespace pfamd
