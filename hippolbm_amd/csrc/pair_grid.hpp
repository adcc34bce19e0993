// pair_grid.hpp -- how pair_kernel (two time steps per pass) covers a grid.
// Host-only and free of HIP, so that the choice can be checked on any machine.
#pragma once

#include <stdint.h>

namespace hlbm {

constexpr int PAIR_TX = 64;  // tile columns along x: one wave per row
// Tile rows: with the ring's two rows and the wave for its columns, the 16 waves
// a workgroup can have.  The ring is stepped twice, so a step costs 16/13 of its
// arithmetic (9 rows: 512^3 FP64 5.1-5.4 ms per step where 13 took 4.7).
constexpr int PAIR_TY = 13;

struct PairGrid {
  int32_t tx, ty, segs;  // tiles along x and y, segments along z
  int32_t planes;        // planes per segment
  uint32_t seed2;        // rounding seed of the second step (StepParams::seed is the first's)
};

// The segments that cost the fewest planes: a CU holds one workgroup at a time
// (registers and LDS), and each segment steps a plane more on either side.
// `cost` is that number of planes times `cus`: the planes the chip steps,
// against nx * ny * nz / (64 * 13) for a grid that fills it exactly.
// Segment counts with the same planes per segment make the same launch, so only
// the first of each is looked at: 2 sqrt(nz) of them, 0.6 us for 512 planes and
// 4 us for 20000, where all of them took 4 and 50.
constexpr int PAIR_CUS = 256;
inline PairGrid pair_grid(int nx, int ny, int nz, int64_t* cost) {
  PairGrid g{(nx + PAIR_TX - 1) / PAIR_TX, (ny + PAIR_TY - 1) / PAIR_TY, 1, nz, 0u};
  *cost = INT64_MAX;
  for (int64_t k = 1; k <= nz;) {
    const int planes = (int)((nz + k - 1) / k), segs = (nz + planes - 1) / planes;
    const int64_t rounds = ((int64_t)g.tx * g.ty * segs + PAIR_CUS - 1) / PAIR_CUS;
    const int64_t c = rounds * (planes + 2) * PAIR_CUS;
    if (c < *cost) {
      *cost = c;
      g.planes = planes;
      g.segs = segs;
    }
    if (planes == 1) break;
    k = (nz + planes - 2) / (planes - 1);  // the fewest segments of at most planes - 1
  }
  return g;
}

}  // namespace hlbm
