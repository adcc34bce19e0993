// pair_grid (pair_grid.hpp) against the search over every segment count, and on
// grids of up to 2^29 planes, where that search would take seconds per call.
#include <cstdio>
#include <random>

#include "../../hippolbm_amd/csrc/pair_grid.hpp"

using namespace hlbm;

static PairGrid every_count(int nx, int ny, int nz, int64_t* cost) {
  PairGrid g{(nx + PAIR_TX - 1) / PAIR_TX, (ny + PAIR_TY - 1) / PAIR_TY, 1, nz, 0u};
  *cost = INT64_MAX;
  for (int k = 1; k <= nz; k++) {
    const int planes = (nz + k - 1) / k, segs = (nz + planes - 1) / planes;
    const int64_t rounds = ((int64_t)g.tx * g.ty * segs + PAIR_CUS - 1) / PAIR_CUS;
    const int64_t c = rounds * (planes + 2) * PAIR_CUS;
    if (c < *cost) {
      *cost = c;
      g.planes = planes;
      g.segs = segs;
    }
  }
  return g;
}

int main() {
  std::mt19937_64 rng(3);
  unsigned long bad = 0, tested = 0;
  auto check = [&](int nx, int ny, int nz) {
    int64_t a, b;
    const PairGrid g = pair_grid(nx, ny, nz, &a), w = every_count(nx, ny, nz, &b);
    tested++;
    bad += a != b || g.tx != w.tx || g.ty != w.ty || g.segs != w.segs || g.planes != w.planes;
  };
  for (int nz = 2; nz <= 700; nz++)
    for (int nx : {2, 64, 65, 130, 512})
      for (int ny : {2, 13, 14, 100, 512}) check(nx, ny, nz);
  for (int k = 0; k < 2000; k++) check(2 + (int)(rng() % 1000), 2 + (int)(rng() % 1000), 2 + (int)(rng() % 30000));
  // (the largest grid of a domain holds fewer than 2^31 nodes)
  int64_t c;
  for (int k = 0; k < 1000; k++) {
    const int nz = (1 << 29) - 1 - (int)(rng() % 1000);
    const PairGrid g = pair_grid(2, 2, nz, &c);
    tested++;
    bad += (int64_t)g.segs * g.planes < nz || (int64_t)(g.segs - 1) * g.planes >= nz;
  }
  std::printf("failures %lu of %lu\n", bad, tested);
  return bad ? 1 : 0;
}
