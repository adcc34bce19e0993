// reduce_parts.hpp: the number of records a reduction of N nodes writes, and the
// scratch that every caller of launch_reduce holds for them.
#include <cstdio>

#include "../../hippolbm_amd/csrc/reduce_parts.hpp"

int main() {
  using namespace hlbm;
  const uint32_t n[] = {0u, 1u, 256u, 257u, 1u << 18, (1u << 18) + 1u, (1u << 31) - 1u, 0xFFFFFF00u, 0xFFFFFF01u, 0xFFFFFFFFu};
  const int want[] = {1, 1, 1, 2, 1024, 1024, 1024, 1024, 1024, 1024};
  int bad = 0;
  for (size_t k = 0; k < sizeof(n) / sizeof(n[0]); k++) {
    const int parts = reduce_parts(n[k]);
    std::printf("%u nodes: %d records\n", n[k], parts);
    bad += parts != want[k] || parts * sizeof(double) * RED_VALUES > RED_SCRATCH_BYTES;
  }
  std::printf("failures %d\n", bad);
  return bad ? 1 : 0;
}
