// NodeDivisors (d3q19.hpp): floor(n / d) from one multiply-high and a shift,
// against the division, at the edges of quotients and on random pairs.
#include <cstdio>
#include <random>

#include "../../hippolbm_amd/csrc/d3q19.hpp"

int main() {
  std::mt19937_64 rng(7);
  const uint64_t top = 1ull << 31;
  unsigned long bad = 0, tested = 0;
  auto check = [&](uint64_t d) {
    if (d < 2 || d >= top) return;
    uint32_t m, s;
    hlbm::node_divisor((uint32_t)d, m, s);
    auto one = [&](uint64_t n) {
      if (n >= top) return;
      tested++;
      bad += hlbm::div_by((uint32_t)n, m, s) != n / d;
    };
    const uint64_t last = (top - 1) / d * d;
    for (uint64_t n : {(uint64_t)0, (uint64_t)1, d - 1, d, d + 1, 2 * d - 1, 2 * d, last - 1, last, top - 1}) one(n);
    for (int k = 0; k < 20; k++) one(rng() % top);
  };
  for (uint64_t d = 2; d < 20000; d++) check(d);
  for (int k = 1; k < 31; k++)
    for (int e = -1; e <= 1; e++) check((1ull << k) + e);
  for (int k = 0; k < 200000; k++) check(rng() % top);
  std::printf("failures %lu of %lu\n", bad, tested);
  return bad ? 1 : 0;
}
