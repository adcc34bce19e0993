// reduce_parts.hpp -- partial records of the simulation_state reduction
// (launch_reduce): how many a grid writes, and the scratch that holds them.
// Host-only and free of HIP, so that the sizes can be checked on any machine.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace hlbm {

constexpr int RED_BLOCK = 256;       // nodes (and threads) per record and sweep
constexpr int RED_VALUES = 7;        // doubles per record
constexpr int RED_MAX_PARTS = 1024;  // workgroups, one record each

// Records that the reduction of N nodes writes, for every 32-bit N.
constexpr int reduce_parts(uint32_t N) {
  const uint64_t parts = ((uint64_t)N + RED_BLOCK - 1) / RED_BLOCK;
  return parts < 1 ? 1 : (parts > RED_MAX_PARTS ? RED_MAX_PARTS : (int)parts);
}

// Scratch for any N: whoever calls launch_reduce allocates this much, whatever
// sizes it means to reduce.
constexpr size_t RED_SCRATCH_BYTES = sizeof(double) * RED_VALUES * RED_MAX_PARTS;

}  // namespace hlbm
