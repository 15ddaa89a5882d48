// Block counts of launches (csrc/launch_size.hpp).  Prints "ok" and returns 0, or names the line.
#include "launch_size.hpp"

#include <stdio.h>

#include <initializer_list>

#define CHECK(cond)                             \
  do {                                          \
    if (!(cond)) {                              \
      printf("line %d: %s\n", __LINE__, #cond); \
      return 1;                                 \
    }                                           \
  } while (0)

using nts::blocks_of_groups;
using nts::kMostBlocks;

int main() {
  CHECK(blocks_of_groups(1, 64, 0) == 1 && blocks_of_groups(4, 64, 0) == 1 && blocks_of_groups(5, 64, 7) == 9);
  CHECK(blocks_of_groups(256, 1, 0) == 1 && blocks_of_groups(257, 1, 0) == 2);
  // rows x tiles of 64 vectors at which a launch would reach 2^32 threads
  const uint64_t most = 4ull * kMostBlocks;
  CHECK(blocks_of_groups(most, 64, 0) == kMostBlocks && blocks_of_groups(most + 1, 64, 0) == kMostBlocks);
  CHECK(blocks_of_groups(most, 64, 2048) == kMostBlocks && blocks_of_groups(most - 4 * 2048, 64, 2048) == kMostBlocks);
  CHECK(blocks_of_groups(most - 4 * 2048 - 4, 64, 2048) == kMostBlocks - 1);
  const struct {
    uint64_t rows, F;
  } wide[] = {{6700000, 602}, {6750000, 602}, {2900000, 1433}, {2449029, 1793}, {33000000, 260}, {67108864, 65}, {4294967294u, 4294967295u}};
  for (const auto &w : wide)
    for (uint32_t first : {0u, 512u, 2048u}) {
      const uint64_t groups = w.rows * ((w.F + 63) / 64);
      const uint64_t blocks = blocks_of_groups(groups, 64, first);
      CHECK(blocks * 256 < 1ull << 32 && blocks > first);
      CHECK((blocks - first) * 4 >= groups || blocks == kMostBlocks);
    }
  printf("ok\n");
  return 0;
}
