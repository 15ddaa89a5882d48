// Sizes of launches that grow with their arguments.  Host logic only.
#pragma once
#include <stdint.h>

namespace nts {

// A launch has fewer than 2^32 threads: blocks of 256, at most.
constexpr uint32_t kMostBlocks = (1u << 24) - 1;

// Blocks of 256 threads for `groups` groups of `lanes` threads each (a power of two up to 256), beside `first` blocks of another
// use; the groups that this leaves out are the next launch's.
inline uint32_t blocks_of_groups(uint64_t groups, uint32_t lanes, uint32_t first) {
  const uint64_t per_block = 256 / lanes, blocks = groups / per_block + (groups % per_block != 0);
  const uint32_t most = kMostBlocks - first;
  return first + (blocks < most ? static_cast<uint32_t>(blocks) : most);
}

}  // namespace nts
