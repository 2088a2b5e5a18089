// Launches of more blocks than one launch can hold.
#pragma once
#include <algorithm>
#include <cstdint>

namespace brille_amd {
// a launch holds fewer than 2^32 threads along x: blocks of 256 of them
constexpr uint64_t kMostBlocks = (1ull << 24) - 1;

// launch(first, count, blocks) over `units` units of work, `per_block` in each
// block of at most 256 threads, in as few launches as that takes
template <typename Launch>
void in_pieces(uint64_t units, uint64_t per_block, Launch&& launch) {
  const uint64_t piece = kMostBlocks * per_block;
  for (uint64_t first = 0; first < units; first += piece) {
    const uint64_t count = std::min(piece, units - first);
    launch(first, count, (unsigned)((count + per_block - 1) / per_block));
  }
}
}  // namespace brille_amd
