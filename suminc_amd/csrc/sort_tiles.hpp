// sort_tiles.hpp -- how the binned layout's ordering (k_bin_sort) cuts its edges.
//
// Edge numbers are 32 bits and go up to 2^32 - 2, so no sum here may pass 2^32.  No HIP
// header: the cuts are tested on the host at that limit.
#pragma once
#include <cstdint>

#include "commit.hpp"

namespace suminc {

constexpr int kSortBlock = 1024, kSortPer = 16;
constexpr uint32_t kSortTile = kSortPer * kSortBlock - 4;  // a chunk may begin up to 3 edges into its first 16 bytes
constexpr uint32_t kSortStep = 8192, kSortBins = 4096;

// Workgroups for m edges: one for every kSortStep of them.
inline uint32_t sort_tiles(uint64_t m) { return (uint32_t)((m + kSortStep - 1) / kSortStep); }

// The end of the chunk that begins at lo < stop, and the next one's beginning.
SUMINC_HOST_DEVICE uint32_t sort_chunk_end(uint32_t lo, uint32_t stop) {
  return stop - lo < kSortTile ? stop : lo + kSortTile;
}

}  // namespace suminc
