// The cuts of the binned layout's ordering (suminc_amd/csrc/sort_tiles.hpp), small and up
// to the largest edge count, 2^32 - 2: exit status 0 and "PASS" when they are right.
#include <cstdio>

#include "../../suminc_amd/csrc/sort_tiles.hpp"

using namespace suminc;

#define CHECK(x)                                  \
  do {                                            \
    if (!(x)) {                                   \
      std::printf("line %d: %s\n", __LINE__, #x); \
      return 1;                                   \
    }                                             \
  } while (0)

// The chunks of [begin, stop) follow each other, fill a workgroup at most and end.
static int walk(uint32_t begin, uint32_t stop) {
  uint32_t count = 0;
  for (uint32_t lo = begin, hi; lo < stop; lo = hi) {
    hi = sort_chunk_end(lo, stop);
    CHECK(hi > lo && hi <= stop && hi - lo <= kSortTile);
    CHECK(hi - (lo & ~3u) <= (uint32_t)kSortBlock * kSortPer);  // what the threads read
    CHECK(hi == stop || hi - lo == kSortTile);
    CHECK(++count <= (stop - begin) / kSortTile + 1);
  }
  return 0;
}

int main() {
  const uint32_t top = 0xFFFFFFFEu;
  const uint32_t lengths[] = {0, 1, 3, kSortTile - 1, kSortTile, kSortTile + 1, 2 * kSortTile, 2 * kSortTile + 5, 131072};
  for (uint32_t len : lengths)
    for (uint32_t off = 0; off < 9; ++off) {
      if (walk(off, off + len) || walk(top - off - len, top - off)) return 1;
    }
  const uint64_t counts[] = {1, kSortStep - 1, kSortStep, kSortStep + 1, top - kSortStep, top - 1, top};
  for (uint64_t m : counts) {
    const uint64_t t = sort_tiles(m);
    CHECK(t * kSortStep >= m && (t - 1) * kSortStep < m);
  }
  std::puts("PASS");
  return 0;
}
