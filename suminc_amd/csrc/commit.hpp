// commit.hpp -- how a traversal's {value, parent} word is replaced by a better one.
//
// Words only decrease while rounds run, and a candidate is tested against a read of the
// word that other threads may have passed meanwhile.  SSSP and BFS take the minimum of
// the whole words: every edge adds at least 1, so on equal values either parent will do
// and the smallest id wins.  SSWP must take strictly better values only: a width passes
// along an edge unchanged, so a parent that replaces another on equal widths may have
// got its own width from this very vertex, and the two would be each other's parents (a
// deletion's repair walks the parents and would leave both stale).  With strict values
// no cycle can close: round a cycle, the vertex replaced last would need a width above
// one that came from its own earlier, smaller width.  So SSWP compares the value with
// the word that it replaces, whatever was read before.
//
// No HIP header: the interleavings are tested on the host.
#pragma once
#include "../../include/suminc.h"

#if defined(__HIPCC__)
#define SUMINC_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define SUMINC_HOST_DEVICE inline
#endif

namespace suminc {

// Cell: fetch_min(x) and compare_exchange(expected, x), each returning the word that was
// there.  seen: the word as the caller last read it, however long ago.  Returns the word
// that cand met (SSWP: or the last one seen, when that already rules cand out): the value
// (high half) fell if it is above cand's.
template <class Cell>
SUMINC_HOST_DEVICE unsigned long long trav_commit(int app, Cell cell, unsigned long long cand,
                                                  unsigned long long seen) {
  if (app != SUMINC_APP_SSWP) return cell.fetch_min(cand);
  unsigned long long now = seen;
  while ((cand >> 32) < (now >> 32)) {  // a failed exchange finds a smaller word: it ends
    const unsigned long long was = cell.compare_exchange(now, cand);
    if (was == now) break;
    now = was;
  }
  return now;
}

}  // namespace suminc
