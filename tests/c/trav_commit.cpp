// Interleavings of trav_commit (suminc_amd/csrc/commit.hpp) with other writers, played on
// the host: exit status 0 and "PASS" when every one ends as it must.
#include <cstdio>
#include <vector>

#include "../../suminc_amd/csrc/commit.hpp"

using suminc::trav_commit;
using u64 = unsigned long long;
static u64 word(u64 value, u64 parent) { return value << 32 | parent; }

// A word; before its k-th access (0, 1, ...) from trav_commit the k-th of `others` is
// committed by another thread under the app's own rule (~0: none).
struct Shared {
  int app;
  u64 now;
  std::vector<u64> others;
  size_t at = 0;
  u64 replaced = ~0ull;  // the word that trav_commit wrote over
  void interfere() {
    if (at < others.size() && others[at] != ~0ull) {
      const u64 x = others[at];
      if (app == SUMINC_APP_SSWP ? (x >> 32) < (now >> 32) : x < now) now = x;
    }
    ++at;
  }
};
struct Cell {
  Shared* s;
  u64 fetch_min(u64 x) const {
    s->interfere();
    const u64 was = s->now;
    if (x < was) {
      s->replaced = was;
      s->now = x;
    }
    return was;
  }
  u64 compare_exchange(u64 expected, u64 x) const {
    s->interfere();
    const u64 was = s->now;
    if (was == expected) {
      s->replaced = was;
      s->now = x;
    }
    return was;
  }
};

#define CHECK(x)                                          \
  do {                                                    \
    if (!(x)) {                                           \
      std::printf("line %d: %s\n", __LINE__, #x);         \
      return 1;                                           \
    }                                                     \
  } while (0)

int main() {
  // every word as it was read, interfering words since and candidate, over small values
  // and parents
  std::vector<u64> words;
  for (u64 v = 0; v < 4; ++v)
    for (u64 p = 0; p < 3; ++p) words.push_back(word(v, p));
  std::vector<u64> others = words;
  others.push_back(~0ull);
  for (int app : {SUMINC_APP_SSSP, SUMINC_APP_BFS, SUMINC_APP_SSWP})
    for (u64 first : words)
      for (u64 a : others)
        for (u64 b : others)
          for (u64 cand : words) {
            Shared s{app, first, {a, b}};
            const u64 met = trav_commit(app, Cell{&s}, cand, first);
            if (app == SUMINC_APP_SSWP) {
              // written over a strictly worse value only, and reported as such
              CHECK((s.replaced != ~0ull) == ((cand >> 32) < (met >> 32)));
              if (s.replaced != ~0ull) CHECK(s.replaced == met && s.now == cand);
            } else {
              CHECK(s.now == (cand < met ? cand : met));
            }
            CHECK((s.now >> 32) <= (cand >> 32));
          }
  // Vertices v = 0, u1 = 2, u2 = 1, all in the frontier, v's row shared by two writers.  B
  // tests v's word and reads u2's; between the two A improves v through u1 to width W, and
  // u2 takes W from v.  B's commit ties with A's and must not make u2 v's parent.
  {
    const u64 W = 5, old = 9;
    Shared v{SUMINC_APP_SSWP, word(old, 7), {}}, u2{SUMINC_APP_SSWP, word(old, 7), {}};
    const u64 b_old = v.now >> 32;
    trav_commit(SUMINC_APP_SSWP, Cell{&v}, word(W, 2), v.now);
    trav_commit(SUMINC_APP_SSWP, Cell{&u2}, word(v.now >> 32, 0), u2.now);
    const u64 best = word(u2.now >> 32, 1);
    CHECK((best >> 32) < b_old);  // B's own test lets it pass
    trav_commit(SUMINC_APP_SSWP, Cell{&v}, best, word(old, 7));
    CHECK((u2.now & 0xFFFFFFFFu) == 0);
    CHECK((v.now & 0xFFFFFFFFu) == 2);
  }
  std::puts("PASS");
  return 0;
}
