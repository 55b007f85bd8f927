// The copying threads of a read-back (suminc_amd/csrc/copiers.hpp): every chunk arrives,
// with threads and without, and whatever allocation fails while they start, nothing ends
// the process: exit status 0 and "PASS".
#include <cstdio>
#include <cstdlib>
#include <new>

#include "../../suminc_amd/csrc/copiers.hpp"

static thread_local long fail_at = -1;  // the allocation of this thread that fails (counted down)
__attribute__((noinline)) void* operator new(std::size_t n) {
  if (fail_at >= 0 && fail_at-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
__attribute__((noinline)) void operator delete(void* p) noexcept { std::free(p); }
__attribute__((noinline)) void operator delete(void* p, std::size_t) noexcept { std::free(p); }

using namespace suminc;

// One read-back of `count` chunks of up to 64 bytes; 0: all there, 1: wrong, 2: bad_alloc.
static int run(size_t count, bool threaded, long fail) {
  static std::vector<unsigned char> slots(kSlots * kChunkBytes);
  std::vector<unsigned char> out(count * 64, 0);
  std::vector<Chunk> chunks;
  for (size_t i = 0; i < count; ++i) chunks.push_back({0, i, 1, &out[i * 64], 1 + i % 64});
  try {
    fail_at = fail;
    Copiers c(chunks, slots.data(), threaded);
    fail_at = -1;
    for (size_t i = 0; i < count; ++i) {
      c.wait_free(i);
      std::memset(&slots[(i % kSlots) * kChunkBytes], (int)(i % 251 + 1), chunks[i].bytes);
      c.post(i);
    }
    c.finish();
  } catch (const std::bad_alloc&) {
    fail_at = -1;
    return 2;
  }
  for (size_t i = 0; i < count; ++i)
    for (size_t b = 0; b < 64; ++b)
      if (out[i * 64 + b] != (b < chunks[i].bytes ? (unsigned char)(i % 251 + 1) : 0)) return 1;
  return 0;
}

int main() {
  const size_t counts[] = {0, 1, 7, 16, 17, 200};
  for (size_t count : counts)
    for (int threaded = 0; threaded < 2; ++threaded)
      for (long fail = -1; fail < 24; ++fail) {
        const int r = run(count, threaded != 0, fail);
        // (without its counters, the first allocation, there is no read-back to fall back to)
        if (r == 1 || (r == 2 && fail != 0)) {
          std::printf("%zu chunks, threads %d, allocation %ld: %d\n", count, threaded, fail, r);
          return 1;
        }
      }
  std::puts("PASS");
  return 0;
}
