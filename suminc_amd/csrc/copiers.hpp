// copiers.hpp -- the threads that copy a read-back's pinned slots to the caller's array
// (readback.hip).  No HIP header: tested on the host.
#pragma once
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace suminc {

// A chunk is large enough to amortise its launch and event (2 MiB cross in 40 us) and
// small enough that every copying thread has one.
constexpr size_t kChunkBytes = size_t(2) << 20;
constexpr int kThreads = 8;
constexpr int kSlots = 2 * kThreads;

struct Chunk {
  int part;
  uint64_t first, count;
  unsigned char* dst;
  size_t bytes;
};

// Copies chunks [0, n) as they become ready; chunk i is thread i % threads' (the calling
// thread's own, as the last step of post(), without threads).
struct Copiers {
  const std::vector<Chunk>& chunks;
  unsigned char* mem;  // the pinned slots
  std::atomic<size_t> ready{0};
  std::atomic<bool> stop{false};
  std::vector<std::atomic<size_t>> done;  // per slot: chunks copied out of it
  std::vector<std::thread> threads;

  Copiers(const std::vector<Chunk>& c, unsigned char* slots, bool threaded) : chunks(c), mem(slots), done(kSlots) {
    if (!threaded) return;
    const unsigned hw = std::thread::hardware_concurrency();
    const int want = (int)std::min<size_t>(std::min<unsigned>(kThreads, hw ? hw : 1u), chunks.size());
    try {
      threads.reserve(want);
      for (int t = 0; t < want; ++t) threads.emplace_back([this, t, want] { work(t, want); });
    } catch (...) {  // no threads or no memory to be had: the calling thread copies
      stop_all();
      threads.clear();
      stop = false;
    }
  }
  ~Copiers() { stop_all(); }
  void stop_all() {
    stop = true;
    for (std::thread& t : threads)
      if (t.joinable()) t.join();
  }
  void copy(size_t i) {
    const Chunk& k = chunks[i];
    std::memcpy(k.dst, mem + (i % kSlots) * kChunkBytes, k.bytes);
    done[i % kSlots].fetch_add(1, std::memory_order_release);
  }
  void work(size_t t, size_t step) {
    for (size_t i = t; i < chunks.size(); i += step) {
      while (ready.load(std::memory_order_acquire) <= i) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      copy(i);
    }
  }
  void post(size_t i) {
    if (threads.empty()) copy(i);
    else ready.store(i + 1, std::memory_order_release);
  }
  void wait_free(size_t i) {  // slot of chunk i is free: every earlier chunk in it was copied
    while (done[i % kSlots].load(std::memory_order_acquire) < i / kSlots) std::this_thread::yield();
  }
  void finish() {
    const size_t n = chunks.size();
    for (size_t s = 0; s < kSlots && s < n; ++s)
      while (done[s].load(std::memory_order_acquire) < (n - s + kSlots - 1) / kSlots) std::this_thread::yield();
  }
};

}  // namespace suminc
