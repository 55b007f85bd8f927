// readback.hip -- results of n values each to pageable host memory.
//
// A hipMemcpy to pageable memory runs at about 10 GB/s here (one thread copies out of
// the runtime's staging buffers, and the first touch of a fresh result array falls into
// it), while a kernel stores to pinned memory at the bus' rate, about 50 GB/s.  So a
// result crosses in chunks: a kernel converts the state and stores a chunk straight to a
// pinned slot, an event says that it is there, and several threads copy the slots to the
// caller's array while the next chunks cross.  MI355X, FP32 state of 2^26 vertices to two
// FP64 arrays (1 GiB): 104 -> 23 ms; 2^22 vertices, distances and parents (32 MiB):
// 2.5 -> 0.95 ms; 1000 vertices: 84 -> 50 us (no allocation).
#include "readback.hpp"

#include <atomic>
#include <mutex>
#include <system_error>
#include <thread>

namespace suminc {

namespace {

// A chunk is large enough to amortise its launch and event (2 MiB cross in 40 us) and
// small enough that every copying thread has one.
constexpr size_t kChunkBytes = size_t(2) << 20;
constexpr int kThreads = 8;
constexpr int kSlots = 2 * kThreads;
// Below this the calling thread copies alone: starting the threads costs 0.1 ms.
constexpr size_t kThreadedBytes = size_t(4) << 20;

struct Ring {
  unsigned char* mem = nullptr;
  hipEvent_t ev[kSlots] = {};
  int device = -1;
  ~Ring() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (mem) (void)hipHostFree(mem);
  }
};

// Rings not in use, shared by the process' contexts: a call takes one (or makes one) and
// gives it back; at most kIdle stay, none after the last context is gone.
constexpr size_t kIdle = 2;
std::mutex g_mu;
std::vector<Ring*> g_idle;
size_t g_contexts = 0;

Ring* ring_take(int device) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (size_t i = 0; i < g_idle.size(); ++i)
      if (g_idle[i]->device == device) {
        Ring* r = g_idle[i];
        g_idle.erase(g_idle.begin() + i);
        return r;
      }
  }
  Ring* r = new (std::nothrow) Ring();
  if (!r) return nullptr;
  r->device = device;
  void* p = nullptr;
  bool ok = hipHostMalloc(&p, kSlots * kChunkBytes, hipHostMallocDefault) == hipSuccess;
  if (ok) r->mem = reinterpret_cast<unsigned char*>(p);
  for (int i = 0; ok && i < kSlots; ++i) ok = hipEventCreateWithFlags(&r->ev[i], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    delete r;
    return nullptr;
  }
  return r;
}

void ring_give(Ring* r) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_contexts && g_idle.size() < kIdle) {
      g_idle.push_back(r);
      return;
    }
  }
  delete r;
}

// Copies chunks [0, n) as they become ready; chunk i is thread i % threads' (the calling
// thread's own, as the last step of post(), without threads).
struct Copiers {
  const std::vector<Chunk>& chunks;
  Ring* ring;
  std::atomic<size_t> ready{0};
  std::atomic<bool> stop{false};
  std::vector<std::atomic<size_t>> done;  // per slot: chunks copied out of it
  std::vector<std::thread> threads;

  Copiers(const std::vector<Chunk>& c, Ring* r, bool threaded) : chunks(c), ring(r), done(kSlots) {
    if (!threaded) return;
    const unsigned hw = std::thread::hardware_concurrency();
    const int want = (int)std::min<size_t>(std::min<unsigned>(kThreads, hw ? hw : 1u), chunks.size());
    try {
      threads.reserve(want);
      for (int t = 0; t < want; ++t) threads.emplace_back([this, t, want] { work(t, want); });
    } catch (const std::system_error&) {  // no threads to be had: the calling thread copies
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
    std::memcpy(k.dst, ring->mem + (i % kSlots) * kChunkBytes, k.bytes);
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

}  // namespace

void readback_context(int change) {
  std::vector<Ring*> gone;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_contexts += change;
    if (!g_contexts) gone.swap(g_idle);
  }
  for (Ring* r : gone) delete r;
}

bool readback_pageable(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

bool readback(suminc_ctx* c, const std::vector<ReadbackPart>& parts, const ReadbackLaunch& launch) {
  for (const ReadbackPart& p : parts)
    if (p.dst && !readback_pageable(p.dst)) return false;
  Ring* ring = ring_take(c->device);
  if (!ring) return false;
  struct Give {
    Ring* r;
    ~Give() { ring_give(r); }
  } give{ring};
  std::vector<Chunk> chunks;
  size_t total = 0;
  for (size_t k = 0; k < parts.size(); ++k) {
    const ReadbackPart& p = parts[k];
    if (!p.dst) continue;
    const size_t per = kChunkBytes / p.elem;
    for (uint64_t b = 0; b < p.count; b += per) {
      const uint64_t m = std::min<uint64_t>(per, p.count - b);
      chunks.push_back({(int)k, b, m, reinterpret_cast<unsigned char*>(p.dst) + b * p.elem, m * p.elem});
      total += m * p.elem;
    }
  }
  // whatever ends this call early, no kernel still stores to the ring when it goes back
  struct Drain {
    hipStream_t s;
    ~Drain() { (void)hipStreamSynchronize(s); }
  } drain{c->stream};
  Copiers copiers(chunks, ring, total >= kThreadedBytes);
  const size_t n = chunks.size();
  size_t sent = 0;
  for (size_t i = 0; i < n; ++i) {
    // keep half of the ring crossing while the other half is copied out
    for (; sent < n && sent < i + kSlots / 2; ++sent) {
      copiers.wait_free(sent);
      const Chunk& k = chunks[sent];
      launch(k.part, k.first, k.count, ring->mem + (sent % kSlots) * kChunkBytes);
      SUMINC_HIP(hipGetLastError());
      SUMINC_HIP(hipEventRecord(ring->ev[sent % kSlots], c->stream));
    }
    SUMINC_HIP(hipEventSynchronize(ring->ev[i % kSlots]));
    copiers.post(i);
  }
  copiers.finish();
  return true;
}

}  // namespace suminc
