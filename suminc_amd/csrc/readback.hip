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

#include <mutex>
#include <utility>

#include "copiers.hpp"

namespace suminc {

namespace {

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

// Rings are shared by the process' contexts: a call takes an idle one, or makes one up to
// kRings, and gives it back; none stays after the last context is gone.  With kRings in use
// a call goes the runtime's way instead: pinning a ring for one call takes longer than that.
// 3.2 MB to each of 8 threads, 12 threads: 0.55 ms, 0.91; with two rings that stay and the
// others made and freed for the call 1.14, 2.14; all the runtime's way 0.93, 1.33.
constexpr size_t kRings = 8;
std::mutex g_mu;
Ring* g_idle[kRings] = {};
size_t g_rings = 0, g_contexts = 0;

Ring* ring_take(int device) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (Ring*& slot : g_idle)
      if (slot && slot->device == device) return std::exchange(slot, nullptr);
    if (g_rings == kRings) return nullptr;
    ++g_rings;
  }
  Ring* r = new (std::nothrow) Ring();
  if (!r) {
    std::lock_guard<std::mutex> lk(g_mu);
    --g_rings;
    return nullptr;
  }
  r->device = device;
  void* p = nullptr;
  bool ok = hipHostMalloc(&p, kSlots * kChunkBytes, hipHostMallocDefault) == hipSuccess;
  if (ok) r->mem = reinterpret_cast<unsigned char*>(p);
  for (int i = 0; ok && i < kSlots; ++i) ok = hipEventCreateWithFlags(&r->ev[i], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    delete r;
    std::lock_guard<std::mutex> lk(g_mu);
    --g_rings;
    return nullptr;
  }
  return r;
}

void ring_give(Ring* r) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (Ring*& slot : g_idle)
      if (g_contexts && !slot) {
        slot = r;
        return;
      }
    --g_rings;
  }
  delete r;
}

}  // namespace

void readback_context(int change) {
  Ring* gone[kRings] = {};
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_contexts += change;
    if (!g_contexts) {
      std::swap(gone, g_idle);
      for (Ring* r : gone) g_rings -= r != nullptr;
    }
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
  Copiers copiers(chunks, ring->mem, total >= kThreadedBytes);
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
