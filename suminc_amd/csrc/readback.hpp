// readback.hpp -- results to pageable host memory through pinned slots (readback.hip).
#pragma once
#include <algorithm>
#include <functional>
#include <vector>

#include "ctx.hpp"

namespace suminc {

struct ReadbackPart {
  void* dst;       // host array of count elements of elem bytes (null: left out)
  uint64_t count;
  size_t elem;
};
// Enqueues on the context's stream the kernel that stores elements
// [first, first + count) of a part at out (pinned memory).
using ReadbackLaunch = std::function<void(int part, uint64_t first, uint64_t count, void* out)>;

// Brings the parts over and returns once they are there; false, with nothing done, when
// one of them is not pageable memory or there is no pinned memory to be had.
bool readback(suminc_ctx* c, const std::vector<ReadbackPart>& parts, const ReadbackLaunch& launch);
bool readback_pageable(const void* p);
// A context was made (1) or is gone (-1): the last one takes the pinned slots with it.
void readback_context(int change);

}  // namespace suminc
