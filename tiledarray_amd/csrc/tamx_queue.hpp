// The item queue of the persistent grouped GEMM kernels.
//
// A launch's items (macro tiles of the result) are split into kRegions
// contiguous ranges, one per XCD: a workgroup drains the range of its own XCD
// (workgroups are dispatched to XCDs round-robin by blockIdx), so the macro
// tiles of one result tile, which share A and B panels, run on one L2; then
// it steals from the other ranges in turn.
//
// The first items of a range belong to its workgroups by their number, with
// no atomic; only the rest is handed out through the range's counter, which
// counts from the first item past them.  Device-wide atomics on one line are
// served one after the other, about 10 ns each.  (When every workgroup took
// every item through a counter, found all eight ranges empty through eight
// more and counted itself out through a ninth, a launch of 1024 workgroups
// spent 70 to 100 us on them however small the product; without them one pass
// of a dense 256^3 product in 64-wide tiles, 16 items, went from 146 to 48 us,
// dense 2048^3 from 370 to 302, 1024 tensor-of-tensor products from 1.73 to
// 1.49 ms.)  So a range with no items past the first ones costs no atomic,
// other ranges are read before they are added to, every counter has a
// 128-byte line of its own, and the planner's last kernel clears them before
// every launch.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tamx {

constexpr int kRegions = 8;       // XCDs of an MI355X
constexpr int kQueueStride = 32;  // int32 from one range's counter to the next
constexpr int kQueueInts = kRegions * kQueueStride;

// Used by one thread of the workgroup; `total` items in the launch.
struct ItemQueue {
  int32_t* counters;
  int32_t total;
  int tried = 0;       // ranges found empty, starting with the own one
  bool first = true;
  bool asked = false;  // `pending` holds an item number of the own range
  int32_t pending = 0;

  __device__ ItemQueue(int32_t* counters_, int32_t total_) : counters(counters_), total(total_) {}

  // The next item of this workgroup, or -1 when there is none left.
  __device__ inline int next() {
    const int home = blockIdx.x % kRegions;
    if (first) {
      first = false;
      const int it = range_begin(home) + (int)(blockIdx.x / kRegions);
      if (it < range_begin(home + 1)) return it;
    }
    for (; tried < kRegions; ++tried) {
      const int r = (home + tried) % kRegions;
      const int rb = owned_end(r);
      const int left = range_begin(r + 1) - rb;
      if (left <= 0) continue;
      int32_t* c = counters + r * kQueueStride;
      if (asked) {
        asked = false;
        if (pending < left) return rb + pending;
        continue;
      }
      if (tried > 0 && __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= left)
        continue;
      const int q = atomicAdd(c, 1);
      if (q < left) return rb + q;
    }
    return -1;
  }

  // Takes the next item of the own range for next() to return.  Called
  // shortly before an item ends, while the other waves still multiply: an item
  // is bound to its workgroup from here on.
  __device__ inline void prefetch() {
    const int home = blockIdx.x % kRegions;
    if (first || asked || tried > 0 || owned_end(home) >= range_begin(home + 1)) return;
    pending = atomicAdd(counters + home * kQueueStride, 1);
    // (waits here: an answer left in flight would have the compiler wait for
    // all loads in flight wherever its register may be live)
    asm volatile("" : "+v"(pending));
    asked = true;
  }

 private:
  // the first item of range r that no workgroup owns
  __device__ inline int owned_end(int r) const {
    return range_begin(r) + (int)((gridDim.x + kRegions - 1 - r) / kRegions);
  }
  __device__ inline int range_begin(int r) const { return (int)((int64_t)total * r / kRegions); }
};

}  // namespace tamx
