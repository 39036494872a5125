// queue.h -- the work queue of the persistent kernels: one wave a workgroup,
// items 0 .. nitems - 1, heaviest first.
//
// Device-scope atomics on one address pass one at a time through memory
// (about 20 ns each here), so a single counter bounds a launch of many short
// items: 8192 waves popping once take 0.17 ms whatever the work.  Here the
// first half of a launch's waves (16 per compute unit by default, which all
// fit at once) have their first item from their block index, with no atomic;
// the other items come from QN counters on lines of their own, each wave
// starting at its own and moving to another when it is used up.  (A wave that
// is not resident from the start must not own an item: it gets to it when
// another wave ends, after the queue is empty.)  A wave sees all counters
// with one load before it moves, and gives a counter up for good when a pop
// comes back past its end, so at most QN pops per wave fail and every wave
// leaves.  Item i belongs to counter i % QN; runs of 8 or 32 consecutive
// items per counter, which keep neighbouring leaves in one XCD's L2, were no
// faster (2% slower at 256^3, which is what moving the pair loops by a few
// bytes can do, see loop_offset in wave.h).  Leaf kernel, one counter and
// now: 0.167 and 0.029 ms for 265 leaves of 32 (1155 entries each), 109.4
// ms either way for 50k leaves of 512 at 256^3; fused adjoint of 256^3, each
// with its loop at its best place, 458.7 and 460.4.
#pragma once

#include "wave.h"

constexpr int QN = 64;       // counters
constexpr int QSTRIDE = 16;  // uint64 per counter: a 128-byte line
constexpr int QWORDS = QN * QSTRIDE;

// The item at position pos of counter k's share.
__device__ __forceinline__ int64_t queue_item(uint64_t pos, int k) {
  return (int64_t)(pos * QN) + k;
}

// Counter values of a queue for a launch of `grid` waves: wave b < grid / 2
// holds position b / QN of counter b % QN from the start.
__device__ __forceinline__ void queue_reset(unsigned long long *q, int k, int64_t grid) {
  if (k < QN) q[k * QSTRIDE] = (unsigned long long)((grid / 2 - k + QN - 1) / QN);
}

// What a wave remembers of the queue between items.  In LDS: held in
// registers through the item's work it cost k_force six VGPRs, which took
// the default shape from 5 waves per SIMD to 4 (110 -> 118 ms at 256^3).
struct QueueState {
  uint64_t used_up;  // counters known to be past their end
  int32_t home;      // -1: the first item has not been taken
};

__device__ __forceinline__ void queue_begin(QueueState *qs) {
  if (lane_id() == 0) {
    qs->used_up = 0;
    qs->home = -1;
  }
}

// The wave's next item; nitems or more when none is left.
__device__ __forceinline__ int64_t queue_pop(unsigned long long *ctr, int64_t nitems,
                                             QueueState *qs) {
  const int l = lane_id();
  __syncthreads();
  // readlane: what is read from LDS is one for the wave, and so is all control
  // flow that follows (scalar registers and loads)
  uint64_t used = readlane_u64(qs->used_up, 0);
  int home = readlane_i32(qs->home, 0);
  int64_t item = nitems;
  bool own = false;
  if (home < 0) {
    const int64_t owners = gridDim.x / 2;
    home = (int)(blockIdx.x % QN);
    own = blockIdx.x < owners;
    if (own) item = queue_item(blockIdx.x / QN, home);
    // when the owners' first items are all there is, nothing is popped
    if (nitems <= owners) used = ~0ull;
  }
  if (!own) {
    int tries = QN + 1;  // each failed pop uses up a counter
    uint64_t pos = 0;
    do {
      if ((used >> home) & 1ull) {
        pos = 0;
        if (!((used >> l) & 1ull))
          pos = __hip_atomic_load(ctr + l * QSTRIDE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        used |= __ballot(queue_item(pos, l) >= nitems);
        if (~used == 0ull) {
          item = nitems;
          break;
        }
        // the next counter after home that is not used up
        const uint64_t left = ~used;
        const uint64_t rot = home ? (left >> home) | (left << (QN - home)) : left;
        home = (home + (int)__builtin_ctzll(rot)) % QN;
      }
      if (l == 0) pos = atomicAdd(ctr + home * QSTRIDE, 1ull);
      item = queue_item(readlane_u64(pos, 0), home);
      if (item >= nitems) used |= 1ull << home;
    } while (item >= nitems && --tries > 0);
  }
  __syncthreads();
  if (l == 0) {
    qs->used_up = used;
    qs->home = home;
  }
  return (int64_t)readlane_u64((uint64_t)item, 0);
}
