// sg_queue.hpp -- device work queues of the batched launches.
//
// A batch's tiles sit in one queue per XCD: queue q holds tiles[start[q] ..
// start[q + 1]); start[] is stored after one counter per queue.  Workgroup b
// of a launch runs on XCD b mod 8 (workgroups are dispatched to the XCDs
// round-robin).  The native batch takes one tile per workgroup (queue_tile).
// The MFMA tiers, whose tiles are several times as many and shorter, run
// persistent workgroups that drain the queues through the atomic counters
// counters[q * kQueueStride] (one 256-byte line each), that of their XCD first
// and then the others in turn (1024 grids: 1.69 ms, with a workgroup per tile
// 1.80 ms).
#pragma once

#include "sg_internal.hpp"

namespace sg {

// A tile of a batched launch: grid (or argument record) index, tile along
// dimension 1, chunk along dimension 2, and the dimension-3 position.
struct BTile {
  int grid, bx, by, bz;
};

constexpr int kQueueStride = 64;
constexpr int kQueueInts = kXcds * kQueueStride + kXcds + 1;

// The tile of this workgroup in a launch from the queues' tiles `first` on, or
// -1 past the end of its queue.
__device__ inline int queue_tile(const int* __restrict__ queues, int first) {
  const int* start = queues + kXcds * kQueueStride;
  const int q = static_cast<int>(blockIdx.x) % kXcds;
  const int i = start[q] + first + static_cast<int>(blockIdx.x) / kXcds;
  return i < start[q + 1] ? i : -1;
}

// Tiles of the longest queue: queue_tile's launches take kXcds times as many
// workgroups.
inline int longest_queue(const int* host_q) {
  const int* start = host_q + kXcds * kQueueStride;
  int most = 0;
  for (int q = 0; q < kXcds; ++q) most = start[q + 1] - start[q] > most ? start[q + 1] - start[q] : most;
  return most;
}

namespace {

[[maybe_unused]] __global__ void queue_reset(int* counters) {
  if (blockIdx.x == 0 && threadIdx.x < kXcds) counters[threadIdx.x * kQueueStride] = 0;
}

// Thread 0 of a workgroup: the next tile, own queue first, or -1 once every
// queue is empty.  `visited` (kept by the caller) counts the queues already
// found empty; they are not asked again.
__device__ inline int pop_tile(int* counters, int home, int& visited) {
  const int* start = counters + kXcds * kQueueStride;
  for (; visited < kXcds; ++visited) {
    const int q = (home + visited) % kXcds;
    const int i = start[q] + atomicAdd(counters + q * kQueueStride, 1);
    if (i < start[q + 1]) return i;
  }
  return -1;
}

}  // namespace

}  // namespace sg
