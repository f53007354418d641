// Per-cell maxima of particles in arbitrary order.
//
// The order leaves no runs to reduce, so every particle would go to memory
// past the caches (an XCD's L2 does not see the other XCDs' atomics): about 30
// G/s over the chip, a few M/s on one word, and clustered cells hold many
// particles.  Two things keep most of them from it:
//  - the particles are taken in ranges up to n/64, n/16, n/4 and n, a launch each.  A
//    launch starts with fresh caches, so an ordinary cached read of the maximum
//    that the ranges before left drops all but about 1 in 5 of 64 random
//    particles of a cell (the read may be stale, but is never above the true
//    value, so nothing is dropped wrongly);
//  - a workgroup sends one particle per cell, picked by an LDS table.
// The volumetric keys of 60k particles 32 us in one launch without either, 11 now;
// of 16M 706 and 471.  (32M particles on 22M cells, a table beyond the caches:
// 1011 and 967.)
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace ilc {

constexpr int kMaxSlots = 1024;

// cellmax[cell] = max(cellmax[cell], v) for the workgroup's threads with valid
// set; slots is LDS, every thread of the workgroup calls
__device__ inline void block_raise_max(uint32_t* __restrict__ cellmax, uint32_t cell, uint32_t v,
                                       bool valid, unsigned long long (&slots)[kMaxSlots]) {
#pragma unroll
  for (int k = 0; k < kMaxSlots / kBlock; ++k) slots[threadIdx.x + k * kBlock] = 0ull;
  __syncthreads();
  valid = valid && v > __hip_atomic_load(cellmax + cell, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
  // the slot's largest (cell, v): a cell that loses its slot to another sends
  // its particles itself
  auto& slot = slots[(cell * 2654435761u) >> 22];
  const unsigned long long mine = (static_cast<unsigned long long>(cell) << 32) | v;
  if (valid) atomicMax(&slot, mine);
  __syncthreads();
  if (valid) {
    const unsigned long long best = slot;
    if (uint32_t(best >> 32) != cell || best == mine)
      if (v > __hip_atomic_load(cellmax + cell, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(cellmax + cell, v);
  }
}

// f(first, last) over the ranges of n particles.  Below a million the extra
// launches cost more than the atomics.
template <class F>
void for_ranges(uint32_t n, F&& f) {
  uint32_t first = 0;
  for (int shift = n < (1u << 20) ? 0 : 6; shift >= 0; shift -= 2) {
    const uint32_t last = shift ? (n >> shift) / kBlock * kBlock : n;
    if (last > first) f(first, last);
    first = last;
  }
}

}  // namespace ilc
