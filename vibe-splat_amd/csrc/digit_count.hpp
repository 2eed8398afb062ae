// Counting a sort's digits where its keys are written (sort.hip): per tile of
// kCountedTile destinations, how many of its keys hold each digit of the next pass.
#pragma once

#include "device.hpp"
#include "kernels.hpp"

namespace vsplat {

// One more key of digit `digit` stored at `at`, for every lane that has one
// (valid; every lane of the wave calls it). Neighbouring keys often share tile
// and digit (a depth key's high bytes are all but constant), and atomics on one
// address are served one after another, some 8 ns each: the first two groups of
// equal lanes add once for all of theirs, and what is left adds lane by lane.
__device__ __forceinline__ void count_digit(uint32_t *__restrict__ counts, uint32_t at, uint32_t digit, bool valid) {
  const uint32_t slot = (at / kCountedTile) * kCountedStride + digit;
  uint64_t left = __ballot(valid);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (left == 0) return;
    const int leader = __builtin_ctzll(left);
    const uint64_t same = __ballot(slot == static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(slot), leader))) & left;
    if (static_cast<int>(threadIdx.x & 63u) == leader) atomicAdd(&counts[slot], static_cast<uint32_t>(__popcll(same)));
    left &= ~same;
  }
  if ((left >> (threadIdx.x & 63u)) & 1u) atomicAdd(&counts[slot], 1u);
}

} // namespace vsplat
