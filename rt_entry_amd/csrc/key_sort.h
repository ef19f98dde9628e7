// Sorting 64-bit keys across a wave, one a lane.
#pragma once
#include <stdint.h>

#include "search_impl.h"

namespace rte {

// compare-exchange of 64-bit keys at lane distance SUB: ascending, or
// descending where DESC(lane) holds
template <int SUB>
__device__ __forceinline__ uint64_t cas_key(uint64_t k, int lane, bool want_larger) {
  const uint32_t lo = (uint32_t)xor_lane<SUB>((int)(uint32_t)k, lane);
  const uint32_t hi = (uint32_t)xor_lane<SUB>((int)(uint32_t)(k >> 32), lane);
  const uint64_t p = ((uint64_t)hi << 32) | lo;
  return (p > k) == want_larger ? p : k;
}
template <int STEP, int SUB>
__device__ __forceinline__ uint64_t sort_keys_step(uint64_t k, int lane) {
  // pairs of a step are descending where (lane & 2 * STEP) == 0
  k = cas_key<SUB>(k, lane, ((lane & SUB) == 0) == ((lane & (2 * STEP)) == 0));
  if constexpr (SUB > 1) return sort_keys_step<STEP, SUB / 2>(k, lane);
  return k;
}
template <int STEP = 1>
__device__ __forceinline__ uint64_t sort_keys_desc(uint64_t k, int lane) {
  k = sort_keys_step<STEP, STEP>(k, lane);
  if constexpr (STEP < 32) return sort_keys_desc<STEP * 2>(k, lane);
  return k;
}
template <int SUB = 32>
__device__ __forceinline__ uint64_t merge_keys_asc(uint64_t k, int lane) {
  k = cas_key<SUB>(k, lane, (lane & SUB) != 0);
  if constexpr (SUB > 1) return merge_keys_asc<SUB / 2>(k, lane);
  return k;
}

}  // namespace rte
