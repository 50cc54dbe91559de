// Stable ranking of 8-bit digits inside a wave and over a workgroup: shared by the sort kernels (bucket_sort.hip) and by the
// workgroups that hash and rank beside the exact causal kernel (unit_ranking.h).
#pragma once

#include "ha_common.h"

namespace {

// lanes of the wave holding the same digit as this lane, restricted to valid lanes.  Per bit: the
// lane's own bit spread over a word (0 or ~0), one ballot, and per mask half one three-input bit
// operation "keep the lanes whose bit equals mine".
__device__ __forceinline__ uint64_t match_digit(int digit, bool valid) {
  const uint64_t all = __ballot(valid);
  uint32_t lo = (uint32_t)all, hi = (uint32_t)(all >> 32);
#pragma unroll
  for (int bit = 0; bit < 8; ++bit) {
    const uint32_t mine = (uint32_t)((int32_t)((uint32_t)digit << (31 - bit)) >> 31);
    const uint64_t b = __ballot(mine != 0u);
    lo &= ~((uint32_t)b ^ mine);
    hi &= ~((uint32_t)(b >> 32) ^ mine);
  }
  return ((uint64_t)hi << 32) | lo;
}

// number of set bits of `mask` below this lane
__device__ __forceinline__ uint32_t rank_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// exclusive scan of one value per thread over a block
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* wave_totals) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  uint32_t incl = v;
#pragma unroll
  for (int off = 1; off < HA_WAVE; off <<= 1) {
    const uint32_t up = __shfl_up(incl, off);
    if (lane >= off) incl += up;
  }
  if (lane == HA_WAVE - 1) wave_totals[wave] = incl;
  __syncthreads();
  uint32_t base = 0;
  for (int w = 0; w < wave; ++w) base += wave_totals[w];
  __syncthreads();
  return base + incl - v;
}

}  // namespace
