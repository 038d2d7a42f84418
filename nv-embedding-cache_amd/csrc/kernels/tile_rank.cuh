// tile_rank.cuh -- pieces of a digit sort inside one workgroup, shared by the
// radix sort's passes and the single-workgroup dedup: the stable rank of a
// key's digit among its wave's keys.
#pragma once

#include "device_common.cuh"

namespace nve_amd {

constexpr int kMaxBins = 512;  // digits of at most 9 bits

// One key per lane, d its digit of RB bits: returns the number of the wave's
// earlier keys of the same digit (those counted in cnt by earlier rounds, then
// the lower lanes) and adds this round's keys to cnt (one word per digit, the
// wave's own).  The lanes sharing a digit are found with one ballot per bit.
template <int RB>
__device__ __forceinline__ uint32_t wave_digit_rank(uint32_t d, bool valid, uint32_t* cnt) {
  const uint64_t valids = __ballot(valid);
  uint32_t lo = (uint32_t)valids, hi = (uint32_t)(valids >> 32);
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const uint64_t m = __ballot((d >> b) & 1u);
    const uint32_t mine = 0u - ((d >> b) & 1u);  // lanes whose bit differs leave
    lo &= ~((uint32_t)m ^ mine);
    hi &= ~((uint32_t)(m >> 32) ^ mine);
  }
  const uint64_t peers = ((uint64_t)hi << 32) | lo;
  const uint32_t before = (uint32_t)__popcll(peers & ((1ull << (threadIdx.x & 63)) - 1ull));
  // a wave's LDS accesses stay in order: every lane reads the count before the
  // first of its digit's lanes adds to it
  const uint32_t seen = cnt[d];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (valid && before == 0) cnt[d] = seen + (uint32_t)__popcll(peers);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  return seen + before;
}

// A word published by a tile: state in the top two bits, a count below.
constexpr uint64_t kStateOwn = 1ull << 62;     // of the tile alone
constexpr uint64_t kStateBefore = 2ull << 62;  // with every tile before it
constexpr uint64_t kStateCount = (1ull << 62) - 1;

__device__ __forceinline__ uint64_t load_state(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_state(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The next tile number: tiles are numbered in the order their workgroups start.
__device__ __forceinline__ uint32_t take_tile(uint64_t* counter) {
  return (uint32_t)atomicAdd(reinterpret_cast<unsigned long long*>(counter), 1ull);
}

}  // namespace nve_amd
