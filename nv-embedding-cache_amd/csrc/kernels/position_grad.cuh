// position_grad.cuh -- the gradient row and weight of key positions of a
// training backprop, computed by the dedup's run outputs on the way.
//
// Reference behaviour restated: compute_normalized_weights and
// compute_pooling_inverse_mapping (cuda_ops/gradient_calculator.cuh:29-82).
#pragma once

#include "backprop_launch.hpp"
#include "device_common.cuh"

namespace nve_amd {

// rows[x] = the gradient row of key position base + x, x < TILE: the bag that holds
// it (Fixed: position / hotness; CSR: the last bag b with offsets[b] <= position,
// when that is below offsets[b + 1]), kNoGradRow outside every bag.  rows: LDS;
// every thread of the workgroup calls it.  The tile's first bag comes from a
// search that reads an offset per thread and step; the bags that start inside
// the tile mark their first positions, and a running maximum spreads the marks.  (A
// search per position is bound by its loads: 9.5 us for 262,144 positions of
// 256 bags, with eight offsets a step 20 us; this takes 4.)  A thread marks at most
// kMarkSteps bags, each step a load's latency (0.8 us): where more bags start in the
// tile (mostly empty ones), every position searches for its own.  The line is
// where the two meet: backprop of 2,000 keys with 4,096, 8,192 and 16,384 bags in a
// tile takes 46.5, 50 and 57 us with marks and 49 with the search, of 100,000 keys 83,
// 86 and 93 us and 81-82.  (All bags marked, 2,000 keys in 1,000,000 bags: 861 us; 57 now.)
constexpr int kMarkSteps = 8;
template <int NT, int TILE>
__device__ __forceinline__ void tile_rows(const PositionGrad& g, int64_t base, uint32_t* rows) {
  constexpr int kPer = TILE / NT;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (g.offsets == nullptr) {
    for (int x = tid; x < TILE; x += NT) {
      const int64_t b = g.hotness > 0 ? (base + x) / g.hotness : -1;
      rows[x] = b >= 0 && b < g.num_bags ? (uint32_t)b : kNoGradRow;
    }
    __syncthreads();
    return;
  }
  __shared__ uint32_t s_max[NT / 64];
  for (int x = tid; x < TILE; x += NT) rows[x] = 0;
  // the first bag with offsets[b] > base, in [lo, hi] (32-bit: num_bags <
  // kNoGradRow; as 64-bit integers the two minima of a step were compiled into
  // selects that shared one condition)
  uint32_t lo = 0, hi = (uint32_t)g.num_bags;
  while (lo < hi) {  // uniform over the workgroup
    const uint32_t step = (hi - lo - 1) / NT + 1;
    const uint64_t at = lo + (uint64_t)step * (uint32_t)(tid + 1) - 1;
    bool le = false;
    if (at < hi) le = load_key(g.offsets, g.key_bytes, (int64_t)at) <= base;
    lo += step * (uint32_t)__syncthreads_count(le);  // at most hi: only offsets below hi count
    hi = hi - lo < step ? hi : lo + step - 1;
  }
  __syncthreads();
  const int64_t first = lo;
  const int64_t end = g.num_bags > 0 ? load_key(g.offsets, g.key_bytes, g.num_bags) - base : 0;
  const int64_t past = first + (int64_t)kMarkSteps * NT;  // the first bag that no thread would mark
  if (past < g.num_bags && load_key(g.offsets, g.key_bytes, past) - base < TILE) {  // uniform
    uint32_t n[kPer];  // bags that start at or before the position, at least `first`
#pragma unroll
    for (int q = 0; q < kPer; ++q) n[q] = lo;
    for (uint32_t half, len = (uint32_t)g.num_bags - lo; len > 0; len -= half) {
      half = (len + 1) / 2;
#pragma unroll
      for (int q = 0; q < kPer; ++q)
        if (load_key(g.offsets, g.key_bytes, (int64_t)n[q] + half - 1) <= base + q * NT + tid) n[q] += half;
    }
#pragma unroll
    for (int q = 0; q < kPer; ++q) rows[q * NT + tid] = n[q] != 0 && q * NT + tid < end ? n[q] - 1u : kNoGradRow;
    __syncthreads();
    return;
  }
  for (int64_t b = first + tid; b < g.num_bags; b += NT) {
    const int64_t x = load_key(g.offsets, g.key_bytes, b) - base;
    if (x >= TILE || x < 0) break;  // non-decreasing offsets: none of the later ones either
    atomicMax(&rows[x], (uint32_t)b + 1u);
  }
  __syncthreads();
  uint32_t v[kPer], m = 0;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    v[q] = rows[tid * kPer + q];
    m = v[q] > m ? v[q] : m;
  }
  uint32_t inc = m;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o);
    if (lane >= o) inc = t > inc ? t : inc;
  }
  if (lane == 63) s_max[wave] = inc;
  uint32_t run = __shfl_up(inc, 1);
  if (lane == 0) run = 0;
  __syncthreads();
  run = run > (uint32_t)first ? run : (uint32_t)first;  // the bag before the first that starts in the tile, + 1
#pragma unroll
  for (int w = 0; w < NT / 64; ++w)
    if (w < wave) run = s_max[w] > run ? s_max[w] : run;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    run = v[q] > run ? v[q] : run;
    rows[tid * kPer + q] = run != 0 && tid * kPer + q < end ? run - 1u : kNoGradRow;
  }
  __syncthreads();
}

// Whether a position's weight needs nothing but its gradient row, so that the
// dedup may carry rows in place of positions.
__host__ __device__ __forceinline__ bool weight_from_row(int mode) {
  return mode != kBackpropWSum && mode != kBackpropWMean;
}

// For the dedup positions first + j * step below n, j < ITEMS: rows[..] = the
// gradient row it reads, nw[..] = its weight (w[p], 1 / count or w[p] / sum of the
// bag's weights; not written where it is 1).  v[j] is its row if `carried`, else
// its key position, whose row row_at gives.
template <int ITEMS, typename R>
__device__ __forceinline__ void position_grads(const PositionGrad& g, bool carried, const R& row_at, int64_t first,
                                               int64_t step, int64_t n, const uint32_t (&v)[ITEMS]) {
  uint32_t row[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
    row[j] = carried || g.mode == kBackpropConcat || first + j * step >= n ? v[j] : row_at(v[j]);
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int64_t i = first + j * step;
    if (i < n) {
      g.rows[i] = row[j];
      if (g.mode >= kBackpropWSum) {
        float w = 1.0f;
        if (row[j] != kNoGradRow) {
          if (g.mode == kBackpropWSum) w = load_weight(g.weights, g.wdt, v[j]);
          else if (g.mode == kBackpropMean) w = 1.0f / g.denom[row[j]];
          else w = load_weight(g.weights, g.wdt, v[j]) / g.denom[row[j]];
        }
        g.nw[i] = w;
      }
    }
  }
}

}  // namespace nve_amd
