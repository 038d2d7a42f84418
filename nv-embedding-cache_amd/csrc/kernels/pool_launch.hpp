// pool_launch.hpp -- per-type-group launchers of the find-and-pool kernel
// (pool_float.hip, pool_quant.hip, pool_ext.hip), called by launch_pool once
// it has chosen the geometry.
#pragma once

#include "launch.hpp"

namespace nve_amd {

// kF32, kF16
hipError_t launch_pool_float(const PoolLaunch& a, const PoolGeometry& g, hipStream_t stream);
// kQI8F32, kQI8F16, kQU8F32, kQU8F16
hipError_t launch_pool_quant(const PoolLaunch& a, const PoolGeometry& g, hipStream_t stream);
// kXI8AF32, kXE4M3F32
hipError_t launch_pool_ext(const PoolLaunch& a, const PoolGeometry& g, hipStream_t stream);

// The sliced kernels (pool_slices.cuh): each lane of a group of g lanes takes vb
// bytes of a row, columns groups cover it, and gpb groups share a bag.
struct PoolSlices {
  int vb, g, columns, gpb;
};
// Whether they serve the launch, and how (pool_split.hip).
bool pool_slices(const PoolLaunch& a, PoolSlices* g);
hipError_t launch_pool_slices(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream);
// kQI8F32, kQI8F16, kQU8F32, kQU8F16
hipError_t launch_pool_slices_quant(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream);
// kXI8AF32, kXE4M3F32
hipError_t launch_pool_slices_ext(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream);

// Lane groups that share a bag, for groups of g lanes (lookup.hip).
int pool_groups_per_bag(const PoolLaunch& a, int g);

}  // namespace nve_amd
