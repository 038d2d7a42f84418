// pool_slices_quant.hip -- the sliced find-and-pool kernels over the
// reference's rowwise int8 / uint8 row formats.
#include "pool_slices.cuh"

namespace nve_amd {

hipError_t launch_pool_slices_quant(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream) {
  switch (a.stored_dtype) {
    case kQI8F32: return launch_slices_sdt<kQI8F32>(a, g, stream);
    case kQI8F16: return launch_slices_sdt<kQI8F16>(a, g, stream);
    case kQU8F32: return launch_slices_sdt<kQU8F32>(a, g, stream);
    case kQU8F16: return launch_slices_sdt<kQU8F16>(a, g, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace nve_amd
