// pool_slices_ext.hip -- the sliced find-and-pool kernels over this build's two
// extra row formats (int8 with fp32 scale and offset; OCP fp8 e4m3 with fp32
// scale).
#include "pool_slices.cuh"

namespace nve_amd {

hipError_t launch_pool_slices_ext(const PoolLaunch& a, const PoolSlices& g, hipStream_t stream) {
  switch (a.stored_dtype) {
    case kXI8AF32: return launch_slices_sdt<kXI8AF32>(a, g, stream);
    case kXE4M3F32: return launch_slices_sdt<kXE4M3F32>(a, g, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace nve_amd
