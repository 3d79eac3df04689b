// The register-resident dK1/dV1 kernel (compiled with -amdgpu-mfma-vgpr-form, see sa2_acc.hpp).
#include "sa2_bwd_kvr.hpp"
#include "sa2_launch.hpp"

namespace sa2 {

void launch_bwd_kvr(bool in_parts, int grid, hipStream_t stream, const KParams &p) {
    if (in_parts) hipLaunchKernelGGL((bwd_kvr_kernel<256, true>), dim3(grid), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((bwd_kvr_kernel<256, false>), dim3(grid), dim3(256), 0, stream, p);
}

}  // namespace sa2
