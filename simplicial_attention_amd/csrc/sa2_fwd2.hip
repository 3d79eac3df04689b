// fwd2_kernel (compiled with -amdgpu-mfma-vgpr-form, see sa2_acc.hpp).
#include "sa2_fwd2.hpp"
#include "sa2_launch.hpp"

namespace sa2 {

void launch_fwd2(bool split, int grid, hipStream_t stream, const KParams &p) {
    if (split) hipLaunchKernelGGL((fwd2_kernel<128, true>), dim3(grid), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((fwd2_kernel<128>), dim3(grid), dim3(256), 0, stream, p);
}

}  // namespace sa2
