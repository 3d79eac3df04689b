// The kernels of head dimension 256 (compiled with -amdgpu-mfma-vgpr-form, see sa2_acc.hpp).
#include "sa2_launch.hpp"
#include "sa2_wide.hpp"
#include "sa2_wide_q.hpp"

namespace sa2 {

void launch_fwd_wide(int grid, hipStream_t stream, const KParams &p) {
    hipLaunchKernelGGL(fwd_wide_kernel<256>, dim3(grid), dim3(256), 0, stream, p);
}

void launch_bwd_wide_q(bool dq, int grid, hipStream_t stream, const KParams &p, float *ws, int halo) {
    if (dq) hipLaunchKernelGGL((bwd_wide_q_kernel<256, true>), dim3(grid), dim3(256), 0, stream, p, ws, halo);
    else hipLaunchKernelGGL((bwd_wide_q_kernel<256, false>), dim3(grid), dim3(256), 0, stream, p, ws, halo);
}

}  // namespace sa2
