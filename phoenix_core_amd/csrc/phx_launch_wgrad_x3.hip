// fp32 filter gradient on bf16 matrix instructions.
#include "phx_kernels_wgx3.h"
#include "phx_launch.h"

namespace phx {

size_t wgrad_x3_lds_bytes() { return WGX3_LDS_BYTES; }

int launch_wgrad_x3(const WgradArgs& a, dim3 grid, hipStream_t st) {
    constexpr auto kernel = qconv_wgrad_x3_kernel;
    if (!BigLds<kernel>::registered) return -1;  // dynamic LDS opt-in at set-up, see BigLds
    hipLaunchKernelGGL(kernel, grid, dim3(WGX3_THREADS), WGX3_LDS_BYTES, st, a);
    return 0;
}

}  // namespace phx
