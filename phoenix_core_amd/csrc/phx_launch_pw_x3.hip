// fp32 pointwise kernel on bf16 matrix instructions and its filter packing.
#include "phx_kernels_pwx3.h"
#include "phx_launch.h"

namespace phx {

int pw_x3_pixels() { return PWX3_PX; }
size_t pw_x3_lds_bytes() { return PWX3_LDS_BYTES; }
size_t pw_x3_image_bytes(int WCO, int co_tiles, int nsteps, int red, int rows) {
    return pwx3_packed_bytes(WCO, co_tiles, nsteps) + split_copy_bytes(1, red, rows);
}

int launch_pw_x3(const FwdVariant& v, const ConvArgs& a, hipStream_t st) {
    const dim3 grid(v.wgs, grid_rows(a.groups));
    if (v.WCO == 1) hipLaunchKernelGGL((qconv_pw_x3_kernel<1>), grid, dim3(WG_THREADS), PWX3_LDS_BYTES, st, a);
    else hipLaunchKernelGGL((qconv_pw_x3_kernel<2>), grid, dim3(WG_THREADS), PWX3_LDS_BYTES, st, a);
    return 0;
}

int launch_pack_filters_pw_x3(int map, int WCO, const PackArgs& a, int blocks, hipStream_t st) {
    const dim3 g(blocks, grid_rows(a.groups)), b(WG_THREADS);
    if (map == MAP_FWD) hipLaunchKernelGGL((pack_filters_pwx3_kernel<MAP_FWD>), g, b, 0, st, a, WCO);
    else hipLaunchKernelGGL((pack_filters_pwx3_kernel<MAP_DGRAD>), g, b, 0, st, a, WCO);
    return 0;
}

}  // namespace phx
