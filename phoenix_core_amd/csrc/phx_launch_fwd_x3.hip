// fp32 forward / input-gradient kernels on bf16 matrix instructions and their filter packing.
#include "phx_kernels_x3.h"
#include "phx_launch.h"

namespace phx {

size_t x3_lds_bytes() { return X3_LDS_BYTES; }
size_t x3_image_bytes(int WCO, int co_tiles, int nchunks, int ngroups, int taps, int red, int rows) {
    return x3_packed_bytes(WCO, co_tiles, nchunks, ngroups * X3_GROUP) + split_copy_bytes(taps, red, rows);
}

template <int S, int NPT>
static int launch_one(const FwdVariant& v, const ConvArgs& a, hipStream_t st) {
    constexpr auto kernel = qconv_fwd_x3_kernel<S, NPT>;
    if (!BigLds<kernel>::registered) return -1;  // dynamic LDS opt-in at set-up, see BigLds
    hipLaunchKernelGGL(kernel, dim3(v.wgs, grid_rows(a.groups)), dim3(WG_THREADS), v.lds_bytes, st, a);
    return 0;
}

int launch_fwd_x3(const FwdVariant& v, const ConvArgs& a, hipStream_t st) {
    if (v.WCO == 1) return v.NTW == 1 ? launch_one<1, 2>(v, a, st) : v.NTW == 2 ? launch_one<1, 4>(v, a, st) : -1;
    return v.NTW == 1 ? launch_one<2, 2>(v, a, st) : v.NTW == 2 ? launch_one<2, 4>(v, a, st) : -1;
}

int launch_pack_filters_x3(int map, int WCO, int ngroups, const PackArgs& a, int blocks, hipStream_t st) {
    const PackLanesArgs la{a, ngroups * X3_GROUP};
    const dim3 g(blocks, grid_rows(a.groups)), b(WG_THREADS);
    if (map == MAP_FWD) hipLaunchKernelGGL((pack_filters_x3_kernel<MAP_FWD>), g, b, 0, st, la, WCO);
    else hipLaunchKernelGGL((pack_filters_x3_kernel<MAP_DGRAD>), g, b, 0, st, la, WCO);
    return 0;
}

}  // namespace phx
