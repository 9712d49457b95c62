// fp16-MFMA forward / input-gradient kernels in factorized form with the product lanes dealt over the waves, and their
// filter packing.
#include "phx_kernels_lanes16.h"
#include "phx_launch.h"

namespace phx {

size_t lanes_lds_bytes() { return LANES_LDS_BYTES; }
size_t lanes_image_bytes(int co_tiles, int nchunks, int ngroups) { return lanes_packed_bytes(co_tiles, nchunks, ngroups * LANES_GROUP); }

int launch_fwd_f16_lanes(const FwdVariant& v, const ConvArgs& a, hipStream_t st) {
#define PHX_CASE(NTW_, CL_)                                                                              \
    if (v.NTW == NTW_ && (a.nhwc != 0) == CL_) {                                                         \
        constexpr auto kernel = qconv_fwd_f16_lanes_kernel<2 * NTW_, CL_>;                               \
        if (!BigLds<kernel>::registered) return -1; /* dynamic LDS opt-in at set-up, see BigLds */       \
        hipLaunchKernelGGL(kernel, dim3(v.wgs, grid_rows(a.groups)), dim3(WG_THREADS), v.lds_bytes, st, a); \
        return 0;                                                                                        \
    }
    PHX_CASE(1, false) PHX_CASE(2, false) PHX_CASE(1, true) PHX_CASE(2, true)
#undef PHX_CASE
    return -1;
}

int launch_pack_filters_lanes(int map, int ngroups, const PackArgs& a, int blocks, hipStream_t st) {
    const PackLanesArgs la{a, ngroups * LANES_GROUP};
    const dim3 g(blocks, grid_rows(a.groups)), b(WG_THREADS);
    if (map == MAP_FWD) hipLaunchKernelGGL((pack_filters_lanes_kernel<MAP_FWD>), g, b, 0, st, la);
    else hipLaunchKernelGGL((pack_filters_lanes_kernel<MAP_DGRAD>), g, b, 0, st, la);
    return 0;
}

}  // namespace phx
