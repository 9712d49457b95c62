// Instantiations of the fp32-MFMA forward / input-gradient kernels and their filter packing.
#include "phx_launch.h"

namespace phx {

template <int MODE>
static int launch_variant(const FwdVariant& v, const ConvArgs& a, hipStream_t st) {
#define PHX_CASE(WCO_, NTW_, CK_, P2_, VS_)                                                                   \
    if (v.WCO == WCO_ && v.NTW == NTW_ && v.CK == CK_ && v.P2LOG == P2_ && v.vstage == VS_) {                 \
        hipLaunchKernelGGL((qconv_fwd_f32_kernel<float, MODE, WCO_, NTW_, CK_, P2_, VS_>), dim3(v.wgs, grid_rows(a.groups)),          \
                           dim3(WG_THREADS), v.lds_bytes, st, a);                                             \
        return 0;                                                                                             \
    }
    // vector staging for every window without zero insertion; the per-position form only in its general shape
#define PHX_CASES(WCO_, NTW_)                                                                       \
    PHX_CASE(WCO_, NTW_, 8, 8, true) PHX_CASE(WCO_, NTW_, 16, 7, true) PHX_CASE(WCO_, NTW_, 32, 6, true) \
    PHX_CASE(WCO_, NTW_, 8, 8, false)
    PHX_CASES(1, 1) PHX_CASES(2, 1) PHX_CASES(4, 1)
    if constexpr (MODE == 16) {
        PHX_CASES(1, 2) PHX_CASES(2, 2) PHX_CASES(4, 2)
    }
#undef PHX_CASES
#undef PHX_CASE
    return -1;
}

// (fp32 tensors only: fp16 tensors run on the fp16 matrix instructions under every policy)
int launch_fwd_f32(const FwdVariant& v, const ConvArgs& a, hipStream_t st) {
    // one kernel for both passes: the input gradient differs only in how its filters are packed
    if (v.pwx3) return launch_pw_x3(v, a, st);
    if (v.x3) return launch_fwd_x3(v, a, st);
    return v.mode == 16 ? launch_variant<16>(v, a, st) : launch_variant<8>(v, a, st);
}

int launch_pack_filters(const FwdVariant& v, const PackArgs& a, int blocks, hipStream_t st) {
    if (v.pwx3) return launch_pack_filters_pw_x3(v.map, v.WCO, a, blocks, st);
    if (v.x3) return launch_pack_filters_x3(v.map, v.WCO, v.ngroups, a, blocks, st);
    const dim3 g(blocks, grid_rows(a.groups)), b(WG_THREADS);
    if (v.mode == 16 && v.map == MAP_FWD) hipLaunchKernelGGL((pack_filters_f32_kernel<float, 16, MAP_FWD>), g, b, 0, st, a);
    else if (v.mode == 16) hipLaunchKernelGGL((pack_filters_f32_kernel<float, 16, MAP_DGRAD>), g, b, 0, st, a);
    else if (v.map == MAP_FWD) hipLaunchKernelGGL((pack_filters_f32_kernel<float, 8, MAP_FWD>), g, b, 0, st, a);
    else hipLaunchKernelGGL((pack_filters_f32_kernel<float, 8, MAP_DGRAD>), g, b, 0, st, a);
    return 0;
}

}  // namespace phx
