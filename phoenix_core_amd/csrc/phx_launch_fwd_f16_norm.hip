// fp16-MFMA forward kernels that apply evaluation-mode batch norm (+ residual, ReLU) to what they store: the instances of the
// chunk-staging and the lane-dealing kernels with NORM (instances of their own: what they add to the epilogue would cost the
// plain kernels registers).  The quaternion ResNet-50 in evaluation mode, 8 images of 224x224: 1717 us with a normalisation
// pass behind each of its 53 convolutions (265 us of kernel time, and as many operator calls of the host, which bounds it),
// 889 us with the passes inside the convolutions; where each pass of the network is waited for, 1815 and 1010.
#include "phx_kernels_lanes16.h"
#include "phx_launch.h"

namespace phx {

bool fwd_f16_takes_norm(const FwdVariant& v, const ConvArgs& a) { return !a.nhwc && (v.lanes || (v.lds_filters && v.chunks)); }

template <auto kernel>
static int launch_one(const FwdVariant& v, const ConvNormArgs& a, hipStream_t st, size_t more_lds = 0) {
    if (!BigLds<kernel>::registered) return -1;  // dynamic LDS opt-in at set-up, see BigLds
    hipLaunchKernelGGL(kernel, dim3(v.wgs, grid_rows(a.groups)), dim3(WG_THREADS), v.lds_bytes + more_lds, st, a);
    return 0;
}

// (the instance that the same variant takes without NORM: launch_fwd_f16)
int launch_fwd_f16_norm(const FwdVariant& v, const ConvArgs& plain, const NormArgs& norm, hipStream_t st) {
    const ConvNormArgs a{plain, norm};
    if (v.lanes) return v.NTW == 1 ? launch_one<qconv_fwd_f16_lanes_kernel<2, false, true>>(v, a, st, LANES_NORM_BYTES) :
                        v.NTW == 2 ? launch_one<qconv_fwd_f16_lanes_kernel<4, false, true>>(v, a, st, LANES_NORM_BYTES) : -1;
#define PHX_CASE(MODE_, WCO_, NTW_, EARLY_, XREAL_) \
    if (v.WCO == WCO_ && v.NTW == NTW_) return launch_one<qconv_fwd_f16_lds_kernel<MODE_, WCO_, NTW_, 8, true, EARLY_, XREAL_, true>>(v, a, st);
    if (v.mode == 8) {
        PHX_CASE(8, 1, 1, false, false) PHX_CASE(8, 1, 2, false, false) PHX_CASE(8, 2, 1, false, false) PHX_CASE(8, 2, 2, false, false)
        return -1;
    }
    if (a.in.ncomp == 1 && !(v.ngroups == 1 && v.NTW == 1)) {
        PHX_CASE(16, 1, 1, false, true) PHX_CASE(16, 1, 2, false, true) PHX_CASE(16, 2, 1, false, true) PHX_CASE(16, 2, 2, false, true)
        PHX_CASE(16, 4, 1, false, true) PHX_CASE(16, 4, 2, false, true)
        return -1;
    }
    if (v.ngroups == 1 && v.NTW == 1 && !tuning_noearly()) {
        PHX_CASE(16, 1, 1, true, false) PHX_CASE(16, 2, 1, true, false)
    }
    PHX_CASE(16, 1, 1, false, false) PHX_CASE(16, 1, 2, false, false) PHX_CASE(16, 2, 1, false, false) PHX_CASE(16, 2, 2, false, false)
    PHX_CASE(16, 4, 1, false, false) PHX_CASE(16, 4, 2, false, false)
#undef PHX_CASE
    return -1;
}

}  // namespace phx
