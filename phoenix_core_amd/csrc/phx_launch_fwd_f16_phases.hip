// The phases of a strided fp16 input gradient in one launch: fp16-MFMA kernel with both operands through LDS, 16-product form.
#include "phx_kernels_f16.h"
#include "phx_launch.h"

namespace phx {

int launch_fwd_f16_phases(const FwdVariant& v, const ConvPhases& a, int phases, hipStream_t st) {
#define PHX_CASE(WCO_)                                                                                          \
    if (v.WCO == WCO_) {                                                                                        \
        constexpr auto kernel = qconv_fwd_f16_lds_kernel<16, WCO_, 1, 8, true, false, false, false, true>;      \
        if (!BigLds<kernel>::registered) return -1; /* dynamic LDS opt-in at set-up, see BigLds */              \
        hipLaunchKernelGGL(kernel, dim3(v.wgs, phases), dim3(WG_THREADS), v.lds_bytes, st, a);                  \
        return 0;                                                                                               \
    }
    PHX_CASE(1) PHX_CASE(2)
#undef PHX_CASE
    return -1;
}

}  // namespace phx
