// Pointwise fp16-MFMA kernels with the packed filter resident in LDS (phx_kernels_pwr16.h): instantiations.
#include "phx_kernels_pwr16.h"
#include "phx_launch.h"

namespace phx {

template <int WCO, int TAIL>
static int launch_pwr_one(const PwxArgsOf<TAIL>& a, int blocks, size_t lds_bytes, hipStream_t st) {
    constexpr auto kernel = qconv_pwr_f16_kernel<WCO, TAIL>;
    if (!BigLds<kernel>::registered) return -1;  // more than 64 KiB of dynamic LDS: opted in per device at set-up, see BigLds
    hipLaunchKernelGGL(kernel, dim3(blocks, grid_rows(a.groups)), dim3(WG_THREADS), lds_bytes, st, a);
    return 0;
}

template <int WCO>
static int launch_pwr_tail(const PwxArgs& a, const NormArgs& norm, int blocks, size_t lds_bytes, hipStream_t st) {
    const PwxNormArgs na{a, norm};
    if (norm.gamma)
        return a.addend ? launch_pwr_one<WCO, PWX_NORM_ADD>(na, blocks, lds_bytes, st) : launch_pwr_one<WCO, PWX_NORM>(na, blocks, lds_bytes, st);
    return a.addend ? launch_pwr_one<WCO, PWX_ADD>(a, blocks, lds_bytes, st) : launch_pwr_one<WCO, PWX_PLAIN>(a, blocks, lds_bytes, st);
}

// LDS of a workgroup: the filter image (K steps x sub-tiles x 4 components x 64 lanes x 16 bytes) and four waves' rings
size_t pwr_lds_bytes(int WCO, int nsteps) {
    return ((size_t)nsteps * WCO * 4 * 64 + 4 * PWR_STAGES * PWR_STAGE_VEC) * 16;
}

int launch_pwr_f16(int WCO, const PwxArgs& a, const NormArgs& norm, int blocks, hipStream_t st) {
    const size_t lds = pwr_lds_bytes(WCO, a.nsteps);
    if (lds > 160 * 1024 || a.co_tiles != 1 || a.nsteps < 2 || a.HW % 8 != 0 || a.GI * 8 != a.HW) return -1;
    if (WCO == 4) return launch_pwr_tail<4>(a, norm, blocks, lds, st);
    if (WCO == 2) return launch_pwr_tail<2>(a, norm, blocks, lds, st);
    if (WCO == 1) return launch_pwr_tail<1>(a, norm, blocks, lds, st);
    return -1;
}

}  // namespace phx
