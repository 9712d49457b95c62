// Launches of the kernel on registers (phx_kernels_reg16.h), one translation unit for each shape of a filter row.
#pragma once

#include "phx_kernels_reg16.h"
#include "phx_launch.h"

namespace phx {

template <int KW, int D, int S, bool CL, bool NORM, bool PHASE = false>
static int launch_reg_one(const RegArgsOf<NORM, PHASE>& a, int waves, int blocks, hipStream_t st) {
    constexpr auto kernel = qconv_reg_f16_kernel<KW, D, S, CL, NORM, PHASE>;
    if (!BigLds<kernel>::registered || waves > reg_waves(KW)) return -1;  // dynamic LDS opt-in at set-up, see BigLds
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * waves), a.kslog ? waves * REG_WAVE_LDS : 0, st, a);
    return 0;
}

template <int KW, int D, int S>
static int launch_reg_row(bool cl, const RegArgs& a, const NormArgs& norm, int waves, int blocks, hipStream_t st) {
    if (norm.gamma) return cl ? -1 : launch_reg_one<KW, D, S, false, true>(RegNormArgs{a, norm}, waves, blocks, st);
    return cl ? launch_reg_one<KW, D, S, true, false>(a, waves, blocks, st) : launch_reg_one<KW, D, S, false, false>(a, waves, blocks, st);
}

}  // namespace phx
