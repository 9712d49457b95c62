// The kernel on registers for filter rows of 3 taps, dilation 1, stride 2.
#include "phx_launch_reg16.h"

namespace phx {

int launch_reg_k3d1s2(bool cl, const RegArgs& a, const NormArgs& norm, int waves, int blocks, hipStream_t st) {
    return launch_reg_row<3, 1, 2>(cl, a, norm, waves, blocks, st);
}

}  // namespace phx
