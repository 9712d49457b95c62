// The kernel on registers for filter rows of 3 taps, dilation 1, stride 1.
#include "phx_launch_reg16.h"

namespace phx {

int launch_reg_k3d1s1(bool cl, const RegArgs& a, const NormArgs& norm, int waves, int blocks, hipStream_t st) {
    return launch_reg_row<3, 1, 1>(cl, a, norm, waves, blocks, st);
}

}  // namespace phx
