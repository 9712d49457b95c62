// The kernel on registers for the phases of a strided input gradient, whose filter rows have 1 to 3 taps.
#include "phx_launch_reg16.h"

namespace phx {

template <int KW>
static int launch_row(bool cl, const RegPhaseArgs& a, int waves, int blocks, hipStream_t st) {
    return cl ? launch_reg_one<KW, 1, 1, true, false, true>(a, waves, blocks, st) : launch_reg_one<KW, 1, 1, false, false, true>(a, waves, blocks, st);
}

int launch_reg_phases(int kw, bool cl, const RegPhaseArgs& a, int waves, int blocks, hipStream_t st) {
    if (kw == 1) return launch_row<1>(cl, a, waves, blocks, st);
    if (kw == 2) return launch_row<2>(cl, a, waves, blocks, st);
    if (kw == 3) return launch_row<3>(cl, a, waves, blocks, st);
    return -1;
}

}  // namespace phx
