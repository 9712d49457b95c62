// The kernel on registers (phx_kernels_reg16.h): which instances there are, and its filter packing.
#include "phx_launch_reg16.h"

namespace phx {

#define PHX_REG_ROWS(X) X(1, 1, 1) X(1, 1, 2) X(3, 1, 1) X(3, 1, 2) X(3, 2, 1) X(5, 1, 1) X(5, 1, 2)  // (taps, dilation, stride) along a row
#define PHX_CASE(K, D, S) int launch_reg_k##K##d##D##s##S(bool cl, const RegArgs& a, const NormArgs& norm, int waves, int blocks, hipStream_t st);
PHX_REG_ROWS(PHX_CASE)
#undef PHX_CASE

bool reg_row_shape(int kw, int dw, int sw) {
#define PHX_CASE(K, D, S) \
    if (kw == K && (dw == D || K == 1) && sw == S) return true;
    PHX_REG_ROWS(PHX_CASE)
#undef PHX_CASE
    return false;
}

int launch_reg_f16(int kw, int dw, int sw, bool cl, const RegArgs& a, const NormArgs& norm, int waves, int blocks, hipStream_t st) {
#define PHX_CASE(K, D, S) \
    if (kw == K && (dw == D || K == 1) && sw == S) return launch_reg_k##K##d##D##s##S(cl, a, norm, waves, blocks, st);
    PHX_REG_ROWS(PHX_CASE)
#undef PHX_CASE
    return -1;
}

template <int MAP>
__global__ void __launch_bounds__(WG_THREADS) pack_filters_reg_kernel(const PackArgs P) {
    pack_filters_reg_body<MAP>(P, (long)blockIdx.x * blockDim.x + threadIdx.x, (long)gridDim.x * blockDim.x);
}

int launch_pack_filters_reg(int map, const PackArgs& a, int blocks, hipStream_t st) {
    hipLaunchKernelGGL(map == MAP_FWD ? pack_filters_reg_kernel<MAP_FWD> : pack_filters_reg_kernel<MAP_DGRAD>, dim3(blocks), dim3(WG_THREADS), 0, st, a);
    return 0;
}

}  // namespace phx
