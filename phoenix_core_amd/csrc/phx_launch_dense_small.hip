// Quaternion Dense for small problems (a classifier head, the reference's own 128 -> 128 benchmark layer): the
// matrix-core kernels serve Dense as a 1x1 convolution on 1x1 images, where a batch of 32..64 rows is a single
// pixel tile -- one or two workgroups walking the whole reduction with a pack kernel in front and a split-K
// reduction behind (55 us per pass for 17 MFLOP).  Below a few million quaternion products plain fp32 FMA threads
// are faster: no packing, no workspace, one launch per pass, or for both gradients.
//   forward          y[q][n][o]  = sum_i sum_p s(p,q) x[p][n][i] w[p^q][i][o] (+ bias[q][o])      (src/dense.hpp:77-180)
//   input gradient   dx[q][n][i] = sum_o sum_p s(p,q) g[p][n][o] conj(w)[p^q][i][o]               (src/dense.hpp:252-377)
//   filter gradient  dw[q][i][o] = sum_n sum_p s(p,q) conj(x)[p][n][i] g[p^q][n][o]
// fp32 accumulation whatever the storage type (at least as exact as every fp16 policy asks for); the same result in
// either product mode.
#include "phx_launch.h"

namespace phx {

// Forward and input gradient share one kernel: out[q][a][b] = sum_k sum_p s(p,q) A[p][a][k] B[p^q][k][b], B the
// filter (conjugated for the input gradient), read at the strides of its layout.  A workgroup makes 16 outputs b of
// one row a; its 256 threads split the reduction 16 ways (short dependent-load chains: a thread's loop is nk / 16
// steps) and meet in LDS.  The 16 lanes that run along the filter's contiguous index read 64-byte runs.
struct DenseRowArgs {
    const void* a;     // [4][na][nk]
    const void* b;     // filter: element (c, k, b) at c * b_cs + k * b_ks + b * b_bs
    const void* bias;  // [4][nb] or null
    void* out;         // [4][na][nb]
    long b_cs, b_ks, b_bs;
    int na, nb, nk;
    int kfast;         // the filter is contiguous along k: lanes run along k (else along b)
};

typedef float DenseSums[4][16][17];

template <typename TS, bool CONJB>
__device__ __forceinline__ void dense_row_body(const DenseRowArgs& P, int block, DenseSums& part) {
    const int tiles_b = (P.nb + 15) >> 4;
    const int a = block / tiles_b, b0 = (block - a * tiles_b) * 16;
    const int lo = threadIdx.x & 15, hi = threadIdx.x >> 4;
    const int bl = P.kfast ? hi : lo, ks = P.kfast ? lo : hi;
    const int b = b0 + bl;
    const bool live = b < P.nb;
    const TS* A = static_cast<const TS*>(P.a) + (long)a * P.nk;
    const TS* B = static_cast<const TS*>(P.b) + (live ? b : 0) * P.b_bs;
    const long acs = (long)P.na * P.nk;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = ks; k < P.nk; k += 16) {
        float av[4], bv[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            av[c] = ldf<TS>(A + c * acs + k);
            const float v = ldf<TS>(B + c * P.b_cs + k * P.b_ks);
            bv[c] = (CONJB && c) ? -v : v;
        }
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] += (qneg(p, q) ? -av[p] : av[p]) * bv[p ^ q];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) part[q][bl][ks] = acc[q];
    __syncthreads();
    if (threadIdx.x < 64) {  // thread = (component, output): sums the 16 reduction slices in a fixed order
        const int q = threadIdx.x >> 4, ob = threadIdx.x & 15;
        if (b0 + ob < P.nb) {
            float sum = 0.f;
#pragma unroll
            for (int s = 0; s < 16; ++s) sum += part[q][ob][s];
            if (P.bias) sum += ldf<TS>(static_cast<const TS*>(P.bias) + q * P.nb + b0 + ob);
            static_cast<TS*>(P.out)[((long)q * P.na + a) * P.nb + b0 + ob] = (TS)sum;
        }
    }
}

// Filter gradient: a workgroup makes 64 neighbouring filter quaternions, its four waves a quarter of the rows each.  Chains of
// dependent loads bound it at these sizes: 32 rows, 128 -> 128 in fp32 took 8.1 us with a thread per quaternion on 64 workgroups
// and both gradients 14.6 in two launches; a quarter of the chain on 256, in one launch with the input gradient, takes 5.6.
constexpr int DENSE_WGRAD = 64;
template <typename TS>
__device__ __forceinline__ void dense_wgrad_body(const DenseSmallArgs& P, int block, DenseSums& sums) {
    float(*part)[4][DENSE_WGRAD] = reinterpret_cast<float(*)[4][DENSE_WGRAD]>(&sums[0][0][0]);  // [slice][component][quaternion]
    static_assert(sizeof(DenseSums) >= sizeof(float) * 4 * 4 * DENSE_WGRAD);
    const int slice = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int idx = block * DENSE_WGRAD + lane;
    const bool live = idx < P.ni * P.no;
    const int i = live ? idx / P.no : 0, o = live ? idx - i * P.no : 0;
    const TS* x = static_cast<const TS*>(P.a) + i;
    const TS* g = static_cast<const TS*>(P.b) + o;
    const long xcs = (long)P.n * P.ni, gcs = (long)P.n * P.no;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int n = slice; n < P.n; n += 4) {
        float cx[4], gv[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float xv = ldf<TS>(x + c * xcs + (long)n * P.ni);
            cx[c] = c ? -xv : xv;  // conjugate
            gv[c] = ldf<TS>(g + c * gcs + (long)n * P.no);
        }
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] += (qneg(p, q) ? -cx[p] : cx[p]) * gv[p ^ q];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) part[slice][q][lane] = acc[q];
    __syncthreads();
    // wave q finishes component q
    const float sum = (part[0][slice][lane] + part[1][slice][lane]) + (part[2][slice][lane] + part[3][slice][lane]);
    if (live) static_cast<TS*>(P.out)[slice * P.wcs + o * P.so + i * P.si] = (TS)sum;
}

template <typename TS, bool CONJB>
__global__ void __launch_bounds__(WG_THREADS) dense_small_row_kernel(const DenseRowArgs P) {
    __shared__ DenseSums part;
    dense_row_body<TS, CONJB>(P, blockIdx.x, part);
}

template <typename TS>
__global__ void __launch_bounds__(WG_THREADS) dense_small_wgrad_kernel(const DenseSmallArgs P) {
    __shared__ DenseSums part;
    dense_wgrad_body<TS>(P, blockIdx.x, part);
}

// Both gradients in one launch: they share the output gradient and nothing else, and a launch costs as much as either.
template <typename TS>
__global__ void __launch_bounds__(WG_THREADS) dense_small_bwd_kernel(const DenseRowArgs R, const DenseSmallArgs W, int row_blocks) {
    __shared__ DenseSums part;
    if ((int)blockIdx.x < row_blocks) dense_row_body<TS, true>(R, blockIdx.x, part);
    else dense_wgrad_body<TS>(W, blockIdx.x - row_blocks, part);
}

static long wgrad_blocks(const DenseSmallArgs& a) { return ((long)a.ni * a.no + DENSE_WGRAD - 1) / DENSE_WGRAD; }
static DenseRowArgs row_args(bool fwd, const DenseSmallArgs& a) {
    DenseRowArgs r{a.a, a.b, fwd ? a.bias : nullptr, a.out, a.wcs, fwd ? a.si : a.so, fwd ? a.so : a.si,
                   a.n, fwd ? a.no : a.ni, fwd ? a.ni : a.no, 0};
    r.kfast = r.b_ks == 1 && r.b_bs != 1;
    return r;
}
static long row_blocks(const DenseRowArgs& r) { return (long)r.na * ((r.nb + 15) / 16); }

int launch_dense_small_bwd(bool half_storage, const DenseSmallArgs& weights, const DenseSmallArgs& data, hipStream_t st) {
    const DenseRowArgs r = row_args(false, data);
    const long rows = row_blocks(r), blocks = rows + wgrad_blocks(weights);
    if (blocks == 0) return 0;
    if (blocks >= (1L << 31)) return -1;
    const dim3 grid((unsigned int)blocks), block(WG_THREADS);
    if (half_storage) hipLaunchKernelGGL(dense_small_bwd_kernel<_Float16>, grid, block, 0, st, r, weights, (int)rows);
    else hipLaunchKernelGGL(dense_small_bwd_kernel<float>, grid, block, 0, st, r, weights, (int)rows);
    return 0;
}

int launch_dense_small(bool half_storage, int pass, const DenseSmallArgs& a, hipStream_t st) {
    if (pass == PHX_PASS_BWD_WEIGHTS) {
        const long blocks = wgrad_blocks(a);
        if (blocks == 0) return 0;
        if (blocks >= (1L << 31)) return -1;
        const dim3 grid((unsigned int)blocks), block(WG_THREADS);
        if (half_storage) hipLaunchKernelGGL(dense_small_wgrad_kernel<_Float16>, grid, block, 0, st, a);
        else hipLaunchKernelGGL(dense_small_wgrad_kernel<float>, grid, block, 0, st, a);
        return 0;
    }
    const bool fwd = pass == PHX_PASS_FWD;
    const DenseRowArgs r = row_args(fwd, a);
    const long blocks = row_blocks(r);
    if (blocks == 0) return 0;
    if (blocks >= (1L << 31)) return -1;
    const dim3 grid((unsigned int)blocks), block(WG_THREADS);
    if (fwd) {
        if (half_storage) hipLaunchKernelGGL((dense_small_row_kernel<_Float16, false>), grid, block, 0, st, r);
        else hipLaunchKernelGGL((dense_small_row_kernel<float, false>), grid, block, 0, st, r);
    } else {
        if (half_storage) hipLaunchKernelGGL((dense_small_row_kernel<_Float16, true>), grid, block, 0, st, r);
        else hipLaunchKernelGGL((dense_small_row_kernel<float, true>), grid, block, 0, st, r);
    }
    return 0;
}

}  // namespace phx
