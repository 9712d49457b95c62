// Quaternion Dense as matrix products on the matrix cores, for any number of rows and units.
//   forward          y[q][n][o]  = sum_i sum_p s(p,q) x[p][n][i] w[p^q][i][o] (+ bias[q][o])      (src/dense.hpp:77-180)
//   input gradient   dx[q][n][i] = sum_o sum_p s(p,q) g[p][n][o] conj(w)[p^q][i][o]               (src/dense.hpp:252-377)
//   filter gradient  dw[q][i][o] = sum_n sum_p s(p,q) conj(x)[p][n][i] g[p^q][n][o]
// The other matrix-core path of Dense is a 1x1 convolution: channels-last for unit counts that are multiples of eight, else
// on n images of one position each, whose windows are gathered one 2-byte value at a time.
//
// A workgroup makes 64 * MT rows x 64 columns of all four components, a wave 32 * MT x 32: sixteen products per 16 reduced
// indices (the negative ones flip the sign bits of the row operand).  Both operands go through LDS as [component][pack of 8
// reduced indices][row] entries of 16 bytes, whichever index is contiguous in memory: a source that is contiguous along the
// reduction is copied, one that is contiguous along its rows is transposed in registers (4 rows x 8 indices a thread).  Ragged
// ends cost no branches per element: the last rows' loads move back inside the matrix, the last reduced indices are rotated
// into place and masked.  The next chunk's loads are in flight during the products; two or three workgroups per CU hide each
// other's barriers.  Problems of few tiles run in slices of the reduction whose fp32 sums a second kernel adds (fixed order).
//
// Measured (us a pass, the convolution kernels or FMA threads / here): fp16 1731 rows, 1056 -> 1689 units forward 672 / 147, input
// gradient 715 / 133, filter gradient 1773 / 143 (16 products of 3.1 G quaternion products: 690 TFLOP/s); 3707, 95 -> 408 86 / 22,
// 64 / 22, 107 / 27; 49, 530 -> 1552 64 / 16, 118 / 15, 46 / 11; fp32 201, 328 -> 264 152 / 20, 103 / 18, 31 / 18.  Bound: the
// latency of a chunk's loads (1.7 us) until two or three workgroups share a CU, then the matrix pipe and LDS alike; under
// 64 rows the launches.  Errors of fp32 below.
//
// fp32 operands are split into three bf16 parts on their way into LDS and multiplied as six products (see phx_kernels_x3.h for
// the arithmetic and for what becomes of values that have no three parts), in 16-product form whatever the mode asks for; the
// five small products have accumulators of their own.  The largest ones have 16 bits and lose nothing under an accumulator, so
// they do not drift as the sums of phx_kernels_x3.h do (1e-9 of the mean result).  Error against fp64, 2-norm, fp32 instructions /
// here: zero-mean values, 4096 rows, 1024 units 8.1e-7 / 4.0e-7; of one sign, forward 8.5e-7 / 3.5e-7.  Filter gradients of one
// sign, which the fp32 instructions sum in more slices, start a chunk's largest products from zero, with one rounding of the
// whole a chunk instead of four: 512 rows, 512 units 7.0e-8 / 7.7e-8 without, 4.9e-8 with; channels-last 96 -> 96 at 56x56, N=32
// 5.4e-8 / 6.2e-8, 4.2e-8 (and 3 % slower); on planes 475 -> 475 at 28x27, N=1 6.6e-8 / 7.6e-8, 3.9e-8 (2-8 % slower: 96 -> 96 at
// 56x56, N=32 260 -> 278 us).
#include <algorithm>

#include "phx_kernels_x3.h"
#include "phx_launch.h"

namespace phx {

template <typename T>
struct DenseTile {  // fp16
    static constexpr int KC = 32, KP = 4, PARTS = 1;  // reduced indices per chunk, packs of eight, parts of a value
};
template <>
struct DenseTile<float> {
    static constexpr int KC = 16, KP = 2, PARTS = 3;
};

typedef u32x2 u32x2_a4 __attribute__((aligned(4)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));

__host__ __device__ constexpr int dense_pitch(int rows) { return rows + 4; }  // entries of a pack's rows (the 4 packs x 4 rows a write covers fill all banks)

// One operand's tile of R rows: element (component, row, k) at base + component * cs + row * rs + k * ks, ks == 1 or (TURN)
// rs == 1.  load() requests a chunk, store() writes it to LDS.
template <typename T, bool TURN, int R>
struct DenseOperand {
    using S = DenseTile<T>;
    static constexpr bool F32 = sizeof(T) == 4;
    static constexpr int ROWS = TURN ? (F32 ? 2 : 4) : 1;                  // rows of a thread's task; a task is 8 reduced indices
    static constexpr int TASKS = 4 * S::KP * (R / ROWS) / WG_THREADS;      // per thread
    static constexpr int LOADS = TURN ? 8 : (F32 ? 2 : 1);                 // per task
    static constexpr int WORDS = TURN ? 2 : 4;                             // 32-bit words per load
    static constexpr int PITCH = dense_pitch(R);
    static constexpr int ENTRIES = S::PARTS * 4 * S::KP * PITCH;
    unsigned int v[TASKS][LOADS][WORDS];

    __device__ __forceinline__ static void task(int e, int& comp, int& kp, int& r) {
        int idx = threadIdx.x + e * WG_THREADS;
        if constexpr (TURN) {  // neighbouring threads along the rows, which are contiguous
            r = idx % (R / ROWS) * ROWS;
            idx /= R / ROWS;
            kp = idx % S::KP;
            comp = idx / S::KP;
        } else {               // ... along the packs of a row
            kp = idx % S::KP;
            idx /= S::KP;
            r = idx % R;
            comp = idx / R;
        }
    }

    __device__ __forceinline__ void load(const T* base, long cs, long rs, long ks, int row0, int rows, int k0, int K) {
#pragma unroll
        for (int e = 0; e < TASKS; ++e) {
            int comp, kp, r;
            task(e, comp, kp, r);
            const int k = k0 + kp * 8;
            const T* src = base + comp * cs;
            if constexpr (TURN) {
                const int row = min(row0 + r, rows - ROWS);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const u32x2 w = *reinterpret_cast<const std::conditional_t<F32, u32x2_a4, u32x2_a2>*>(src + (long)min(k + i, K - 1) * ks + row);
                    v[e][i][0] = w[0];
                    v[e][i][1] = w[1];
                }
            } else {
                src += (long)min(row0 + r, rows - 1) * rs;
                constexpr int N = 16 / sizeof(T);  // values per load
#pragma unroll
                for (int h = 0; h < LOADS; ++h) {
                    const u32x4 w = *reinterpret_cast<const std::conditional_t<F32, u32x4_a4, u32x4_a2>*>(src + min(k + h * N, K - N));
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[e][h][i] = w[i];
                }
            }
        }
    }

    // tail: the chunk reaches past the last reduced index
    __device__ __forceinline__ void store(u32x4* lds, int row0, int rows, int k0, int K, bool tail) {
#pragma unroll
        for (int e = 0; e < TASKS; ++e) {
            int comp, kp, r;
            task(e, comp, kp, r);
            const int left = K - (k0 + kp * 8);  // reduced indices of the task
            const int row = TURN ? min(row0 + r, rows - ROWS) - row0 : r;
#pragma unroll
            for (int j = 0; j < ROWS; ++j) {
                if (TURN && row + j < 0) continue;  // (a tile of fewer rows than the task)
                u32x4* dst = lds + (comp * S::KP + kp) * PITCH + row + j;
                if constexpr (!F32) {
                    u32x4 w;
                    if constexpr (TURN) {
#pragma unroll
                        for (int m = 0; m < 4; ++m)
                            w[m] = __builtin_amdgcn_perm(v[e][2 * m + 1][j >> 1], v[e][2 * m][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
                    } else {
                        w = u32x4{v[e][0][0], v[e][0][1], v[e][0][2], v[e][0][3]};
                        if (tail && left < 8) w = rotate_halves(w, left & 7);  // (loaded so as to end at the last index)
                    }
                    if (tail) w &= expand_half_mask(interval_bits(0, left));
                    *dst = w;
                } else {
                    float x[8];
                    if constexpr (TURN) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) x[i] = __builtin_bit_cast(float, v[e][i][j]);
                    } else {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            u32x4 w = {v[e][h][0], v[e][h][1], v[e][h][2], v[e][h][3]};
                            const int n = left - 4 * h;
                            if (tail && n < 4) {
                                if (n & 2) w = u32x4{w[2], w[3], w[0], w[1]};
                                if (n & 1) w = u32x4{w[3], w[0], w[1], w[2]};
                            }
#pragma unroll
                            for (int i = 0; i < 4; ++i) x[4 * h + i] = __builtin_bit_cast(float, (unsigned int)w[i]);
                        }
                    }
                    if (tail) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) x[i] = i < left ? x[i] : 0.f;
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] *= SPLIT_SCALE;
#pragma unroll
                    for (int part = 0; part < 3; ++part) {
                        u32x4 w;
#pragma unroll
                        for (int m = 0; m < 4; ++m) {
                            w[m] = pack_bf16(x[2 * m], x[2 * m + 1]);
                            if (part < 2) {
                                x[2 * m] -= bf16_low(w[m]);
                                x[2 * m + 1] -= bf16_high(w[m]);
                            }
                        }
                        dst[part * (4 * S::KP * PITCH)] = w;
                    }
                }
            }
        }
    }
};

// sign of row component p with column component p ^ q in output q
constexpr bool dense_negative(int pass, int p, int q) {
    return qneg(p, q) != (pass == PHX_PASS_BWD_DATA && (p ^ q) > 0) != (pass == PHX_PASS_BWD_WEIGHTS && p > 0);
}

struct GemmArgsPlanes : DenseGemmArgs {
    GemmPlanes planes;
};
template <bool PLANES>
using GemmArgsOf = std::conditional_t<PLANES, GemmArgsPlanes, DenseGemmArgs>;

// fp32: the four components of result (m, n), without the bias, over the chunks [first, end) in fp32 FMA (see split_bad in
// phx_kernels_x3.h)
template <int PASS, bool PLANES>
__device__ __forceinline__ void dense_fp32(const GemmArgsOf<PLANES>& P, int first, int end, int m, int n, float (&y)[4]) {
    constexpr int KC = DenseTile<float>::KC;
#pragma unroll
    for (int q = 0; q < 4; ++q) y[q] = 0.f;
    for (int c = first; c < end; ++c) {
        const float* a = static_cast<const float*>(P.a) + m * P.ars;
        const float* b = static_cast<const float*>(P.b) + n * P.brs;
        int k0 = c * KC;
        if constexpr (PLANES) {
            const int img = c / P.planes.chunks;
            a += img * P.planes.aimg;
            b += img * P.planes.bimg;
            k0 = (c - img * P.planes.chunks) * KC;
        }
#pragma unroll 4
        for (int k = k0; k < min(k0 + KC, P.K); ++k) {
            float x[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = a[i * P.acs + k * P.aks];
                w[i] = b[i * P.bcs + k * P.bks];
            }
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q) y[q] = fmaf(dense_negative(PASS, p, q) ? -x[p] : x[p], w[p ^ q], y[q]);
        }
        if (all_nan(y)) return;
    }
}

// ROWTURN, COLTURN: the operand is contiguous along its rows, not along the reduction.  PLANES: the filter gradient of a pointwise
// convolution on image planes: the reduction runs over the pixels of one image after the other, and results are contiguous along
// m, so the matrix instructions take their operands the other way round.
template <typename T, int PASS, bool ROWTURN, bool COLTURN, bool PLANES, int MT>
__global__ void __launch_bounds__(WG_THREADS, 2) dense_gemm_kernel(const GemmArgsOf<PLANES> P) {
    using S = DenseTile<T>;
    constexpr bool F32 = sizeof(T) == 4;
    static_assert(!PLANES || PASS == PHX_PASS_BWD_WEIGHTS, "planes: the filter gradient");
    using Rows = DenseOperand<T, ROWTURN, 64 * MT>;
    using Cols = DenseOperand<T, COLTURN, 64>;
    extern __shared__ u32x4 ldsd[];
    u32x4* const rl = ldsd;
    u32x4* const cl = ldsd + Rows::ENTRIES;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = lane & 31, kk = lane >> 5, wm = wave & 1, wn = wave >> 1;
    int bid = xcd_remap(blockIdx.x, gridDim.x);  // (the column tiles of one row tile read the same rows)
    const int n0 = bid % P.tiles_n * 64;
    bid /= P.tiles_n;
    const int m0 = bid % P.tiles_m * (64 * MT), z = bid / P.tiles_m;
    const T* a = static_cast<const T*>(P.a);
    const T* b = static_cast<const T*>(P.b);
    // the slice's chunks; planes: chunk c is one of image c / planes.chunks
    const int first = z * P.kper, end = min(P.chunks, first + P.kper);
    int load_img = 0, load_k = first * S::KC;
    if constexpr (PLANES) {
        load_img = first / P.planes.chunks;
        load_k = (first - load_img * P.planes.chunks) * S::KC;
    }

    Rows rows;
    Cols cols;
    auto load = [&] {  // the next chunk; the cursor moves on
        const T *la = a, *lb = b;
        if constexpr (PLANES) {
            la += load_img * P.planes.aimg;
            lb += load_img * P.planes.bimg;
        }
        rows.load(la, P.acs, P.ars, P.aks, m0, P.M, load_k, P.K);
        cols.load(lb, P.bcs, P.brs, P.bks, n0, P.N, load_k, P.K);
        load_k += S::KC;
        if (PLANES && load_k >= P.K) {
            load_k = 0;
            ++load_img;
        }
    };
    f32x16 acc[MT][4], low[F32 ? 4 : 1];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t][q][r] = 0.f;
            if constexpr (F32) low[q][r] = 0.f;
        }
    }
    const u32x4* const ra = rl + kk * Rows::PITCH + wm * 32 * MT + j;
    const u32x4* const ca = cl + kk * Cols::PITCH + wn * 32 + j;
    auto negated = [](const u32x4 v) { return v ^ u32x4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u}; };

    int k = load_k;  // of the chunk being stored and multiplied
    load();
    for (int c = first; c < end; ++c) {
        const bool tail = k + S::KC > P.K;
        if (c > first) __syncthreads();
        rows.store(rl, m0, P.M, k, P.K, tail);
        cols.store(cl, n0, P.N, k, P.K, tail);
        __syncthreads();
        k = load_k;
        if (c + 1 < end) load();
#pragma unroll
        for (int ks = 0; ks < S::KP / 2; ++ks) {
            if constexpr (!F32) {
                f16x8 w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] = __builtin_bit_cast(f16x8, ca[(i * S::KP + 2 * ks) * Cols::PITCH]);
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const u32x4 v = ra[(p * S::KP + 2 * ks) * Rows::PITCH + t * 32];
                        const f16x8 x = __builtin_bit_cast(f16x8, v), nx = __builtin_bit_cast(f16x8, negated(v));
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const f16x8 xs = dense_negative(PASS, p, q) ? nx : x;
                            acc[t][q] = PLANES ? __builtin_amdgcn_mfma_f32_32x32x16_f16(xs, w[p ^ q], acc[t][q], 0, 0, 0)
                                               : __builtin_amdgcn_mfma_f32_32x32x16_f16(w[p ^ q], xs, acc[t][q], 0, 0, 0);
                        }
                    }
            } else {
                bf16x8 w[3][4];
#pragma unroll
                for (int part = 0; part < 3; ++part)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        w[part][i] = __builtin_bit_cast(bf16x8, ca[((part * 4 + i) * S::KP + 2 * ks) * Cols::PITCH]);
                // (the filter gradient's largest products below)
                constexpr int TERMS = PASS == PHX_PASS_BWD_WEIGHTS ? 5 : 6;
                const auto product = [](const bf16x8& x, const bf16x8& y, const f32x16& sum) {
                    return PLANES ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, sum, 0, 0, 0) : __builtin_amdgcn_mfma_f32_32x32x16_bf16(y, x, sum, 0, 0, 0);
                };
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    bf16x8 x[3], nx[3];
#pragma unroll
                    for (int part = 0; part < 3; ++part) {
                        const u32x4 v = ra[((part * 4 + p) * S::KP + 2 * ks) * Rows::PITCH];
                        x[part] = __builtin_bit_cast(bf16x8, v);
                        nx[part] = __builtin_bit_cast(bf16x8, negated(v));
                    }
#pragma unroll
                    for (int term = 0; term < TERMS; ++term) {
                        constexpr int wp[6] = {2, 0, 1, 1, 0, 0}, xp[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            f32x16& sum = term < 5 ? low[q] : acc[0][q];
                            sum = product(dense_negative(PASS, p, q) ? nx[xp[term]] : x[xp[term]], w[wp[term]][p ^ q], sum);
                        }
                    }
                }
                if constexpr (TERMS == 5) {  // summed from zero: one rounding of the whole a chunk
                    __builtin_amdgcn_sched_barrier(0);  // (the other parts' registers come free)
                    u32x4 h[4];
#pragma unroll
                    for (int p = 0; p < 4; ++p) h[p] = ra[(p * S::KP + 2 * ks) * Rows::PITCH];
#pragma unroll
                    for (int q = 0; q < 4; q += 2) {
                        f32x16 sum[2];
#pragma unroll
                        for (int r = 0; r < 16; ++r) sum[0][r] = sum[1][r] = 0.f;
#pragma unroll
                        for (int p = 0; p < 4; ++p)
#pragma unroll
                            for (int i = 0; i < 2; ++i)
                                sum[i] = product(__builtin_bit_cast(bf16x8, dense_negative(PASS, p, q + i) ? negated(h[p]) : h[p]), w[0][p ^ (q + i)], sum[i]);
#pragma unroll
                        for (int i = 0; i < 2; ++i) acc[0][q + i] += sum[i];
                    }
                }
            }
        }
    }

    float bad = 0.f;
    // accumulator register 4 g + e: column 8 g + 4 kk + e of the wave's 32 at row j (PLANES: row 8 g + 4 kk + e at column j)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int lane_index = PLANES ? n0 + wn * 32 + j : m0 + (wm * MT + t) * 32 + j;
        if (lane_index >= (PLANES ? P.N : P.M)) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int run = (PLANES ? m0 + (wm * MT + t) * 32 : n0 + wn * 32) + 8 * g + 4 * kk, length = PLANES ? P.M : P.N;
                const int m = PLANES ? run : lane_index, n = PLANES ? lane_index : run;
                const bool whole = run + 3 < length;
                f32x4 y = {acc[t][q][4 * g], acc[t][q][4 * g + 1], acc[t][q][4 * g + 2], acc[t][q][4 * g + 3]};
                if constexpr (F32) {
                    y = (y + f32x4{low[q][4 * g], low[q][4 * g + 1], low[q][4 * g + 2], low[q][4 * g + 3]}) * SPLIT_RESULT;
#pragma unroll
                    for (int e = 0; e < 4; ++e) split_check(bad, y[e]);
                }
                if (P.partial) {  // [slice][component][m][n], PLANES [n][m]
                    float* dst = P.partial + (((long)z * 4 + q) * (PLANES ? P.N : P.M) + lane_index) * length + run;
                    if (whole) *reinterpret_cast<f32x4_a4*>(dst) = y;
                    else
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (run + e < length) dst[e] = y[e];
                    continue;
                }
                const long step = PLANES ? P.ors : P.ons;
                typedef T t4 __attribute__((ext_vector_type(4)));
                if constexpr (PASS == PHX_PASS_FWD) {
                    if (P.bias) {
                        const T* bias = static_cast<const T*>(P.bias) + q * P.N + n;
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[e] += n + e < P.N ? (float)bias[e] : 0.f;
                    }
                }
                t4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (T)y[e];
                T* dst = static_cast<T*>(P.out) + q * P.ocs + m * P.ors + n * P.ons;
                if (step == 1 && whole)
                    *reinterpret_cast<std::conditional_t<F32, u32x4_a4, u32x2_a2>*>(dst) = __builtin_bit_cast(std::conditional_t<F32, u32x4, u32x2>, o);
                else
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (run + e < length) dst[e * step] = o[e];
            }
    }
    if constexpr (F32) {
        if (bad != bad) {  // (rare) results that are not finite, once more
            const int lane_index = PLANES ? n0 + wn * 32 + j : m0 + wm * 32 + j, length = PLANES ? P.M : P.N;
#pragma unroll 1
            for (int i = 0; i < 16; ++i) {
                const int run = (PLANES ? m0 + wm * 32 : n0 + wn * 32) + 8 * (i >> 2) + 4 * kk + (i & 3);
                if (run >= length) break;
                const int m = PLANES ? run : lane_index, n = PLANES ? lane_index : run;
                float* const dst = P.partial ? P.partial + ((long)z * 4 * (PLANES ? P.N : P.M) + lane_index) * length + run
                                             : static_cast<float*>(P.out) + m * P.ors + n * P.ons;
                const long cs = P.partial ? (long)(PLANES ? P.N : P.M) * length : P.ocs;
                bool again = false;
#pragma unroll
                for (int q = 0; q < 4; ++q) again = again || split_bad(dst[q * cs]);
                if (!again) continue;
                float y[4];
                dense_fp32<PASS, PLANES>(P, first, end, m, n, y);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (PASS == PHX_PASS_FWD && !P.partial && P.bias) y[q] += static_cast<const float*>(P.bias)[q * P.N + n];
                    dst[q * cs] = y[q];
                }
            }
        }
    }
}

// out = the sum of the slices' partial results (+ bias), one rounding
template <typename T, bool PLANES>
__global__ void __launch_bounds__(WG_THREADS) dense_gemm_sum_kernel(const DenseGemmArgs P) {
    const long count = 4L * P.M * P.N, stride = (long)gridDim.x * blockDim.x;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += stride) {
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
        int z = 0;
        for (; z + 4 <= P.Z; z += 4)
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[i] += P.partial[(z + i) * count + e];
        for (; z < P.Z; ++z) sum[0] += P.partial[z * count + e];
        float y = (sum[0] + sum[1]) + (sum[2] + sum[3]);
        const int length = PLANES ? P.M : P.N, lines = PLANES ? P.N : P.M;
        const long row = e / length;
        const int run = (int)(e - row * length), q = (int)(row / lines), line = (int)(row - (long)q * lines);
        const int m = PLANES ? run : line, n = PLANES ? line : run;
        if (P.bias) y += (float)static_cast<const T*>(P.bias)[q * P.N + n];
        static_cast<T*>(P.out)[q * P.ocs + m * P.ors + n * P.ons] = (T)y;
    }
}

// Tiles and reduction slices, by an estimate of the time: a workgroup's chunks of reduced indices, its start and stores, and
// for more than one slice the partial results' way to memory and back in a second kernel.  A chunk of a lone workgroup takes
// the latency of its loads, those of two or three on one CU overlap.  Times from M, N, K = 64 ... 4096 (us a chunk, one to three
// workgroups on a CU: fp16 64 rows 1.7 / 2.8 / 3.9, 128 rows 3.9 / 4.8; fp32 3.4 / 5.7).
void dense_gemm_plan(bool half_storage, DenseGemmArgs& a, GemmPlanes* planes) {
    const int KC = half_storage ? DenseTile<_Float16>::KC : DenseTile<float>::KC;
    a.chunks = (a.K + KC - 1) / KC;
    if (planes) {
        planes->chunks = a.chunks;
        a.chunks *= planes->images;
    }
    a.tiles_n = (a.N + 63) / 64;
    double best = 1e30;
    for (int mt = 1; mt <= (half_storage ? 2 : 1); ++mt) {
        const int tiles_m = (a.M + 64 * mt - 1) / (64 * mt), most = half_storage && mt == 1 ? 3 : 2;
        const double first = !half_storage ? 3.4 : mt == 2 ? 3.9 : 1.7, more = !half_storage ? 2.3 : mt == 2 ? 0.9 : 1.1;
        const int limit = std::min(a.chunks, planes ? 512 : 64);
        for (int Z = 1, per = a.chunks; Z <= limit; Z = (a.chunks + per - 2) / (per - 1)) {  // (the slice counts that leave no slice empty)
            per = (a.chunks + Z - 1) / Z;
            const long load = ((long)tiles_m * a.tiles_n * Z + 255) / 256, full = load / most, rest = load % most;
            double us = 4.0 + per * (full * (first + (most - 1) * more) + (rest > 0 ? first + (rest - 1) * more : 0.0));
            if (Z > 1) us += 4.0 + (Z + 0.5) * 32.0 * a.M * a.N / 3.0e6;
            if (us < best) {
                best = us;
                a.MT = mt; a.tiles_m = tiles_m; a.Z = Z; a.kper = per;
            }
            if (per == 1) break;
        }
    }
}

template <typename T, int PASS, bool ROWTURN, bool COLTURN, bool PLANES, int MT>
static int launch_one(const GemmArgsOf<PLANES>& a, hipStream_t st) {
    constexpr size_t lds = (size_t)(DenseOperand<T, ROWTURN, 64 * MT>::ENTRIES + DenseOperand<T, COLTURN, 64>::ENTRIES) * 16;
    static_assert(lds <= 64 * 1024, "no opt-in for dynamic LDS");
    hipLaunchKernelGGL((dense_gemm_kernel<T, PASS, ROWTURN, COLTURN, PLANES, MT>), dim3((unsigned)((long)a.tiles_m * a.tiles_n * a.Z)),
                       dim3(WG_THREADS), lds, st, a);
    return 0;
}

template <typename T, bool PLANES>
static int launch_sum(const DenseGemmArgs& a, hipStream_t st) {
    if (a.Z == 1) return 0;
    const long count = 4L * a.M * a.N;
    const dim3 grid((unsigned)std::min<long>((count + WG_THREADS - 1) / WG_THREADS, 1 << 14));
    hipLaunchKernelGGL((dense_gemm_sum_kernel<T, PLANES>), grid, dim3(WG_THREADS), 0, st, a);
    return 0;
}

template <typename T, int MT>
static int launch_pass(int pass, const DenseGemmArgs& a, hipStream_t st) {
    const bool turn = a.bks != 1;
    if (pass == PHX_PASS_FWD)
        return turn ? launch_one<T, PHX_PASS_FWD, false, true, false, MT>(a, st) : launch_one<T, PHX_PASS_FWD, false, false, false, MT>(a, st);
    if (pass == PHX_PASS_BWD_DATA)
        return turn ? launch_one<T, PHX_PASS_BWD_DATA, false, true, false, MT>(a, st) : launch_one<T, PHX_PASS_BWD_DATA, false, false, false, MT>(a, st);
    return launch_one<T, PHX_PASS_BWD_WEIGHTS, true, true, false, MT>(a, st);
}

int launch_dense_gemm(bool half_storage, int pass, const DenseGemmArgs& a, hipStream_t st) {
    // (a load's 16 bytes lie inside a row of units, a task's rows inside the units that are contiguous)
    if (a.M < 1 || a.K < 1 || a.N < 8 || (pass == PHX_PASS_BWD_WEIGHTS ? a.M : a.K) < 8 || (a.Z > 1) != (a.partial != nullptr)) return -1;
    const int rc = !half_storage ? launch_pass<float, 1>(pass, a, st) : a.MT == 2 ? launch_pass<_Float16, 2>(pass, a, st) : launch_pass<_Float16, 1>(pass, a, st);
    if (rc != 0) return rc;
    return half_storage ? launch_sum<_Float16, false>(a, st) : launch_sum<float, false>(a, st);
}

int launch_planes_gemm(const DenseGemmArgs& plain, const GemmPlanes& planes, hipStream_t st) {
    const GemmArgsPlanes a{plain, planes};
    if (a.M < 1 || a.K < 4 || a.N < 1 || a.MT != 1 || (a.Z > 1) != (a.partial != nullptr)) return -1;  // (loads of four pixels inside a plane)
    if (const int rc = launch_one<float, PHX_PASS_BWD_WEIGHTS, false, false, true, 1>(a, st)) return rc;
    return launch_sum<float, true>(a, st);
}

}  // namespace phx
