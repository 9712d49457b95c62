// Factorized (8-product) fp32 filter gradient on bf16 matrix instructions: every operand as the sum of three bf16 values.
#pragma once

#include "phx_kernels_x3.h"

namespace phx {

// The products of phx_kernels_x3.h (six of the nine of two three-part sums, 32x32x16 instructions), contracted over output
// pixels: rows = output channels (gradient), columns = input channels (input under a tap).
//   grid.x = 64 output x 32 input channels, a filter row kh and up to three neighbouring kw, a slice of the reduction; partial
//   sums as qconv_wgrad_f32_kernel's, added by reduce_wgrad_kernel.  Wave i owns product lane i of the whole tile.
//   A K step is two segments of 8 pixels of an output row (lists as in the fp16 kernel: ceil(wo / 8) to a row), the K halves
//   of an instruction.  The gradient of a segment is 8 values a channel and the input 10, those of all three taps: a tap's
//   operand is the segment's 16 bytes and the two values behind them, shifted in registers, so that the input is taken apart
//   once for three taps.
// A thread makes the eight lanes and their three parts of one component quadruple of four pixels (waves 0-3: gradient, 4-6:
// input), some 260 instructions, from values loaded a step ahead, into the other half of a double buffer.  The two waves of a
// SIMD take turns: one starts a step with its staging (the gradient's), the other with its products, so that one's products run
// beside the other's arithmetic.
//
// Rounding: the instructions' sums drop their lowest bits downwards, the same way whatever the sign, which over thousands of
// steps adds up.  Every K step's six products therefore start from zero and are added to the accumulator by an ordinary
// addition, and every other reduction slice runs on the negated gradient.  Errors against fp64 (relative 2-norm, standard normal
// values, here / fp32 instructions): 3x3, 128 x 48 channels at 9x9 1.8e-7 / 3.4e-7, 16 x 512 at 7x7 2.4e-7 / 4.7e-7, 4 x 256 at
// 14x14 1.6e-7 / 2.9e-7; without the negation 6.3e-7, 2.4e-7, 2.0e-7; accumulated by the instructions 1.5-2 times as much again.
// A pass of one slice has no other to make up for it, and needs none: 512 x 512 at 14x14, N=32 6.2e-7 / 1.36e-6, half of it drift
// (which grows with the root of the steps, as the roundings do, since each step's sum starts from zero).
//
// Bound: the two pipes of a SIMD together.  64 channels at 56x56, N=64 (1399 us on fp32 instructions, 770 here): a step of
// 2.5 us holds 72 products of 32 clocks and 700 vector instructions of 4, which overlap in part: 610 us without the staging,
// 450 without the products.  (Tried, against 800 with the gradient's products first: the additions dealt between the products 850,
// subtracting parts by dot2 instructions 868, neighbouring waves in turn 858.)
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));

constexpr int WGX3_TPW = 3;                              // taps of a filter row
constexpr int WGX3_CO = 64, WGX3_CI = 32;                // channel tile
constexpr int WGX3_THREADS = 512;
constexpr int WGX3_G = 8 * 3 * 2 * WGX3_CO * 16;         // bytes: [lane][part][segment][co] x 8 pixels
constexpr int WGX3_XSEG = WGX3_CI * 16 + WGX3_CI * 4;    // a segment: [ci] x 8 pixels, [ci] x the 2 behind them
constexpr int WGX3_X = 8 * 3 * 2 * WGX3_XSEG;
constexpr int WGX3_BUF = WGX3_G + WGX3_X;
constexpr int WGX3_LDS_BYTES = 2 * WGX3_BUF;
constexpr int WGX3_PITCH = WGX3_CI + 1;                  // epilogue: [lane][co][ci]
static_assert(8 * WGX3_CO * WGX3_PITCH * 4 <= WGX3_LDS_BYTES && WGX3_LDS_BYTES <= 160 * 1024, "LDS of the split filter gradient");

// tap (kh, kw) of channels (co, ci), over the segments of reduction slice zi, in fp32
__device__ __forceinline__ void wgrad_fp32(const WgradArgs& P, int zi, int kh, int kw, int co, int ci, float (&y)[4]) {
    const long xplane = (long)P.x.Hd * P.x.Wd, gplane = (long)P.g.Hd * P.g.Wd;
    const int rows = P.g.Hd;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = 0.f;
    for (int tile = zi; tile < P.ntiles; tile += P.zsplit)
        for (int seg = 2 * tile; seg < 2 * tile + 2; ++seg) {
            const int line = seg / P.cpr, img = line / rows, ho = line - img * rows, h = ho * P.sh + kh * P.dh - P.pt;
            if (img >= P.g.N || h < 0 || h >= P.x.Hd) continue;
            const float* const x = static_cast<const float*>(P.x.base) + ((long)img * P.x.Cs + ci) * xplane + (long)h * P.x.Wd;
            const float* const g = static_cast<const float*>(P.g.base) + ((long)img * P.g.Cs + co) * gplane + (long)ho * P.g.Wd;
            const int c0 = (seg - line * P.cpr) * 8;
            const int shift = kw - P.pl, end = min(min(c0 + 8, P.g.Wd), P.x.Wd - shift);  // (columns whose input lies in the image)
#pragma unroll 4
            for (int c = max(c0, -shift); c < end; ++c) {
                float xv[4], gv[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    xv[i] = x[i * P.x.comp_stride + c + shift];
                    gv[i] = g[i * P.g.comp_stride + c];
                }
#pragma unroll
                for (int p = 0; p < 4; ++p)
#pragma unroll
                    for (int r = 0; r < 4; ++r) y[r] = fmaf(qneg(p, p ^ r) ? -xv[p] : xv[p], gv[p ^ r], y[r]);
            }
            if (all_nan(y)) return;
        }
}

__global__ void __launch_bounds__(WGX3_THREADS, 1) qconv_wgrad_x3_kernel(const WgradArgs P0) {
    const WgradArgs P = group_view(P0);
    extern __shared__ u32x4 ldswgx3[];
    char* const lds = reinterpret_cast<char*>(ldswgx3);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kk = lane >> 5;
    // workgroups that share a reduction slice read the same tensors: keep them on one XCD
    int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int cot = bid % P.co_tiles;  bid /= P.co_tiles;
    const int cit = bid % P.ci_tiles;  bid /= P.ci_tiles;
    const int ngroups = P.groups_per_row * P.Kh;
    const int grp = bid % ngroups;
    const int zi = bid / ngroups;
    const int kh = grp / P.groups_per_row;
    const int kw0 = (grp % P.groups_per_row) * WGX3_TPW;
    const int nkw = (P.Kw - kw0 < WGX3_TPW) ? P.Kw - kw0 : WGX3_TPW;

    // The thread's task: four pixels of a channel, all components.  A wave's tasks are of one kind; neighbouring threads take
    // the pixels of the two segments, which mostly lie side by side.
    const bool grad = wave < 4, tail = wave == 6, idle = wave == 7;
    const int seg = tail ? tid & 1 : (tid >> 1) & 1;
    const int half = tail ? 2 : tid & 1;                                  // 4-pixel group of the segment (2: the input's last two)
    const int ch = grad ? tid >> 2 : tail ? lane >> 1 : (tid - 256) >> 2;  // channel of the tile
    const int chan = (grad ? cot * WGX3_CO : cit * WGX3_CI) + ch;
    const int Hd = grad ? P.g.Hd : P.x.Hd, Wd = grad ? P.g.Wd : P.x.Wd;
    const int C = grad ? P.g.C : P.x.C, Cs = grad ? P.g.Cs : P.x.Cs, N = P.g.N;
    const long plane = (long)Hd * Wd, cs = grad ? P.g.comp_stride : P.x.comp_stride;
    const unsigned int* const base = static_cast<const unsigned int*>(grad ? P.g.base : P.x.base);
    const long total = 3 * cs + ((long)(N - 1) * Cs + C) * plane;
    const int row_step = grad ? 1 : P.sh, row0 = grad ? 0 : kh * P.dh - P.pt;
    const int col0 = (grad ? 0 : kw0 - P.pl) + half * 4;
    // where it writes: lane 0, part 0 of the first buffer
    const unsigned int wr = grad ? ((seg * WGX3_CO + (ch ^ (seg * 8))) * 16 + half * 8)
                                 : WGX3_G + seg * WGX3_XSEG + (tail ? WGX3_CI * 16 + ch * 4 : ch * 16 + half * 8);

    // segments 2 * tile + seg of the list, as (image, output row, 8-pixel chunk): stepped with carries
    const int first = 2 * zi + seg, step = 2 * P.zsplit, rows = P.g.Hd;
    int cc = first % P.cpr, ho = (first / P.cpr) % rows, img = first / (P.cpr * rows);
    const int step_c = step % P.cpr, step_h = (step / P.cpr) % rows, step_n = step / (P.cpr * rows);

    const unsigned int sign = (unsigned int)zi << 31;  // odd slices: on the negated gradient
    u32x4 v[4] = {};        // (finite where nothing is loaded: multiplied by zero)
    unsigned int keep = 0;  // pixels of the task inside the image
    auto issue = [&]() {    // requests the values of the current tile; steps to the workgroup's next one
        const int r = ho * row_step + row0, c = cc * 8 + col0;
        keep = 0;
        if (img < N && chan < C && r >= 0 && r < Hd && !idle) keep = interval_bits<4>(-c, Wd - c);
        if (tail) keep &= 3;
        const long off = ((long)img * Cs + chan) * plane + (long)r * Wd + c;
        if (keep) {
            if (off >= 0 && off + 3 * cs + 4 <= total) {
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const u32x4_a4*>(base + off + q * cs);
            } else {  // a tensor's first and last values, one by one (those outside the image: any that the tensor has)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[q][k] = base[((keep >> k) & 1) ? off + q * cs + k : 0];
            }
        }
        cc += step_c;
        if (cc >= P.cpr) { cc -= P.cpr; ++ho; }
        ho += step_h;
        if (ho >= rows) { ho -= rows; ++img; }
        img += step_n;
    };
    // the eight lanes of the task's values in three parts each (ROLE 0: gradient, 1: input, 2: input, the segment's last two)
    auto convert_as = [&](auto role, int buf) {
        constexpr int ROLE = decltype(role)::value, PX = ROLE == 2 ? 2 : 4;
        constexpr int PART = ROLE == 0 ? 2 * WGX3_CO * 16 : 2 * WGX3_XSEG;
        char* const dst = lds + buf * WGX3_BUF + wr;
        float lanes[PX][8];
#pragma unroll
        for (int k = 0; k < PX; ++k) {
            const float m = ((keep >> k) & 1) ? (ROLE == 0 && sign ? -SPLIT_SCALE : SPLIT_SCALE) : 0.f;
            float e[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) e[q] = __builtin_bit_cast(float, (unsigned int)v[q][k]) * m;
            if constexpr (ROLE == 0) lanes_grad(e, lanes[k], 0.5f);
            else lanes_left(e, lanes[k]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float a[PX];
#pragma unroll
            for (int k = 0; k < PX; ++k) a[k] = lanes[k][i];
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                unsigned int two[PX / 2];
#pragma unroll
                for (int k = 0; k < PX / 2; ++k) {
                    two[k] = pack_bf16(a[2 * k], a[2 * k + 1]);
                    a[2 * k] -= bf16_low(two[k]);
                    a[2 * k + 1] -= bf16_high(two[k]);
                }
                if constexpr (ROLE == 2) *reinterpret_cast<unsigned int*>(dst + (i * 3 + t) * PART) = two[0];
                else *reinterpret_cast<u32x2*>(dst + (i * 3 + t) * PART) = u32x2{two[0], two[1]};
            }
        }
    };
    auto convert = [&](int buf) {
        if (grad) convert_as(std::integral_constant<int, 0>{}, buf);
        else if (wave < 6) convert_as(std::integral_constant<int, 1>{}, buf);
        else if (tail) convert_as(std::integral_constant<int, 2>{}, buf);
    };

    f32x16 acc[2][WGX3_TPW];  // [32 output channels][tap]; rows = output channels, columns = input channels
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < WGX3_TPW; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[s][t][r] = 0.f;

    // the wave's products of a staged K step
    auto products = [&](int buf) {
        const char* const gs = lds + buf * WGX3_BUF + wave * (3 * 2 * WGX3_CO * 16) + (kk * WGX3_CO + (j ^ (kk * 8))) * 16;
        const char* const xs = lds + buf * WGX3_BUF + WGX3_G + (wave * 6 + kk) * WGX3_XSEG;
        // (read in the order of use)
        bf16x8 A[3][2], B[3][WGX3_TPW];
        u32x4 w[3];
        unsigned int w4[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int s = 0; s < 2; ++s) A[2 - p][s] = *reinterpret_cast<const bf16x8*>(gs + (2 - p) * (2 * WGX3_CO * 16) + s * 512);
            w[p] = *reinterpret_cast<const u32x4*>(xs + p * 2 * WGX3_XSEG + j * 16);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) w4[p] = *reinterpret_cast<const unsigned int*>(xs + p * 2 * WGX3_XSEG + WGX3_CI * 16 + j * 4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            B[p][0] = __builtin_bit_cast(bf16x8, w[p]);
            B[p][1] = __builtin_bit_cast(bf16x8, u32x4{__builtin_amdgcn_alignbit(w[p][1], w[p][0], 16), __builtin_amdgcn_alignbit(w[p][2], w[p][1], 16),
                                                       __builtin_amdgcn_alignbit(w[p][3], w[p][2], 16), __builtin_amdgcn_alignbit(w4[p], w[p][3], 16)});
            B[p][2] = __builtin_bit_cast(bf16x8, u32x4{w[p][1], w[p][2], w[p][3], w4[p]});
        }
        constexpr int GP[6] = {2, 1, 1, 0, 0, 0}, XP[6] = {0, 1, 0, 2, 1, 0};  // parts: the largest product last
#pragma unroll
        for (int t = 0; t < WGX3_TPW; ++t) {
            if (t < nkw) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    f32x16 sum;
#pragma unroll
                    for (int r = 0; r < 16; ++r) sum[r] = 0.f;
#pragma unroll
                    for (int i = 0; i < 6; ++i)
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[GP[i]][s], B[XP[i]][t], sum, 0, 0, 0);
                    acc[s][t] += sum;
                }
            }
        }
    };

    if (zi < P.ntiles) {
        issue();
        convert(0);
        if (zi + P.zsplit < P.ntiles) issue();
        wg_barrier_no_vmem_wait();
        int buf = 0;
        for (int tile = zi; tile < P.ntiles; tile += P.zsplit, buf ^= 1) {
            const auto turn = [&] {  // (ahead of the other wave's arithmetic)
                __builtin_amdgcn_s_setprio(2);
                products(buf);
                __builtin_amdgcn_s_setprio(0);
            };
            const bool more = tile + P.zsplit < P.ntiles, more2 = more && tile + 2 * P.zsplit < P.ntiles;
            if (wave >= 4) turn();
            if (more) convert(buf ^ 1);
            if (more2) issue();
            if (wave < 4) turn();
            wg_barrier_no_vmem_wait();
        }
    }

    // partial[z][tap][r][co][ci]: the waves' lanes meet in LDS, tap by tap
    const long tap_stride = 4L * P.CoP * P.CiP, comp = (long)P.CoP * P.CiP;
    float* const dst = P.partial + ((long)zi * P.Kh * P.Kw + kh * P.Kw + kw0) * tap_stride;
    float* const xch = reinterpret_cast<float*>(lds);
    float bad = 0.f;
#pragma unroll
    for (int t = 0; t < WGX3_TPW; ++t) {
        if (t >= nkw) continue;
        if (t > 0) wg_barrier_no_vmem_wait();  // the previous tap has been read
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                xch[(wave * WGX3_CO + s * 32 + 4 * kk + 8 * (e >> 2) + (e & 3)) * WGX3_PITCH + j] = acc[s][t][e];
        wg_barrier_no_vmem_wait();
#pragma unroll
        for (int k = 0; k < WGX3_CO * WGX3_CI / WGX3_THREADS; ++k) {
            const int co = (tid >> 5) + k * (WGX3_THREADS / 32);
            float l[8], y[4];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                l[i] = __builtin_bit_cast(float, __builtin_bit_cast(unsigned int, xch[(i * WGX3_CO + co) * WGX3_PITCH + j]) ^ sign);
            merge_right_grad(l, y);
            float* const d = dst + t * tap_stride + (long)(cot * WGX3_CO + co) * P.CiP + cit * WGX3_CI + j;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                y[r] *= SPLIT_RESULT;
                split_check(bad, y[r]);
                d[r * comp] = y[r];
            }
        }
    }
    if (bad != bad) {  // (rare; see phx_kernels_x3.h) sums that are not finite, once more in fp32
        constexpr int ROUNDS = WGX3_CO * WGX3_CI / WGX3_THREADS;
#pragma unroll 1
        for (int i = 0; i < ROUNDS * nkw; ++i) {
            const int t = i / ROUNDS, row = cot * WGX3_CO + (tid >> 5) + (i - t * ROUNDS) * (WGX3_THREADS / 32), column = cit * WGX3_CI + j;
            if (row >= P.g.C || column >= P.x.C) continue;
            float* const d = dst + t * tap_stride + (long)row * P.CiP + column;
            bool again = false;
#pragma unroll
            for (int r = 0; r < 4; ++r) again = again || split_bad(d[r * comp]);
            if (!again) continue;
            float y[4];
            wgrad_fp32(P, zi, kh, kw0 + t, row, column, y);
#pragma unroll
            for (int r = 0; r < 4; ++r) d[r * comp] = y[r];
        }
    }
}

}  // namespace phx
