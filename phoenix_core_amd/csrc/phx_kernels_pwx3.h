// Factorized (8-product) fp32 pointwise kernel on bf16 matrix instructions: every operand as the sum of three bf16 values.
#pragma once

#include "phx_kernels_x3.h"

namespace phx {

// The products of phx_kernels_x3.h (six of the nine of two three-part sums, 32x32x16 instructions) for one tap at unit stride.
//   Tile: S * 32 output channels (rows) x 64 pixels (columns); wave v owns the two product lanes made from one pair of
//   components, as in qconv_fwd_x3_kernel, so every lane of every input value is formed and taken apart once for the tile.
//   A K step is 16 input channels.  A thread loads what its own operands need and no other thread reads: two neighbouring
//   pixels (the two column tiles) of 8 channels (its K half) of the wave's two components, 8 bytes a load, and keeps everything
//   in registers: the loop has no LDS and no barrier, and two workgroups share a CU.  Filters stream through L2.
//   A lane's filters are requested as the taking apart of its activations begins, a step's activations a lane's products ahead.
//   Pixels come in pairs of an image's plane; the last pair of an odd plane repeats the pixel before it (and stores the same
//   value to it).
// Measured (us a pass with its packing, fp32 instructions / here): N=32, 64 -> 64 channels at 56x56 107 / 72, N=16, 256 -> 64 at
// 28x28 71 / 37, 64 -> 256 57 / 40, 256 -> 256 at 14x14 73 / 41, N=64, 128 -> 128 at 28x28 171 / 102, 16 -> 16 at 56x56 45 / 34,
// N=8, 512 -> 512 at 7x7 80 / 36, N=2, 20 -> 33 at 5x7 18 / 14; the scaling of the values 1-2 % more since.  (With both lanes' filters held a step ahead, 17 registers
// spilled: 85 at 64 -> 64.)  Errors against fp64, relative 2-norm: 256 channels 3.4e-7 (fp32 instructions 4.1e-7), 512 in slices
// 2.5e-7 (4.1e-7), 64 1.7e-7 (2.2e-7).
// Bound: memory where channels are few (64 -> 64: 206 MB in 65 us), else the two pipes of a SIMD: a K step is 48 products of 32
// clocks and 230 vector instructions of 4 a wave.
constexpr int PWX3_STEP = 16;
constexpr int PWX3_PX = 64;
constexpr int PWX3_STRETCH = SPLIT_STRETCH / PWX3_STEP;  // K steps between two changes of sign
constexpr int PWX3_LDS_BYTES = 8 * 32 * PWX3_PX * 4;  // the epilogue's exchange of the product lanes
constexpr int pwx3_vectors(int S) { return 2 * 3 * S * 64; }  // 16-byte vectors of a wave's filters per K step: [lane][part][sub-tile][64]

__host__ __device__ inline size_t pwx3_packed_bytes(int S, int co_tiles, int nsteps) { return (size_t)co_tiles * 4 * nsteps * pwx3_vectors(S) * 16; }

typedef u32x2 u32x2_a4 __attribute__((aligned(4)));

template <int S>
__global__ void __launch_bounds__(WG_THREADS, 2) qconv_pw_x3_kernel(const ConvArgs P0) {
    const ConvArgs P = slice_view(P0, PWX3_STEP);
    extern __shared__ float ldspwx3[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kk = lane >> 5;
    int bid = xcd_remap(blockIdx.x, gridDim.x);  // (the channel tiles of one pixel tile share an XCD)
    const int ct = bid % P.co_tiles, pt = bid / P.co_tiles;
    const int plane = P.in.Hd * P.in.Wd, pairs = (plane + 1) >> 1, npairs = P.in.N * pairs;
    // first pixel of pair q of the tile, and its image (pairs behind the last one repeat it)
    auto pair = [&](int q, int& img) {
        const int i = min(pt * (PWX3_PX / 2) + q, npairs - 1);
        img = i / pairs;
        return min(2 * (i - img * pairs), plane - 2);
    };

    // activations: 32-bit byte offsets (the host keeps larger tensors off this kernel)
    const int ca = (0x78 >> (2 * wave)) & 3, cb = (0x78 >> (2 * ((wave + 1) & 3))) & 3;
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(P.in.base), 0, -1, 0x00020000);
    const unsigned int chan = (unsigned int)plane * 4, abase = (unsigned int)(ca * P.in.comp_stride * 4), bbase = (unsigned int)(cb * P.in.comp_stride * 4);
    unsigned int xoff;
    {
        int img;
        const int p = pair(j, img);
        xoff = ((unsigned int)img * P.in.Cs * plane + p) * 4;
    }
    u32x2 xa[8], xb[8];
    auto load_x = [&](int step) {
        const int c0 = step * PWX3_STEP;
        if (c0 + PWX3_STEP <= P.in.C) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const unsigned int o = xoff + kk * (8 * chan), s = (unsigned int)(c0 + i) * chan;
                xa[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xbuf, o, abase + s, 0));
                xb[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xbuf, o, bbase + s, 0));
            }
        } else {  // (channels past the tensor meet zero filters, any value of this pixel will do)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const unsigned int o = xoff + min(c0 + kk * 8 + i, P.in.C - 1) * chan;
                xa[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xbuf, o, abase, 0));
                xb[i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xbuf, o, bbase, 0));
            }
        }
    };
    // filters: this wave's stream of operands
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<u32x4*>(static_cast<const u32x4*>(P.wpk) + (long)(ct * 4 + wave) * P.nchunks * pwx3_vectors(S)), 0, -1, 0x00020000);
    bf16x8 A[3][S];  // of one lane: [part][sub-tile]
    auto load_a = [&](int step, int l) {
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
            for (int s = 0; s < S; ++s)
                A[t][s] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                    wbuf, lane * 16, (unsigned int)step * (pwx3_vectors(S) * 16) + ((l * 3 + t) * S + s) * 1024, 0));
    };

    f32x16 acc[2][S][2];  // [lane][sub-tile][pixel of the pair]
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[l][s][t][r] = 0.f;

    load_x(0);
    constexpr int FP[6] = {2, 0, 1, 1, 0, 0}, XP[6] = {0, 2, 1, 0, 1, 0};  // parts of filter and input: the largest product last
    float result = SPLIT_RESULT;
    for (int step = 0; step < P.nchunks; ++step) {
        if (step > 0 && step % PWX3_STRETCH == 0) {  // (see Drift in phx_kernels_x3.h)
            result = -result;
#pragma unroll
            for (int l = 0; l < 2; ++l)
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t) acc[l][s][t] = -acc[l][s][t];
        }
        const bool more = step + 1 < P.nchunks;
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            load_a(step, l);  // (on their way while the activations are taken apart)
            bf16x8 B[3][2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                unsigned int part[3][4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const unsigned int ua = xa[2 * q + i][t], ub = xb[2 * q + i][t];
                        const float a = __builtin_bit_cast(float, ua), b = __builtin_bit_cast(float, ub);
                        v[i] = fmaf(a, SPLIT_SCALE, l ? -SPLIT_SCALE * b : SPLIT_SCALE * b);
                    }
#pragma unroll
                    for (int u = 0; u < 3; ++u) {
                        part[u][q] = pack_bf16(v[0], v[1]);
                        v[0] -= bf16_low(part[u][q]);
                        v[1] -= bf16_high(part[u][q]);
                    }
                }
#pragma unroll
                for (int u = 0; u < 3; ++u) B[u][t] = __builtin_bit_cast(bf16x8, u32x4{part[u][0], part[u][1], part[u][2], part[u][3]});
            }
            if (l == 1 && more) load_x(step + 1);
            __builtin_amdgcn_sched_barrier(0);  // (another wave's products run beside the taking apart)
#pragma unroll
            for (int i = 0; i < 6; ++i)
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[l][s][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[FP[i]][s], B[XP[i]][t], acc[l][s][t], 0, 0, 0);
        }
    }

    // Epilogue, one round per filter sub-tile: the waves' product lanes meet in LDS, [product lane][32 channels][64 pixels], and
    // are read back four pixels (two pairs) of a channel at a time, merged and stored.
    float* const out = static_cast<float*>(P.out);
    const float* const bias = static_cast<const float*>(P.bias);
    const int g = tid & 15, row0 = tid >> 4;
    int img[2], p[2];
    bool ok[2];
    long o[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        ok[h] = pt * (PWX3_PX / 2) + 2 * g + h < npairs;
        p[h] = pair(2 * g + h, img[h]);
        o[h] = (long)img[h] * P.CoutS * plane + p[h];
    }
    const bool joined = ok[1] && o[1] == o[0] + 2;
    float bad = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (s > 0) wg_barrier_no_vmem_wait();  // the previous round has been read
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            float* const dst = ldspwx3 + lanes_product(wave, l) * (32 * PWX3_PX) + 4 * kk * PWX3_PX + 2 * j;
#pragma unroll
            for (int e = 0; e < 16; ++e)
                *reinterpret_cast<f32x2*>(dst + (8 * (e >> 2) + (e & 3)) * PWX3_PX) = f32x2{acc[l][s][0][e], acc[l][s][1][e]};
        }
        wg_barrier_no_vmem_wait();
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int row = row0 + 16 * r, co = (ct * S + s) * 32 + row;
            f32x4 in[8], y[4];
#pragma unroll
            for (int i = 0; i < 8; ++i) in[i] = *reinterpret_cast<const f32x4*>(ldspwx3 + (i * 32 + row) * PWX3_PX + 4 * g);
            if (co >= P.Cout || !ok[0]) continue;
            merge_output(in, y);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                y[q] *= result;
#pragma unroll
                for (int k = 0; k < 4; ++k) split_check(bad, y[q][k]);
                if (bias) y[q] += bias[q * P.CoutS + co];
                float* const d = out + q * P.out_cs + (long)co * plane;
                if (joined) {
                    *reinterpret_cast<f32x4_a4*>(d + o[0]) = y[q];
                } else {
                    const f32x2 lo = {y[q][0], y[q][1]}, hi = {y[q][2], y[q][3]};
                    *reinterpret_cast<u32x2_a4*>(d + o[0]) = __builtin_bit_cast(u32x2, lo);
                    if (ok[1]) *reinterpret_cast<u32x2_a4*>(d + o[1]) = __builtin_bit_cast(u32x2, hi);
                }
            }
        }
    }
    if (bad != bad) {  // (rare; see phx_kernels_x3.h)
        const f32x4* const copy = reinterpret_cast<const f32x4*>(static_cast<const char*>(P.wpk) + pwx3_packed_bytes(S, P.co_tiles, P.nchunks));
#pragma unroll 1
        for (int i = 0; i < 4 * 2 * S; ++i) {
            const int co = ct * S * 32 + row0 + 16 * (i >> 2), h = (i >> 1) & 1, pixel = p[h] + (i & 1), y = pixel / P.in.Wd;
            if (co < P.Cout && ok[h]) conv_again(P, copy, img[h], y, pixel - y * P.in.Wd, co);
        }
    }
}

// Filter packing: [filter tile of S * 32][wave][K step][lane][part][sub-tile][64] x 8 bf16 (conjugated / transposed for MAP_DGRAD),
// then the fp32 copy (phx_kernels_x3.h).  One thread per (tile, K step, sub-tile, row, channel of the step): eight product lanes from the same four filter values.
template <int MAP>
__device__ __forceinline__ void pack_filters_pwx3_body(const PackArgs& P, int S, long first, long stride) {
    const long total = (long)P.row_tiles * P.nchunks * S * 32 * PWX3_STEP;
    const float* w = static_cast<const float*>(P.w);
    __bf16* outh = static_cast<__bf16*>(P.out);
    f32x4* const copy = reinterpret_cast<f32x4*>(static_cast<char*>(P.out) + pwx3_packed_bytes(S, P.row_tiles, P.nchunks));
    for (long idx = first; idx < total; idx += stride) {
        const int i = idx & 7, r = (idx >> 3) & 31, k8 = (idx >> 8) & 1;
        long s = idx >> 9;
        const int sub = s % S; s /= S;
        const int step = s % P.nchunks;
        const int tile = s / P.nchunks;
        const int row = (tile * S + sub) * 32 + r, red = step * PWX3_STEP + k8 * 8 + i;
        float R[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (row < P.rows && red < P.red) {
            const int o = (MAP == MAP_DGRAD) ? red : row, in = (MAP == MAP_DGRAD) ? row : red;
            const int kh = (MAP == MAP_DGRAD) ? P.khm : 0, kw = (MAP == MAP_DGRAD) ? P.kwm : 0;
            const long off = o * P.so + in * P.si + kh * P.skh + kw * P.skw;
            float wv[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) wv[c] = ((MAP == MAP_DGRAD && c > 0) ? -1.f : 1.f) * w[c * P.wcs + off];
            copy[(long)red * P.rows + row] = f32x4{wv[0], wv[1], wv[2], wv[3]};
#pragma unroll
            for (int c = 0; c < 4; ++c) wv[c] *= ((step / PWX3_STRETCH) & 1) ? -SPLIT_SCALE : SPLIT_SCALE;
            lanes_right(wv, R);
        }
#pragma unroll
        for (int wave = 0; wave < 4; ++wave)
#pragma unroll
            for (int l = 0; l < 2; ++l) {
                const float v = lanes_negated(wave, l) ? -R[lanes_product(wave, l)] : R[lanes_product(wave, l)];
                const __bf16 h = (__bf16)v, m = (__bf16)(v - (float)h), lo = (__bf16)(v - (float)h - (float)m);
                __bf16* dst = outh + ((((long)(tile * 4 + wave) * P.nchunks + step) * 2 + l) * (3 * S) + sub) * 512 + (k8 * 32 + r) * 8 + i;
                dst[0] = h;
                dst[S * 512] = m;
                dst[2 * S * 512] = lo;
            }
    }
}

template <int MAP>
__global__ void __launch_bounds__(WG_THREADS) pack_filters_pwx3_kernel(const PackArgs A0, int S) {
    const PackArgs A = slice_view(A0, PWX3_STEP);
    pack_filters_pwx3_body<MAP>(A, S, (long)blockIdx.x * blockDim.x + threadIdx.x, (long)gridDim.x * blockDim.x);
}

}  // namespace phx
