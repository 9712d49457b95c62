// Factorized (8-product) fp32 forward / input-gradient kernel on bf16 matrix instructions: every operand as the sum of three
// bf16 values.
#pragma once

#include "phx_kernels_lanes16.h"

namespace phx {

// An fp32 value v is h + m + l with h = bf16(v), m = bf16(v - h), l = bf16(v - h - m): 8 bits each, exact but for what lies
// below 2^-26 of it.  Of the nine products of two such sums the six of at least 2^-18 are formed (the largest one left out is
// below 2^-26 of the whole, a quarter of an fp32 rounding):
//     (h | m) x (h | h) = hh + mh,   (h | m) x (m | m) = hm + mm,   (l | h) x (h | l) = lh + hl       (filter x activation)
// each as one 32x32x16 instruction over 8 channels of two parts (K halves | ), whose products are exact and whose sums are
// fp32.  Three instructions of 32 clocks take the place of four fp32 instructions of 64.  Error against fp64 of whole passes,
// relative 2-norm, this kernel / the fp32 instructions: standard normal values, 576 products a result 5.1e-7 / 5.9e-7, 2304
// 1.03e-6 / 1.18e-6, 12800 2.2e-6 / 2.7e-6; of one sign 4.7e-7 / 6.2e-7, 7.9e-7 / 1.24e-6, 1.6e-6 / 2.6e-6: it rounds a fraction as often.
//
// Range.  The parts have fp32's exponents, so m and l of a value below 2^-109 would end in bf16's subnormals, an infinity (or a
// value that rounds to one) leaves inf - inf in m, and m * inf may have the other sign than h * inf.  So
//   - operands are scaled by 2^24 ahead of the split, results by 2^-48: every fp32 value below 2^104, subnormals too, is then the
//     sum of its parts;
//   - whatever lies beyond (infinities, operands of 2^104 or more, sums of 2^80 or more) makes the results that it reaches
//     infinite or not a number, and no others: those are formed once more, in fp32 FMA, by the threads that stored them
//     (split_bad; the packed filters carry an fp32 copy for it).  NaN is what remains where the operands say so.
//
// Drift.  The instructions' sums drop what lies 2^-30 or so below them downwards, whatever their sign: in a chain of n of them
// n * 2^-31 of the whole beside the sqrt(n) * 2^-25 of its roundings (error against fp64 / that of the fp32 instructions, zero-mean
// operands: 4608 products 0.89, 12800 0.92, 25088 0.96, 51200 1.03).  So every 2304 products the accumulators change their sign,
// and the filters of every other such stretch are packed negated: what one stretch loses the next one gains
// (0.86, 0.83, 0.82, 0.78).  A change takes 3 k clocks of the 440 k of a stretch.
//
// The tile and the lanes are those of qconv_fwd_f16_lanes_kernel: S * 32 output channels x NPT * 32 pixels, wave v owns the two
// product lanes made from one pair of components.  A chunk is 8 channels, and its three parts of eight lanes do not fit LDS
// twice, so a chunk is worked on in two phases, the waves' sum lanes and then their difference lanes, each with a buffer of
// its own: while one is read the other is staged from the same activations, kept in registers.
//
// Measured (us a pass, fp32 instructions / here): 3x3, N=64, 64 channels at 56x56 1177 / 650-720; N=2, 256 at 75x75 1235 / 617;
// N=36, 144 -> 136 at 10x10 310 / 109; N=8, 32 at 56x56 82 / 47; 5x5, N=16, 104 -> 40 at 58x7 629 / 178; N=1, 24 at 9x9 61 / 26.
// Bound: the matrix pipe.  At 64 channels, 56x56 the 677 k clocks of products a SIMD would take 376 us at 1.8 GHz; 1568 tiles are
// 6.1 rounds of 256 workgroups run as 7, of 93 us each, 111 k clocks of them products.
constexpr int X3_CK = 8;
constexpr int X3_UPITCH = 265;                   // 16-byte entries: 256 positions, 8 zeros, odd
constexpr int X3_BUF = 12 * X3_UPITCH;           // one phase: 3 parts x 4 waves
constexpr int X3_LDS_BYTES = 8 * 32 * (128 + 4) * 4;  // the epilogue's exchange is larger than the two buffers
static_assert(2 * X3_BUF * 16 <= X3_LDS_BYTES, "LDS of the split kernel");
constexpr int x3_step(int S) { return 128 * S; }  // 16-byte vectors of a wave's filter operands per phase and tap: [2 operands][sub-tile][64]
constexpr int X3_GROUP = 3;                      // taps per group = taps in the filter register ring

constexpr int SPLIT_STRETCH = 2304;               // products between two changes of sign
__host__ __device__ constexpr int x3_stretch(int taps3) { return taps3 * X3_CK < SPLIT_STRETCH ? SPLIT_STRETCH / (taps3 * X3_CK) : 1; }  // in chunks

__host__ __device__ inline size_t x3_packed_bytes(int S, int co_tiles, int nchunks, int taps3) {  // (in front of the fp32 copy)
    return ((size_t)co_tiles * 4 * nchunks * 2 * taps3 + X3_GROUP) * x3_step(S) * 16;
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));

__device__ __forceinline__ unsigned int pack_bf16(float a, float b) {
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float bf16_low(unsigned int v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float bf16_high(unsigned int v) { return __builtin_bit_cast(float, v & 0xffff0000u); }

constexpr float SPLIT_SCALE = 0x1p24f, SPLIT_RESULT = 0x1p-48f;

// bad stays zero as long as every y is finite, and is NaN from the first one on that is not
__device__ __forceinline__ void split_check(float& bad, float y) { bad = fmaf(y, 0.f, bad); }
__device__ __forceinline__ bool split_bad(float y) { return !(fabsf(y) < __builtin_inff()); }
__device__ __forceinline__ bool all_nan(const float (&y)[4]) { return y[0] != y[0] && y[1] != y[1] && y[2] != y[2] && y[3] != y[3]; }

// y += x (x) w, in fp32
__device__ __forceinline__ void add_product(const float (&x)[4], const f32x4& w, float (&y)[4]) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] = fmaf(qneg(p, q) ? -x[p] : x[p], w[p ^ q], y[q]);
}

// The packed image's fp32 copy of the filter, [tap][reduced channel][output channel] x 4 components (conjugated / mirrored /
// transposed for MAP_DGRAD), and the four components of one output from it
inline size_t split_copy_bytes(int taps, int red, int rows) { return (size_t)taps * red * rows * 16; }
__device__ __forceinline__ void conv_fp32(const ConvArgs& P, const f32x4* copy, int n, int ho, int wo, int co, float (&y)[4]) {
    const long plane = (long)P.in.Hd * P.in.Wd;
#pragma unroll
    for (int q = 0; q < 4; ++q) y[q] = 0.f;
    for (int tap = 0; tap < P.taps; ++tap) {
        const int kh = tap / P.Kw, h = ho * P.sh - P.pt + kh * P.dh, w = wo * P.sw - P.pl + (tap - kh * P.Kw) * P.dw;
        if (h < 0 || h >= P.in.Hd || w < 0 || w >= P.in.Wd) continue;
        const float* src = static_cast<const float*>(P.in.base) + (long)n * P.in.Cs * plane + (long)h * P.in.Wd + w;
        const f32x4* f = copy + (long)tap * P.in.C * P.Cout + co;
#pragma unroll 4
        for (int c = 0; c < P.in.C; ++c, src += plane, f += P.Cout) {
            const float x[4] = {src[0], src[P.in.comp_stride], src[2 * P.in.comp_stride], src[3 * P.in.comp_stride]};
            add_product(x, *f, y);
        }
        if (all_nan(y)) return;
    }
}

// output (n, ho, wo, co) once more if what has been stored is not finite
__device__ __forceinline__ void conv_again(const ConvArgs& P, const f32x4* copy, int n, int ho, int wo, int co) {
    float* const out = static_cast<float*>(P.out) + (((long)n * P.CoutS + co) * P.Hout + ho) * P.Wout + wo;
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) bad = bad || split_bad(out[q * P.out_cs]);
    if (!bad) return;
    float y[4];
    conv_fp32(P, copy, n, ho, wo, co, y);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (P.bias) y[q] += static_cast<const float*>(P.bias)[q * P.CoutS + co];
        out[q * P.out_cs] = y[q];
    }
}

template <int S, int NPT>
__global__ void __launch_bounds__(WG_THREADS, 1) qconv_fwd_x3_kernel(const ConvArgs P0) {
    const ConvArgs P = slice_view(P0, X3_CK);
    constexpr int TG = X3_GROUP;
    constexpr int PX = NPT * 32, STEP = x3_step(S);
    extern __shared__ u32x4 ldsx3[];  // [2][X3_BUF]; the epilogue's exchange

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kk = lane >> 5;

    int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int ct = bid % P.co_tiles;
    bid /= P.co_tiles;
    const int tw = bid % P.tiles_w;
    bid /= P.tiles_w;
    const int th = bid % P.tiles_h;
    const int tn = bid / P.tiles_h;
    const bool tall = P.in.tall != 0;  // (flat tiling, see qconv_fwd_f16_lds_kernel)
    const int q0 = th * PX, R0 = tall ? q0 / P.Wout : 0;
    const int n0 = tall ? R0 / P.in.tall : tn * P.NB;
    const int y0 = tall ? R0 - n0 * P.in.tall : th * P.TH, c0 = tall ? q0 - R0 * P.Wout : tw * P.TW;

    // Filters: this wave's stream of operands, [chunk][phase][tap], through L2 into a ring of three taps.
    const int ngroups = (P.taps + TG - 1) / TG;  // per phase, at least 3
    const long nsteps = (long)P.nchunks * 2 * ngroups * TG;
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<u32x4*>(static_cast<const u32x4*>(P.wpk) + (ct * 4 + wave) * nsteps * STEP), 0, -1, 0x00020000);
    unsigned int wstep = 0;  // bytes to the current tap
    bf16x8 A[TG][2][S], B[3][NPT];  // [tap][operand][sub-tile]; [instruction of the three][pixel tile]
    auto load_a = [&](int o, int s, int ahead) {
        return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wbuf, lane * 16 + (o * S + s) * 1024,
                                                                               wstep + ahead * (STEP * 16), 0));
    };

    // Staging: a thread holds 4 consecutive positions of one component and 8 channels; four neighbouring threads 16 positions
    // (64 contiguous bytes a load), the sixteen of a DPP row the components in the order x0, x2, x3, x1, so that each finds
    // its partner four threads on.
    const int p = (tid >> 2) & 3, ch = wave * 16 + ((lane >> 4) << 2) + (lane & 3);
    const int w0 = (tall ? 0 : c0) * P.sw - P.pl;
    const int cpr = P.HTW >> 2;
    const int row = small_div(ch, __builtin_amdgcn_rcpf(cpr)), cc = ch - row * cpr;
    unsigned int bits = 0;   // positions of the task inside the image
    bool careful = false;    // the loads of four positions would leave the tensor
    long element = 0;        // the task's first position, channel 0
    const long plane_in = (long)P.in.Hd * P.in.Wd;
    if (ch < P.NB * P.HTH * cpr) {
        const int nb = tall ? 0 : small_div(row, __builtin_amdgcn_rcpf(P.HTH)), hr = row - nb * P.HTH;
        int img = n0 + nb, vh = y0 * P.sh - P.pt + hr;
        if (tall) {  // (rows above the image belong to the one before, or are its gap)
            const int d = small_div(vh + P.in.tall, __builtin_amdgcn_rcpf(P.in.tall));
            img += d - 1;
            vh -= (d - 1) * P.in.tall;
        }
        const int vw = w0 + cc * 4;
        if (img >= 0 && img < P.in.N && vh >= 0 && vh < P.in.Hd) bits = interval_bits<4>(-vw, P.in.Wd - vw);
        const int comp = (0x78 >> (2 * p)) & 3;
        element = comp * P.in.comp_stride + ((long)img * P.in.Cs * P.in.Hd + vh) * P.in.Wd + vw;
        const long size = 3 * P.in.comp_stride + ((long)(P.in.N - 1) * P.in.Cs + P.in.C) * plane_in;
        careful = bits && (element < 0 || element + (long)(P.in.C - 1) * plane_in + 4 > size);
    }
    // (32-bit byte offsets: the host keeps larger tensors off this kernel; tasks that load nothing read the tensor's start)
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(P.in.base), 0, -1, 0x00020000);
    const unsigned int xoff = (bits && !careful) ? (unsigned int)(element * 4) : 0u;
    const unsigned int xstep = (unsigned int)(plane_in * 4);  // to the next channel
    const bool any_careful = __any(careful);
    u32x4 stage[X3_CK];
    auto load_stage = [&](int chan, int i) {  // (channels past the tensor meet zero filters, any value of this position will do)
        const int c = chan + i;
        stage[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, xoff, c < P.in.C ? c * xstep : 0u, 0));
    };
    // a tensor's first and last rows: value by value
    auto fill_careful = [&](int chan) {
        if (!careful) return;
        const unsigned int* src = static_cast<const unsigned int*>(P.in.base) + element;
#pragma unroll
        for (int i = 0; i < X3_CK; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int c = chan + i < P.in.C ? chan + i : 0;
                stage[i][k] = ((bits >> k) & 1) ? src[(long)c * plane_in + k] : 0u;
            }
    };
    float keep[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) keep[k] = ((bits >> k) & 1) ? SPLIT_SCALE : 0.f;
    // Position k of the task, channels 2q and 2q + 1, in nine steps of one to three instructions, which go between the
    // products: scaled, or cleared outside the image (a value there that is not finite is one more reason for conv_again), the partner's, sum (l = 0) or difference, the three parts; behind the last pair
    // the parts' eight channels go to LDS.
    float e[2], f[2];
    unsigned int part[3][4];
    u32x4* const wunit = ldsx3 + p * X3_UPITCH + ch * 4;
    auto slice = [&](int l, int k, int q, int u) {
        if (u == 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i) e[i] = __builtin_bit_cast(float, (unsigned int)stage[2 * q + i][k]) * keep[k];
        } else if (u == 1) {
#pragma unroll
            for (int i = 0; i < 2; ++i)  // row_ror:12 = from four threads on
                f[i] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, e[i]), 0x12C, 0xf, 0xf, true));
        } else if (u == 2) {
#pragma unroll
            for (int i = 0; i < 2; ++i) e[i] = l ? e[i] - f[i] : e[i] + f[i];
        } else if (u == 3 || u == 5 || u == 7) {
            part[(u - 3) / 2][q] = pack_bf16(e[0], e[1]);
            if (u < 7) f[0] = bf16_low(part[(u - 3) / 2][q]);
        } else if (u == 4 || u == 6) {
            e[0] -= f[0];
            e[1] -= bf16_high(part[(u - 4) / 2][q]);
        } else if (q == 3) {
#pragma unroll
            for (int t = 0; t < 3; ++t)
                wunit[l * X3_BUF + t * (4 * X3_UPITCH) + k] = u32x4{part[t][0], part[t][1], part[t][2], part[t][3]};
        }
    };

    // prologue: the first chunk, the first taps' filters
#pragma unroll
    for (int i = 0; i < X3_CK; ++i) load_stage(0, i);
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int s = 0; s < S; ++s) A[tg][o][s] = load_a(o, s, tg);

    // window offset, output offset and validity of a pixel of the tile
    const float rcp_w = __builtin_amdgcn_rcpf(tall ? P.Wout : P.TW), rcp_h = __builtin_amdgcn_rcpf(tall ? P.in.tall : P.TH * P.TW);
    auto decode_at = [&](int pix, int& off, int& n, int& ho, int& wo) -> bool {
        bool valid;
        if (tall) {
            const int x = c0 + pix, r = small_div(x, rcp_w), y = y0 + r, d = small_div(y, rcp_h);
            n = n0 + d; ho = y - d * P.in.tall; wo = x - r * P.Wout;
            valid = n < P.in.N && ho < P.Hout;
            off = valid ? r * P.HTW + wo : 0;
        } else {
            const int nb = small_div(pix, rcp_h), rem = pix - nb * (P.TH * P.TW), r = small_div(rem, rcp_w), c = rem - r * P.TW;
            n = n0 + nb; ho = y0 + r; wo = c0 + c;
            valid = nb < P.NB && n < P.in.N && ho < P.Hout && wo < P.Wout;
            off = valid ? (nb * P.HTH + r * P.sh) * P.HTW + c * P.sw : 0;
        }
        return valid;
    };
    auto decode = [&](int pix, int& off, long& oaddr) -> bool {
        int n, ho, wo;
        const bool valid = decode_at(pix, off, n, ho, wo);
        oaddr = ((long)n * P.CoutS * P.Hout + ho) * P.Wout + wo;
        return valid;
    };
    unsigned int poff[NPT];  // bytes into a phase's buffer: the wave's lane, part h
#pragma unroll
    for (int t = 0; t < NPT; ++t) {
        long unused;
        int off;
        decode(t * 32 + j, off, unused);
        poff[t] = (off + wave * X3_UPITCH) * 16;
    }
    const unsigned int outer = kk * (8 * X3_UPITCH * 16);  // the third instruction's halves: h and l

    f32x16 acc[2][S][NPT];  // [lane][filter sub-tile][pixel tile]; rows = pixels, columns = output channels
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int t = 0; t < NPT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[l][s][t][r] = 0.f;
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int t = 0; t < NPT; ++t) asm volatile("" : "+a"(acc[l][s][t]));  // (cleared while the loads are on their way)
    if (any_careful) fill_careful(0);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int u = 0; u < 9; ++u) slice(0, k, q, u);
    wg_barrier_no_vmem_wait();

    unsigned int addr[NPT];
    auto read_b = [&](int l, int t, int i) {  // operand of instruction i
        const unsigned int a = addr[t] + l * (X3_BUF * 16) + (i == 1 ? 4 * X3_UPITCH * 16 : i == 2 ? outer : 0u);
        return *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(ldsx3) + a);
    };

    // One group of three taps of phase l.  PH 1: requests the next chunk's activations; PH 2, 3: a phase's last two groups,
    // which stage two positions each, for the other phase.  The products of a tap are the three instructions one after the
    // other over all tiles; the operands of one are read during the one before.
    int tap = 0, kh = 0, kw = 0;
    auto group = [&](auto lane_tag, auto phase_tag, int chan_next) {
        constexpr int L = decltype(lane_tag)::value, PH = decltype(phase_tag)::value;
        constexpr int MF = S * NPT;  // products of an instruction kind
#pragma unroll
        for (int tg = 0; tg < TG; ++tg) {
            ++tap;
            if (++kw == P.Kw) { kw = 0; ++kh; }
            const int off = tap < P.taps ? kh * P.dh * P.HTW + kw * P.dw : 0;  // (of the next tap; padded taps have zero filters)
            const bool last = PH == 3 && tg == TG - 1;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
#pragma unroll
                for (int m = 0; m < MF; ++m) {
                    const int t = m / S, s = m % S;
                    acc[L][s][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(B[i][t], A[tg][i == 2][s], acc[L][s][t], 0, 0, 0);
                    if (m < NPT) {
                        if (i == 2 && !last) addr[m] = poff[m] + off * 16;
                        if (i < 2 || !last) B[(i + 1) % 3][m] = read_b(L, m, (i + 1) % 3);
                    }
                    // requests to memory, at most one per two products: the filters of three taps on as their registers
                    // come free
                    if (i == 0 && tg > 0 && (m & 1) && m / 2 < S) A[tg - 1][1][m / 2] = load_a(1, m / 2, TG - 1);
                    if (i == 2 && (m & 1) && m / 2 < S) A[tg][0][m / 2] = load_a(0, m / 2, TG);
                    if (i == 2 && tg == TG - 1 && m == MF - 1) {
#pragma unroll
                        for (int r = 0; r < S; ++r) A[tg][1][r] = load_a(1, r, TG);
                    }
                    const int g = (tg * 3 + i) * MF + m;
                    if constexpr (PH == 1) {
                        constexpr int W = MF == 8 ? 3 : 2;
                        if (g % W == 0 && g / W < X3_CK) load_stage(chan_next, g / W);
                    }
                    if constexpr (PH >= 2) {
                        constexpr int PIECES = 8 / MF;  // steps of the staging behind a product: 72 in all
#pragma unroll
                        for (int a = 0; a < PIECES; ++a) {
                            const int x = g * PIECES + a;
                            slice(1 - L, (PH - 2) * 2 + x / 36, (x / 9) % 4, x % 9);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            wstep += STEP * 16;
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int t = 0; t < NPT; ++t) asm volatile("" : "+a"(acc[L][s][t]));
        }
    };
    auto start_phase = [&](int l) {
        tap = 0; kh = 0; kw = 0;
#pragma unroll
        for (int t = 0; t < NPT; ++t) {
            addr[t] = poff[t];
            B[0][t] = read_b(l, t, 0);
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    const int stretch = x3_stretch(ngroups * TG);
    int left = stretch;
    float result = SPLIT_RESULT;
    for (int chunk = 0; chunk < P.nchunks; ++chunk) {
        if (left-- == 0) {
            left = stretch - 1;
            result = -result;
#pragma unroll
            for (int l = 0; l < 2; ++l)
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int t = 0; t < NPT; ++t) {
                        asm volatile("" : "+a"(acc[l][s][t]));
                        acc[l][s][t] = -acc[l][s][t];
                        asm volatile("" : "+a"(acc[l][s][t]));
                        __builtin_amdgcn_sched_barrier(0);  // (a tile at a time leaves the accumulator file)
                    }
        }
        const int chan_next = (chunk + 1) * X3_CK;  // (behind the last chunk: loads of channel 0, into a buffer nobody reads)
        start_phase(0);
        for (int g = 2; g < ngroups; ++g) group(I0{}, I0{}, 0);
        group(I0{}, I2{}, 0);
        group(I0{}, I3{}, 0);
        wg_barrier_no_vmem_wait();
        start_phase(1);
        group(I1{}, I1{}, chan_next);
        for (int g = 3; g < ngroups; ++g) group(I1{}, I0{}, 0);
        if (any_careful) fill_careful(chan_next);
#pragma unroll
        for (int i = 0; i < X3_CK; ++i) asm volatile("" : "+v"(stage[i]));  // (the staging stays between the products)
        group(I1{}, I2{}, 0);
        group(I1{}, I3{}, 0);
        wg_barrier_no_vmem_wait();
    }

    // Epilogue, one round per filter sub-tile: the waves' product lanes meet in LDS and are read back eight pixels of a channel
    // at a time, merged and stored as two 16-byte words.
    float* const xch = reinterpret_cast<float*>(ldsx3);
    float* const out = static_cast<float*>(P.out);
    const float* const bias = static_cast<const float*>(P.bias);
    const long plane_out = (long)P.Hout * P.Wout;
    constexpr int PITCH = PX + 4;                      // [product lane][32 channels][PX pixels + 4]
    constexpr int SLAB = 32 * PITCH;
    constexpr int GR = PX / 8;                         // groups of eight pixels side by side
    constexpr int ROWS = WG_THREADS / GR;              // rows the threads cover at once
    const int g8 = tid % GR, row0 = tid / GR;
    long o8[2] = {0, 0};                               // offset of the two halves of the group (the same for every channel)
    bool run4[2] = {false, false};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        int off;
        long end;
        const bool a = decode(g8 * 8 + 4 * h, off, o8[h]), b = decode(g8 * 8 + 4 * h + 3, off, end);
        run4[h] = a && b && end == o8[h] + 3;
    }
    float bad = 0.f;  // (pixels behind the tile's last one count as well: conv_again looks)
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (s > 0) wg_barrier_no_vmem_wait();  // the previous round has been read
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            float* const dst = xch + lanes_product(wave, l) * SLAB;
#pragma unroll
            for (int t = 0; t < NPT; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x16& a = acc[l][s][t];
                    // (the two halves of a group trade places in every other 64 pixels: see qconv_fwd_f16_lanes_kernel)
                    *reinterpret_cast<f32x4*>(dst + j * PITCH + t * 32 + 8 * g + 4 * (kk ^ (t >> 1))) =
                        f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
                }
        }
        wg_barrier_no_vmem_wait();
#pragma unroll
        for (int pass = 0; pass < 32 / ROWS; ++pass) {
            const int r = row0 + pass * ROWS, co = (ct * S + s) * 32 + r;
            f32x4 lanes[8][2];
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    lanes[i][h] = *reinterpret_cast<const f32x4*>(xch + i * SLAB + r * PITCH + g8 * 8 + 4 * (h ^ (g8 >> 3)));
            if (co >= P.Cout) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4 y[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float in[8], c[4];
#pragma unroll
                    for (int i = 0; i < 8; ++i) in[i] = lanes[i][h][k];
                    merge_output(in, c);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        y[q][k] = c[q] * result;
                        split_check(bad, y[q][k]);
                    }
                }
                if (bias) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) y[q] += bias[q * P.CoutS + co];
                }
                if (run4[h]) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) *reinterpret_cast<f32x4_a4*>(out + q * P.out_cs + o8[h] + co * plane_out) = y[q];
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        int off;
                        long o;
                        if (decode(g8 * 8 + 4 * h + k, off, o)) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) out[q * P.out_cs + o + co * plane_out] = y[q][k];
                        }
                    }
                }
            }
        }
    }
    if (bad != bad) {  // (rare)
        const f32x4* const copy = reinterpret_cast<const f32x4*>(static_cast<const char*>(P.wpk) + x3_packed_bytes(S, P.co_tiles, P.nchunks, ngroups * TG));
#pragma unroll 1
        for (int i = 0; i < 8 * S * (32 / ROWS); ++i) {
            const int co = ct * S * 32 + row0 + (i >> 3) * ROWS;
            int off, n, ho, wo;
            if (co < P.Cout && decode_at(g8 * 8 + (i & 7), off, n, ho, wo)) conv_again(P, copy, n, ho, wo, co);
        }
    }
}

// Filter packing: [filter tile of S * 32][wave][chunk][phase][tap, padded to whole groups][operand (h | m), (l | h)][sub-tile][64] x 8
// bf16 (conjugated / mirrored / transposed for MAP_DGRAD), then the fp32 copy.  One thread per (tile, chunk, tap, sub-tile, row,
// channel of the chunk): eight product lanes from the same four filter values.
template <int MAP>
__device__ __forceinline__ void pack_filters_x3_body(const PackLanesArgs& A, int S, long first, long stride) {
    const PackArgs& P = A.base;
    const int taps = P.Kh * P.Kw;
    const long total = (long)P.row_tiles * P.nchunks * A.taps3 * S * 32 * 8;
    const float* w = static_cast<const float*>(P.w);
    __bf16* outh = static_cast<__bf16*>(P.out);
    f32x4* const copy = reinterpret_cast<f32x4*>(static_cast<char*>(P.out) + x3_packed_bytes(S, P.row_tiles, P.nchunks, A.taps3));
    const int stretch = x3_stretch(A.taps3);
    for (long idx = first; idx < total; idx += stride) {
        const int i = idx & 7, r = (idx >> 3) & 31;
        long s = idx >> 8;
        const int sub = s % S; s /= S;
        const int tap = s % A.taps3; s /= A.taps3;
        const int chunk = s % P.nchunks;
        const int tile = s / P.nchunks;
        const int row = (tile * S + sub) * 32 + r;
        const int red = chunk * X3_CK + i;
        float R[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (tap < taps && row < P.rows && red < P.red) {
            int kh = tap / P.Kw, kw = tap - kh * P.Kw;
            if (MAP == MAP_DGRAD) { kh = P.khm - kh * P.khs; kw = P.kwm - kw * P.kws; }
            const int o = (MAP == MAP_DGRAD) ? red : row;
            const int in = (MAP == MAP_DGRAD) ? row : red;
            const long off = o * P.so + in * P.si + kh * P.skh + kw * P.skw;
            float wv[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) wv[c] = ((MAP == MAP_DGRAD && c > 0) ? -1.f : 1.f) * w[c * P.wcs + off];
            copy[((long)tap * P.red + red) * P.rows + row] = f32x4{wv[0], wv[1], wv[2], wv[3]};
#pragma unroll
            for (int c = 0; c < 4; ++c) wv[c] *= ((chunk / stretch) & 1) ? -SPLIT_SCALE : SPLIT_SCALE;
            lanes_right(wv, R);
        }
#pragma unroll
        for (int wave = 0; wave < 4; ++wave)
#pragma unroll
            for (int l = 0; l < 2; ++l) {
                const float v = lanes_negated(wave, l) ? -R[lanes_product(wave, l)] : R[lanes_product(wave, l)];
                const __bf16 h = (__bf16)v, m = (__bf16)(v - (float)h), lo = (__bf16)(v - (float)h - (float)m);
                const long step = (((long)(tile * 4 + wave) * P.nchunks + chunk) * 2 + l) * A.taps3 + tap;
                __bf16* dst = outh + ((step * 2 * S + sub) * 64 + r) * 8 + i;
                dst[0] = h;
                dst[32 * 8] = m;
                dst[S * 64 * 8] = lo;
                dst[S * 64 * 8 + 32 * 8] = h;
            }
    }
}

template <int MAP>
__global__ void __launch_bounds__(WG_THREADS) pack_filters_x3_kernel(const PackLanesArgs A0, int S) {
    PackLanesArgs A = A0;
    A.base = slice_view(A0.base, X3_CK);
    pack_filters_x3_body<MAP>(A, S, (long)blockIdx.x * blockDim.x + threadIdx.x, (long)gridDim.x * blockDim.x);
}

}  // namespace phx
