// Factorized (8-product) fp16 forward / input-gradient kernel with the product lanes dealt over the waves.
#pragma once

#include <type_traits>

#include "phx_kernels_f16.h"

namespace phx {

// Workgroup = 64 output channels x NPT*32 pixels; wave v owns the two product lanes made from one pair of components
// (the sum and the difference) for the whole tile: 2 lanes x 2 filter sub-tiles x NPT pixel tiles of 32x32 accumulators.
//   - The left lanes are formed ONCE per staged chunk, on their way into LDS, and not once per tap and wave in front of
//     the products: four lane groups of a DPP row stage the four components of the same positions, each thread fetches
//     its partner's value with one DPP rotation and writes the sum and the difference.
//   - No two waves of a workgroup read the same filter operand, so filters go from L2 straight into registers, two taps
//     ahead or more, and LDS holds activations alone: two buffers of a 16-channel chunk's eight lanes (the next chunk is
//     staged between the products of this one), one barrier per chunk.
//   - Per 16 matrix instructions a wave reads 8 operands from LDS and 4 from L2 and adds nothing.
// The product lanes meet in the epilogue, through LDS.
//
// Measured (full16, 8-product, forward, on the box where the kernel that forms the lanes in front of the products takes
// the second time): 3x3, N=128, 128 channels at 28x28 282 / 392 us, 256 at 14x14 270 / 405, 512 at 7x7 409 / 594; N=64, 64
// at 28x28 55 / 67; 5x5, N=4, 256 at 28x28 110 / 157.  Bit for bit the same results.
// Bound: a tile of 128 channels x 9 taps takes 83 k clocks of which the 1152 products, at 32 clocks, would take 37 k.  The
// products run at one per 39 clocks where nothing is staged and one per 47 in the last four taps of a chunk, between the
// staging's vector instructions and stores; 12 k clocks are the start (arguments, tile arithmetic, first loads), 13 k the
// epilogue.  Persistent workgroups that request the next tile's first activations in front of the epilogue measured no gain:
// 6.6 tiles per CU round up to 7.
//
// Component pairs (left lanes as in lanes_left, up to a sign that the packed filter takes along):
//   wave 0: (x0, x2) -> L2, L1    wave 1: (x2, x3) -> L7, -L4    wave 2: (x3, x1) -> L0, L3    wave 3: (x1, x0) -> L5, -L6
// Units of a staged chunk, unit (l * 2 + pack) * 4 + wave: 256 positions in order (a wave reads runs of them: no swizzle that
// helped the stores would leave those free of bank conflicts), 8 zeros, and an odd pitch that spreads the four units a DPP
// row stores to.
constexpr int LANES_UPITCH = 265;             // 16-byte entries
constexpr int LANES_BUF = 16 * LANES_UPITCH;  // one chunk: 4 waves x 2 lanes x 2 packs of 8 channels
constexpr int LANES_LDS_BYTES = 8 * 128 * 36 * 4;  // the epilogue's exchange (channels-last) is larger than the two buffers
constexpr int LANES_NORM_BYTES = 64 * 16;      // behind it: the factors of the tile's channels (NORM)
static_assert(2 * LANES_BUF * 16 <= LANES_LDS_BYTES && 8 * 32 * (128 + 4) * 4 <= LANES_LDS_BYTES, "LDS of the lanes kernel");
constexpr int LANES_STEP = 256;               // 16-byte vectors of one wave's filter operands per tap: [lane][sub-tile][64]
constexpr int LANES_GROUP = 3;                // taps per group = taps in a filter register ring

__host__ __device__ constexpr int lanes_product(int wave, int l) { return (0x65304712 >> (4 * (2 * wave + l))) & 7; }
__host__ __device__ constexpr bool lanes_negated(int wave, int l) { return l == 1 && (wave & 1); }

// bytes of the packed image: one stream of tap operands per (filter tile, wave), and what the last stream's register
// rings read past its end
inline size_t lanes_packed_bytes(int co_tiles, int nchunks, int taps3) {
    return ((size_t)co_tiles * 4 * nchunks * taps3 + LANES_GROUP + 1) * LANES_STEP * 16;
}

// a / b for 0 <= a < 2^20 and the reciprocal of 1 <= b < 2^20
__device__ __forceinline__ int small_div(int a, float rcp_b) { return (int)(((float)a + 0.5f) * rcp_b); }

// NORM (planes only): P0.norm is applied to what is stored.
template <int NPT, bool CL, bool NORM = false>
__global__ void __launch_bounds__(WG_THREADS, 1) qconv_fwd_f16_lanes_kernel(const ConvArgsOf<NORM> P0) {
    const ConvArgs P = group_view(P0);
    constexpr int TG = LANES_GROUP;
    constexpr int CK = F16_CK;
    constexpr int PX = NPT * 32;
    extern __shared__ f16x8 lds16[];  // [2][LANES_BUF]; the epilogue's exchange

    PHX_PHASES_BEGIN(6)
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
    // Origin of the tile; flat tiling (P.in.tall, see qconv_fwd_f16_lds_kernel): position q0 of the tall image is column
    // c0 of row y0 of image n0.
    f32x4* const factors = reinterpret_cast<f32x4*>(lds16 + LANES_LDS_BYTES / 16);  // (formed in front of the first barrier, read in the epilogue)
    if constexpr (NORM) {
        if (tid < 64) factors[tid] = ct * 64 + tid < P.Cout ? norm_factors(P0.norm, ct * 64 + tid) : f32x4{};
    }
    const bool tall = P.in.tall != 0;
    const int q0 = th * PX, R0 = tall ? q0 / P.Wout : 0;
    const int n0 = tall ? R0 / P.in.tall : tn * P.NB;
    const int y0 = tall ? R0 - n0 * P.in.tall : th * P.TH, c0 = tall ? q0 - R0 * P.Wout : tw * P.TW;

    // Filters: this wave's stream of tap operands, through L2 into registers (scalar offsets, no address arithmetic).
    const int ngroups = (P.taps + TG - 1) / TG;  // per chunk, at least 3
    const long nsteps = (long)P.nchunks * ngroups * TG;
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<f16x8*>(static_cast<const f16x8*>(P.wpk) + (ct * 4 + wave) * nsteps * LANES_STEP), 0, -1, 0x00020000);
    unsigned int wstep = 0;  // bytes to the current tap
    // Two rings of a group's operands: X for a chunk's first group, Y for the others.  The loads that bring the next chunk's
    // activations from HBM are issued in the first group, and what is requested behind them is not delivered before them:
    // with one ring, two taps ahead, every chunk waited for HBM (78 clocks per matrix instruction in the first group
    // instead of 50).
    f16x8 X[TG][2][2], Y[TG][2][2], B[2][NPT];
    auto load_a = [&](int l, int s, int ahead) {
        return __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(wbuf, lane * 16 + (l * 2 + s) * 1024,
                                                                              wstep + ahead * (LANES_STEP * 16), 0));
    };

    // Staging: four neighbouring threads hold 4 x 8 consecutive positions (64 contiguous bytes a load) of one component and
    // 8 channels, the sixteen of a DPP row the four components in the order x0, x2, x3, x1, so that each finds its partner
    // four threads on.
    const int p = (tid >> 2) & 3, pack = wave >> 1, ch = (wave & 1) * 16 + ((lane >> 4) << 2) + (lane & 3);
    // Rows of even length: the window starts at an even column, so that every load is aligned to 4 bytes.  (A wave's 16-byte
    // loads at odd multiples of 2 bytes take the CU's address unit four times as long: 38 % of the time of this kernel's
    // products were spent behind its 8 activation loads per chunk.)
    const int w0 = (tall ? 0 : c0) * P.sw - P.pl, colshift = P.even ? w0 & 1 : 0;
    const int cpr = P.HTW >> 3;
    const int row = small_div(ch, __builtin_amdgcn_rcpf(cpr)), cc = ch - row * cpr;
    const bool task = ch < P.NB * P.HTH * cpr;
    unsigned int bits = 0;   // positions of the task inside the image
    bool careful = false;    // the tensor is too small for loads of eight positions
    int rot = 0;             // the loads start this many positions (modulo 8) behind the task's first one (see StageChunk)
    long element = 0;        // the task's first position, channel 0
    {
        const int nb = tall ? 0 : small_div(row, __builtin_amdgcn_rcpf(P.HTH)), hr = row - nb * P.HTH;
        int img = n0 + nb, vh = y0 * P.sh - P.pt + hr;
        if (tall) {  // (rows above the image belong to the one before, or are its gap)
            const int d = small_div(vh + P.in.tall, __builtin_amdgcn_rcpf(P.in.tall));
            img += d - 1;
            vh -= (d - 1) * P.in.tall;
        }
        const int vw = w0 - colshift + (CL ? cc : cc * 8);
        if (task && img >= 0 && img < P.in.N && vh >= 0 && vh < P.in.Hd) {
            if constexpr (CL) {
#pragma unroll
                for (int k = 0; k < 8; ++k) bits |= (unsigned int)(vw + k * cpr >= 0 && vw + k * cpr < P.in.Wd) << k;
            } else {
                bits = interval_bits(-vw, P.in.Wd - vw);
            }
        }
        const long comp = ((0x78 >> (2 * p)) & 3) * P.in.comp_stride;
        const long size = 3 * P.in.comp_stride + ((long)(P.in.N - 1) * P.in.Cs + P.in.C) * P.in.Hd * P.in.Wd;  // (planes)
        if constexpr (CL) {
            element = comp + (((long)img * P.in.Hd + vh) * P.in.Wd + vw) * P.in.Cs;
        } else {
            element = comp + ((long)img * P.in.Cs * P.in.Hd + vh) * P.in.Wd + vw;
            if (bits) {
                const long sh = inside_shift(element, (long)(P.in.C - 1) * P.in.Hd * P.in.Wd, size);
                careful = sh == NO_SHIFT;
                if (!careful) {
                    element += sh;
                    rot = (int)sh & 7;
                }
            }
        }
    }
    // (32-bit byte offsets: the host keeps larger tensors off this kernel; tasks that load nothing read the tensor's start)
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(P.in.base), 0, -1, 0x00020000);
    const unsigned int xoff = CL || (bits && !careful) ? (unsigned int)(element * 2) : 0u;  // (channels-last: added up modulo 2^32)
    const unsigned int xstep = (CL ? cpr * P.in.Cs : P.in.Hd * P.in.Wd) * 2;  // CL: to the next position, else to the next channel
    const int first = (CL && task) ? row * P.HTW + cc : ch * 8;  // first position and distance of the task's positions
    const int pstep = (CL && task) ? cpr : 1;                    // (threads without a task clear positions behind the window)
    const bool any_careful = !CL && __any(careful || rot);
    u32x4 stage[8];
    auto load_stage = [&](int chan, int i) {  // (channels past the tensor meet zero filters, any finite value will do)
        unsigned int off;
        if constexpr (CL) {
            const unsigned int o = ((bits >> i) & 1u) && chan + pack * 8 < P.in.C ? xoff + (chan + pack * 8) * 2 + i * xstep : 0u;
            stage[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, o, 0, 0));
        } else {
            const int c = chan + pack * 8 + i;
            stage[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, xoff, c < P.in.C ? c * xstep : 0u, 0));
        }
    };
    // Threads whose loads were moved to stay inside the tensor (its first and last rows) rotate their values into place,
    // or fill them one by one.
    auto fill_careful = [&](int chan) {
        if (rot) {
#pragma unroll
            for (int i = 0; i < 8; ++i) stage[i] = rotate_halves(stage[i], rot);
        }
        if (!careful) return;
        const _Float16* src = static_cast<const _Float16*>(P.in.base) + element;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            _Float16 e[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {  // channel i, position k
                const int c = chan + pack * 8 + i;
                e[k] = c < P.in.C && ((bits >> k) & 1) ? src[(long)c * P.in.Hd * P.in.Wd + k] : (_Float16)0;
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) stage[i][m] = __builtin_bit_cast(unsigned int, f16x2{e[2 * m], e[2 * m + 1]});
        }
    };
    // Position jj of the task: v = its 8 channels, cleared outside the image (step 0), the partner's value (1), sum (2),
    // difference (3), both to LDS (4).  (Planes: the byte permutes that gather a position's channels clear it, too.)
    u32x4 v, pv, sum, dif;
    unsigned int select[CL ? 1 : 8];
    if constexpr (!CL) {
#pragma unroll
        for (int k = 0; k < 8; ++k) select[k] = (bits >> k) & 1 ? ((k & 1) ? 0x07060302u : 0x05040100u) : 0x0c0c0c0cu;
    }
    f16x8* const wunit = lds16 + (pack * 4 + p) * LANES_UPITCH + first;  // sum lane; the difference lane eight units behind
    auto slice = [&](int jj, int piece, int chan, int buf) {
        if (piece == 0) {
            if constexpr (CL) {
                const unsigned int keep = chan + pack * 8 < P.in.C ? (unsigned int)((int)(bits << (31 - jj)) >> 31) : 0u;
#pragma unroll
                for (int m = 0; m < 4; ++m) v[m] = stage[jj][m] & keep;
            } else {
#pragma unroll
                for (int m = 0; m < 4; ++m) v[m] = __builtin_amdgcn_perm(stage[2 * m + 1][jj >> 1], stage[2 * m][jj >> 1], select[jj]);
            }
        } else if (piece == 1) {
#pragma unroll
            for (int m = 0; m < 4; ++m)  // row_ror:12 = from four threads on
                pv[m] = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v[m], 0x12C, 0xf, 0xf, true);
        } else if (piece == 2) {
            sum = __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, v) + __builtin_bit_cast(f16x8, pv));
        } else if (piece == 3) {
            dif = __builtin_bit_cast(u32x4, sub8_pinned(__builtin_bit_cast(f16x8, v), __builtin_bit_cast(f16x8, pv)));
        } else {
            f16x8* q = wunit + buf * LANES_BUF + jj * pstep;
            q[0] = __builtin_bit_cast(f16x8, sum);
            q[8 * LANES_UPITCH] = __builtin_bit_cast(f16x8, dif);
        }
    };

    {   // the zeros behind the window's last row (P.even, see the host)
        const int unit = tid & 15, entry = 256 + ((tid >> 4) & 7), buf = tid >> 7;
        lds16[buf * LANES_BUF + unit * LANES_UPITCH + entry] = f16x8{};
    }
    // prologue: the first chunk, the first taps' filters
#pragma unroll
    for (int i = 0; i < 8; ++i) load_stage(0, i);
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
            for (int s = 0; s < 2; ++s) X[tg][l][s] = load_a(l, s, tg);
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Y[0][l][s] = load_a(l, s, TG);
        }

    // window offset, output offset and validity of a pixel of the tile
    const float rcp_w = __builtin_amdgcn_rcpf(tall ? P.Wout : P.TW), rcp_h = __builtin_amdgcn_rcpf(tall ? P.in.tall : P.TH * P.TW);
    auto decode = [&](int pix, int& off, long& oaddr) -> bool {
        int n, ho, wo;
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
        oaddr = CL ? (((long)n * P.Hout + ho) * P.Wout + wo) * P.CoutS : ((long)n * P.CoutS * P.Hout + ho) * P.Wout + wo;
        return valid;
    };
    int poff[NPT];
#pragma unroll
    for (int t = 0; t < NPT; ++t) {
        long unused;
        decode(t * 32 + j, poff[t], unused);
        poff[t] = (poff[t] + colshift + (kk * 4 + wave) * LANES_UPITCH) * 16;  // bytes into a chunk buffer: the wave's sum lane, pack kk
    }

    // [lane][filter sub-tile][pixel tile]; rows = pixels, columns = output channels (channels-last: the other way round), so
    // that a register quad is four consecutive elements of the output's memory order
    f32x16 acc[2][2][NPT];
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int t = 0; t < NPT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[l][s][t][r] = 0.f;

#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int t = 0; t < NPT; ++t) asm volatile("" : "+a"(acc[l][s][t]));  // (cleared while the loads are on their way)
    if (any_careful) fill_careful(0);
#pragma unroll
    for (int jj = 0; jj < 8; ++jj)
#pragma unroll
        for (int piece = 0; piece < 5; ++piece) slice(jj, piece, 0, 0);
    wg_barrier_no_vmem_wait();

    unsigned int addr[NPT], next[NPT];
    unsigned int xcur = 0;  // bytes to the current chunk buffer
    auto address = [&](int off, int t) { return poff[t] + (xcur + off * 16); };
    auto read_b = [&](unsigned int a, int l) {
        return *reinterpret_cast<const f16x8*>(reinterpret_cast<const char*>(lds16) + a + l * (8 * LANES_UPITCH * 16));
    };

    // One group of three taps.  PH 1: a chunk's first, with the requests for the second group's filters and for the next
    // chunk's activations; PH 0: products alone; PH 2: a chunk's last but one, PH 3 its last, which request the next chunk's
    // first filters; the last four taps stage the next chunk, one position per half tap.  A half tap is one lane's
    // products; its operands are requested during the half before (a chunk's first: behind the barrier).
    int tap = 0, kh = 0, kw = 0;
    auto group = [&](auto phase, int chan_next, int buf_next) {
        constexpr int PH = decltype(phase)::value;
        constexpr int MF = 2 * NPT;  // products of a half tap
#pragma unroll
        for (int tg = 0; tg < TG; ++tg) {
            ++tap;
            if (++kw == P.Kw) { kw = 0; ++kh; }
            const int off = tap < P.taps ? kh * P.dh * P.HTW + kw * P.dw : 0;  // (of the next tap; padded taps have zero filters)
            const bool last = PH == 3 && tg == TG - 1;
            if constexpr (PH == 2) {
                if (tg == TG - 1) {
                    if (any_careful) fill_careful(chan_next);
#pragma unroll
                    for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(stage[i]));  // (the staging stays between the products)
                }
            }
#pragma unroll
            for (int l = 0; l < 2; ++l) {
#pragma unroll
                for (int m = 0; m < MF; ++m) {
                    const int t = m >> 1, s = m & 1;
                    const f16x8 a = PH == 1 ? X[tg][l][s] : Y[tg][l][s];
                    if constexpr (CL) acc[l][s][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, B[l][t], acc[l][s][t], 0, 0, 0);
                    else acc[l][s][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(B[l][t], a, acc[l][s][t], 0, 0, 0);
                    const int g = (tg * 2 + l) * MF + m;
                    if (l == 0) {
                        if (m < NPT) B[1][m] = read_b(addr[m], 1);
                        else if (!last) next[m - NPT] = address(off, m - NPT);
                    } else {
                        if (m < NPT && !last) B[0][m] = read_b(next[m], 0);
                    }
                    // Requests to memory: at most one per two products, or the four waves' requests queue up in front of
                    // the CU's cache and hold up the products.  (wstep moves on with the taps.)
                    constexpr int W = NPT == 4 ? 3 : 1;  // products from one to the next
                    if constexpr (PH == 1) {
                        // the second group's filters of tap 1, the next chunk's activations, the filters of tap 2
                        const int x = g % W == 0 ? g / W : 16;
                        if (x < 4) Y[1][x >> 1][x & 1] = load_a(x >> 1, x & 1, TG + 1 - tg);
                        else if (x < 12) load_stage(chan_next, x - 4);
                        else if (x < 16) Y[2][(x >> 1) & 1][x & 1] = load_a((x >> 1) & 1, x & 1, TG + 2 - tg);
                    } else if constexpr (PH == 3) {
                        // the next chunk's first group, and the first tap of its second one (whose slot is free by then)
                        const int x = g % W == 0 ? g / W : 16;
                        if (x < 12) X[x >> 2][(x >> 1) & 1][x & 1] = load_a((x >> 1) & 1, x & 1, TG - tg + (x >> 2));
                        else if (x < 16) Y[0][(x >> 1) & 1][x & 1] = load_a((x >> 1) & 1, x & 1, TG - tg + (x >> 2));
                    } else {
                        // the next group's: a slot is free once its last product is issued
                        if (l == 0 && tg > 0 && (m == 1 || m == 3)) Y[tg - 1][1][m >> 1] = load_a(1, m >> 1, TG - 1);
                        if (l == 1 && (m == 1 || m == 3)) Y[tg][0][m >> 1] = load_a(0, m >> 1, TG);
                        if (l == 1 && tg == TG - 1 && m == MF - 1) {
                            Y[tg][1][0] = load_a(1, 0, TG);
                            Y[tg][1][1] = load_a(1, 1, TG);
                        }
                    }
                    if constexpr (PH >= 2) {
                        const int half = PH == 2 ? (tg - TG + 1) * 2 + l : (tg + 1) * 2 + l;  // of the last four taps
                        if (half >= 0) {
                            if (NPT == 4 && m < 5) slice(half, m, chan_next, buf_next);
                            if (NPT == 2 && m < 3) {
                                slice(half, 2 * m, chan_next, buf_next);
                                if (m < 2) slice(half, 2 * m + 1, chan_next, buf_next);
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            wstep += LANES_STEP * 16;
#pragma unroll
            for (int t = 0; t < NPT; ++t) addr[t] = next[t];
#pragma unroll
            for (int l = 0; l < 2; ++l)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int t = 0; t < NPT; ++t) asm volatile("" : "+a"(acc[l][s][t]));
        }
    };

    int cur = 0;
    for (int chunk = 0; chunk < P.nchunks; ++chunk) {
        xcur = cur * (LANES_BUF * 16);
        const int buf_next = cur ^ 1;
        const int chan_next = (chunk + 1) * CK;  // (behind the last chunk: loads from the tensor's first bytes, into a buffer nobody reads)
#pragma unroll
        for (int t = 0; t < NPT; ++t) {
            addr[t] = address(0, t);
            next[t] = addr[t];
            B[0][t] = read_b(addr[t], 0);
        }
        tap = 0; kh = 0; kw = 0;
        PHX_STAMP(0)
        group(std::integral_constant<int, 1>{}, chan_next, buf_next);
        PHX_STAMP(1)
        for (int g = 3; g < ngroups; ++g) group(std::integral_constant<int, 0>{}, chan_next, buf_next);
        group(std::integral_constant<int, 2>{}, chan_next, buf_next);
        PHX_STAMP(2)
        group(std::integral_constant<int, 3>{}, chan_next, buf_next);
        PHX_STAMP(3)
        wg_barrier_no_vmem_wait();
        PHX_STAMP(4)
        cur ^= 1;
    }

    // Epilogue, one round per filter sub-tile: the waves' product lanes meet in LDS and are read back eight elements of the
    // output's memory order at a time, merged and stored as 16 bytes.
    float* const xch = reinterpret_cast<float*>(lds16);
    _Float16* const out = static_cast<_Float16*>(P.out);
    const _Float16* const bias = static_cast<const _Float16*>(P.bias);
    const long plane_out = (long)P.Hout * P.Wout;
    // [product lane][32 channels][PX pixels + 4], channels-last [product lane][PX pixels][32 channels + 4]
    constexpr int PITCH = CL ? 36 : PX + 4;
    constexpr int SLAB = (CL ? PX : 32) * PITCH;
    constexpr int GR = CL ? 4 : PX / 8;                // groups of eight elements side by side
    constexpr int ROWS = WG_THREADS / GR;              // rows the threads cover at once
    const int g8 = tid % GR, row0 = tid / GR;
    long o8[2] = {0, 0};         // offset of the two halves of the group (planes: the same for every channel)
    bool run8 = false, run4[2] = {false, false};
    if constexpr (!CL) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int off;
            long end;
            const bool a = decode(g8 * 8 + 4 * h, off, o8[h]), b = decode(g8 * 8 + 4 * h + 3, off, end);
            run4[h] = a && b && end == o8[h] + 3;
        }
        run8 = run4[0] && run4[1] && o8[1] == o8[0] + 4;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (s > 0) wg_barrier_no_vmem_wait();  // the previous round has been read
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            float* const dst = xch + lanes_product(wave, l) * SLAB;
#pragma unroll
            for (int t = 0; t < NPT; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x16& a = acc[l][s][t];
                    // (planes: the two halves of a group trade places in every other 64 pixels: the sixteen groups that are
                    // read at once then fill all banks)
                    *reinterpret_cast<f32x4*>(dst + (CL ? (t * 32 + j) * PITCH + 8 * g + 4 * kk : j * PITCH + t * 32 + 8 * g + 4 * (kk ^ (t >> 1)))) =
                        f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
                }
        }
        wg_barrier_no_vmem_wait();
#pragma unroll
        for (int pass = 0; pass < (CL ? PX : 32) / ROWS; ++pass) {
            const int r = row0 + pass * ROWS;
            f32x4 lanes[8][2];
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) 
                    lanes[i][h] = *reinterpret_cast<const f32x4*>(xch + i * SLAB + r * PITCH + g8 * 8 + 4 * (CL ? h : h ^ (g8 >> 3)));
            const int co = (ct * 2 + s) * 32 + (CL ? g8 * 8 : r);
            if (co >= P.Cout) continue;
            float c[8][4];
            f16x8 y[4];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float in[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) in[i] = lanes[i][e >> 2][e & 3];
                merge_output(in, c[e]);
            }
            if (bias) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 8; ++e) c[e][q] += (float)bias[q * P.CoutS + co + (CL ? e : 0)];
            }
            if constexpr (NORM && !CL) {
                const f32x4 f = factors[s * 32 + r];
                const _Float16* const res = static_cast<const _Float16*>(P0.norm.res);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) c[e][q] = norm_result<_Float16>(f, c[e][q]);
                    if (res) {
                        f16x8 rv = {};
                        const long at = q * P.out_cs + co * plane_out;
                        if (run8) {
                            rv = __builtin_bit_cast(f16x8, load16_a2(res + at + o8[0]));
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                int off;
                                long o;
                                if (decode(g8 * 8 + e, off, o)) rv[e] = res[at + o];
                            }
                        }
#pragma unroll
                        for (int e = 0; e < 8; ++e) c[e][q] += (float)rv[e];
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) c[e][q] = relu_if(P0.norm.relu, c[e][q]);
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 8; ++e) y[q][e] = (_Float16)c[e][q];
            if constexpr (CL) {
                int off;
                if (decode(r, off, o8[0])) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<u32x4_a2*>(out + q * P.out_cs + o8[0] + co) = __builtin_bit_cast(u32x4, y[q]);
                }
            } else if (run8) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<u32x4_a2*>(out + q * P.out_cs + o8[0] + co * plane_out) = __builtin_bit_cast(u32x4, y[q]);
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (run4[h]) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const u32x4 w = __builtin_bit_cast(u32x4, y[q]);
                            *reinterpret_cast<u32x2_a2*>(out + q * P.out_cs + o8[h] + co * plane_out) = u32x2{w[2 * h], w[2 * h + 1]};
                        }
                    } else {
#pragma unroll
                        for (int e = 4 * h; e < 4 * h + 4; ++e) {
                            int off;
                            long o;
                            if (decode(g8 * 8 + e, off, o)) {
#pragma unroll
                                for (int q = 0; q < 4; ++q) out[q * P.out_cs + o + co * plane_out] = y[q][e];
                            }
                        }
                    }
                }
            }
        }
    }
    PHX_STAMP(5)
    PHX_PHASES_REPORT("fwd_f16_lanes: start + first operands / loads group / staging group / last group / barrier / epilogue", 6)
}

// Filter packing: [filter tile of 64][wave][chunk][tap, padded to whole groups][lane of the wave][sub-tile][64] x 8 halves
// (conjugated / mirrored / transposed for MAP_DGRAD, lanes formed in fp32 and rounded once).  One thread per (tile, chunk,
// tap, sub-tile, MFMA lane, channel of the pack): eight product lanes from the same four filter values.
struct PackLanesArgs {
    PackArgs base;  // row_tiles: tiles of 64 output channels
    int taps3;      // taps padded to whole groups
};

template <int MAP>
__device__ __forceinline__ void pack_filters_lanes_body(const PackLanesArgs& A, long first, long stride) {
    const PackArgs& P = A.base;
    const int taps = P.Kh * P.Kw;
    const long total = (long)P.row_tiles * P.nchunks * A.taps3 * 2 * 64 * 8;
    const _Float16* w = static_cast<const _Float16*>(P.w);
    _Float16* outh = static_cast<_Float16*>(P.out);
    for (long idx = first; idx < total; idx += stride) {
        const int i = idx & 7, lane = (idx >> 3) & 63, sub = (idx >> 9) & 1;
        long s = idx >> 10;
        const int tap = s % A.taps3; s /= A.taps3;
        const int chunk = s % P.nchunks;
        const int tile = s / P.nchunks;
        const int row = (tile * 2 + sub) * 32 + (lane & 31);
        const int red = chunk * F16_CK + (lane >> 5) * 8 + i;
        float R[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (tap < taps && row < P.rows && red < P.red) {
            int kh = tap / P.Kw, kw = tap - kh * P.Kw;
            if (MAP == MAP_DGRAD) { kh = P.khm - kh * P.khs; kw = P.kwm - kw * P.kws; }
            const int o = (MAP == MAP_DGRAD) ? red : row;
            const int in = (MAP == MAP_DGRAD) ? row : red;
            const long off = o * P.so + in * P.si + kh * P.skh + kw * P.skw;
            float wv[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) wv[c] = ((MAP == MAP_DGRAD && c > 0) ? -1.f : 1.f) * (float)w[c * P.wcs + off];
            lanes_right(wv, R);
        }
        const long step = (long)chunk * A.taps3 + tap;
#pragma unroll
        for (int wave = 0; wave < 4; ++wave)
#pragma unroll
            for (int l = 0; l < 2; ++l) {
                const float r = R[lanes_product(wave, l)];
                const long vec = (((long)(tile * 4 + wave) * P.nchunks * A.taps3 + step) * 4 + l * 2 + sub) * 64 + lane;
                outh[vec * 8 + i] = (_Float16)(lanes_negated(wave, l) ? -r : r);
            }
    }
}

template <int MAP>
__global__ void __launch_bounds__(WG_THREADS) pack_filters_lanes_kernel(const PackLanesArgs A0) {
    PackLanesArgs A = A0;
    A.base = group_view(A0.base);
    pack_filters_lanes_body<MAP>(A, (long)blockIdx.x * blockDim.x + threadIdx.x, (long)gridDim.x * blockDim.x);
}

}  // namespace phx
