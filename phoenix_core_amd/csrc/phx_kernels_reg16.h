// fp16 convolutions of few output tiles (small batches, small images): 16-product kernel whose operands go from memory to
// registers without LDS.
#pragma once

#include "phx_kernels_f32.h"

namespace phx {

// A layer of a few hundred to some thousand output pixels is a handful of workgroups of the LDS kernels, and each of them
// waits a dozen times for a staged chunk and a barrier: 13-20 us whatever the layer's arithmetic, of which the whole chip would
// make half a microsecond.  Here a WAVE is on its own: it owns 16 pairs of neighbouring output pixels x 16 output channels x the
// four components (eight 16x16 accumulator tiles), loads the activations of a whole filter row of a chunk of 32 input channels
// straight into registers, forms the operands of all its taps from them with one byte permutation a register, and multiplies.
// 1 to 8 waves (KS) share a tile, each taking every KS-th (chunk, filter row) of its reduction, and add their accumulators
// through LDS once at the end; Z workgroups can share it through fp32 partial sums.  So a small problem becomes a thousand waves
// that each wait for memory a few times.
//
// Operands.  Channels-first: lane (pair r, channel group kg) loads, for each of its eight channels, the SPAN pixels that the pair
// reads under a filter row, one load of 4, 8 or 16 bytes; tap kw of pixel e is pixel kw * D + e * S of it, and the operand
// register of channels (2m, 2m+1) is one v_perm of the two channels' registers.  What is padding gets a permutation that selects
// zeros.  Channels-last: a pixel's eight channels are one 16-byte load, the operand itself; each pixel of the span is loaded
// once for all taps.  Filters are packed in operand order (pack_filters_reg_body).
// At unit stride and equal widths the pairs go through the plane's pixels regardless of its rows (the input pixel of output
// pixel q is q + a constant under each tap); otherwise each row has its own pairs.
struct RegArgs {
    const _Float16* in;
    long in_cs;             // elements between input components
    const f16x8* wpk;
    const _Float16* bias;   // [4][Cout] or null
    _Float16* out;
    long out_cs;
    float* partial;         // Z > 1: [Z][elements of out], else null
    const _Float16* addend; // input gradient: a tensor laid out like out that is added to the rounded result, or null
    int N, Cin, Cout, Hin, Win, Hout, Wout;
    int Kh, sh, dh, pt, pl;
    int flat;               // pairs go through the whole plane
    int rpr, tpi;           // pairs of an output row; tiles of a plane
    int tiles, co_tiles, items;  // pixel tiles (N * tpi); output-channel tiles; (chunk, filter row) steps of the reduction
    int kslog;              // log2 of the waves that share a tile
    int Z, zitems;          // workgroups that share a tile, and the items of each
};
struct RegNormArgs : RegArgs {
    NormArgs norm;
};
// The phases of a strided input gradient in one launch: the results whose row is oh and whose column ow modulo the stride, a unit-
// stride correlation of the gradient with the filter's taps that reach them.  Each phase has tiles of its own and writes its
// results where they belong; one that no tap reaches writes zeros (and the addend).
constexpr int REG_PHASES_MAX = 4;
struct RegPhase {
    int first;              // its first tile
    int Kh, kw, dh, pt, pl; // filter rows; taps of a row (at most the kernel's, those behind them are zero); as in RegArgs
    int Hout, Wout;         // its results
    int oh, ow;             // ... and where they lie
    int flat, rpr, tpi, items, zitems;
    int image;              // its packed filters, 16-byte vectors behind the first one's
};
struct RegPhaseArgs : RegArgs {
    RegPhase phase[REG_PHASES_MAX];
    int phases, step_h, step_w;  // and the strides; Hout, Wout: the whole result
};
template <bool NORM, bool PHASE = false>
using RegArgsOf = std::conditional_t<PHASE, RegPhaseArgs, std::conditional_t<NORM, RegNormArgs, RegArgs>>;

// Pixels that a pair reads under a filter row, as a power of two.  (Memory bounds a CU: its L1 hands out some 30 bytes a clock
// of these loads.  Runs of four pixels with 16-byte loads measured the same rate per pixel, 0.84 against 0.76 us for the 3x3
// items of four pixels on a CU, with twice the start-up and half the waves.)
constexpr int REG_PX = 2;
constexpr int reg_span(int kw, int d, int s) { return (kw - 1) * d + s + 1 <= 2 ? 2 : (kw - 1) * d + s + 1 <= 4 ? 4 : 8; }
constexpr int REG_TM = 16;     // pairs and output channels of a wave's tile
constexpr int REG_CK = 32;     // input channels of a chunk
constexpr int REG_SUMS = 32;   // a wave's accumulators per lane: 4 components x 2 pixels x 4 rows
constexpr size_t REG_WAVE_LDS = REG_SUMS * 64 * sizeof(float);
constexpr int reg_waves(int kw) { return kw <= 3 ? 8 : 4; }  // most waves of a workgroup: 256 or 512 registers a wave

template <int W>
struct RegWords {
    unsigned int v[W];
};

// W words from an address with 2-byte alignment
template <int W>
__device__ __forceinline__ RegWords<W> reg_load(const char* base, unsigned int off) {
    RegWords<W> r;
    const _Float16* p = reinterpret_cast<const _Float16*>(base + off);
    if constexpr (W == 1) {
        r.v[0] = load4_a2(p);
    } else if constexpr (W == 2) {
        const u32x2 t = load8_a2(p);
        r.v[0] = t[0]; r.v[1] = t[1];
    } else {
        const u32x4 t = load16_a2(p);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.v[i] = t[i];
    }
    return r;
}

// the halves of r from place n on, moved to place 0 (n < 0: moved up by -n places); zeros take the places left
template <int W>
__device__ __forceinline__ RegWords<W> reg_shift(const RegWords<W>& a, int n) {
    RegWords<W> r;
    const int down = n > 0 ? 16 * n : 0, up = n < 0 ? -16 * n : 0;
    if constexpr (W == 1) {
        r.v[0] = (a.v[0] >> down) << up;
    } else if constexpr (W == 2) {
        const unsigned long long t = (((unsigned long long)a.v[1] << 32 | a.v[0]) >> down) << up;
        r.v[0] = (unsigned int)t; r.v[1] = (unsigned int)(t >> 32);
    } else {
        unsigned __int128 t = 0;
#pragma unroll
        for (int i = W - 1; i >= 0; --i) t = t << 32 | a.v[i];
        t = (t >> down) << up;
#pragma unroll
        for (int i = 0; i < W; ++i) r.v[i] = (unsigned int)(t >> (32 * i));
    }
    return r;
}

// KW taps a filter row, dilation D and stride S along the row; CL: channels-last tensors; PHASE: see RegPhase
template <int KW, int D, int S, bool CL, bool NORM, bool PHASE = false>
__global__ void __launch_bounds__(64 * reg_waves(KW)) qconv_reg_f16_kernel(const RegArgsOf<NORM, PHASE> P0) {
    static_assert(!(CL && NORM) && !(PHASE && NORM), "channels-last passes and input gradients take no norm");
    [[maybe_unused]] RegArgs one;  // (PHASE: this tile's phase as a correlation of its own)
    [[maybe_unused]] RegPhase phase;
    const auto& P = [&]() -> const auto& {
        if constexpr (PHASE) return one;
        else return P0;
    }();
    if constexpr (PHASE) one = P0;
    constexpr int PX = REG_PX, SPAN = reg_span(KW, D, S);
    constexpr int W = CL ? 4 : SPAN / 2;                  // words of a load
    constexpr int NL = CL ? (KW - 1) * D + (PX - 1) * S + 1 : 8;     // loads of a component's part of an item
    extern __shared__ float red[];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int KS = 1 << P.kslog;
    const int rank = wave & (KS - 1);
    const int subs = ((int)blockDim.x >> 6) >> P.kslog;   // tiles of a workgroup

    const int wg = xcd_remap(blockIdx.x, gridDim.x);
    const int co_t = wg % P.co_tiles;
    const int rest = wg / P.co_tiles;
    const int groups = (P.tiles + subs - 1) / subs;
    const int z = rest / groups;
    int tile = (rest - z * groups) * subs + (wave >> P.kslog);
    const bool live = tile < P.tiles;
    if constexpr (PHASE) {
        int which = 0;
#pragma unroll
        for (int i = 1; i < REG_PHASES_MAX; ++i)
            if (live && i < P0.phases && tile >= P0.phase[i].first) which = i;
        phase = P0.phase[which];
        tile -= phase.first;
        one.Kh = phase.Kh; one.dh = phase.dh; one.pt = phase.pt; one.pl = phase.pl;
        one.Hout = phase.Hout; one.Wout = phase.Wout;
        one.flat = phase.flat; one.rpr = phase.rpr; one.tpi = phase.tpi; one.items = phase.items; one.zitems = phase.zitems;
        one.wpk += phase.image;
    }
    const int img = live ? tile / P.tpi : 0;
    const int first_pair = (tile - img * P.tpi) * REG_TM;
    const int pair = first_pair + r;

    // the pair's pixels: (ho[e], wo[e]), q0 the first one's place in the plane
    const int HWin = P.Hin * P.Win, HWout = P0.Hout * P0.Wout;  // (PHASE: of the whole result)
    auto pixel = [&](int h, int w) __attribute__((always_inline)) {  // a result's place in its plane
        if constexpr (PHASE) return (h * P0.step_h + phase.oh) * P0.Wout + w * P0.step_w + phase.ow;
        else return h * P0.Wout + w;
    };
    int ho[PX], wo[PX];
    bool ok[PX];
    const int per_row = P.flat ? P.Wout : P.rpr * PX;  // pixels of a row as the pairs count them
    ho[0] = pair * PX / per_row; wo[0] = pair * PX - ho[0] * per_row;
    const int q0 = ho[0] * P.Wout + wo[0];
#pragma unroll
    for (int e = 1; e < PX; ++e) {
        const bool wrap = P.flat && wo[e - 1] + 1 == P.Wout;
        ho[e] = ho[e - 1] + wrap;
        wo[e] = wrap ? 0 : wo[e - 1] + 1;
    }
    unsigned int cols[PX];  // bit kw: the tap's column lies in the image
#pragma unroll
    for (int e = 0; e < PX; ++e) {
        ok[e] = live && ho[e] < P.Hout && wo[e] < P.Wout;
        cols[e] = 0;
#pragma unroll
        for (int kw = 0; kw < KW; ++kw) {
            const int iw = wo[e] * S - P.pl + kw * D;
            if (ok[e] && iw >= 0 && iw < P.Win && (!PHASE || kw < phase.kw)) cols[e] |= 1u << kw;
        }
    }

    f32x4 acc[4][PX];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < PX; ++e) acc[q][e] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int first = z * P.zitems + rank, last = min(P.items, (z + 1) * P.zitems);
    // (byte offsets are unsigned and start SPAN pixels in front of the tensor: a span may start in front of its plane)
    constexpr int LEAD = CL ? 0 : SPAN;
    const char* in = reinterpret_cast<const char*>(P.in + (long)img * P.Cin * HWin - LEAD);
    const unsigned int comp_bytes = (unsigned int)(P.in_cs * 2), plane_bytes = (unsigned int)HWin * 2;

    RegWords<W> act[4][NL];
    f16x8 filt[KW][4];
    // what an item's loads need of this lane
    struct Item {
        int start;             // the span's first pixel, in the planes' pixel sequence
        int base, dup;         // the lane's first channel; how many of its eight belong to the group before it (last chunk)
        unsigned int taps[PX]; // the taps of each pixel that are not padding
        int moved;             // pixels by which a span that leaves the tensor is moved back inside
    };
    auto locate = [&](int item) {
        Item it;
        const int chunk = item / P.Kh, kh = item - chunk * P.Kh;
        const int want = chunk * REG_CK + kg * 8;
        it.base = min(want, P.Cin - 8);
        it.dup = want - it.base;
        it.moved = 0;
        unsigned int any = 0;
#pragma unroll
        for (int e = 0; e < PX; ++e) {
            const int ih = ho[e] * P.sh - P.pt + kh * P.dh;
            it.taps[e] = (ih >= 0 && ih < P.Hin) ? cols[e] : 0u;
            any |= it.taps[e];
        }
        const int o = (ho[0] * P.sh - P.pt + kh * P.dh) * P.Win + wo[0] * S - P.pl;
        it.start = any ? o : 0;
        if constexpr (!CL) {
            // (a span that sticks out of its plane reads its neighbours', which nothing selects; only in front of the first plane of
            // the tensor and behind the last one there are none: load_act moves the spans of those two)
            if ((it.start < 0 && it.base == 0 && img == 0) || (it.start + SPAN > HWin && it.base + 8 == P.Cin && img == P.N - 1))
                it.moved = it.start - min(max(it.start, 0), HWin - SPAN);
        }
        return it;
    };
    auto load_act = [&](const Item& it, int p) {
        if constexpr (CL) {
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                // the pixel is read where a tap of either pixel selects it
                bool use = false;
#pragma unroll
                for (int e = 0; e < PX; ++e)
#pragma unroll
                    for (int kw = 0; kw < KW; ++kw)
                        if (kw * D + e * S == j) use = use || ((it.taps[e] >> kw) & 1u);
                act[p][j] = reg_load<W>(in, p * comp_bytes + (unsigned int)((use ? (it.start + j) * P.Cin : 0) + it.base) * 2u);
            }
        } else {
            const unsigned int off = p * comp_bytes + (unsigned int)(it.base * HWin + it.start + LEAD) * 2u;
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                const bool end = (p == 0 && j == 0 && it.moved < 0) || (p == 3 && j == 7 && it.moved > 0);
                act[p][j] = reg_load<W>(in, off + j * plane_bytes - (end ? it.moved * 2 : 0));
            }
        }
    };
    const f16x8* wbase = P.wpk + (long)co_t * P.items * (KW * 4 * 64) + lane;
    auto load_filter = [&](int item, int kw) {
#pragma unroll
        for (int w = 0; w < 4; ++w) filt[kw][w] = wbase[((long)item * KW + kw) * (4 * 64) + w * 64];
    };

    // rare corrections of loaded activations, behind branches that whole waves take or skip
    auto correct = [&](const Item& it) {
        if constexpr (!CL) {
            if (__any(it.moved != 0)) {
                act[0][0] = reg_shift<W>(act[0][0], min(it.moved, 0));
                act[3][7] = reg_shift<W>(act[3][7], max(it.moved, 0));
            }
        }
        if (__any(it.dup != 0)) {
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int j = 0; j < NL; ++j) {
                    if constexpr (CL) {
                        const u32x4 keep = expand_half_mask(0xFFu << min(it.dup, 8));
#pragma unroll
                        for (int i = 0; i < W; ++i) act[p][j].v[i] &= keep[i];
                    } else {
#pragma unroll
                        for (int i = 0; i < W; ++i) act[p][j].v[i] = j < it.dup ? 0u : act[p][j].v[i];
                    }
                }
        }
    };

    auto operand = [&](const Item& it, int p, int kw, int e) -> f16x8 {
        u32x4 x;
        const int at = kw * D + e * S;
        const bool on = (it.taps[e] >> kw) & 1u;
        if constexpr (CL) {
#pragma unroll
            for (int m = 0; m < 4; ++m) x[m] = on ? act[p][at].v[m] : 0u;
        } else {
            const unsigned int sel = on ? ((at & 1) ? 0x07060302u : 0x05040100u) : 0x0C0C0C0Cu;
#pragma unroll
            for (int m = 0; m < 4; ++m) x[m] = __builtin_amdgcn_perm(act[p][2 * m + 1].v[at / 2], act[p][2 * m].v[at / 2], sel);
        }
        return __builtin_bit_cast(f16x8, x);
    };

    if (live && first < last) {
        Item it = locate(first);
#pragma unroll
        for (int p = 0; p < 4; ++p) load_act(it, p);
#pragma unroll
        for (int kw = 0; kw < KW; ++kw) load_filter(first, kw);
        for (int item = first; item < last; item += KS) {
            correct(it);
            // a component's activations of the next item are loaded into the registers that its last product has left
            const bool more = item + KS < last;
            const Item nit = more ? locate(item + KS) : it;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
#pragma unroll
                for (int kw = 0; kw < KW; ++kw) {
                    f16x8 x[PX];
#pragma unroll
                    for (int e = 0; e < PX; ++e) x[e] = operand(it, p, kw, e);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const f16x8 w = qneg(p, q) ? neg8(filt[kw][p ^ q]) : filt[kw][p ^ q];
#pragma unroll
                        for (int e = 0; e < PX; ++e)
                            acc[q][e] = CL ? __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x[e], acc[q][e], 0, 0, 0)
                                           : __builtin_amdgcn_mfma_f32_16x16x32_f16(x[e], w, acc[q][e], 0, 0, 0);
                    }
                    if (p == 3 && more) load_filter(item + KS, kw);
                }
                if (more) load_act(nit, p);
            }
            it = nit;
        }
    }

    // The waves of a tile add their sums.  Wave `rank` finishes the components q with q % min(KS, 4) == rank % 4 and, of eight
    // waves, the rows i0 and i0 + 1 of them.
    const int qmask = min(KS, 4) - 1;
    const int i0 = reg_waves(KW) > 4 && KS > 4 ? (rank >> 2) * 2 : 0;
    const float* sums = red + (wave - rank) * (REG_SUMS * 64) + lane;
    if (KS > 1) {
        float* mine = red + wave * (REG_SUMS * 64) + lane;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < PX; ++e)
#pragma unroll
                for (int i = 0; i < 4; ++i) mine[((q * PX + e) * 4 + i) * 64] = acc[q][e][i];
        __syncthreads();
    }
    if (!live) return;

    // Row 4 kg + i, column r of a tile; channels-first the rows are pairs, channels-last output channels.  NI of the rows: v[PX i + e].
    const long elements = 4 * P.out_cs;
    typedef float sums_t __attribute__((ext_vector_type(4 * PX)));
    auto finish = [&](auto ni, int q, const sums_t v) __attribute__((always_inline)) {
        constexpr int NI = decltype(ni)::value;
        if constexpr (CL) {
            const int co = co_t * REG_TM + 4 * kg + i0;
#pragma unroll
            for (int e = 0; e < PX; ++e) {
                if (!ok[e]) continue;
                const long at = q * P.out_cs + ((long)img * HWout + (PHASE ? pixel(ho[e], wo[e]) : q0 + e)) * P.Cout + co;
                _Float16 h[NI];
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    if (co + i >= P.Cout) continue;
                    if (P.partial) { P.partial[z * elements + at + i] = v[PX * i + e]; continue; }
                    h[i] = (_Float16)(v[PX * i + e] + (P.bias ? (float)P.bias[q * P.Cout + co + i] : 0.f));
                    if (P.addend) h[i] = (_Float16)((float)h[i] + (float)P.addend[at + i]);
                }
                if (P.partial) continue;
                typedef _Float16 run_t __attribute__((ext_vector_type(NI), aligned(2)));
                if (NI > 1 && co + NI <= P.Cout) {
                    run_t t;
#pragma unroll
                    for (int i = 0; i < NI; ++i) t[i] = h[i];
                    *reinterpret_cast<run_t*>(P.out + at) = t;
                } else {
#pragma unroll
                    for (int i = 0; i < NI; ++i)
                        if (co + i < P.Cout) P.out[at + i] = h[i];
                }
            }
        } else {
            const int co = co_t * REG_TM + r;
            if (co >= P.Cout) return;
            const long plane = q * P.out_cs + ((long)img * P.Cout + co) * HWout;
            const float b = P.bias ? (float)P.bias[q * P.Cout + co] : 0.f;
            [[maybe_unused]] f32x4 nf;
            [[maybe_unused]] NormTail tail;
            const _Float16* more = P.addend;
            if constexpr (NORM) {
                tail = norm_tail_of(P.norm);
                nf = norm_factors(P.norm, co);
                more = static_cast<const _Float16*>(P.norm.res);
            }
            auto result = [&](float sum, float other) __attribute__((always_inline)) {
                float o = sum + b;
                if constexpr (NORM) {
                    o = norm_half(nf, (_Float16)o, tail);
                    if (more) o = __builtin_fmaf((float)other, tail.one, o);
                    return (_Float16)relu_at(tail, o);
                } else {
                    const _Float16 h = (_Float16)o;
                    return more ? (_Float16)((float)h + other) : h;
                }
            };
            const int r0 = first_pair + 4 * kg + i0;  // the first of NI pairs
            // (rows of an odd number of pixels end in half a pair, unless the pairs go through the plane)
            const bool whole = !PHASE && (P.flat || P.Wout % PX == 0);  // (uniform)
            if (whole && PX * (r0 + NI) <= HWout) {
                const long at = plane + PX * r0;
                if (P.partial) {
                    typedef float part_t __attribute__((ext_vector_type(PX), aligned(4)));
#pragma unroll
                    for (int i = 0; i < NI; ++i) {
                        part_t t;
#pragma unroll
                        for (int e = 0; e < PX; ++e) t[e] = v[PX * i + e];
                        reinterpret_cast<part_t*>(P.partial + z * elements + at)[i] = t;
                    }
                    return;
                }
                constexpr int V = PX * NI < 8 ? PX * NI : 8;
                typedef _Float16 run_t __attribute__((ext_vector_type(V), aligned(2)));
#pragma unroll
                for (int g = 0; g < PX * NI / V; ++g) {
                    run_t h, other{};
                    if (more) other = reinterpret_cast<const run_t*>(more + at)[g];
#pragma unroll
                    for (int i = 0; i < V; ++i) h[i] = result(v[V * g + i], (float)other[i]);
                    reinterpret_cast<run_t*>(P.out + at)[g] = h;
                }
                return;
            }
            auto store = [&](int px, float sum) __attribute__((always_inline)) {
                const long at = plane + px;
                if (P.partial) P.partial[z * elements + at] = sum;
                else P.out[at] = result(sum, more ? (float)more[at] : 0.f);
            };
            if (whole) {
#pragma unroll
                for (int i = 0; i < PX * NI; ++i)
                    if (PX * r0 + i < HWout) store(PX * r0 + i, v[i]);
            } else {
                int row = PX * r0 / per_row, col = PX * r0 - row * per_row;
#pragma unroll
                for (int i = 0; i < PX * NI; ++i) {
                    if (row < P.Hout && col < P.Wout) store(pixel(row, col), v[i]);
                    if (++col == per_row) { col = 0; ++row; }
                }
            }
        }
    };
    auto finish_sums = [&](auto ni) __attribute__((always_inline)) {  // of the ranks, in their order
        constexpr int NI = decltype(ni)::value;
        for (int q = rank & qmask; q < 4; q += qmask + 1) {
            sums_t v = {};
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int e = 0; e < PX; ++e)
#pragma unroll
                    for (int i = 0; i < NI; ++i) v[PX * i + e] += sums[k * (REG_SUMS * 64) + ((q * PX + e) * 4 + i0 + i) * 64];
            finish(ni, q, v);
        }
    };
    if (KS == 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            sums_t v;
#pragma unroll
            for (int e = 0; e < PX; ++e)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[PX * i + e] = acc[q][e][i];
            finish(std::integral_constant<int, 4>{}, q, v);
        }
    } else if (reg_waves(KW) <= 4 || KS <= 4) {
        finish_sums(std::integral_constant<int, 4>{});
    } else if constexpr (reg_waves(KW) > 4) {
        finish_sums(std::integral_constant<int, 2>{});
    }
}

// Filter packing: one 16-byte vector per (output-channel tile, chunk, filter row, tap, component, lane); lane (row r,
// channel group kg) holds channels min(32 chunk + 8 kg, red - 8) .. + 7 of that row, zero where those belong to the group
// before it (the last chunk's groups are moved back to end at the last channel) and behind the last row.
template <int MAP>
__device__ __forceinline__ void pack_filters_reg_body(const PackArgs& P, long first, long stride) {
    const long total = (long)P.row_tiles * P.nchunks * P.Kh * P.Kw * 4 * 64;
    const _Float16* w = static_cast<const _Float16*>(P.w);
    f16x8* outv = reinterpret_cast<f16x8*>(P.out);
    for (long idx = first; idx < total; idx += stride) {
        const int lane = idx & 63;
        long s = idx >> 6;
        const int c = s & 3; s >>= 2;
        int kw = s % P.Kw; s /= P.Kw;
        int kh = s % P.Kh; s /= P.Kh;
        const int chunk = s % P.nchunks;
        const int row = (int)(s / P.nchunks) * REG_TM + (lane & 15);
        const int want = chunk * REG_CK + (lane >> 4) * 8, base = min(want, P.red - 8);
        if (MAP == MAP_DGRAD) {
            kh = P.khm - kh * P.khs;
            kw = P.kwm - kw * P.kws;  // (negative: a tap that the phase does not have)
        }
        const float sgn = (MAP == MAP_DGRAD && c > 0) ? -1.f : 1.f;
        const long at = c * P.wcs + kh * P.skh + kw * P.skw;
        f16x8 vec;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int red = base + i;
            float v = 0.f;
            if (row < P.rows && red >= want && kw >= 0) v = sgn * (float)w[at + (MAP == MAP_DGRAD ? red * P.so + row * P.si : row * P.so + red * P.si)];
            vec[i] = (_Float16)v;
        }
        outv[idx] = vec;
    }
}

}  // namespace phx
