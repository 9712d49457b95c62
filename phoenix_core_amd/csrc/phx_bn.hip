// Batch normalisation (+ optional residual and ReLU) over [rows, C, H*W] activations, training and evaluation: the
// entry points of include/phx_bn.h.  HBM-bound streaming kernels; a channel's rows are split over many workgroups and
// the per-split partial sums are combined in a fixed order, so results do not depend on scheduling.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>

#include "../../include/phx_bn.h"
#include "phx_device.h"
#include "phx_launch.h"

namespace phx {

struct BnArgs {
    const void* x;
    const void* dy;      // backward only
    const void* res;     // optional residual added in front of the ReLU (null = none)
    void* out;           // y (forward) or dx (backward)
    void* dres;          // backward with a residual: its gradient (the gradient behind the ReLU)
    const float* gamma;
    const float* beta;
    float* partial;      // [C][S][2]
    float* save_mean;
    float* save_invstd;
    float* run_mean;
    float* run_var;
    float* dgamma;
    float* dbeta;
    int rows, C, hw;
    int S, rows_per_split;  // splits of the row range per channel
    int nchunk;             // 16-byte chunks per (row, channel) plane, the last one possibly partial
    float eps, momentum;
    int relu;
    int total, per_split;   // bn_held_kernel: chunks of a channel and those of a split,
    int rows_step, chunks_step;  // a workgroup's threads' chunks as rows and what is left,
    int waits;              // how often a workgroup looks for its channel's other partial sums
};

template <typename TS>
struct Vec;
template <>
struct Vec<_Float16> {
    static constexpr int N = 8;
};
template <>
struct Vec<float> {
    static constexpr int N = 4;
};

// One 16-byte chunk of a plane as floats; elements past the end of the plane read as zero.  Planes of fp16
// tensors start at 2-byte alignment in general (odd H*W), which the 16-byte access tolerates.
template <typename TS>
__device__ __forceinline__ void load_chunk(const TS* p, int n, float (&v)[Vec<TS>::N]) {
    constexpr int V = Vec<TS>::N;
    if (n == V) {
        const u32x4 raw = load16_a2(reinterpret_cast<const _Float16*>(p));
        if constexpr (sizeof(TS) == 2) {
            const f16x8 h = __builtin_bit_cast(f16x8, raw);
#pragma unroll
            for (int i = 0; i < V; ++i) v[i] = (float)h[i];
        } else {
            const f32x4 f = __builtin_bit_cast(f32x4, raw);
#pragma unroll
            for (int i = 0; i < V; ++i) v[i] = f[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] = i < n ? (float)p[i] : 0.f;
    }
}

template <typename TS>
__device__ __forceinline__ void store_chunk(TS* p, int n, const float (&v)[Vec<TS>::N]) {
    constexpr int V = Vec<TS>::N;
    if (n == V) {
        u32x4 raw;
        if constexpr (sizeof(TS) == 2) {
            f16x8 h;
#pragma unroll
            for (int i = 0; i < V; ++i) h[i] = (_Float16)v[i];
            raw = __builtin_bit_cast(u32x4, h);
        } else {
            f32x4 f;
#pragma unroll
            for (int i = 0; i < V; ++i) f[i] = v[i];
            raw = __builtin_bit_cast(u32x4, f);
        }
        *reinterpret_cast<__attribute__((address_space(1))) u32x4_a2*>((__attribute__((address_space(1))) _Float16*)p) = raw;
    } else {
        for (int i = 0; i < n; ++i) p[i] = (TS)v[i];
    }
}

// Sum of two values over the workgroup (256 threads), result in every thread.
template <int T = 256>
__device__ __forceinline__ void wg_sum2(float& a, float& b, float (*red)[2]) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        a += __shfl_xor(a, off, 64);
        b += __shfl_xor(b, off, 64);
    }
    const int wave = threadIdx.x >> 6;
    __syncthreads();  // red may still be read from a previous use
    if ((threadIdx.x & 63) == 0) { red[wave][0] = a; red[wave][1] = b; }
    __syncthreads();
    a = red[0][0] + red[1][0] + red[2][0] + red[3][0];
    b = red[0][1] + red[1][1] + red[2][1] + red[3][1];
#pragma unroll
    for (int w = 4; w < T / 64; ++w) { a += red[w][0]; b += red[w][1]; }
}

// The channel's totals from its S partial pairs (fixed order inside the reduction tree).
__device__ __forceinline__ void channel_totals(const BnArgs& P, int c, float& t0, float& t1, float (*red)[2]) {
    t0 = 0.f; t1 = 0.f;
    if ((int)threadIdx.x < P.S) {
        t0 = P.partial[((long)c * P.S + threadIdx.x) * 2];
        t1 = P.partial[((long)c * P.S + threadIdx.x) * 2 + 1];
    }
    wg_sum2(t0, t1, red);
}

// MODE 0: sum (x - K), sum (x - K)^2 (forward statistics) with the shift K = the channel's first element: the
// variance is E[(x-K)^2] - E[x-K]^2 whatever K is, and with K inside the data's range the two terms are of the size
// of the variance itself -- the plain E[x^2] - E[x]^2 loses every significant bit of a channel whose mean is large
// against its spread (activations behind a ReLU or a residual add, in fp16).
// MODE 1: sum dy', sum dy' * xhat with dy' the gradient behind the optional ReLU (backward sums).
template <typename TS, int MODE>
__global__ void __launch_bounds__(256) bn_sums_kernel(const BnArgs P) {
    constexpr int V = Vec<TS>::N;
    __shared__ float red[4][2];
    const int c = blockIdx.x, s = blockIdx.y;
    const int b0 = s * P.rows_per_split;
    const int nb = min(P.rows_per_split, P.rows - b0);
    const TS* x = static_cast<const TS*>(P.x);
    const TS* dy = static_cast<const TS*>(P.dy);
    const TS* res = static_cast<const TS*>(P.res);
    float mean = 0.f, invstd = 0.f, g = 0.f, be = 0.f;
    if constexpr (MODE == 1) { mean = P.save_mean[c]; invstd = P.save_invstd[c]; g = P.gamma[c]; be = P.beta[c]; }
    const float shift = (MODE == 0) ? (float)x[(long)c * P.hw] : 0.f;
    float a0 = 0.f, a1 = 0.f;
    const int total = nb * P.nchunk;
    for (int idx = threadIdx.x; idx < total; idx += 256) {
        const int b = idx / P.nchunk, ch = idx - b * P.nchunk;
        long off = ((long)(b0 + b) * P.C + c) * P.hw + ch * V;
        int n = min(V, P.hw - ch * V);
        // The last chunk of a plane that is not a whole number of chunks is read as the full chunk that ENDS at the
        // plane's end (one 16-byte load like the others, no element-wise path that every lane of the wave would walk
        // through); its first `seen` elements belong to the chunk before and are left out of the sums.
        int seen = 0;
        if (n < V && P.hw >= V) { seen = V - n; off -= seen; n = V; }
        float xv[V];
        load_chunk<TS>(x + off, n, xv);
        if constexpr (MODE == 0) {
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const float d = (i < n && i >= seen) ? xv[i] - shift : 0.f;
                a0 += d;
                a1 += d * d;
            }
        } else {
            float dv[V], rv[V];
            load_chunk<TS>(dy + off, n, dv);
            if (res) load_chunk<TS>(res + off, n, rv);
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const float xh = (xv[i] - mean) * invstd;
                const float dm = (P.relu && g * xh + be + (res ? rv[i] : 0.f) <= 0.f) ? 0.f : dv[i];
                dv[i] = dm;
                const float d = i < seen ? 0.f : dm;
                a0 += d;
                a1 += d * xh;  // (elements past the plane carry dy = 0)
            }
            // With a residual, the gradient behind the ReLU is the residual's gradient: written here, it also saves
            // the apply kernel the reads of dy and the residual and the mask.
            if (P.dres) store_chunk<TS>(static_cast<TS*>(P.dres) + off, n, dv);
        }
    }
    wg_sum2(a0, a1, red);
    if (threadIdx.x == 0) {
        P.partial[((long)c * P.S + s) * 2] = a0;
        P.partial[((long)c * P.S + s) * 2 + 1] = a1;
    }
}

// MODE 0: y = gamma * xhat + beta (ReLU optional); split 0 also records the statistics.
// MODE 1: dx = gamma * invstd * (dy' - mean(dy') - xhat * mean(dy' * xhat)); split 0 writes dgamma, dbeta.
template <typename TS, int MODE>
__global__ void __launch_bounds__(256) bn_apply_kernel(const BnArgs P) {
    constexpr int V = Vec<TS>::N;
    __shared__ float red[4][2];
    const int c = blockIdx.x, s = blockIdx.y;
    const int b0 = s * P.rows_per_split;
    const int nb = min(P.rows_per_split, P.rows - b0);
    const float m = (float)P.rows * (float)P.hw;
    float t0, t1;
    channel_totals(P, c, t0, t1, red);
    const float g = P.gamma[c], be = P.beta[c];
    float mean, invstd;
    if constexpr (MODE == 0) {
        const float shifted = t0 / m;  // mean of x - K, K as in bn_sums_kernel
        mean = (float)static_cast<const TS*>(P.x)[(long)c * P.hw] + shifted;
        const float var = fmaxf(t1 / m - shifted * shifted, 0.f);
        invstd = 1.f / sqrtf(var + P.eps);
        if (s == 0 && threadIdx.x == 0) {
            P.save_mean[c] = mean;
            P.save_invstd[c] = invstd;
            if (P.run_mean) P.run_mean[c] = (1.f - P.momentum) * P.run_mean[c] + P.momentum * mean;
            if (P.run_var) P.run_var[c] = (1.f - P.momentum) * P.run_var[c] + P.momentum * var * (m > 1.f ? m / (m - 1.f) : 1.f);
        }
    } else {
        mean = P.save_mean[c];
        invstd = P.save_invstd[c];
        if (s == 0 && threadIdx.x == 0) { P.dbeta[c] = t0; P.dgamma[c] = t1; }
    }
    const float k0 = t0 / m, k1 = t1 / m, scale = g * invstd;
    const TS* x = static_cast<const TS*>(P.x);
    const TS* dy = static_cast<const TS*>(P.dy);
    const TS* res = static_cast<const TS*>(P.res);
    TS* out = static_cast<TS*>(P.out);
    TS* dres = static_cast<TS*>(P.dres);
    const int total = nb * P.nchunk;
    for (int idx = threadIdx.x; idx < total; idx += 256) {
        const int b = idx / P.nchunk, ch = idx - b * P.nchunk;
        long off = ((long)(b0 + b) * P.C + c) * P.hw + ch * V;
        int n = min(V, P.hw - ch * V);
        // (a plane's last, partial chunk: the full chunk ending at the plane's end instead, as in bn_sums_kernel; the
        // elements it shares with the chunk before are computed and stored twice, with the same values)
        if (n < V && P.hw >= V) { off -= V - n; n = V; }
        float xv[V], ov[V], rv[V];
        load_chunk<TS>(x + off, n, xv);
        if (res && (MODE == 0 || !dres)) load_chunk<TS>(res + off, n, rv);
        if constexpr (MODE == 0) {
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const float y = scale * (xv[i] - mean) + be + (res ? rv[i] : 0.f);
                ov[i] = (P.relu && y < 0.f) ? 0.f : y;
            }
        } else {
            float dv[V];
            if (dres) {  // the masked gradient, as bn_sums_kernel left it
                load_chunk<TS>(dres + off, n, dv);
#pragma unroll
                for (int i = 0; i < V; ++i) ov[i] = scale * (dv[i] - k0 - (xv[i] - mean) * invstd * k1);
            } else {
                load_chunk<TS>(dy + off, n, dv);
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const float xh = (xv[i] - mean) * invstd;
                    const float d = (P.relu && g * xh + be + (res ? rv[i] : 0.f) <= 0.f) ? 0.f : dv[i];
                    ov[i] = scale * (d - k0 - xh * k1);
                }
            }
        }
        store_chunk<TS>(out + off, n, ov);
    }
}

// ---- both passes in one: a workgroup holds its part of a channel in registers ----
// The two kernels above read x (and dy) twice, with the whole tensor between the two reads: 2.0 GB for the two 128-channel norms
// of a bottleneck block at 128 images of 28x28 where 1.3 are needed.  Here a workgroup keeps the chunks that it has summed (and
// the forward pass's residual, requested with them), publishes its two sums, waits for those of its channel's other
// workgroups, which are its neighbours in the launch, and applies the result to what it holds.  206 MB of a forward pass take
// 44 us (4.7 TB/s, a copy's 5.05), backward 309 MB 72 us; what is missing is the wait, a store and a load behind the tensor's own
// traffic, which the other workgroups of the CU fill in part.  (Neighbouring channels on one XCD: 49 and 102 us; the residual
// of the backward pass requested three chunks ahead: 139 us for 128.)
//
// A pair of sums is one 64-bit word, written and read by relaxed atomics of the device's scope, and differs from BN_NONE, which
// a launch in front sets the words to: nothing else passes between workgroups, so no cache is written back or dropped.
// A thread's elements are summed by the chunk and the channel's words in double.  Against fp64, root mean square over the channels of
// fp16 [256, 64, 56, 56], 1/deviation: 1.8e-7 with one chain a thread and fp32 words (1.5e-7 in two launches), 4.4e-8 now; the mean in
// deviations 4.8e-8 and 1.0e-8; dgamma over the root of its terms 2.7e-7 (2.6e-7) and 1.3e-7; the times are the same.
// No workgroup depends on another's progress: one that has looked P.waits times (some milliseconds) without seeing all words
// forms them itself from memory, in the order of their owners.  What is written is therefore never what is read (one_pass).
constexpr unsigned long long BN_NONE = ~0ull;
constexpr int BN_HELD_ONE = 16, BN_HELD_TWO = 8;  // chunks a thread holds of a single tensor, of each of two

__global__ void __launch_bounds__(256) bn_none_kernel(unsigned long long* words, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) words[i] = BN_NONE;
}

template <typename TS>
__device__ __forceinline__ void unpack_chunk(const u32x4 raw, float (&v)[Vec<TS>::N]) {
    if constexpr (sizeof(TS) == 2) {
        const f16x8 h = __builtin_bit_cast(f16x8, raw);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (float)h[i];
    } else {
        const f32x4 f = __builtin_bit_cast(f32x4, raw);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = f[i];
    }
}
template <typename TS>
__device__ __forceinline__ u32x4 pack_chunk(const float (&v)[Vec<TS>::N]) {
    if constexpr (sizeof(TS) == 2) {
        f16x8 h;
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = (_Float16)v[i];
        return __builtin_bit_cast(u32x4, h);
    } else {
        f32x4 f;
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = v[i];
        return __builtin_bit_cast(u32x4, f);
    }
}
template <typename TS>
__device__ __forceinline__ u32x4 load_raw(const TS* p) { return load16_a2(reinterpret_cast<const _Float16*>(p)); }
template <typename TS>
__device__ __forceinline__ void store_raw(TS* p, u32x4 raw) {
    *reinterpret_cast<__attribute__((address_space(1))) u32x4_a2*>((__attribute__((address_space(1))) _Float16*)p) = raw;
}

// A thread's walk over the chunks first, first + T, ... of channel c: the element offset of each, and how many of its
// elements belong to the chunk before (a plane's last chunk ends where the plane ends; hw >= a chunk here).
struct ChunkWalk {
    int row, chunk;
    __device__ __forceinline__ ChunkWalk(const BnArgs& P, int first) : row(first / P.nchunk), chunk(first - row * P.nchunk) {}
    template <int V>
    __device__ __forceinline__ unsigned int offset(const BnArgs& P, int c, int& seen) const {
        seen = max(chunk * V + V - P.hw, 0);
        return ((unsigned int)row * P.C + c) * (unsigned int)P.hw + (unsigned int)(chunk * V - seen);
    }
    __device__ __forceinline__ void next(const BnArgs& P) {
        chunk += P.chunks_step;
        row += P.rows_step;
        if (chunk >= P.nchunk) { chunk -= P.nchunk; ++row; }
    }
};

template <typename TS, int MODE, bool RES, int HELD, int T>
__global__ void __launch_bounds__(T, 4) bn_held_kernel(const BnArgs P) {
    constexpr int V = Vec<TS>::N;
    __shared__ float red[T / 64][2];
    __shared__ double totals[2];
    const int tid = threadIdx.x;
    const int c = blockIdx.x / P.S, s = blockIdx.x - c * P.S;
    const TS* x = static_cast<const TS*>(P.x);
    const TS* dy = static_cast<const TS*>(P.dy);
    const TS* res = static_cast<const TS*>(P.res);
    const float g = P.gamma[c], be = P.beta[c];
    float mean = 0.f, invstd = 0.f;
    if constexpr (MODE == 1) { mean = P.save_mean[c]; invstd = P.save_invstd[c]; }
    const float shift = MODE == 0 ? (float)x[(long)c * P.hw] : 0.f;

    u32x4 hx[HELD], hd[HELD];  // hd: dy, then the gradient behind the ReLU (MODE 1); the residual (forward pass)
    // One chunk's part of the sums.  MODE 1 leaves the gradient behind the ReLU in `d`.
    const auto add = [&](u32x4 xc, u32x4& d, unsigned int off, int seen, float& a0, float& a1) {
        float xv[V], dv[V], rv[V];
        unpack_chunk<TS>(xc, xv);
        if constexpr (MODE == 1) unpack_chunk<TS>(d, dv);
        if constexpr (MODE == 1 && RES) unpack_chunk<TS>(load_raw(res + off), rv);
        float c0 = 0.f, c1 = 0.f;  // (a chunk's own sums: a thread's 64 to 128 elements one behind the other round more)
#pragma unroll
        for (int i = 0; i < V; ++i) {
            if constexpr (MODE == 0) {
                const float e = i < seen ? 0.f : xv[i] - shift;
                c0 += e;
                c1 += e * e;
            } else {
                const float xh = (xv[i] - mean) * invstd;
                dv[i] = (P.relu && g * xh + be + (RES ? rv[i] : 0.f) <= 0.f) ? 0.f : dv[i];
                const float e = i < seen ? 0.f : dv[i];
                c0 += e;
                c1 += e * xh;
            }
        }
        a0 += c0;
        a1 += c1;
        if constexpr (MODE == 1) d = pack_chunk<TS>(dv);  // (values of the tensor's type: exact)
    };

    const int mine = min(P.per_split, P.total - s * P.per_split);  // chunks of this workgroup
    const ChunkWalk start(P, s * P.per_split + tid);
    ChunkWalk walk = start;
    int seen;
#pragma unroll
    for (int k = 0; k < HELD; ++k, walk.next(P)) {
        if (k * T + tid < mine) {
            const unsigned int off = walk.offset<V>(P, c, seen);
            hx[k] = load_raw(x + off);
            if constexpr (MODE == 1) hd[k] = load_raw(dy + off);
            else if constexpr (RES) hd[k] = load_raw(res + off);
        }
    }
    float a0 = 0.f, a1 = 0.f;
    walk = start;
    asm volatile("" : "+v"(walk.row), "+v"(walk.chunk));
#pragma unroll
    for (int k = 0; k < HELD; ++k, walk.next(P)) {
        if (k * T + tid < mine) {
            const unsigned int off = walk.offset<V>(P, c, seen);
            add(hx[k], hd[k], off, seen, a0, a1);
            if (MODE == 1 && RES && P.dres) store_raw(static_cast<TS*>(P.dres) + off, hd[k]);
        }
    }
    // the channel's totals
    const auto word = [](float a, float b) {
        const unsigned long long w = (unsigned long long)__float_as_uint(b) << 32 | __float_as_uint(a);
        return w == BN_NONE ? 0x7fc000007fc00000ull : w;  // (a NaN for a NaN)
    };
    unsigned long long* words = reinterpret_cast<unsigned long long*>(P.partial) + (long)c * P.S;
    wg_sum2<T>(a0, a1, red);
    if (tid == 0) __hip_atomic_store(words + s, word(a0, a1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long w = tid < P.S ? BN_NONE : 0;
    for (int i = 0; i < P.waits && w == BN_NONE; ++i) {
        w = __hip_atomic_load(words + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (w == BN_NONE) __builtin_amdgcn_s_sleep(10);
    }
    if (__syncthreads_or(w == BN_NONE)) {
        for (int t = 0; t < P.S; ++t) {
            const int count = min(P.per_split, P.total - t * P.per_split);
            ChunkWalk again(P, t * P.per_split + tid);
            a0 = a1 = 0.f;
            for (int i = tid; i < count; i += T, again.next(P)) {
                const unsigned int off = again.offset<V>(P, c, seen);
                u32x4 d{};
                if constexpr (MODE == 1) d = load_raw(dy + off);
                add(load_raw(x + off), d, off, seen, a0, a1);
            }
            wg_sum2<T>(a0, a1, red);
            if (tid == t) w = word(a0, a1);
        }
    }
    // (the words are the first wave's; in double: the last additions, and the variance's difference, are what a statistic's error is made of)
    if (tid < 64) {
        double t0 = __uint_as_float((unsigned int)w), t1 = __uint_as_float((unsigned int)(w >> 32));  // (zeros past the splits)
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            t0 += __shfl_xor(t0, off, 64);
            t1 += __shfl_xor(t1, off, 64);
        }
        if (tid == 0) { totals[0] = t0; totals[1] = t1; }
    }
    __syncthreads();
    const double t0 = totals[0], t1 = totals[1];

    // (what the sums formed of the held values -- conversions, offsets -- is formed again: kept, it would take more registers than they do)
    walk = start;
    asm volatile("" : "+v"(walk.row), "+v"(walk.chunk));
#pragma unroll
    for (int k = 0; k < HELD; ++k) {
        asm volatile("" : "+v"(hx[k]));
        if constexpr (MODE == 1 || RES) asm volatile("" : "+v"(hd[k]));
    }
    const float m = (float)P.rows * (float)P.hw;
    const double each = 1.0 / ((double)P.rows * P.hw), m0 = t0 * each, m1 = t1 * each;
    [[maybe_unused]] const float k0 = (float)m0, k1 = (float)m1;
    if constexpr (MODE == 0) {
        mean = (float)(shift + m0);
        const float var = fmaxf((float)(m1 - m0 * m0), 0.f);
        invstd = 1.f / sqrtf(var + P.eps);
        if (s == 0 && tid == 0) {
            P.save_mean[c] = mean;
            P.save_invstd[c] = invstd;
            if (P.run_mean) P.run_mean[c] = (1.f - P.momentum) * P.run_mean[c] + P.momentum * mean;
            if (P.run_var) P.run_var[c] = (1.f - P.momentum) * P.run_var[c] + P.momentum * var * (m > 1.f ? m / (m - 1.f) : 1.f);
        }
    } else if (s == 0 && tid == 0) {
        P.dbeta[c] = (float)t0;
        P.dgamma[c] = (float)t1;
    }
    const float scale = g * invstd;
#pragma unroll
    for (int k = 0; k < HELD; ++k, walk.next(P)) {
        if (k * T + tid < mine) {
            float xv[V], dv[V], ov[V];
            unpack_chunk<TS>(hx[k], xv);
            if constexpr (MODE == 1 || RES) unpack_chunk<TS>(hd[k], dv);
#pragma unroll
            for (int i = 0; i < V; ++i) {
                if constexpr (MODE == 0) {
                    const float y = scale * (xv[i] - mean) + be + (RES ? dv[i] : 0.f);
                    ov[i] = (P.relu && y < 0.f) ? 0.f : y;
                } else {
                    ov[i] = scale * (dv[i] - k0 - (xv[i] - mean) * invstd * k1);
                }
            }
            store_raw(static_cast<TS*>(P.out) + walk.offset<V>(P, c, seen), pack_chunk<TS>(ov));
        }
    }
}

// Evaluation: y = gamma / sqrt(running_var + eps) * (x - running_mean) + beta (+ residual, ReLU), one pass.
//
// Bound by HBM at the large layers and by its launch at the deep ones (a 512-channel 7x7 layer of 8 images is 1.6 MB).
// The tensor is walked as one run of 16-byte chunks whatever H*W is, not plane by plane: planes of 7x7 fp16 elements
// start at odd multiples of 2 bytes, where a 16-byte access costs about four times an aligned one, and would leave each
// one's last chunk partial.  A workgroup owns BN_EVAL_CHUNKS chunks per thread; the factors of the planes its run
// touches are formed once into LDS.  Measured on the 53 layers of the quaternion ResNet-50 at 8 images, fp16 (1.6 to
// 13 MB each): 290 us in all, 5.5 a layer (4 where it is 1.6 MB), against 940 us as a library normalisation (13 us each), an
// addition (4.4) and a ReLU (3.8) behind each other.  The three also rounded to fp16 one after the other; this pass rounds once
// (logits of that network against fp64, two sets of weights: 2-norm error 2.52e-3 and 2.86e-3 against 2.58e-3 and 2.98e-3).
// FEW_PIXELS: planes of fewer elements than a chunk, whose elements look up their plane one by one; otherwise a chunk lies
// in at most two planes.
constexpr int BN_EVAL_CHUNKS = 2;

struct BnEvalArgs {
    const void* x;
    const void* res;
    void* out;
    const float *gamma, *beta, *mean, *var;
    long total;  // elements
    int C, hw;
    float eps;
    int relu;
};

template <typename TS, bool FEW_PIXELS>
__global__ void __launch_bounds__(256) bn_eval_kernel(const BnEvalArgs P) {
    constexpr int V = Vec<TS>::N;
    constexpr int RUN = 256 * V * BN_EVAL_CHUNKS;      // elements of a workgroup
    extern __shared__ f32x4 factors[];                 // [plane of the run]: scale, mean, beta
    const long e0 = (long)blockIdx.x * RUN;
    const long plane0 = e0 / P.hw;
    const int r0 = (int)(e0 - plane0 * P.hw);          // first element's place in its plane
    const int count = (int)min((long)RUN, P.total - e0);
    const TS* x = static_cast<const TS*>(P.x) + e0;
    const TS* res = static_cast<const TS*>(P.res) + e0;
    TS* out = static_cast<TS*>(P.out) + e0;
    // requested before the factors are formed, so that the two waits overlap
    float xv[BN_EVAL_CHUNKS][V], rv[BN_EVAL_CHUNKS][V];
#pragma unroll
    for (int k = 0; k < BN_EVAL_CHUNKS; ++k) {
        const int t = (k * 256 + threadIdx.x) * V;
        if (t < count) {
            load_chunk<TS>(x + t, min(V, count - t), xv[k]);
            if (P.res) load_chunk<TS>(res + t, min(V, count - t), rv[k]);
        }
    }
    const int planes = (r0 + count - 1) / P.hw + 1;
    for (int i = threadIdx.x; i < planes; i += 256) {
        const int c = (int)((plane0 + i) % P.C);
        factors[i] = f32x4{P.gamma[c] / sqrtf(P.var[c] + P.eps), P.mean[c], P.beta[c], 0.f};
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BN_EVAL_CHUNKS; ++k) {
        const int t = (k * 256 + threadIdx.x) * V;
        if (t >= count) continue;
        const int n = min(V, count - t);
        int i = (r0 + t) / P.hw;
        int left = (i + 1) * P.hw - (r0 + t);          // elements of the chunk in front of the next plane
        f32x4 f0 = factors[i], f1 = f0;
        if (!FEW_PIXELS && left < n) f1 = factors[i + 1];
        float ov[V];
#pragma unroll
        for (int e = 0; e < V; ++e) {
            if (FEW_PIXELS && e < n && left == 0) {
                ++i;
                left = P.hw;
                f0 = factors[i];
            }
            const bool second = !FEW_PIXELS && e >= left;
            if (FEW_PIXELS) --left;
            // (the mean is taken off first: a scaled mean folded into beta would cancel against a large x)
            float y = (second ? f1[0] : f0[0]) * (xv[k][e] - (second ? f1[1] : f0[1])) + (second ? f1[2] : f0[2]);
            if (P.res) y += rv[k][e];
            ov[e] = (P.relu && y < 0.f) ? 0.f : y;
        }
        store_chunk<TS>(out + t, n, ov);
    }
}

template <typename TS>
static void launch_eval(const BnEvalArgs& a, hipStream_t st) {
    constexpr int V = Vec<TS>::N, RUN = 256 * V * BN_EVAL_CHUNKS;
    const dim3 grid((unsigned)((a.total + RUN - 1) / RUN));
    const size_t lds = (size_t)((RUN - 1 + a.hw - 1) / a.hw + 1) * sizeof(f32x4);  // (64 KB at H*W = 1 in fp16)
    if (a.hw < V) hipLaunchKernelGGL((bn_eval_kernel<TS, true>), grid, dim3(256), lds, st, a);
    else hipLaunchKernelGGL((bn_eval_kernel<TS, false>), grid, dim3(256), lds, st, a);
}

int bn_eval_status(const phx_bn_desc* d) {
    if ((d->dtype != PHX_F32 && d->dtype != PHX_F16) || d->rows < 0 || d->c <= 0 || d->hw < 0 || !(d->eps >= 0.f))
        return PHX_ERR_INVALID_ARGUMENT;
    if (d->rows == 0 || d->hw == 0) return PHX_OK;
    // (the kernel multiplies a run's plane numbers by hw in 32 bits; a launch has fewer than 2^32 threads)
    const long run = 256L * BN_EVAL_CHUNKS * (d->dtype == PHX_F16 ? Vec<_Float16>::N : Vec<float>::N);
    if (d->hw >= 1 << 30 || (long)d->rows * d->c > (run << 24) / d->hw - 1) return PHX_ERR_NOT_SUPPORTED;
    return PHX_OK;
}

static int plan(const phx_bn_desc* d, BnArgs& a) {
    if (!d || (d->dtype != PHX_F32 && d->dtype != PHX_F16) || d->rows < 0 || d->c <= 0 || d->hw < 0 || !(d->eps > 0.f))
        return PHX_ERR_INVALID_ARGUMENT;
    if ((long)d->rows * ((d->hw + 3) / 4) >= (1L << 31)) return PHX_ERR_NOT_SUPPORTED;  // chunk indices are 32-bit
    a.rows = d->rows; a.C = d->c; a.hw = d->hw; a.eps = d->eps; a.momentum = d->momentum; a.relu = d->relu;
    const int V = d->dtype == PHX_F16 ? 8 : 4;
    a.nchunk = (d->hw + V - 1) / V;
    // enough workgroups to fill the chip several times over, at most 256 splits (one partial per thread)
    // (fewer, longer-lived workgroups on the small layers -- at least four chunks per thread -- measured slower)
    int S = (2048 + d->c - 1) / d->c;
    S = std::max(1, std::min(S, std::min(std::max(d->rows, 1), 256)));
    a.rows_per_split = (std::max(d->rows, 1) + S - 1) / S;
    a.S = (std::max(d->rows, 1) + a.rows_per_split - 1) / a.rows_per_split;
    return PHX_OK;
}

// The plan of bn_held_kernel: its workgroup's threads, or 0 for sizes it does not take or where it is not the faster one.
// A thread holds 16 chunks, of one tensor or eight each of two (64 of 128 registers; half as many in twice the workgroups took
// 1.3 times as long).  Measured, us, two launches / one pass, forward, forward with residual, backward, backward with residual:
//   fp16 [512, 128, 28, 28] 55/44 74/69 87/72 147/128     fp16 [512, 64, 28, 28] 30/23 37/35 46/36 60/50
//   fp16 [256, 512, 7, 7]   16/14 21/18 27/19  35/25      fp32 [512, 128, 28, 28] 115/94 155/136 209/138 289/232
//   fp16 [64, 64, 28, 28]    9/11 10/11 10/10  12/12      fp32 [64, 64, 28, 28] 11/11 11/11 12/11 17/16
// * The backward pass gains from 8 MB on; the forward pass, whose second reading of x the 256 MB cache serves in part, from
//   32 MB, or 16 MB where a channel's workgroups are few ([128, 256, 14, 14], 12.8 MB in fp16 and 26 in fp32: 12/12, 14/14 and
//   16/14, 21/18).
// * A channel of many workgroups waits longer: from 50 on they have 512 threads (fp32 [256, 64, 56, 56], backward, 98 of 256
//   threads or 49 of 512: 157 or 137 us, two launches 209) and beyond 64 of those the two launches are as fast ([256, 16, 112, 112]
//   in fp16 83/90), as they are for a forward pass with a residual of more than 40 that the cache holds ([256, 64, 56, 56] in
//   fp16 68/70; 567/454 at 695 MB).
static int plan_held(BnArgs& a, int dtype, bool backward, bool residual) {
    const int pinned = tuning_bn_held();
    if (pinned == 0) return 0;
    const int V = dtype == PHX_F16 ? Vec<_Float16>::N : Vec<float>::N;
    const long elements = (long)a.rows * a.C * a.hw, bytes = elements * (dtype == PHX_F16 ? 2 : 4), total = (long)a.rows * a.nchunk;
    if (a.hw < V || elements >= 1L << 31) return 0;  // (offsets are 32-bit)
    const int chunks = !backward && !residual ? BN_HELD_ONE : BN_HELD_TWO;
    int threads = 256;
    if ((total + 256 * chunks - 1) / (256 * chunks) > (!backward && residual ? 40 : 50)) {
        if (!backward && residual && bytes < 160000000 && pinned < 0) return 0;
        threads = 512;
    }
    const long held = (long)threads * chunks;
    // (no fewer workgroups than the GPU holds at once, as long as each has a chunk a thread)
    long S = std::max((total + held - 1) / held, std::min((1024L + a.C - 1) / a.C, (total + threads - 1) / threads));
    const long per = std::min(held, ((total + S - 1) / S + 63) / 64 * 64);
    S = (total + per - 1) / per;
    if (S > 64) return 0;
    if (pinned < 0 && bytes < (backward ? 8000000 : S <= 8 ? 16000000 : 32000000)) return 0;
    a.S = (int)S;
    a.total = (int)total;
    a.per_split = (int)per;
    a.rows_step = threads / a.nchunk;
    a.chunks_step = threads % a.nchunk;
    a.waits = tuning_bn_waits();
    return threads;
}

template <typename TS, int T>
static void launch_held(const BnArgs& a, bool backward, hipStream_t st) {
    const int words = a.C * a.S;
    hipLaunchKernelGGL(bn_none_kernel, dim3((words + 255) / 256), dim3(256), 0, st, reinterpret_cast<unsigned long long*>(a.partial), words);
    const dim3 grid(words);
    if (!backward && !a.res) hipLaunchKernelGGL((bn_held_kernel<TS, 0, false, BN_HELD_ONE, T>), grid, dim3(T), 0, st, a);
    else if (!backward) hipLaunchKernelGGL((bn_held_kernel<TS, 0, true, BN_HELD_TWO, T>), grid, dim3(T), 0, st, a);
    else if (!a.res) hipLaunchKernelGGL((bn_held_kernel<TS, 1, false, BN_HELD_TWO, T>), grid, dim3(T), 0, st, a);
    else hipLaunchKernelGGL((bn_held_kernel<TS, 1, true, BN_HELD_TWO, T>), grid, dim3(T), 0, st, a);
}

// What the calling thread's last call ran (phx_bn_last_kernel_name puts it into words)
struct BnRan {
    const char* pass = "";
    bool half, residual;
    int threads, splits;  // of one pass; threads 0: two launches
};
static thread_local BnRan g_bn_ran;

// One pass where its plan takes the call, the workspace holds its words and nothing that it writes is read.
template <typename TS>
static bool one_pass(BnArgs a, bool backward, size_t workspace_bytes, hipStream_t st) {
    const int threads = plan_held(a, sizeof(TS) == 2 ? PHX_F16 : PHX_F32, backward, a.res != nullptr);
    if (!threads || (size_t)a.C * a.S * 8 > workspace_bytes || reinterpret_cast<uintptr_t>(a.partial) % 8) return false;
    const size_t bytes = sizeof(TS) * (size_t)a.rows * a.C * a.hw;
    for (const void* w : {static_cast<const void*>(a.out), static_cast<const void*>(a.dres)})
        for (const void* r : {a.x, a.dy, a.res})
            if (!apart(w, bytes, r, bytes)) return false;
    if (!apart(a.out, bytes, a.dres, bytes)) return false;
    if (threads == 256) launch_held<TS, 256>(a, backward, st);
    else launch_held<TS, 512>(a, backward, st);
    g_bn_ran.threads = threads;
    g_bn_ran.splits = a.S;
    return true;
}

template <typename TS>
static void launch_all(const BnArgs& a, bool backward, size_t workspace_bytes, hipStream_t st) {
    g_bn_ran = {backward ? "bwd" : "fwd", sizeof(TS) == 2, a.res != nullptr, 0, a.S};
    if (one_pass<TS>(a, backward, workspace_bytes, st)) return;
    const dim3 grid(a.C, a.S);
    if (!backward) {
        hipLaunchKernelGGL((bn_sums_kernel<TS, 0>), grid, dim3(256), 0, st, a);
        hipLaunchKernelGGL((bn_apply_kernel<TS, 0>), grid, dim3(256), 0, st, a);
    } else {
        hipLaunchKernelGGL((bn_sums_kernel<TS, 1>), grid, dim3(256), 0, st, a);
        hipLaunchKernelGGL((bn_apply_kernel<TS, 1>), grid, dim3(256), 0, st, a);
    }
}

}  // namespace phx

using namespace phx;

extern "C" {

const char* phx_bn_last_kernel_name(void) {
    static thread_local char name[64];
    const BnRan& r = g_bn_ran;
    if (!*r.pass) return "";
    const int n = snprintf(name, sizeof(name), "bn_%s_%s%s", r.pass, r.half ? "f16" : "f32", r.residual ? "_res" : "");
    if (r.threads) snprintf(name + n, sizeof(name) - n, "_held%d_s%d", r.threads, r.splits);
    else if (r.splits) snprintf(name + n, sizeof(name) - n, "_two_s%d", r.splits);
    return name;
}

size_t phx_bn_workspace_bytes(const phx_bn_desc* desc) {
    BnArgs a{};
    if (plan(desc, a) != PHX_OK) return 0;
    int splits = a.S;
    for (int pass = 0; pass < 4 && desc->rows > 0 && desc->hw > 0; ++pass) {
        BnArgs held = a;
        if (plan_held(held, desc->dtype, pass & 1, pass & 2)) splits = std::max(splits, held.S);
    }
    return ((size_t)a.C * splits * 2 * sizeof(float) + 255) / 256 * 256;
}

int phx_bn_fwd_train(const phx_bn_desc* desc, phx_stream_t stream, const void* x, const void* residual_or_null,
                     const float* gamma, const float* beta, void* y, float* save_mean, float* save_invstd,
                     float* running_mean_or_null, float* running_var_or_null, void* workspace, size_t workspace_bytes) {
    BnArgs a{};
    const int rc = plan(desc, a);
    if (rc != PHX_OK) return rc;
    if (desc->rows == 0 || desc->hw == 0) return PHX_OK;
    if (!x || !gamma || !beta || !y || !save_mean || !save_invstd) return PHX_ERR_INVALID_ARGUMENT;
    if (!workspace || workspace_bytes < (size_t)a.C * a.S * 2 * sizeof(float)) return PHX_ERR_WORKSPACE;
    a.x = x; a.res = residual_or_null; a.out = y; a.gamma = gamma; a.beta = beta; a.partial = static_cast<float*>(workspace);
    a.save_mean = save_mean; a.save_invstd = save_invstd; a.run_mean = running_mean_or_null; a.run_var = running_var_or_null;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (desc->dtype == PHX_F16) launch_all<_Float16>(a, false, workspace_bytes, st);
    else launch_all<float>(a, false, workspace_bytes, st);
    if (hipGetLastError() != hipSuccess) return PHX_ERR_RUNTIME;
    return PHX_OK;
}

int phx_bn_fwd_eval(const phx_bn_desc* desc, phx_stream_t stream, const void* x, const void* residual_or_null,
                    const float* gamma, const float* beta, const float* running_mean, const float* running_var, void* y) {
    if (!desc) return PHX_ERR_INVALID_ARGUMENT;
    if (desc->rows >= 0 && desc->c > 0 && (desc->rows == 0 || desc->hw == 0)) return bn_eval_status(desc);
    if (!x || !gamma || !beta || !running_mean || !running_var || !y) return PHX_ERR_INVALID_ARGUMENT;
    if (const int rc = bn_eval_status(desc)) return rc;
    BnEvalArgs a{x, residual_or_null, y, gamma, beta, running_mean, running_var, (long)desc->rows * desc->c * desc->hw,
                 desc->c, desc->hw, desc->eps, desc->relu};
    hipStream_t st = static_cast<hipStream_t>(stream);
    g_bn_ran = {"eval", desc->dtype == PHX_F16, residual_or_null != nullptr, 0, 0};
    if (desc->dtype == PHX_F16) launch_eval<_Float16>(a, st);
    else launch_eval<float>(a, st);
    if (hipGetLastError() != hipSuccess) return PHX_ERR_RUNTIME;
    return PHX_OK;
}

int phx_bn_bwd(const phx_bn_desc* desc, phx_stream_t stream, const void* x, const void* residual_or_null, const void* dy,
               const float* gamma, const float* beta, const float* save_mean, const float* save_invstd, void* dx,
               void* dresidual_or_null, float* dgamma, float* dbeta, void* workspace, size_t workspace_bytes) {
    BnArgs a{};
    const int rc = plan(desc, a);
    if (rc != PHX_OK) return rc;
    if (!dgamma || !dbeta) return PHX_ERR_INVALID_ARGUMENT;
    if (desc->rows == 0 || desc->hw == 0) return PHX_OK;
    if (!x || !dy || !gamma || !beta || !save_mean || !save_invstd || !dx) return PHX_ERR_INVALID_ARGUMENT;
    if (!workspace || workspace_bytes < (size_t)a.C * a.S * 2 * sizeof(float)) return PHX_ERR_WORKSPACE;
    if (residual_or_null && !desc->relu) return PHX_ERR_INVALID_ARGUMENT;  // without the ReLU its gradient is dy itself
    a.x = x; a.res = residual_or_null; a.dres = dresidual_or_null; a.dy = dy; a.out = dx; a.gamma = gamma; a.beta = beta; a.partial = static_cast<float*>(workspace);
    a.save_mean = const_cast<float*>(save_mean); a.save_invstd = const_cast<float*>(save_invstd);
    a.dgamma = dgamma; a.dbeta = dbeta;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (desc->dtype == PHX_F16) launch_all<_Float16>(a, true, workspace_bytes, st);
    else launch_all<float>(a, true, workspace_bytes, st);
    if (hipGetLastError() != hipSuccess) return PHX_ERR_RUNTIME;
    return PHX_OK;
}

}  // extern "C"
