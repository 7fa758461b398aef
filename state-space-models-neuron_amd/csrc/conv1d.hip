// Causal depthwise conv1d (+activation), forward and backward, for gfx950.
//
// Replaces the reference's NKI kernels conv1d_with_transpose (mamba2/conv1d_grouped.py:66-125),
// conv1d_with_transpose_bwd (:129-194) and conv1d_grouped_kernel_grad (:198-262).
//
// The op is HBM-bandwidth bound (8 FLOP + one SiLU per element), so the fast path is a
// streaming kernel on the channels-last (b, l, C) layout the mixer uses: one thread owns
// a short vector of channels (8 bytes forward, 4 backward in bf16) and walks TL consecutive tokens
// with the k-1 token history in registers, so every element is loaded once (plus a (k-1)/TL halo)
// and all global accesses are lane-contiguous along channels.  No transposes (the reference needs two per
// tile because its engine wants channels on partitions).
//
// The backward recomputes the pre-activation, forms g = dy * act'(z) and emits dx with a
// k-1 token lag, so the cross-segment halo is exact (the reference zero-pads g per tile and
// loses that contribution).  dw/db are reduced in fp32: registers -> LDS per block ->
// per-block partials in the workspace -> one small second-stage kernel.  No float atomics.
//
// The channel-major (b, C, l) layout of ConvNKI has its own kernels (conv_*_cm_kernel): a lane owns consecutive tokens
// of one row, so the taps of an output come from the lane's own window and nothing is loaded per tap.
//
// A generic path (any strides, k <= 8) covers the rest with one thread per output element.
#include <algorithm>

#include "sums.hpp"

namespace m2 {
namespace {

constexpr int kMaxK = 8;
#ifndef M2_CONV_UNR
#define M2_CONV_UNR 4
#endif
#ifndef M2_CONV_VF
#define M2_CONV_VF 8
#endif
#ifndef M2_CONV_VB
#define M2_CONV_VB 4
#endif
// Bytes of channels per thread in the fast path (VF forward, VB backward; at least two channels).  The backward carries five
// sums, two 3-token windows and the taps per channel: with two channels per thread it needs 96 registers (five waves per
// SIMD), with four 160 (three waves), and the narrower form is the faster one although its loads are 4-byte ones.
constexpr int kUNR = M2_CONV_UNR;    // tokens whose loads are in flight together
#ifndef M2_CONV_CVT
#define M2_CONV_CVT 64
#endif
#ifndef M2_CONV_SEG
#define M2_CONV_SEG 4
#endif
#ifndef M2_CONV_NT
#define M2_CONV_NT 1
#endif
constexpr int kCVT = M2_CONV_CVT;    // channel vectors per block (x dimension)
constexpr int kSEG = M2_CONV_SEG;    // token segments per block (y dimension)
static_assert(kUNR >= 3, "the dx lag fits one load group");

// Tokens per thread.  A thread is a chain of load groups, so where the threads do not fill the chip short segments win, and their
// halo (three tokens more read; six in the backward, and three more activations) and, in the backward, their partial rows only count
// once it is full.  The lines below come from 389 timings (256 to 10240 channels, 24 to 18746 tokens, batches of 1 to 16, both types,
// with the tensors in the caches and not); per band the geometric mean of the time over that of the best of the three forms, threads
// counted at 16 tokens forward and at 32 backward:
//   forward           4 |    8 |   16          backward (with its sum)             8 |   16 |   32
//   to 24K         1.00 | 1.09 | 1.37          to 16K                           1.01 | 1.12 | 1.49
//   24K to 48K     1.02 | 1.02 | 1.11          16K to 64K                       1.06 | 1.04 | 1.27
//   48K to 96K     1.03 | 1.01 | 1.09          64K to 128K                      1.10 | 1.03 | 1.04
//   96K to 192K    1.08 | 1.01 | 1.03          128K to 1M, to 2560 channels     1.15 | 1.05 | 1.01
//   above          1.15 | 1.00 | 1.05          128K to 1M, more channels        1.09 | 1.01 | 1.05
//                                              above                            1.21 | 1.03 | 1.00
//                                              192 partial rows and more        1.32 | 1.07 | 1.00
// Few channels and many partial rows want long segments for the sum's sake: it has a workgroup per 13 channels, and each of its
// threads walks a quarter of the rows.  In us, sizes beside the lines: b3 l1111 C2304 forward 10.1 | 8.7 | 8.8, backward 21.9 | 20.4 |
// 20.0; b6 l808 C2304 12.0 | 11.8 | 11.5 and 28.0 | 25.9 | 24.0; b12 l669 C4352 30.1 | 25.4 | 27.4 and 60.0 | 54.0 | 57.6; b4 l18746
// C256 18.0 | 16.4 | 17.4 and 83.0 | 57.3 | 49.5; b2 l4096 C10240 68.7 | 57.3 | 59.8 and 135.4 | 115.6 | 112.9.  A size on the wrong
// side of a line: b8 l333 C5376, backward 29.6 | 28.7 | 26.6.
constexpr int64_t kMaxSegs = (int64_t)65535 * kSEG;      // what the grid holds: the longest sequences keep the longest segments
int64_t conv_fwd_tokens(int64_t batch, int64_t seqlen, int64_t vectors) {
    const int64_t threads = batch * ceil_div(seqlen, (int64_t)16) * vectors;
    return ceil_div(seqlen, (int64_t)8) > kMaxSegs ? 16 : (threads <= 48 * 1024 ? 4 : 8);
}
int64_t conv_bwd_tokens(int64_t batch, int64_t seqlen, int64_t channels) {
    const int64_t threads = batch * ceil_div(seqlen, (int64_t)32) * ceil_div(channels, (int64_t)2), rows16 = batch * ceil_div(seqlen, (int64_t)(16 * kSEG));
    const bool long_ones = rows16 > 192 || threads > (channels <= 2560 ? 128 * 1024 : 1024 * 1024);
    const int64_t tl = threads <= 16 * 1024 ? 8 : (long_ones ? 32 : 16);
    return ceil_div(seqlen, tl) > kMaxSegs ? 32 : tl;
}
// f<tokens per thread>
template <typename F> void with_fwd_tokens(int64_t tl, F&& f) {
    if (tl == 4) f(std::integral_constant<int, 4>{});
    else if (tl == 8) f(std::integral_constant<int, 8>{});
    else f(std::integral_constant<int, 16>{});
}
template <typename F> void with_bwd_tokens(int64_t tl, F&& f) {
    if (tl == 8) f(std::integral_constant<int, 8>{});
    else if (tl == 16) f(std::integral_constant<int, 16>{});
    else f(std::integral_constant<int, 32>{});
}

// streaming loads/stores of the activations (optionally non-temporal: nothing is re-read soon enough to be worth caching)
// The vectors promise the alignment of an element only: gfx950 issues the same wide access either way, so rows that start
// anywhere (an odd number of channels, of tokens, or of columns in front of a slice) take the vector kernels as well.
template <int BYTES> struct StreamVec;
template <> struct StreamVec<16> { typedef uint32_t type __attribute__((ext_vector_type(4), aligned(2))); };
template <> struct StreamVec<8> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(2))); };
template <> struct StreamVec<4> { typedef uint32_t type __attribute__((aligned(2))); };
template <typename T, int V>
__device__ __forceinline__ RawVec<T, V> ld_stream(const T* __restrict__ p) {
    using S = typename StreamVec<V * (int)sizeof(T)>::type;
    RawVec<T, V> r;
    const S v = M2_CONV_NT ? __builtin_nontemporal_load(reinterpret_cast<const S*>(p)) : *reinterpret_cast<const S*>(p);
    *reinterpret_cast<S*>(&r) = v;
    return r;
}
template <typename T, int V>
__device__ __forceinline__ void st_stream(T* __restrict__ p, const float (&in)[V]) {
    using S = typename StreamVec<V * (int)sizeof(T)>::type;
    S raw;
    T* e = reinterpret_cast<T*>(&raw);
#pragma unroll
    for (int i = 0; i < V; ++i) e[i] = from_f32<T>(in[i]);
    if (M2_CONV_NT) __builtin_nontemporal_store(raw, reinterpret_cast<S*>(p)); else *reinterpret_cast<S*>(p) = raw;
}
// cached load of V elements from anywhere (windows that neighbours read too)
template <typename T, int V>
__device__ __forceinline__ void ld_elems(const T* __restrict__ p, float (&out)[V]) {
    using S = typename StreamVec<V * (int)sizeof(T)>::type;
    const S v = *reinterpret_cast<const S*>(p);
    const T* e = reinterpret_cast<const T*>(&v);
#pragma unroll
    for (int i = 0; i < V; ++i) out[i] = to_f32(e[i]);
}

// N neighbouring elements, as they lie
template <typename T, int N> using Tokens = T __attribute__((ext_vector_type(N)));
template <typename T, int N>
__device__ __forceinline__ Tokens<T, N> ld_whole(const T* __restrict__ p) {
    using S = typename StreamVec<N * (int)sizeof(T)>::type;
    return __builtin_bit_cast(Tokens<T, N>, *reinterpret_cast<const S*>(p));
}

__device__ __forceinline__ float ld_param(const void* p, int pd, int64_t i) {
    return pd == M2_F32 ? reinterpret_cast<const float*>(p)[i] : to_f32(reinterpret_cast<const bf16_t*>(p)[i]);
}
// The 4 taps and the bias of V consecutive channels with 16-byte loads, all in flight together (w is (C, 4) contiguous).
template <typename WT, int V>
__device__ __forceinline__ void load_taps(const void* __restrict__ w, const void* __restrict__ bias, int64_t c0,
                                          float (&wv)[4][V], float (&bv)[V]) {
    constexpr int TV = (V * 4 * (int)sizeof(WT)) < 16 ? V * 4 : 16 / (int)sizeof(WT);     // elements per tap load (<= 16 bytes)
    constexpr int PER = 16 / (int)sizeof(WT);
    static_assert((V * 4) % TV == 0, "taps of one thread must fill whole vectors");
    const WT* wp = static_cast<const WT*>(w) + c0 * 4;
    float flat[V * 4];
#pragma unroll
    for (int i = 0; i < V * 4 / TV; ++i) {
        float tmp[TV];
        ld_elems<WT, TV>(wp + i * TV, tmp);
#pragma unroll
        for (int e = 0; e < TV; ++e) flat[i * TV + e] = tmp[e];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) wv[i][j] = flat[j * 4 + i];
        bv[j] = 0.f;
    }
    if (bias) {
        constexpr int BV = V < PER ? V : PER;      // at most 16 bytes per load
#pragma unroll
        for (int i = 0; i < V / BV; ++i) {
            float tmp[BV];
            ld_elems<WT, BV>(static_cast<const WT*>(bias) + c0 + i * BV, tmp);
#pragma unroll
            for (int e = 0; e < BV; ++e) bv[i * BV + e] = tmp[e];
        }
    }
}

// ------------------------------------------------------------------------------------------
// Fast path, channels-last, k == 4.
// grid: x = ceil(CV / kCVT), y = ceil(nseg / kSEG), z = batch; block (kCVT, kSEG).
// PREFILL: the decode cache `state` ([b][C][W], oldest first) holds the inputs in front of the sequence (kContinuing) and takes
// its last W ones (kTail).  The thread of a strip's first segment does both, so nobody reads a cache entry that another thread
// has renewed; a kernel of its own behind this one took 4-5 us of every prefill (77 -> 73 us for 200 tokens of a 2560-channel
// layer).  Only where no two threads share channels (C a multiple of V), else conv_tail_kernel follows.
constexpr int kContinuing = 1, kTail = 2;
template <typename T, typename WT, int V, int ACT, bool PREFILL, int TL>
__global__ void __launch_bounds__(kCVT * kSEG)
conv_fwd_cl_kernel(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias, T* state, int W, int flags,
                   T* __restrict__ y, int64_t l, int64_t C, int64_t xsb, int64_t xsl, int64_t ysb, int64_t ysl) {
    static_assert(TL % kUNR == 0, "segments are whole load groups");
    const int64_t cv = (int64_t)blockIdx.x * kCVT + threadIdx.x;
    const int64_t seg = (int64_t)blockIdx.y * kSEG + threadIdx.y;
    const int64_t b = blockIdx.z;
    const int64_t t0 = seg * TL;
    if (cv * V >= C || t0 >= l) return;
    const int64_t c0 = cv * V < C - V ? cv * V : C - V;     // the last vector ends with the row (it may repeat channels: same values)

    const T* xp = x + b * xsb + c0;
    T* yp = y + b * ysb + c0;
    // A cache of four columns (the usual one): a channel's are one vector, the first segment's thread asks for its channels' and for the
    // sequence's last four inputs ahead of everything, and the columns leave in one store each (read, sorted and stored one by one
    // behind the segment they kept its workgroups 2 to 3 us longer than the others)
    const bool quick = PREFILL && (flags & kTail) && W == 4 && l >= 4 && t0 == 0;
    RawVec<T, V> last[4];
    Tokens<T, 4> was[V];
    if (quick) {
#pragma unroll
        for (int q = 0; q < 4; ++q) last[q] = ld_stream<T, V>(xp + (l - 4 + q) * xsl);
        if (flags & kContinuing) {
#pragma unroll
            for (int j = 0; j < V; ++j) was[j] = ld_whole<T, 4>(state + (b * C + c0 + j) * 4);
        }
    }
    float wv[4][V], bv[V];
    load_taps<WT, V>(w, bias, c0, wv, bv);
    float h0[V], h1[V], h2[V];   // x[t-3], x[t-2], x[t-1]
#pragma unroll
    for (int j = 0; j < V; ++j) h0[j] = h1[j] = h2[j] = 0.f;
    if (t0 - 3 >= 0) ld_elems<T, V>(xp + (t0 - 3) * xsl, h0);
    if (t0 - 2 >= 0) ld_elems<T, V>(xp + (t0 - 2) * xsl, h1);
    if (t0 - 1 >= 0) ld_elems<T, V>(xp + (t0 - 1) * xsl, h2);
    if (PREFILL && (flags & kContinuing) && t0 == 0) {
        // the inputs in front of the sequence come out of the decode cache (three short reads per channel in the first
        // segment only; putting cache and sequence behind one another in memory first took 35 us of 145 at b8 l333 C5376)
        if (quick) {
#pragma unroll
            for (int j = 0; j < V; ++j) { h0[j] = to_f32(was[j][1]); h1[j] = to_f32(was[j][2]); h2[j] = to_f32(was[j][3]); }
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const T* hp = state + (b * C + c0 + j) * W + (W - 3);
                h0[j] = to_f32(hp[0]); h1[j] = to_f32(hp[1]); h2[j] = to_f32(hp[2]);
            }
        }
    }
    if (quick) {      // (what was there has been read above)
        T* sp = state + (b * C + c0) * 4;
#pragma unroll
        for (int j = 0; j < V; ++j) {
            Tokens<T, 4> v;
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = reinterpret_cast<const T*>(&last[q])[j];
            *reinterpret_cast<typename StreamVec<4 * (int)sizeof(T)>::type*>(sp + j * 4) = __builtin_bit_cast(typename StreamVec<4 * (int)sizeof(T)>::type, v);
        }
    }
    // the last W inputs, four columns at a time; where the sequence is shorter, what is left of the cache (or zeros) moves up
    auto leave_tail = [&] {
        if (!PREFILL || !(flags & kTail) || t0 != 0 || quick) return;
        T* sp = state + (b * C + c0) * W;
        for (int w0 = 0; w0 < W; w0 += 4) {
            T v[4][V];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int wq = w0 + q < W ? w0 + q : W - 1;
                const int64_t t = l - W + wq;
                if (t >= 0) {
                    const RawVec<T, V> r = ld_stream<T, V>(xp + t * xsl);
                    const T* e = reinterpret_cast<const T*>(&r);
#pragma unroll
                    for (int j = 0; j < V; ++j) v[q][j] = e[j];
                } else {
#pragma unroll
                    for (int j = 0; j < V; ++j) v[q][j] = flags & kContinuing ? sp[j * W + wq + l] : from_f32<T>(0.f);
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (w0 + q < W) {
#pragma unroll
                    for (int j = 0; j < V; ++j) sp[j * W + w0 + q] = v[q][j];
                }
        }
    };
    auto step = [&](const RawVec<T, V>& r, T* __restrict__ yq) {
        float out[V], cur[V];
        cvtv<T, V>(r, cur);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            float z = bv[j] + wv[0][j] * h0[j] + wv[1][j] * h1[j] + wv[2][j] * h2[j] + wv[3][j] * cur[j];
            out[j] = act_f<ACT>(z);
            h0[j] = h1[j]; h1[j] = h2[j]; h2[j] = cur[j];
        }
        st_stream<T, V>(yq, out);
    };
    // software pipeline: the loads of group g+1 are issued before group g is computed and stored
    RawVec<T, V> nxt[kUNR];
    if (t0 + TL <= l) {
        // whole segment inside the sequence: no per-token predicates, so the wait before a group's compute can leave
        // the previous group's stores in flight
        const T* xq = xp + t0 * xsl;
        T* yq = yp + t0 * ysl;
#pragma unroll
        for (int u = 0; u < kUNR; ++u) nxt[u] = ld_stream<T, V>(xq + u * xsl);
        for (int g = 0; g < TL / kUNR - 1; ++g) {
            RawVec<T, V> raw[kUNR];
            xq += kUNR * xsl;
#pragma unroll
            for (int u = 0; u < kUNR; ++u) { raw[u] = nxt[u]; nxt[u] = ld_stream<T, V>(xq + u * xsl); }
#pragma unroll
            for (int u = 0; u < kUNR; ++u) step(raw[u], yq + u * ysl);
            yq += kUNR * ysl;
        }
#pragma unroll
        for (int u = 0; u < kUNR; ++u) step(nxt[u], yq + u * ysl);
        leave_tail();
        return;
    }
    const int64_t t1 = l;
#pragma unroll
    for (int u = 0; u < kUNR; ++u)
        if (t0 + u < t1) nxt[u] = ld_stream<T, V>(xp + (t0 + u) * xsl);
    for (int64_t tg = t0; tg < t1; tg += kUNR) {
        RawVec<T, V> raw[kUNR];
#pragma unroll
        for (int u = 0; u < kUNR; ++u) raw[u] = nxt[u];
#pragma unroll
        for (int u = 0; u < kUNR; ++u)
            if (tg + kUNR + u < t1) nxt[u] = ld_stream<T, V>(xp + (tg + kUNR + u) * xsl);
#pragma unroll
        for (int u = 0; u < kUNR; ++u)
            if (tg + u < t1) step(raw[u], yp + (tg + u) * ysl);
    }
    leave_tail();
}

// Backward fast path.  Each thread marches t over [t0, t0+TL+3): at step t it forms g[t] and
// emits dx[t-3] = w3 g[t-3] + w2 g[t-2] + w1 g[t-1] + w0 g[t]  (dx[s] = sum_i w[i] g[s+3-i]).
// Partials: part[(blockIdx.z * gridDim.y + blockIdx.y)][c][0..4] = (dw0..dw3, db).
template <typename T, typename WT, int V, int ACT, int TL>
__global__ void __launch_bounds__(kCVT * kSEG)
conv_bwd_cl_kernel(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias,
                   const T* __restrict__ dy, T* __restrict__ dx, float* __restrict__ part,
                   int64_t l, int64_t C, int64_t xsb, int64_t xsl, int64_t gsb, int64_t gsl,
                   int64_t dsb, int64_t dsl) {
    static_assert(TL % kUNR == 0, "segments are whole load groups");
    __shared__ float red[kSEG][5][kCVT * V + 1];
    const int64_t cv = (int64_t)blockIdx.x * kCVT + threadIdx.x;
    const int64_t seg = (int64_t)blockIdx.y * kSEG + threadIdx.y;
    const int64_t b = blockIdx.z;
    const int64_t c0 = cv * V < C - V ? cv * V : C - V;     // the last vector ends with the row (it may repeat channels: same values)
    const int64_t t0 = seg * TL;
    const bool active = (cv * V < C) && (t0 < l);

    float acc[5][V];
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) acc[i][j] = 0.f;

    if (active) {
        float wv[4][V], bv[V];
        load_taps<WT, V>(w, bias, c0, wv, bv);
        const T* xp = x + b * xsb + c0;
        const T* gp = dy + b * gsb + c0;
        T* dp = dx + b * dsb + c0;
        float h0[V], h1[V], h2[V];   // x[t-3..t-1]
        float g0[V], g1[V], g2[V];   // g[t-3..t-1]
#pragma unroll
        for (int j = 0; j < V; ++j) h0[j] = h1[j] = h2[j] = g0[j] = g1[j] = g2[j] = 0.f;
        if (t0 - 3 >= 0) ld_elems<T, V>(xp + (t0 - 3) * xsl, h0);
        if (t0 - 2 >= 0) ld_elems<T, V>(xp + (t0 - 2) * xsl, h1);
        if (t0 - 1 >= 0) ld_elems<T, V>(xp + (t0 - 1) * xsl, h2);
        // one token: g[t] from x[t-3..t] and dy[t]; the weight/bias sums if the token is this thread's own; dx[t-3] to dq if emit
        auto step = [&](const RawVec<T, V>& rx, const RawVec<T, V>& rg, bool own, bool emit, T* __restrict__ dq) {
            float g[V], cur[V], gy[V];
            cvtv<T, V>(rx, cur);
            cvtv<T, V>(rg, gy);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                float z = bv[j] + wv[0][j] * h0[j] + wv[1][j] * h1[j] + wv[2][j] * h2[j] + wv[3][j] * cur[j];
                g[j] = gy[j] * act_grad_f<ACT>(z);     // gy == 0 beyond the sequence end
                if (own) {
                    acc[0][j] += h0[j] * g[j];
                    acc[1][j] += h1[j] * g[j];
                    acc[2][j] += h2[j] * g[j];
                    acc[3][j] += cur[j] * g[j];
                    acc[4][j] += g[j];
                }
            }
            if (emit) {
                float o[V];
#pragma unroll
                for (int j = 0; j < V; ++j)
                    o[j] = wv[3][j] * g0[j] + wv[2][j] * g1[j] + wv[1][j] * g2[j] + wv[0][j] * g[j];
                st_stream<T, V>(dq, o);
            }
#pragma unroll
            for (int j = 0; j < V; ++j) {
                h0[j] = h1[j]; h1[j] = h2[j]; h2[j] = cur[j];
                g0[j] = g1[j]; g1[j] = g2[j]; g2[j] = g[j];
            }
        };
        // software pipeline: the loads of group g+1 are issued before group g is computed and stored
        RawVec<T, V> nx[kUNR], ng[kUNR];
        if (t0 + TL + kUNR <= l) {
            // the segment and its 3 lag tokens lie inside the sequence: no per-token predicates
            const T* xq = xp + t0 * xsl;
            const T* gq = gp + t0 * gsl;
            T* dq = dp + (t0 - 3) * dsl;
#pragma unroll
            for (int u = 0; u < kUNR; ++u) { nx[u] = ld_stream<T, V>(xq + u * xsl); ng[u] = ld_stream<T, V>(gq + u * gsl); }
            for (int grp = 0; grp < TL / kUNR; ++grp) {
                RawVec<T, V> rawx[kUNR], rawg[kUNR];
                xq += kUNR * xsl;
                gq += kUNR * gsl;
#pragma unroll
                for (int u = 0; u < kUNR; ++u) {
                    rawx[u] = nx[u]; rawg[u] = ng[u];
                    nx[u] = ld_stream<T, V>(xq + u * xsl); ng[u] = ld_stream<T, V>(gq + u * gsl);
                }
#pragma unroll
                for (int u = 0; u < kUNR; ++u) step(rawx[u], rawg[u], true, grp > 0 || u >= 3, dq + u * dsl);
                dq += kUNR * dsl;
            }
#pragma unroll
            for (int u = 0; u < 3; ++u) step(nx[u], ng[u], false, true, dq + u * dsl);
        } else {
            const int64_t tseg = (t0 + TL < l) ? t0 + TL : l;      // end of this thread's own tokens
            const int64_t tend = tseg + 3;                            // march 3 further for the dx lag
#pragma unroll
            for (int u = 0; u < kUNR; ++u) {
                const int64_t t = t0 + u;
                if (t < tend && t < l) { nx[u] = ld_stream<T, V>(xp + t * xsl); ng[u] = ld_stream<T, V>(gp + t * gsl); }
                else { nx[u] = RawVec<T, V>{}; ng[u] = RawVec<T, V>{}; }
            }
            for (int64_t tg = t0; tg < tend; tg += kUNR) {
                RawVec<T, V> rawx[kUNR], rawg[kUNR];
#pragma unroll
                for (int u = 0; u < kUNR; ++u) { rawx[u] = nx[u]; rawg[u] = ng[u]; }
#pragma unroll
                for (int u = 0; u < kUNR; ++u) {
                    const int64_t t = tg + kUNR + u;
                    if (t < tend && t < l) { nx[u] = ld_stream<T, V>(xp + t * xsl); ng[u] = ld_stream<T, V>(gp + t * gsl); }
                    else { nx[u] = RawVec<T, V>{}; ng[u] = RawVec<T, V>{}; }
                }
#pragma unroll
                for (int u = 0; u < kUNR; ++u) {
                    const int64_t t = tg + u;
                    if (t < tend) step(rawx[u], rawg[u], t < tseg, t - 3 >= t0, dp + (t - 3) * dsl);
                }
            }
        }
    }
    // block reduction over the kSEG token segments
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) red[threadIdx.y][i][threadIdx.x * V + j] = acc[i][j];
    __syncthreads();
    const int tid = threadIdx.y * kCVT + threadIdx.x;
    const int64_t pslot = (int64_t)blockIdx.z * gridDim.y + blockIdx.y;
    for (int e = tid; e < 5 * kCVT * V; e += kCVT * kSEG) {
        const int i = e / (kCVT * V), cc = e % (kCVT * V);
        const int64_t cb = (int64_t)blockIdx.x * kCVT * V + cc / V * V;      // first channel of the owning thread
        const int64_t c = (cb < C - V ? cb : C - V) + cc % V;
        if (cb < C) {
            float s = 0.f;
#pragma unroll
            for (int r = 0; r < kSEG; ++r) s += red[r][i][cc];
            part[(pslot * C + c) * 5 + i] = s;
        }
    }
}

// Zero fill (a kernel rather than a memset node, so that a caller may capture the call in a graph).
__global__ void conv_zero_kernel(uint16_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// Second stage: sum the per-block partials.
__global__ void __launch_bounds__(256)
conv_reduce_partials_kernel(const float* __restrict__ part, int64_t nslots, int64_t C, int k,
                            void* __restrict__ dw, void* __restrict__ db, int pd) {
    conv_sum_body(part, nslots, C, k, dw, db, pd, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// ------------------------------------------------------------------------------------------
// Channel-major path, k == 4: tokens contiguous in x, y (and dx).
//
// The kernels take N tokens of a row with one vector access.  Where the row's last vector is cut by its end, the lanes that hold it read the
// row's last N tokens instead (ld_whole) and move the ones that are theirs down (move_down): no lane's branch stands in front of a load.
// (With one, a row's first and last lanes made their whole wave wait for one load after the other.)  Rows shorter than a vector
// (ld_short) have kernels of their own, WHOLE false: as a branch of the same kernel they made the others wait for the taps before they asked
// for x (fp32 forward, b4 C256 l2048 5.0 us, 4.3 without).

// `v` without its first `gone` tokens (the same number for the whole launch), zeros behind the others, in the lanes that `cut` says.
// By words and then by half of one: a 64-bit shift by a lane's amount gave wrong high words here where the compiler had put the amount
// into a wave's last register.
template <typename T, int N>
__device__ __forceinline__ Tokens<T, N> move_down(const Tokens<T, N>& v, int gone, bool cut) {
    if (gone <= 0) return v;
    constexpr int W = N * (int)sizeof(T) / 4;
    uint32_t old[W], w[W + 1];
    __builtin_memcpy(old, &v, sizeof(v));
    if (gone >= N) {
#pragma unroll
        for (int i = 0; i < W; ++i) w[i] = 0;
    } else {
#pragma unroll
        for (int i = 0; i < W; ++i) w[i] = old[i];
        w[W] = 0;
        const int words = gone * (int)sizeof(T) / 4;
#pragma unroll
        for (int by = W / 2; by > 0; by /= 2)
            if (words & by) {
#pragma unroll
                for (int i = 0; i < W; ++i) w[i] = i + by < W ? w[i + by] : 0u;
            }
        if (sizeof(T) == 2 && (gone & 1)) {
#pragma unroll
            for (int i = 0; i < W; ++i) w[i] = (w[i] >> 16) | (w[i + 1] << 16);
        }
    }
    uint32_t o[W];
#pragma unroll
    for (int i = 0; i < W; ++i) o[i] = cut ? w[i] : old[i];
    Tokens<T, N> r;
    __builtin_memcpy(&r, o, sizeof(r));
    return r;
}
// the same N tokens one by one, for rows shorter than a vector
template <typename T, int N>
__device__ __forceinline__ Tokens<T, N> ld_short(const T* __restrict__ row, int64_t t, int64_t l) {
    Tokens<T, N> r;
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = (t + i >= 0 && t + i < l) ? row[t + i] : from_f32<T>(0.f);
    return r;
}
// The last four tokens of the lane below's V, which stand in front of this lane's own; lane 0 keeps `own`.
template <typename T, int V>
__device__ __forceinline__ Tokens<T, 4> tokens_below(const Tokens<T, 4>& own, const Tokens<T, V>& v) {
    constexpr int W = (int)sizeof(T), F = (V - 4) * W / 4;      // words of four tokens; the first of them in v
    uint32_t o[W], all[V * W / 4];
    __builtin_memcpy(o, &own, sizeof(own));
    __builtin_memcpy(all, &v, sizeof(v));
#pragma unroll
    for (int i = 0; i < W; ++i) o[i] = __builtin_amdgcn_update_dpp(o[i], all[F + i], 0x138, 0xF, 0xF, false);      // wave_shr:1
    Tokens<T, 4> r;
    __builtin_memcpy(&r, o, sizeof(r));
    return r;
}
template <typename T, int N>
__device__ __forceinline__ void st_tokens(T* __restrict__ row, int64_t t, int64_t l, const float (&in)[N]) {
    if (t + N <= l) {
        st_stream<T, N>(row + t, in);
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (t + i < l) row[t + i] = from_f32<T>(in[i]);
    }
}
template <typename WT>
__device__ __forceinline__ void ld_row_taps(const void* __restrict__ w, const void* __restrict__ bias, int64_t c, float (&wv)[4], float& bv) {
    ld_elems<WT, 4>(static_cast<const WT*>(w) + c * 4, wv);
    bv = bias ? to_f32(static_cast<const WT*>(bias)[c]) : 0.f;
}

// One thread per 16-byte piece of a row: its own tokens, and the 4 before them from the lane below, eight
// waves' worth of pieces per SIMD in flight.  HBM bound, kernel alone in a stream of them with its inputs cold: b4 C5376 l2048 bf16 30 us (176 MB,
// 5.9 TB/s; 37 with a branch in front of the row ends' loads), fp32 58.3 (62 with the four tokens loaded and behind the taps).
template <typename T, typename WT, int ACT, bool WHOLE>
__global__ void __launch_bounds__(256)
conv_fwd_cm_kernel(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias, T* __restrict__ y,
                   int64_t l, uint32_t C, uint32_t pieces, uint32_t total, int64_t xsb, int64_t xsc, int64_t ysb, int64_t ysc) {
    constexpr int V = VecTraits<T>::kVec;
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= total) return;
    const uint32_t row = idx / pieces, b = row / C, c = row - b * C;
    const int64_t t0 = (int64_t)(idx - row * pieces) * V;
    const T* xr = x + b * xsb + c * xsc;
    float h[4], cur[V], wv[4], bv, o[V];
    Tokens<T, 4> rh{};
    Tokens<T, V> rc;
    const int gone = WHOLE ? (int)((int64_t)pieces * V - l) : 0;      // what the row's last piece lacks
    const bool cut = WHOLE && idx - row * pieces == pieces - 1;
    if constexpr (WHOLE) {
        rc = ld_whole<T, V>(xr + t0 - (cut ? gone : 0));
        if ((threadIdx.x & 63) == 0 && t0 > 0) rh = ld_whole<T, 4>(xr + t0 - 4);
    } else {
        rc = ld_short<T, V>(xr, t0, l);
    }
    ld_row_taps<WT>(w, bias, c, wv, bv);
    if constexpr (WHOLE) {
        rh = tokens_below<T, V>(rh, rc);
        if (gone > 0 && __any(cut)) rc = move_down<T, V>(rc, gone, cut);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = t0 > 0 ? to_f32(rh[i]) : 0.f;
#pragma unroll
    for (int i = 0; i < V; ++i) cur[i] = to_f32(rc[i]);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        float z = bv;
#pragma unroll
        for (int k = 0; k < 4; ++k) z += wv[k] * (i + k < 3 ? h[1 + i + k] : cur[i + k - 3]);
        o[i] = act_f<ACT>(z);
    }
    st_tokens<T, V>(y + b * ysb + c * ysc, t0, l, o);
}

// One wave per (channel, split): its lanes walk the channel's pieces of two vectors of tokens over all rows of the batch,
// so the sums of dw and db stay in registers until the end, and the next piece is on its way while this one is computed.  The 1, 2 or
// 4 (`inner`) splits of a channel inside a workgroup meet in LDS and finish it there; only with more of them (long channels) do fp32
// partials go to conv_reduce_partials_kernel, whose launch is 2 to 4 us.  Where a channel has no more than 32 pieces, `lanes` of the wave (a
// power of two) take it and the others the channels behind it.
// A lane recomputes the three tokens behind its own for the dx lag: 3 in 16
// (bf16) more activations, against a cross-lane exchange that would break at every row end.
// What bounds it: the vector units (some 40 us of activations recomputed, at b4 C5376 l2048 bf16) beside 264 MB of traffic (44 us), in
// waves of their own each waiting for its loads: 94 -> 67 us there, cold and in a stream of them, without a lane's branch in front of the loads and
// with the next piece under way (in a row of forward and backward passes of autograd, which find some of their inputs cached, 71 -> 61; five waves a
// SIMD spill: 77); 3 x 4097 rows of 1001 38 -> 27, 10240 rows of 77 19.7 -> 5.9.
template <typename T, typename WT, int ACT, bool WHOLE>
__global__ void __launch_bounds__(256, 4)
conv_bwd_cm_kernel(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias, const T* __restrict__ dy,
                   T* __restrict__ dx, float* __restrict__ part, void* __restrict__ dw, void* __restrict__ db,
                   int64_t l, uint32_t C, uint32_t lanes, uint32_t inner, uint32_t outer, uint32_t pieces, uint32_t per_split, uint32_t total,
                   int64_t xsb, int64_t xsc, int64_t gsb, int64_t gsc, int64_t dsb, int64_t dsc) {
    constexpr int V = VecTraits<T>::kVec, N = 2 * V;
    constexpr int pd = std::is_same<WT, float>::value ? M2_F32 : M2_BF16;
    __shared__ float red[4][5];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & (lanes - 1), sub = wave & (inner - 1);
    const uint32_t unit = lanes < 64 ? (blockIdx.x * 256u + threadIdx.x) >> __builtin_ctz(lanes) : (blockIdx.x * 4u + wave) >> __builtin_ctz(inner);      // powers of two
    const bool live = unit < C * outer;            // the last workgroup may have fewer channels
    const uint32_t part_row = live && outer > 1 ? unit / C : 0, c = live ? unit - part_row * C : 0, split = part_row * inner + sub;
    const uint32_t end = !live ? 0 : (split + 1) * per_split < total ? (split + 1) * per_split : total;
    float wv[4], bv, acc[5];
    ld_row_taps<WT>(w, bias, c, wv, bv);
#pragma unroll
    for (int k = 0; k < 5; ++k) acc[k] = 0.f;
    struct Piece { Tokens<T, 4> xa, xd, gc; Tokens<T, V> xb, xc, ga, gb; };
    auto load = [&](uint32_t p) {
        const uint32_t b = p / pieces;
        const int64_t t0 = (int64_t)(p - b * pieces) * N;
        const T* xr = x + b * xsb + c * xsc;
        const T* gr = dy + b * gsb + c * gsc;
        Piece q;
        if constexpr (WHOLE) {
            // what the row's last piece lacks of its two vectors, and the piece before it of the four tokens behind it
            const int lacks = (int)((int64_t)pieces * N - l);
            const bool last = t0 + N >= l, near = t0 + N + 4 > l;
            const int64_t tb = t0 + V > l ? l - V : t0, tc = t0 + N > l ? l - V : t0 + V, td = near ? l - 4 : t0 + N;
            q.xb = ld_whole<T, V>(xr + tb); q.ga = ld_whole<T, V>(gr + tb); q.xc = ld_whole<T, V>(xr + tc); q.gb = ld_whole<T, V>(gr + tc);
            q.xa = ld_whole<T, 4>(xr + (t0 > 0 ? t0 - 4 : 0)); q.xd = ld_whole<T, 4>(xr + td); q.gc = ld_whole<T, 4>(gr + td);
            if (lacks > 0 && __any(near)) {
                q.xb = move_down<T, V>(q.xb, lacks - V, last); q.ga = move_down<T, V>(q.ga, lacks - V, last);
                q.xc = move_down<T, V>(q.xc, lacks, last); q.gb = move_down<T, V>(q.gb, lacks, last);
                q.xd = move_down<T, 4>(q.xd, lacks - (N - 4), near); q.gc = move_down<T, 4>(q.gc, lacks - (N - 4), near);
            }
        } else {
            q.xb = ld_short<T, V>(xr, t0, l); q.ga = ld_short<T, V>(gr, t0, l);
            q.xc = q.gb = (T)0.f;
            q.xa = q.xd = q.gc = (T)0.f;
        }
        return q;
    };
    Piece next{};
    uint32_t p = split * per_split + lane;
    if (p < end) next = load(p);
    for (; p < end; p += lanes) {
        const Piece q = next;
        if (p + lanes < end) next = load(p + lanes);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t b = p / pieces;
        const int64_t t0 = (int64_t)(p - b * pieces) * N;
        const bool more = t0 + N < l;
        T* dr = dx + b * dsb + c * dsc;
        float xw[N + 8], g[N + 4];                 // x[t0 - 4 ...], dy -> g = dy * act'(z) from t0 on
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            xw[i] = t0 > 0 ? to_f32(q.xa[i]) : 0.f;
            xw[4 + N + i] = more ? to_f32(q.xd[i]) : 0.f;
            g[N + i] = more ? to_f32(q.gc[i]) : 0.f;
        }
#pragma unroll
        for (int i = 0; i < V; ++i) {
            xw[4 + i] = to_f32(q.xb[i]); xw[4 + V + i] = to_f32(q.xc[i]);
            g[i] = to_f32(q.ga[i]); g[V + i] = to_f32(q.gb[i]);
        }
#pragma unroll
        for (int i = 0; i < N + 3; ++i) {
            const float z = bv + wv[0] * xw[i + 1] + wv[1] * xw[i + 2] + wv[2] * xw[i + 3] + wv[3] * xw[i + 4];
            g[i] *= act_grad_f<ACT>(z);            // dy is 0 behind the row's end
            if (i < N) {
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[k] += xw[i + 1 + k] * g[i];
                acc[4] += g[i];
            }
        }
        float oa[V], ob[V];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float o = wv[3] * g[i] + wv[2] * g[i + 1] + wv[1] * g[i + 2] + wv[0] * g[i + 3];
            if (i < V) oa[i] = o; else ob[i - V] = o;
        }
        st_tokens<T, V>(dr, t0, l, oa);
        if (t0 + V < l) st_tokens<T, V>(dr, t0 + V, l, ob);
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        float v = acc[k];
        if (lanes > 1) v = lane_xor_add<1>(v);
        if (lanes > 2) v = lane_xor_add<2>(v);
        if (lanes > 4) v = lane_xor_add<4>(v);
        if (lanes > 8) v = lane_xor_add<8>(v);
        if (lanes > 16) v = lane_xor_add<16>(v);
        if (lanes > 32) v = lane_xor_add<32>(v);
        acc[k] = v;
    }
    if (lanes < 64) {                              // a channel's only lanes
        if (live && lane == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) st_param(dw, pd, (int64_t)c * 4 + k, acc[k]);
            if (db) st_param(db, pd, c, acc[4]);
        }
        return;
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) red[wave][k] = acc[k];
    }
    __syncthreads();
    if (const uint32_t k = threadIdx.x & 63; live && sub == 0 && k < 5) {
        float v = 0.f;
        for (uint32_t q = 0; q < inner; ++q) v += red[wave + q][k];
        if (outer > 1) part[((int64_t)part_row * C + c) * 5 + k] = v;
        else if (k < 4) st_param(dw, pd, (int64_t)c * 4 + k, v);
        else if (db) st_param(db, pd, c, v);
    }
}

// ------------------------------------------------------------------------------------------
// Generic path: any strides / layout, k <= 8, one thread per output element.
template <typename T>
__global__ void conv_fwd_generic_kernel(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias,
                                        const T* __restrict__ hist, int W, T* __restrict__ y, int64_t nb, int64_t l, int64_t C, int k,
                                        int64_t xsb, int64_t xsl, int64_t xsc, int64_t ysb, int64_t ysl, int64_t ysc,
                                        int pd, int act, int t_fastest) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nb * l * C) return;
    int64_t b, t, c;
    if (t_fastest) { t = idx % l; c = (idx / l) % C; b = idx / (l * C); }
    else { c = idx % C; t = (idx / C) % l; b = idx / (l * C); }
    float z = bias ? ld_param(bias, pd, c) : 0.f;
    for (int i = 0; i < k; ++i) {
        const int64_t tt = t - (k - 1) + i;
        if (tt >= 0) z += ld_param(w, pd, c * k + i) * to_f32(x[b * xsb + tt * xsl + c * xsc]);
        else if (hist) z += ld_param(w, pd, c * k + i) * to_f32(hist[(b * C + c) * W + W + tt]);
    }
    const float o = act == M2_ACT_SILU ? silu_f(z) : (act == M2_ACT_RELU ? (z > 0.f ? z : 0.f) : z);
    y[b * ysb + t * ysl + c * ysc] = from_f32<T>(o);
}

// The last W inputs of a sequence into the decode cache [b][C][W], oldest first; one thread per channel.  Where the sequence
// is shorter than W, what is left of the cache (or zeros) moves up; a thread reads ahead of what it writes.
template <typename T>
__global__ void __launch_bounds__(256)
conv_tail_kernel(const T* __restrict__ x, T* state, int W, int keep, int64_t nb, int64_t l, int64_t C, int64_t xsb, int64_t xsl, int64_t xsc) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= nb * C) return;
    const int64_t b = idx / C, c = idx % C;
    T* sp = state + idx * W;
    for (int w = 0; w < W; ++w) {
        const int64_t t = l - W + w;
        sp[w] = t >= 0 ? x[b * xsb + t * xsl + c * xsc] : (keep ? sp[w + l] : from_f32<T>(0.f));
    }
}

template <typename T>
__device__ __forceinline__ float conv_g_at(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias,
                                           const T* __restrict__ dy, int64_t b, int64_t t, int64_t c, int k,
                                           int64_t xsb, int64_t xsl, int64_t xsc, int64_t gsb, int64_t gsl, int64_t gsc,
                                           int pd, int act) {
    float z = bias ? ld_param(bias, pd, c) : 0.f;
    for (int i = 0; i < k; ++i) {
        const int64_t tt = t - (k - 1) + i;
        if (tt >= 0) z += ld_param(w, pd, c * k + i) * to_f32(x[b * xsb + tt * xsl + c * xsc]);
    }
    const float d = act == M2_ACT_SILU ? silu_grad_f(z) : (act == M2_ACT_RELU ? (z > 0.f ? 1.f : 0.f) : 1.f);
    return to_f32(dy[b * gsb + t * gsl + c * gsc]) * d;
}

template <typename T>
__global__ void conv_bwd_dx_generic_kernel(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias,
                                           const T* __restrict__ dy, T* __restrict__ dx, int64_t nb, int64_t l, int64_t C, int k,
                                           int64_t xsb, int64_t xsl, int64_t xsc, int64_t gsb, int64_t gsl, int64_t gsc,
                                           int64_t dsb, int64_t dsl, int64_t dsc, int pd, int act, int t_fastest) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nb * l * C) return;
    int64_t b, t, c;
    if (t_fastest) { t = idx % l; c = (idx / l) % C; b = idx / (l * C); }
    else { c = idx % C; t = (idx / C) % l; b = idx / (l * C); }
    float s = 0.f;
    for (int i = 0; i < k; ++i) {
        const int64_t tt = t + (k - 1) - i;
        if (tt < l) s += ld_param(w, pd, c * k + i) * conv_g_at(x, w, bias, dy, b, tt, c, k, xsb, xsl, xsc, gsb, gsl, gsc, pd, act);
    }
    dx[b * dsb + t * dsl + c * dsc] = from_f32<T>(s);
}

// one block per channel; threads stride over (b, t)
template <typename T>
__global__ void __launch_bounds__(256)
conv_bwd_dw_generic_kernel(const T* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias,
                           const T* __restrict__ dy, void* __restrict__ dw, void* __restrict__ db,
                           int64_t nb, int64_t l, int k, int64_t xsb, int64_t xsl, int64_t xsc,
                           int64_t gsb, int64_t gsl, int64_t gsc, int pd, int act) {
    __shared__ float red[4][kMaxK + 1];
    const int64_t c = blockIdx.x;
    float acc[kMaxK + 1];
#pragma unroll
    for (int i = 0; i <= kMaxK; ++i) acc[i] = 0.f;
    for (int64_t e = threadIdx.x; e < nb * l; e += blockDim.x) {
        const int64_t b = e / l, t = e % l;
        const float g = conv_g_at(x, w, bias, dy, b, t, c, k, xsb, xsl, xsc, gsb, gsl, gsc, pd, act);
#pragma unroll
        for (int i = 0; i < kMaxK; ++i) {
            if (i < k) {
                const int64_t tt = t - (k - 1) + i;
                if (tt >= 0) acc[i] += to_f32(x[b * xsb + tt * xsl + c * xsc]) * g;
            }
        }
        acc[kMaxK] += g;
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i <= kMaxK; ++i) {
        const float s = warp_sum(acc[i]);
        if (lane == 0) red[wave][i] = s;
    }
    __syncthreads();
    if (threadIdx.x <= kMaxK) {
        const int i = threadIdx.x;
        const float s = red[0][i] + red[1][i] + red[2][i] + red[3][i];
        if (i < k) st_param(dw, pd, c * k + i, s);
        else if (i == kMaxK && db) st_param(db, pd, c, s);
    }
}

// elements per thread: 16-byte vectors forward, 8-byte vectors backward (the backward carries twice the
// per-channel state in registers; halving the vector keeps its occupancy up)
template <typename T> constexpr int conv_vec(bool bwd) {
    const int v = (int)((bwd ? M2_CONV_VB : M2_CONV_VF) / sizeof(T));
    return v < 2 ? 2 : v;
}

// Channels-last kernels: unit channel strides; a row must hold one vector.
template <int V>
bool channels_last_ok(const m2_conv1d_params* p, bool bwd) {
    return p->k == 4 && p->x_stride_c == 1 && p->y_stride_c == 1 && p->channels >= V && (!bwd || p->dx_stride_c == 1);
}
// Channel-major kernels: unit token strides; the flattened pieces are counted in 32 bits.
bool channel_major_ok(const m2_conv1d_params* p, bool bwd) {
    return p->k == 4 && p->x_stride_l == 1 && p->y_stride_l == 1 && (!bwd || p->dx_stride_l == 1) &&
           p->channels < (int64_t(1) << 24) && p->batch * p->channels * ceil_div(p->seqlen, (int64_t)4) < (int64_t(1) << 31);
}

// calls f<parameter type, activation>
template <typename F>
void conv_dispatch(const m2_conv1d_params* p, F&& f) {
    auto act = [&](auto wt) {
        using WT = decltype(wt);
        if (p->activation == M2_ACT_SILU) f(WT{}, std::integral_constant<int, M2_ACT_SILU>{});
        else if (p->activation == M2_ACT_RELU) f(WT{}, std::integral_constant<int, M2_ACT_RELU>{});
        else f(WT{}, std::integral_constant<int, M2_ACT_NONE>{});
    };
    if (p->param_dtype == M2_F32) act(float{}); else act(bf16_t{});
}

int check_common(const m2_conv1d_params* p) {
    M2_REQUIRE(p, M2_ERR_NULL, "conv1d: params is NULL");
    M2_REQUIRE(p->batch >= 0 && p->seqlen >= 0 && p->channels >= 0, M2_ERR_SHAPE, "conv1d: negative dimension");
    M2_REQUIRE(p->k >= 1 && p->k <= kMaxK, M2_ERR_SHAPE, "conv1d: kernel size %d not in [1, %d]", p->k, kMaxK);
    M2_REQUIRE(p->dtype == M2_F32 || p->dtype == M2_BF16, M2_ERR_DTYPE, "conv1d: bad dtype %d", p->dtype);
    M2_REQUIRE(p->param_dtype == M2_F32 || p->param_dtype == M2_BF16, M2_ERR_DTYPE, "conv1d: bad param dtype %d", p->param_dtype);
    M2_REQUIRE(p->activation >= M2_ACT_NONE && p->activation <= M2_ACT_RELU, M2_ERR_SHAPE, "conv1d: bad activation %d", p->activation);
    M2_REQUIRE(p->batch <= 65535, M2_ERR_SHAPE, "conv1d: batch %lld > 65535", (long long)p->batch);
    return M2_OK;
}

// state: null, or the decode cache of W >= k - 1 inputs, [b][C][W], oldest first: in front of the sequence where `continuing`,
// and its last ones afterwards
template <typename T>
int launch_fwd(const m2_conv1d_params* p, void* state_, int W, bool continuing, hipStream_t st) {
    T* state = static_cast<T*>(state_);
    const T* hist = continuing ? state : nullptr;
    bool tail = state != nullptr;      // still to be left by conv_tail_kernel
    const int64_t nb = p->batch, l = p->seqlen, C = p->channels;
    const T* x = static_cast<const T*>(p->x);
    T* y = static_cast<T*>(p->y);
    constexpr int V = conv_vec<T>(false);
    if (channels_last_ok<V>(p, false)) {
        const int64_t CV = ceil_div(C, (int64_t)V), tl = conv_fwd_tokens(nb, l, CV), nseg = ceil_div(l, tl);
        dim3 grid((unsigned)ceil_div(CV, kCVT), (unsigned)ceil_div(nseg, kSEG), (unsigned)nb), block(kCVT, kSEG);
        M2_REQUIRE(grid.y <= 65535, M2_ERR_SHAPE, "conv1d: sequence too long for the grid");
        const bool fold = tail && C % V == 0;
        const int flags = (continuing ? kContinuing : 0) | (fold ? kTail : 0);
        conv_dispatch(p, [&](auto wt, auto act) {
            with_fwd_tokens(tl, [&](auto t) {
                auto k = state ? conv_fwd_cl_kernel<T, decltype(wt), V, decltype(act)::value, true, decltype(t)::value>
                               : conv_fwd_cl_kernel<T, decltype(wt), V, decltype(act)::value, false, decltype(t)::value>;
                k<<<grid, block, 0, st>>>(x, p->w, p->bias, state, W, flags, y, l, C, p->x_stride_b, p->x_stride_l, p->y_stride_b, p->y_stride_l);
            });
        });
        tail = tail && !fold;
    } else if (!hist && channel_major_ok(p, false)) {
        const int64_t pieces = ceil_div(l, (int64_t)VecTraits<T>::kVec), total = nb * C * pieces;
        conv_dispatch(p, [&](auto wt, auto act) {
            auto go = [&](auto k) {
                k<<<(unsigned)ceil_div(total, (int64_t)256), 256, 0, st>>>(x, p->w, p->bias, y, l, (uint32_t)C, (uint32_t)pieces, (uint32_t)total, p->x_stride_b, p->x_stride_c,
                                                                          p->y_stride_b, p->y_stride_c);
            };
            if (l >= VecTraits<T>::kVec) go(conv_fwd_cm_kernel<T, decltype(wt), decltype(act)::value, true>);
            else go(conv_fwd_cm_kernel<T, decltype(wt), decltype(act)::value, false>);
        });
    } else {
        const int64_t total = nb * l * C;
        const int tf = (p->x_stride_l == 1 && p->x_stride_c != 1) ? 1 : 0;
        conv_fwd_generic_kernel<T><<<(unsigned)ceil_div(total, 256), 256, 0, st>>>(
            x, p->w, p->bias, hist, W, y, nb, l, C, p->k, p->x_stride_b, p->x_stride_l, p->x_stride_c,
            p->y_stride_b, p->y_stride_l, p->y_stride_c, p->param_dtype, p->activation, tf);
    }
    const int rc = check_launch("conv1d_fwd");
    if (rc || !tail) return rc;
    conv_tail_kernel<T><<<(unsigned)ceil_div(nb * C, (int64_t)256), 256, 0, st>>>(x, state, W, continuing, nb, l, C, p->x_stride_b, p->x_stride_l, p->x_stride_c);
    return check_launch("conv1d_tail");
}

// slots: null, or where the number of partial rows goes that are left in the workspace instead of summed (0: dw and db are there)
template <typename T>
int launch_bwd(const m2_conv1d_params* p, int64_t* slots, hipStream_t st) {
    const int64_t nb = p->batch, l = p->seqlen, C = p->channels;
    const T* x = static_cast<const T*>(p->x);
    const T* dy = static_cast<const T*>(p->dy);
    T* dx = static_cast<T*>(p->dx);
    constexpr int V = conv_vec<T>(true);
    if (channels_last_ok<V>(p, true)) {
        const int64_t CV = ceil_div(C, (int64_t)V), tl = conv_bwd_tokens(nb, l, C), nseg = ceil_div(l, tl);
        dim3 grid((unsigned)ceil_div(CV, kCVT), (unsigned)ceil_div(nseg, kSEG), (unsigned)nb), block(kCVT, kSEG);
        M2_REQUIRE(grid.y <= 65535, M2_ERR_SHAPE, "conv1d: sequence too long for the grid");
        const int64_t nslots = (int64_t)grid.y * grid.z;
        const size_t need = (size_t)nslots * C * 5 * sizeof(float);
        M2_REQUIRE(p->workspace && p->workspace_bytes >= need, M2_ERR_WORKSPACE,
                   "conv1d_bwd: workspace %zu bytes < %zu needed", p->workspace_bytes, need);
        float* part = static_cast<float*>(p->workspace);
        conv_dispatch(p, [&](auto wt, auto act) {
            with_bwd_tokens(tl, [&](auto t) {
                conv_bwd_cl_kernel<T, decltype(wt), V, decltype(act)::value, decltype(t)::value><<<grid, block, 0, st>>>(
                    x, p->w, p->bias, dy, dx, part, l, C, p->x_stride_b, p->x_stride_l, p->y_stride_b, p->y_stride_l, p->dx_stride_b, p->dx_stride_l);
            });
        });
        int rc = check_launch("conv1d_bwd");
        if (rc) return rc;
        if (slots) { *slots = nslots; return M2_OK; }
        conv_reduce_partials_kernel<<<(unsigned)ceil_div(C * 5 * 4, (int64_t)256), 256, 0, st>>>(part, nslots, C, 4, p->dw, p->db, p->param_dtype);
        return check_launch("conv1d_bwd_reduce");
    }
    if (channel_major_ok(p, true)) {
        const int64_t pieces = ceil_div(l, (int64_t)(2 * VecTraits<T>::kVec)), total = nb * pieces;
        int64_t lanes = 64;
        while (lanes > 1 && lanes / 2 >= total) lanes /= 2;
        const int64_t rounds = ceil_div(total, lanes);
        // A channel's rounds over the four waves of one workgroup; where they are many, over several workgroups, whose partials cost a launch
        // more, in as many rounds a wave as take the least time: a chain of rounds (1.6 us each) or, beyond one workgroup per CU, what a
        // CU's workgroups do at 1.2 us a round; chains of more than three lose an eighth to that.  Four waves | one | two | four rounds, us: 17 x 20
        // channels x 795 bf16 10.9 | 7.8 | 9.5, fp32 11.5 | 7.3 | 8.2 | 10.0; 35 x 3 x 2818 bf16 38.9 | 8.7 | 10.0 | 12.2; 31 x 188 x 9665 bf16 141 |
        // 115 | 108 | 114, fp32 209 | 169 | 174 | 196; 25 x 118 x 1798 bf16 23 | 16.0 | 15.5 | 17.4; 4 x 5376 x 2048 fp32 139 | 122 | 127; 1 x 5646 x 4789
        // fp32 82 | 93 | 101; 7 x 412 x 1279 fp32 13.8 | 16.7 | 17.5 | 15.4.  Up to eight rounds the launch is not earned: 4 x 5376 x 2048
        // bf16 68 | 72, 1 x 16 x 8192 6.2 | 6.8.
        int64_t inner = rounds >= 3 ? 4 : rounds, outer = 1, r = ceil_div(rounds, inner);
        if (rounds > 8) {
            auto cost = [&](int64_t k, int64_t n) {
                const float us = (float)k * std::max(1.6f, 1.2f * (float)(C * n) / (float)device_cus());
                return (k > 3 ? 1.13f * us : us) + (n > 1 ? 3.f + 0.04f * (float)n : 0.f);
            };
            float least = cost(r, 1);
            for (int64_t k = 1; ceil_div(rounds, k) > 4; k *= 2) {
                const int64_t n = ceil_div(rounds, 4 * k);
                const float us = cost(k, n);
                if (us < least) { least = us; outer = n; r = k; }
            }
        }
        const int64_t per_split = r * lanes;
        float* part = static_cast<float*>(p->workspace);
        M2_REQUIRE(outer == 1 || (part && p->workspace_bytes >= (size_t)(outer * C * 5) * sizeof(float)), M2_ERR_WORKSPACE,
                   "conv1d_bwd: workspace %zu bytes < %zu needed", p->workspace_bytes, (size_t)(outer * C * 5) * sizeof(float));
        conv_dispatch(p, [&](auto wt, auto act) {
            auto go = [&](auto k) {
                k<<<(unsigned)(lanes < 64 ? ceil_div(C * lanes, (int64_t)256) : ceil_div(C * outer * inner, (int64_t)4)), 256, 0, st>>>(
                    x, p->w, p->bias, dy, dx, part, p->dw, p->db, l, (uint32_t)C, (uint32_t)lanes, (uint32_t)inner, (uint32_t)outer, (uint32_t)pieces, (uint32_t)per_split,
                    (uint32_t)total, p->x_stride_b, p->x_stride_c, p->y_stride_b, p->y_stride_c, p->dx_stride_b, p->dx_stride_c);
            };
            if (l >= VecTraits<T>::kVec) go(conv_bwd_cm_kernel<T, decltype(wt), decltype(act)::value, true>);
            else go(conv_bwd_cm_kernel<T, decltype(wt), decltype(act)::value, false>);
        });
        int rc = check_launch("conv1d_bwd");
        if (rc || outer == 1) return rc;
        conv_reduce_partials_kernel<<<(unsigned)ceil_div(C * 5 * 4, (int64_t)256), 256, 0, st>>>(part, outer, C, 4, p->dw, p->db, p->param_dtype);
        return check_launch("conv1d_bwd_reduce");
    }
    const int64_t total = nb * l * C;
    const int tf = (p->x_stride_l == 1 && p->x_stride_c != 1) ? 1 : 0;
    conv_bwd_dx_generic_kernel<T><<<(unsigned)ceil_div(total, 256), 256, 0, st>>>(
        x, p->w, p->bias, dy, dx, nb, l, C, p->k, p->x_stride_b, p->x_stride_l, p->x_stride_c,
        p->y_stride_b, p->y_stride_l, p->y_stride_c, p->dx_stride_b, p->dx_stride_l, p->dx_stride_c,
        p->param_dtype, p->activation, tf);
    int rc = check_launch("conv1d_bwd_dx");
    if (rc) return rc;
    conv_bwd_dw_generic_kernel<T><<<(unsigned)C, 256, 0, st>>>(x, p->w, p->bias, dy, p->dw, p->db, nb, l, p->k,
                                                                p->x_stride_b, p->x_stride_l, p->x_stride_c,
                                                                p->y_stride_b, p->y_stride_l, p->y_stride_c, p->param_dtype, p->activation);
    return check_launch("conv1d_bwd_dw");
}

}  // namespace
}  // namespace m2

extern "C" int m2_conv1d_fwd(const m2_conv1d_params* p, void* stream) {
    using namespace m2;
    int rc = check_common(p);
    if (rc) return rc;
    if (p->batch == 0 || p->seqlen == 0 || p->channels == 0) return M2_OK;
    M2_REQUIRE(p->x && p->w && p->y, M2_ERR_NULL, "conv1d_fwd: x, w and y are required");
    M2_DISPATCH_DTYPE(p->dtype, T, return launch_fwd<T>(p, nullptr, 0, false, static_cast<hipStream_t>(stream)));
    return M2_OK;
}

extern "C" int m2_conv1d_prefill(const m2_conv1d_params* p, void* conv_state, int32_t W, int32_t continuing, void* stream) {
    using namespace m2;
    int rc = check_common(p);
    if (rc) return rc;
    if (p->batch == 0 || p->seqlen == 0 || p->channels == 0) return M2_OK;
    M2_REQUIRE(p->x && p->w && p->y && conv_state, M2_ERR_NULL, "conv1d_prefill: x, w, y and conv_state are required");
    M2_REQUIRE(W >= p->k - 1, M2_ERR_SHAPE, "conv1d_prefill: the cache holds %d inputs, needs %d", W, p->k - 1);
    M2_DISPATCH_DTYPE(p->dtype, T, return launch_fwd<T>(p, conv_state, W, continuing != 0, static_cast<hipStream_t>(stream)));
    return M2_OK;
}

extern "C" size_t m2_conv1d_bwd_workspace_bytes(int64_t batch, int64_t seqlen, int64_t channels, int32_t k) {
    using namespace m2;
    (void)k;
    const int64_t nseg = ceil_div(seqlen, conv_bwd_tokens(batch, seqlen, channels));
    return (size_t)(ceil_div(nseg, kSEG) * batch * channels * 5) * sizeof(float) + 16;
}

namespace m2 {
namespace {
int conv1d_bwd(const m2_conv1d_params* p, int64_t* slots, void* stream) {
    int rc = check_common(p);
    if (rc) return rc;
    M2_REQUIRE(p->dw, M2_ERR_NULL, "conv1d_bwd: dw is required");
    if (p->channels == 0) return M2_OK;
    if (p->batch == 0 || p->seqlen == 0) {
        // empty reduction: gradients of the parameters are zero
        hipStream_t st = static_cast<hipStream_t>(stream);
        const size_t esz = p->param_dtype == M2_F32 ? 4 : 2;
        const int64_t nw = p->channels * p->k * (int64_t)(esz / 2), nb = p->channels * (int64_t)(esz / 2);     // 16-bit words
        conv_zero_kernel<<<(unsigned)ceil_div(nw, (int64_t)256), 256, 0, st>>>(static_cast<uint16_t*>(p->dw), nw);
        if (p->db) conv_zero_kernel<<<(unsigned)ceil_div(nb, (int64_t)256), 256, 0, st>>>(static_cast<uint16_t*>(p->db), nb);
        return check_launch("conv1d_bwd_zero");
    }
    M2_REQUIRE(p->x && p->w && p->dy && p->dx, M2_ERR_NULL, "conv1d_bwd: x, w, dy, dx are required");
    M2_DISPATCH_DTYPE(p->dtype, T, return launch_bwd<T>(p, slots, static_cast<hipStream_t>(stream)));
    return M2_OK;
}
}  // namespace
}  // namespace m2

extern "C" int m2_conv1d_bwd(const m2_conv1d_params* p, void* stream) { return m2::conv1d_bwd(p, nullptr, stream); }

extern "C" int m2_conv1d_bwd_partial(const m2_conv1d_params* p, int64_t* slots, void* stream) {
    using namespace m2;
    M2_REQUIRE(slots, M2_ERR_NULL, "conv1d_bwd_partial: slots is required");
    *slots = 0;
    return conv1d_bwd(p, slots, stream);
}
