// Elementwise glue of the mixer core as HBM-bound kernels: softplus(dt + dt_bias) and the gated, grouped RMSNorm,
// forward and backward (mamba2/fused_kernel.py:33-73 softplus_with_bias(_bwd), :76-175 rmsnorm(_bwd); torch twins
// mamba2/mamba2_mixer.py:36-38, 88-105).  Every tensor is read once and written once; all arithmetic is fp32.
//
//   softplus:  out = v < 10 ? log(1 + e^v) : v,  v = dt + bias[h]              (threshold form, mamba2_mixer.py:36-38)
//              d_in = d_out * (v < 10 ? sigmoid(v) : 1),   d_bias[h] = sum over rows of d_in
//   rmsnorm:   h = x * silu(z);   out = w * h * rsqrt(mean_group(h^2) + eps)    per group of d / n_groups channels
//              backward (fused_kernel.py:159-171):  var = mean(h^2) + eps, r = rsqrt(var), gw = g w,
//              cf = mean(h gw) / var,  d_h = r (gw - cf h),  dx = d_h silu(z),  dz = d_h x silu'(z),  dw = sum_rows g h r
//
// A (row, group) is handled by a part of a wave (several groups of up to 32 vectors), by one wave (groups of up to 2048
// channels) or by the four or five waves of a workgroup (up to 8192), its channels in registers as 16-byte vectors; a workgroup takes many rows, so the per-channel weight
// and -- in the backward -- the dw accumulators stay in registers across rows.  dw and d_bias leave as per-block
// partials in a caller-owned workspace and are summed in a fixed order by a second small kernel (no atomics).
#include <initializer_list>

#include "sums.hpp"

namespace m2 {
namespace {

// ------------------------------------------------------------------------------------------ softplus
template <typename T>
__global__ void __launch_bounds__(256)
softplus_fwd_kernel(const T* __restrict__ dt, int64_t dt_sr, const float* __restrict__ bias, T* __restrict__ out, int64_t out_sr,
                    int64_t rows, int64_t nheads) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= rows * nheads) return;
    const int64_t row = idx / nheads, h = idx % nheads;
    const float v = to_f32(dt[row * dt_sr + h]) + bias[h];
    out[row * out_sr + h] = from_f32<T>(softplus_f(v));
}

constexpr int kSpRows = 16;      // rows per workgroup of the softplus backward
// 256 threads = 4 row phases x 64 heads; a workgroup walks kSpRows rows and leaves one partial row of d_bias
template <typename T>
__global__ void __launch_bounds__(256)
softplus_bwd_kernel(const T* __restrict__ dt, int64_t dt_sr, const float* __restrict__ bias, const T* __restrict__ d_out, int64_t do_sr,
                    T* __restrict__ d_in, int64_t di_sr, float* __restrict__ partial, int64_t rows, int64_t nheads) {
    __shared__ float red[4][64];
    const int hl = threadIdx.x & 63, ph = threadIdx.x >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * kSpRows;
    const int64_t r1 = r0 + kSpRows < rows ? r0 + kSpRows : rows;
    for (int64_t h0 = 0; h0 < nheads; h0 += 64) {
        const int64_t h = h0 + hl;
        float acc = 0.f;
        if (h < nheads) {
            const float bh = bias[h];
#pragma unroll 4
            for (int64_t r = r0 + ph; r < r1; r += 4) {
                const float v = to_f32(dt[r * dt_sr + h]) + bh;
                const float g = to_f32(d_out[r * do_sr + h]) * (v < kSoftplusThreshold ? sigmoid_f(v) : 1.f);
                d_in[r * di_sr + h] = from_f32<T>(g);
                acc += g;
            }
        }
        red[ph][hl] = acc;
        __syncthreads();
        if (ph == 0 && h < nheads) partial[(int64_t)blockIdx.x * nheads + h] = (red[0][hl] + red[1][hl]) + (red[2][hl] + red[3][hl]);
        __syncthreads();
    }
}

template <int V>
__global__ void __launch_bounds__(1024)
column_sum_kernel(const float* __restrict__ partial, float* __restrict__ out, int64_t nrows, int64_t ncols) {
    column_sum_body<V>(partial, nrows, ncols, blockIdx.x, [&](int64_t c, float v) { out[c] = v; });
}
int launch_column_sum(const float* partial, float* out, int64_t nrows, int64_t ncols, hipStream_t st) {
    const unsigned blocks = (unsigned)ceil_div(ncols, (int64_t)kSumCols);
    if (ncols % 4 == 0 && aligned16(partial)) column_sum_kernel<4><<<blocks, 1024, 0, st>>>(partial, out, nrows, ncols);
    else column_sum_kernel<1><<<blocks, 1024, 0, st>>>(partial, out, nrows, ncols);
    return check_launch("column_sum_kernel");
}

// ------------------------------------------------------------------------------------------ gated RMSNorm
struct NormArgs {
    const void* x; int64_t x_sr;            // [rows][d], channels contiguous
    const void* z; int64_t z_sr;            // gate, or null
    const float* w;                         // [d]
    void* out; int64_t out_sr; int out_f32; // forward output
    const void* g; int64_t g_sr;            // backward: d_out
    void* dx; int64_t dx_sr;
    void* dz; int64_t dz_sr;
    float* partial;                         // backward: [partial rows][d]
    int64_t rows, d, gw, groups, rows_per_block;    // gw = channels per group
    float eps;
};

template <typename T> struct GlueVec;
template <> struct GlueVec<bf16_t> { static constexpr int V = 8; };
template <> struct GlueVec<float> { static constexpr int V = 4; };

// The gate lies in rows of the packed projection, whose width is any number of elements (10 * 1024 + 256 + 13 heads): its vectors promise
// the alignment of an element only.  gfx950 issues the same 16-byte access either way: 8192 rows of
// 2112 channels in rows of 4513, 24.6 us against 23.6 for aligned rows (16384 x 5056: 100 and 92); 13115 rows of
// 1664 24.6 and 24.4, where a copy in front took 22.
typedef uint32_t AnyVec __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ uint4 load_any(const void* p) {
    const AnyVec v = *static_cast<const AnyVec*>(p);
    return uint4{v[0], v[1], v[2], v[3]};
}
template <typename T>
__device__ __forceinline__ void unpack_vec(const uint4 raw, float (&v)[GlueVec<T>::V]) {
    if constexpr (sizeof(T) == 2) {
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[2 * q] = __builtin_bit_cast(float, w[q] << 16);
            v[2 * q + 1] = __builtin_bit_cast(float, w[q] & 0xffff0000u);
        }
    } else {
        v[0] = __builtin_bit_cast(float, raw.x); v[1] = __builtin_bit_cast(float, raw.y);
        v[2] = __builtin_bit_cast(float, raw.z); v[3] = __builtin_bit_cast(float, raw.w);
    }
}
template <typename T>
__device__ __forceinline__ void store_vec(T* p, const float (&v)[GlueVec<T>::V]) {
    if constexpr (sizeof(T) == 2) {
        T e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) e[q] = from_f32<T>(v[q]);
        *reinterpret_cast<uint4*>(p) = *reinterpret_cast<const uint4*>(e);
    } else {
        *reinterpret_cast<floatx4*>(p) = floatx4{v[0], v[1], v[2], v[3]};
    }
}

// sum over runs of LPG lanes
template <int LPG>
__device__ __forceinline__ float lanes_sum(float v) {
    if constexpr (LPG == 64) return warp_sum(v);
    if constexpr (LPG >= 32) v = lane_xor_add<16>(v);
    if constexpr (LPG >= 16) v = lane_xor_add<8>(v);
    v = lane_xor_add<4>(v); v = lane_xor_add<2>(v); v = lane_xor_add<1>(v);
    return v;
}
// two sums over the lanes or, where WPG waves share a (row, group), over those; `slot` alternates between two LDS rows so that one barrier
// per reduction is enough
template <int WPG, int LPG>
__device__ __forceinline__ void group_sum2(float& a, float& b, float (*red)[2][16], int slot) {
    a = lanes_sum<LPG>(a); b = lanes_sum<LPG>(b);
    if constexpr (WPG > 1) {
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) { red[slot][0][wave] = a; red[slot][1][wave] = b; }
        __syncthreads();
        a = red[slot][0][0]; b = red[slot][1][0];
#pragma unroll
        for (int q = 1; q < WPG; ++q) { a += red[slot][0][q]; b += red[slot][1][q]; }      // fixed order
    }
}

// grid (row blocks, groups).  WPG = waves per (row, group): 1 (256 threads, each wave its own rows) or 4 or 5 (the whole
// workgroup of WPG waves shares a row).  LPG < 64: a wave takes 64 / LPG neighbouring groups of its row, LPG lanes each, and the
// grid has as many fewer columns.  NV = vectors per lane.  GATED: z given.  EXACT: the group is exactly WPG x 64 x NV
// vectors wide, so no lane is idle and nothing is masked (5120 channels of a 16-bit type = 5 waves x 2 vectors).
template <typename T, int WPG, int NV, bool BWD, bool GATED, bool EXACT, int LPG = 64>
__global__ void __launch_bounds__(WPG == 1 ? 256 : WPG * 64)
rmsnorm_gated_kernel(const NormArgs a) {
    constexpr int V = GlueVec<T>::V;
    constexpr int TPG = WPG * 64;                 // threads per (row, group)
    __shared__ float red[2][2][16];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    static_assert(LPG == 64 || (WPG == 1 && NV == 1 && !EXACT), "several groups per wave: one vector a lane, idle lanes masked");
    constexpr int SUB = 64 / LPG;                 // groups per wave
    const int tl = WPG > 1 ? tid : lane % LPG;    // index inside the (row, group)
    const int64_t grp = (int64_t)blockIdx.y * SUB + (SUB > 1 ? lane / LPG : 0), groups = a.groups;
    const bool spare = SUB > 1 && grp >= groups;  // lanes behind the last group
    const int64_t c0 = (spare ? groups - 1 : grp) * a.gw;      // first channel of the group
    const int nvec = spare ? 0 : (int)(a.gw / V);
    const float inv_n = 1.f / (float)a.gw;

    // The weights as vectors (a caller's tensor: on any element); idle lanes take the group's first: their x is zeroed, and with it every product.
    // Element by element, each in a branch, they cost a few rows 0.4 us: 64 rows of 8 x 256 channels 3.15 -> 2.7, 1101 of 2560 7.9 -> 6.6.
    typedef float AnyFloat4 __attribute__((ext_vector_type(4), aligned(4)));
    float w[NV][V], dw[BWD ? NV : 1][V];
#pragma unroll
    for (int it = 0; it < NV; ++it) {
        const int vi = it * TPG + tl;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            if constexpr (NV == 1 || !EXACT) {
                const AnyFloat4 v = *reinterpret_cast<const AnyFloat4*>(a.w + c0 + (int64_t)((EXACT || vi < nvec) ? vi : 0) * V + e / 4 * 4);
                w[it][e] = v[e % 4];
            } else {
                w[it][e] = a.w[c0 + (int64_t)vi * V + e];
            }
            if (BWD) dw[it][e] = 0.f;
        }
    }
    // Rows are dealt out round-robin: workgroup i (WPG > 1; wave 4 i + w for WPG == 1) takes rows i, i + G, i + 2 G, ... with G
    // the number of workgroups (waves), so that at any moment the rows in flight over the whole chip are neighbours in
    // memory and every memory channel is in use.  (A contiguous block of rows per workgroup puts all workgroups a fixed
    // power-of-two-rich distance apart, and they then walk through the same channels together: 3.6 TB/s for the loads alone.)
    const int64_t r1 = a.rows;
    const int64_t RSTEP = WPG > 1 ? (int64_t)gridDim.x : (int64_t)gridDim.x * 4;
    int slot = 0;
    // WPG > 1: every wave takes every row of the workgroup (uniform trip count, barriers inside); WPG == 1: each wave its own rows.
    // the raw vectors of the next row are loaded before this row is reduced (the row after the last: the first once more)
    constexpr bool gated = GATED;
    // Two register sets, a row loaded a whole iteration before it is used: the forward always; the backward where the
    // workgroup is alone on its compute unit anyway (five waves: up to 256 registers each).  Otherwise the backward loads
    // the next row behind the first pass over the current one.
    constexpr bool TWO = !BWD || WPG == 5;
    struct RowRegs { uint4 x[NV], z[NV], g[BWD ? NV : 1]; };
    RowRegs ra, rb;
    const int64_t rfirst = WPG > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wave;
    auto load_row = [&](int64_t r, RowRegs& q) {
        uint4 (&rx)[NV] = q.x; uint4 (&rz)[NV] = q.z; uint4 (&rg)[BWD ? NV : 1] = q.g;
        const int64_t rr = r < r1 ? r : rfirst;
        const T* xr = static_cast<const T*>(a.x) + rr * a.x_sr + c0;
        const T* zr = gated ? static_cast<const T*>(a.z) + rr * a.z_sr + c0 : xr;
        const T* gr = BWD ? static_cast<const T*>(a.g) + rr * a.g_sr + c0 : xr;
#pragma unroll
        for (int it = 0; it < NV; ++it) {
            const int vi = it * TPG + tl;
            const int64_t off = (int64_t)((EXACT || vi < nvec) ? vi : 0) * V;      // idle lanes read the first vector and ignore it
            rx[it] = *reinterpret_cast<const uint4*>(xr + off);
            if (gated) rz[it] = load_any(zr + off);
            if (BWD) rg[it] = *reinterpret_cast<const uint4*>(gr + off);
        }
    };
    if (rfirst < r1) load_row(rfirst, ra);
    auto do_row = [&](int64_t r, RowRegs& q) {
        uint4 (&rx)[NV] = q.x; uint4 (&rz)[NV] = q.z; uint4 (&rg)[BWD ? NV : 1] = q.g;
        const bool zr = gated;
        float h[NV][V], xs[BWD ? NV : 1][V], zs[BWD ? NV : 1][V], gs[BWD ? NV : 1][V];
        float ss = 0.f, dot = 0.f;
#pragma unroll
        for (int it = 0; it < NV; ++it) {
            const int vi = it * TPG + tl;
            float xv[V], zv[V], gv[V];
            // an idle lane's x is zeroed as a raw vector (four selects): h, and with it every sum, is then zero there
            uint4 rxv = rx[it];
            if (!EXACT && vi >= nvec) rxv = uint4{0u, 0u, 0u, 0u};
            unpack_vec<T>(rxv, xv);
            if (gated) unpack_vec<T>(rz[it], zv);
            if (BWD) unpack_vec<T>(rg[it], gv);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float gate = zr ? silu_f(zv[e]) : 1.f;
                h[it][e] = xv[e] * gate;
                ss += h[it][e] * h[it][e];
                if (BWD) {
                    xs[it][e] = xv[e]; zs[it][e] = zr ? zv[e] : 0.f; gs[it][e] = gv[e];
                    dot += h[it][e] * gv[e] * w[it][e];
                }
            }
        }
        if (!TWO) load_row(r + RSTEP, q);
        group_sum2<WPG, LPG>(ss, dot, red, slot);
        slot ^= 1;
        const float var = ss * inv_n + a.eps;
        const float rinv = __builtin_amdgcn_rsqf(var);
        if (!BWD) {
#pragma unroll
            for (int it = 0; it < NV; ++it) {
                const int vi = it * TPG + tl;
                if (!EXACT && vi >= nvec) continue;
                float o[V];
#pragma unroll
                for (int e = 0; e < V; ++e) o[e] = w[it][e] * (h[it][e] * rinv);
                if (a.out_f32) {
                    float* op = static_cast<float*>(a.out) + r * a.out_sr + c0 + (int64_t)vi * V;
#pragma unroll
                    for (int q = 0; q < V / 4; ++q) *reinterpret_cast<floatx4*>(op + 4 * q) = floatx4{o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]};
                } else {
                    store_vec<T>(static_cast<T*>(a.out) + r * a.out_sr + c0 + (int64_t)vi * V, o);
                }
            }
        } else {
            const float cf = dot * inv_n / var;
#pragma unroll
            for (int it = 0; it < NV; ++it) {
                const int vi = it * TPG + tl;
                if (!EXACT && vi >= nvec) continue;
                float ox[V], oz[V];
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const float gwv = gs[it][e] * w[it][e];
                    const float dh = rinv * (gwv - cf * h[it][e]);
                    if (zr) {
                        const float z = zs[it][e];
                        const float s = sigmoid_f(z);
                        ox[e] = dh * (z * s);
                        oz[e] = dh * xs[it][e] * (s * (1.f + z * (1.f - s)));
                    } else {
                        ox[e] = dh; oz[e] = 0.f;
                    }
                    dw[it][e] += gs[it][e] * (h[it][e] * rinv);
                }
                store_vec<T>(static_cast<T*>(a.dx) + r * a.dx_sr + c0 + (int64_t)vi * V, ox);
                if (zr && a.dz) store_vec<T>(static_cast<T*>(a.dz) + r * a.dz_sr + c0 + (int64_t)vi * V, oz);
            }
        }
    };
    if constexpr (!TWO) {
        for (int64_t r = rfirst; r < r1; r += RSTEP) do_row(r, ra);
    } else {
        // rows in pairs, one per register set; a row's loads are issued before the row in front of it is processed
        for (int64_t r = rfirst; r < r1; r += 2 * RSTEP) {
            load_row(r + RSTEP, rb);
            do_row(r, ra);
            if (r + RSTEP < r1) {      // uniform over the workgroup when it shares its rows (WPG > 1)
                load_row(r + 2 * RSTEP, ra);
                do_row(r + RSTEP, rb);
            }
        }
    }
    if (BWD) {
        // one partial row per workgroup: each lane owns its channels, or (WPG == 1) the four waves' sums meet in LDS first
        float* pp = a.partial + (int64_t)blockIdx.x * a.d + c0;
        if constexpr (WPG == 1) {
            __shared__ __align__(16) float sums[4][64 * NV * V];
#pragma unroll
            for (int it = 0; it < NV; ++it)
#pragma unroll
                for (int q = 0; q < V / 4; ++q)
                    *reinterpret_cast<floatx4*>(&sums[wave][(it * 64 + lane) * V + 4 * q]) = floatx4{dw[it][4 * q], dw[it][4 * q + 1], dw[it][4 * q + 2], dw[it][4 * q + 3]};
            __syncthreads();
            if constexpr (SUB > 1) {
                const int e = tid * 4, v = e / V % LPG;
                const int64_t g = (int64_t)blockIdx.y * SUB + e / V / LPG;
                if (e < 64 * V && g < groups && (int64_t)v * V < a.gw)
                    *reinterpret_cast<floatx4*>(a.partial + (int64_t)blockIdx.x * a.d + g * a.gw + v * V + e % V) =
                        (*reinterpret_cast<const floatx4*>(&sums[0][e]) + *reinterpret_cast<const floatx4*>(&sums[1][e])) +
                        (*reinterpret_cast<const floatx4*>(&sums[2][e]) + *reinterpret_cast<const floatx4*>(&sums[3][e]));
                return;
            }
            for (int e = tid * 4; e < nvec * V; e += 256 * 4)
                *reinterpret_cast<floatx4*>(pp + e) = (*reinterpret_cast<const floatx4*>(&sums[0][e]) + *reinterpret_cast<const floatx4*>(&sums[1][e])) +
                                                      (*reinterpret_cast<const floatx4*>(&sums[2][e]) + *reinterpret_cast<const floatx4*>(&sums[3][e]));
            return;
        }
#pragma unroll
        for (int it = 0; it < NV; ++it) {
            const int vi = it * TPG + tl;
            if (!EXACT && vi >= nvec) continue;
#pragma unroll
            for (int q = 0; q < V / 4; ++q)
                *reinterpret_cast<floatx4*>(pp + (int64_t)vi * V + 4 * q) = floatx4{dw[it][4 * q], dw[it][4 * q + 1], dw[it][4 * q + 2], dw[it][4 * q + 3]};
        }
    }
}

// waves per (row, group) and vectors per lane for a group of `nvec` 16-byte vectors; false if it does not fit
bool norm_shape(int64_t nvec, int vec_elems, int* wpg, int* nv) {
    if (nvec <= 0) return false;
    if (nvec <= 256) { *wpg = 1; *nv = (int)((nvec + 63) / 64); return true; }
    // a group that five waves cover with no idle lane (5120 channels: the 2.7B width) takes five
    if (nvec % 320 == 0 && (nvec / 320 == 2 || nvec / 320 == 4) && nvec * vec_elems <= 8192) { *wpg = 5; *nv = (int)(nvec / 320); return true; }
    // up to 8192 channels per group in either type: 4 vectors of 8 per lane (16-bit), 8 vectors of 4 (fp32)
    if (nvec * vec_elems <= 8192) { *wpg = 4; *nv = (int)((nvec + 255) / 256); return true; }
    return false;
}

// Lanes per group: a wave, or a half, a quarter or an eighth of one for several groups of so few vectors.  With a wave per group of 64
// channels 56 of 64 lanes idle and every access is a piece of 128 bytes.  Time of 53445 rows of 8 x 64 channels
// 115 -> 29 us and, backward, 223 -> 52; 16384 x 8 x 128 38 -> 19 and 69 -> 31; 16384 x 8 x 192 38 -> 26 and 70 -> 43; 16384 x 2 x
// 256 13.1 -> 11.9 and 23 -> 19; up to about 1000 rows the same.
int norm_lanes(int64_t nvec, int64_t groups) {
    if (nvec > 32) return 64;
    int lanes = 8;
    while (lanes < nvec || (lanes < 64 && 64 / lanes > groups)) lanes *= 2;
    return lanes;
}
// columns of a launch's grid
int64_t norm_columns(int64_t nvec, int64_t groups) { return ceil_div(groups, (int64_t)(64 / norm_lanes(nvec, groups))); }

// Rows per workgroup.  A workgroup (or, with a wave per row, each of its four waves) is a chain of rows, dealt round-robin, and the chip
// likes a few of them per CU: one more than fit run alone at the end, and in the backward every one leaves a partial row of dw.
// Workgroups per CU by the form of a row, from 990 sizes (64 to 16000 rows, groups of 64 to 8192 channels, both types; one | two | three | four
// per CU, us; `all`: rows times columns of the grid):
//   forward, a wave per row, one vector a lane: four (8192 x 8 x 512 52.3 | 35.0 | 32.7 | 33.4, 6500 x 512 6.9 | 6.1 | 6.2 | 5.7); two vectors: two
//     (16384 x 1024 20.5 | 18.2 | 19.0 | 19.3); more: one (8192 x 2048 18.4 | 19.1 | 20.6 | 20.5).  16-bit rows that are few enough for chains of up
//     to three go one to a wave instead where the busiest CU then has fewer: 2100 x 1024 5.1 | 5.2, a row each 4.9; 513 x 8 x 1024 7.0, 6.4; not
//     3700 x 1024 6.3 | 5.9, 6.1.  fp32 does not gain by it (600 x 8 x 512 6.2, a row each 6.8).
//   backward, a wave per row, up to one and a half vectors a lane: two for many rows or where a partial row is short, else one (9001 x 2 x 320 fp32
//     28.8 | 24.2 | 24.9 | 27.1, 1500 x 512 bf16 6.9 | 7.2, 3001 x 512 8.4 | 8.9 | 9.1, 6500 x 512 11.6 | 11.7; 400 x 8 x 512 8.65 | 8.3); more vectors:
//     one (3333 x 2048 19.5 | 20.9 | 21.0 | 26.0, 9001 x 512 fp32 19.8 | 21.1 | 22.2).
//   a workgroup per row, two vectors a lane, idle lanes: two (6500 x 2560 27.8 | 22.6 | 21.4 | 21.6, backward 9001 x 2560 52.8 | 47.0 | 54.5 | 49.9),
//     the backward of few rows one (1500 x 2560 14.2 | 14.3, 1800 16.3 | 15.6).
//   ... no idle lane: forward a row each up to five per CU (1101 x 5120 9.3 | 9.2, each 8.6; 1300: 10.3 | 9.6, 9.5; 1500: 10.5 | 10.05, 10.5), then
//     two of 16-bit rows up to 35 rows per CU (6500 x 5120 36.4 | 33.3 | 34.6 | 37.2, 12001 67.2 | 70.6), else one, and the backward one
//     (2664 x 5120 32.0 | 36.4 | 38.1 | 38.9).
//   ... more vectors a lane: one (2664 x 7168 24.1 | 25.5 | 28.3 | 30.8).
int64_t norm_rows_per_workgroup(int64_t rows, int64_t groups, int64_t nvec, int vec_elems, bool bwd) {
    int wpg = 1, nv = 1;
    if (!norm_shape(nvec, vec_elems, &wpg, &nv)) return ceil_div(rows, (int64_t)512);      // refused before any launch
    const int64_t columns = norm_columns(nvec, groups), all = rows * columns, cus = device_cus();
    if (wpg == 1) {
        const int64_t per_cu = bwd ? (nvec <= 96 && (all > 20 * cus || columns >= 4) ? 2 : 1) : (nv == 1 ? 4 : nv == 2 ? 2 : 1);
        const int64_t chain = ceil_div(all, 4 * per_cu * cus);      // rows per wave
        auto busiest = [&](int64_t c) { return ceil_div(ceil_div(rows, 4 * c) * columns, cus) * c; };
        if (!bwd && nv <= 2 && vec_elems == 8 && chain <= 3 && busiest(1) < busiest(chain)) return 4;
        return 4 * chain;
    }
    const bool exact = (int64_t)wpg * 64 * nv == nvec;
    int64_t per_cu = 1;
    if (nv == 2 && !exact) per_cu = !bwd || all > 6 * cus ? 2 : 1;
    if (nv == 2 && exact && !bwd) {
        if (all <= 5 * cus) return 1;
        if (vec_elems == 8 && all <= 35 * cus) per_cu = 2;
    }
    return ceil_div(all, per_cu * cus);
}

template <typename T, bool BWD>
int launch_norm(const NormArgs& a, int64_t groups, hipStream_t st) {
    constexpr int V = GlueVec<T>::V;
    int wpg = 0, nv = 0;
    if (!norm_shape(a.gw / V, V, &wpg, &nv))
        return fail(M2_ERR_SHAPE, "rmsnorm_gated: %lld channels per group exceed the supported 8192", (long long)a.gw);
    const dim3 grid((unsigned)ceil_div(a.rows, a.rows_per_block), (unsigned)norm_columns(a.gw / V, groups));
    const bool exact = (int64_t)wpg * 64 * nv == a.gw / V, gated = a.z != nullptr;
    const int lanes = norm_lanes(a.gw / V, groups);
#define M2_NORM_PART(L) if (lanes == L) { \
        if (gated) rmsnorm_gated_kernel<T, 1, 1, BWD, true, false, L><<<grid, 256, 0, st>>>(a); \
        else rmsnorm_gated_kernel<T, 1, 1, BWD, false, false, L><<<grid, 256, 0, st>>>(a); \
        return check_launch("rmsnorm_gated_kernel"); }
    M2_NORM_PART(8) M2_NORM_PART(16) M2_NORM_PART(32)
#undef M2_NORM_PART
#define M2_NORM_LAUNCH(W, N, G, E) { rmsnorm_gated_kernel<T, W, N, BWD, G, E><<<grid, (W == 1 ? 256 : W * 64), 0, st>>>(a); return check_launch("rmsnorm_gated_kernel"); }
#define M2_NORM_CASE(W, N) if (wpg == W && nv == N) { \
        if (gated) { if (exact) M2_NORM_LAUNCH(W, N, true, true) else M2_NORM_LAUNCH(W, N, true, false) } \
        else { if (exact) M2_NORM_LAUNCH(W, N, false, true) else M2_NORM_LAUNCH(W, N, false, false) } }
    M2_NORM_CASE(1, 1) M2_NORM_CASE(1, 2) M2_NORM_CASE(1, 3) M2_NORM_CASE(1, 4)
    M2_NORM_CASE(4, 2) M2_NORM_CASE(4, 3) M2_NORM_CASE(4, 4)
    M2_NORM_CASE(5, 2) M2_NORM_CASE(5, 4)
    if constexpr (sizeof(T) == 4) { M2_NORM_CASE(4, 5) M2_NORM_CASE(4, 6) M2_NORM_CASE(4, 7) M2_NORM_CASE(4, 8) }
#undef M2_NORM_CASE
#undef M2_NORM_LAUNCH
    return fail(M2_ERR_SHAPE, "rmsnorm_gated: no kernel for %d waves x %d vectors", wpg, nv);
}

// Block boundary of a decode step: residual += delta; out = weight * residual * rsqrt(mean(residual^2) + eps).
// One workgroup per row, the row (up to 8192 channels) stays in registers between the sum of squares and the output.
template <typename T>
__global__ void __launch_bounds__(256)
add_rmsnorm_kernel(float* __restrict__ res, int64_t res_sr, const T* __restrict__ delta, int64_t delta_sr, const float* __restrict__ w,
                   T* __restrict__ out, int64_t out_sr, int d, float eps) {
    constexpr int NV = 8;
    __shared__ float red[4];
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x;
    float* rr = res + row * res_sr;
    const T* dr = delta ? delta + row * delta_sr : nullptr;
    T* orow = out + row * out_sr;
    const int nvec = d / 4;
    floatx4 v[NV];
    float ss = 0.f;
#pragma unroll
    for (int it = 0; it < NV; ++it) {
        const int vi = it * 256 + tid;
        v[it] = floatx4{0.f, 0.f, 0.f, 0.f};
        if (vi < nvec) {
            floatx4 r = *reinterpret_cast<const floatx4*>(rr + vi * 4);
            if (dr) {
                if constexpr (sizeof(T) == 2) {
                    const uint2 raw = *reinterpret_cast<const uint2*>(dr + vi * 4);
                    r[0] += __builtin_bit_cast(float, raw.x << 16); r[1] += __builtin_bit_cast(float, raw.x & 0xffff0000u);
                    r[2] += __builtin_bit_cast(float, raw.y << 16); r[3] += __builtin_bit_cast(float, raw.y & 0xffff0000u);
                } else {
                    const floatx4 dv = *reinterpret_cast<const floatx4*>(dr + vi * 4);
                    r[0] += dv[0]; r[1] += dv[1]; r[2] += dv[2]; r[3] += dv[3];
                }
                *reinterpret_cast<floatx4*>(rr + vi * 4) = r;
            }
            v[it] = r;
            ss += (r[0] * r[0] + r[1] * r[1]) + (r[2] * r[2] + r[3] * r[3]);
        }
    }
    ss = warp_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    const float rinv = rsqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)d + eps);
#pragma unroll
    for (int it = 0; it < NV; ++it) {
        const int vi = it * 256 + tid;
        if (vi < nvec) {
            const floatx4 wv = *reinterpret_cast<const floatx4*>(w + vi * 4);
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = wv[e] * (v[it][e] * rinv);
            if constexpr (sizeof(T) == 2) {
                T e4[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) e4[e] = from_f32<T>(o[e]);
                *reinterpret_cast<uint2*>(orow + vi * 4) = *reinterpret_cast<const uint2*>(e4);
            } else {
                *reinterpret_cast<floatx4*>(orow + vi * 4) = floatx4{o[0], o[1], o[2], o[3]};
            }
        }
    }
}

// Parameter casts of a mixer layer: a few thousand values, one launch instead of one per parameter and operation (each
// such launch costs the host 4-5 us; the layer's step had seven in front of its kernels and eight behind them).
__device__ __forceinline__ float ld_as_f32(const void* p, int dt, int64_t i) {
    return dt == M2_F32 ? static_cast<const float*>(p)[i] : to_f32(static_cast<const bf16_t*>(p)[i]);
}
struct MixerParams { const void *A_log, *D, *dt_bias, *norm; int a, d, b, w; };
__global__ void __launch_bounds__(256)
mixer_params_kernel(const MixerParams p, float* __restrict__ out, int64_t nheads, int64_t channels) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < nheads) {
        out[i] = -expf(ld_as_f32(p.A_log, p.a, i));
        if (p.D) out[nheads + i] = ld_as_f32(p.D, p.d, i);
        out[2 * nheads + i] = ld_as_f32(p.dt_bias, p.b, i);
    }
    if (i < channels) out[3 * nheads + i] = ld_as_f32(p.norm, p.w, i);
}
// The sums behind a layer's backward in one launch: the norm weight's partial rows, the conv's partials, and the per-head gradients
// in their parameters' types (dA_log = dA A where A is given).  Each of them had been a launch of its own, 3-5 us plus the gap in front
// of it for a few hundred kilobytes (training step of a 768-channel layer on 500 tokens: 23 launches 210 us, 21 launches 202; b3 l1111 h32 with recompute 217 -> 214).
struct ParamSums {
    const float* norm; int64_t norm_rows, channels; void* d_norm; int norm_dtype;
    const float* conv; int64_t conv_slots, conv_channels; void *dw, *db; int conv_dtype;
    int64_t nheads; const float *A, *dA, *dD, *d_dt_bias; void *o_A, *o_D, *o_dt_bias; int a, d, b;
    unsigned n_norm, n_conv;      // workgroups of the first two parts
};
template <int V>
__global__ void __launch_bounds__(1024)
param_sums_kernel(const ParamSums p) {
    if (blockIdx.x < p.n_norm) {
        column_sum_body<V>(p.norm, p.norm_rows, p.channels, blockIdx.x, [&](int64_t c, float v) { st_param(p.d_norm, p.norm_dtype, c, v); });
    } else if (blockIdx.x < p.n_norm + p.n_conv) {
        conv_sum_body(p.conv, p.conv_slots, p.conv_channels, 4, p.dw, p.db, p.conv_dtype, (int64_t)(blockIdx.x - p.n_norm) * 1024 + threadIdx.x);
    } else {
        const int64_t i = (int64_t)(blockIdx.x - p.n_norm - p.n_conv) * 1024 + threadIdx.x;
        if (i >= p.nheads) return;
        st_param(p.o_A, p.a, i, p.A ? p.dA[i] * p.A[i] : p.dA[i]);
        if (p.o_D) st_param(p.o_D, p.d, i, p.dD[i]);
        st_param(p.o_dt_bias, p.b, i, p.d_dt_bias[i]);
    }
}

int check_norm_common(const m2_rmsnorm_params* p, const char* what) {
    M2_REQUIRE(p, M2_ERR_NULL, "%s: NULL params", what);
    M2_REQUIRE(p->rows >= 0 && p->channels > 0 && p->n_groups > 0 && p->channels % p->n_groups == 0, M2_ERR_SHAPE,
               "%s: rows %lld, channels %lld, groups %d", what, (long long)p->rows, (long long)p->channels, (int)p->n_groups);
    M2_REQUIRE(p->dtype == M2_F32 || p->dtype == M2_BF16, M2_ERR_DTYPE, "%s: unsupported dtype %d", what, (int)p->dtype);
    const int V = p->dtype == M2_F32 ? 4 : 8;
    M2_REQUIRE((p->channels / p->n_groups) % V == 0, M2_ERR_SHAPE, "%s: channels per group must be a multiple of %d", what, V);
    return M2_OK;
}

// any_z: the gate may start on any element
int check_norm_fwd(const m2_rmsnorm_params* p, bool any_z) {
    const int rc = check_norm_common(p, "rmsnorm_gated_fwd");
    if (rc || p->rows == 0) return rc;
    M2_REQUIRE(p->x && p->weight && p->out, M2_ERR_NULL, "rmsnorm_gated_fwd: x, weight and out are required");
    const int V = p->dtype == M2_F32 ? 4 : 8;
    M2_REQUIRE(aligned16(p->x) && aligned16(p->out) && p->x_stride_row % V == 0 && p->out_stride_row % 4 == 0 &&
                   (p->out_f32 || p->out_stride_row % V == 0) && (!p->z || any_z || (aligned16(p->z) && p->z_stride_row % V == 0)),
               M2_ERR_ALIGN, "rmsnorm_gated_fwd: pointers must be 16-byte aligned and row strides multiples of %d elements", V);
    int wpg = 0, nv = 0;
    const int64_t gw = p->channels / p->n_groups;
    M2_REQUIRE(norm_shape(gw / V, V, &wpg, &nv), M2_ERR_SHAPE, "rmsnorm_gated: %lld channels per group exceed the supported 8192", (long long)gw);
    return M2_OK;
}
int norm_fwd(const m2_rmsnorm_params* p, bool any_z, void* stream) {
    const int rc = check_norm_fwd(p, any_z);
    if (rc || p->rows == 0) return rc;
    const int V = p->dtype == M2_F32 ? 4 : 8;
    NormArgs a{};
    a.x = p->x; a.x_sr = p->x_stride_row; a.z = p->z; a.z_sr = p->z_stride_row; a.w = p->weight;
    a.out = p->out; a.out_sr = p->out_stride_row; a.out_f32 = p->out_f32 || p->dtype == M2_F32;
    a.rows = p->rows; a.d = p->channels; a.gw = p->channels / p->n_groups; a.groups = p->n_groups; a.eps = p->eps;
    a.rows_per_block = norm_rows_per_workgroup(p->rows, p->n_groups, a.gw / V, V, false);
    hipStream_t st = static_cast<hipStream_t>(stream);
    M2_DISPATCH_DTYPE(p->dtype, T, return (launch_norm<T, false>(a, p->n_groups, st)));
    return M2_OK;
}
int norm_bwd_partial(const m2_rmsnorm_params* p, bool any_z, int64_t* rows, void* stream) {
    int rc = check_norm_common(p, "rmsnorm_gated_bwd");
    if (rc) return rc;
    M2_REQUIRE(rows, M2_ERR_NULL, "rmsnorm_gated_bwd_partial: rows is required");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int V = p->dtype == M2_F32 ? 4 : 8;
    int64_t prows = 0;
    if (p->rows > 0) {
        M2_REQUIRE(p->x && p->weight && p->d_out && p->dx, M2_ERR_NULL, "rmsnorm_gated_bwd: x, weight, d_out and dx are required");
        M2_REQUIRE(!p->z || p->dz, M2_ERR_NULL, "rmsnorm_gated_bwd: dz is required when z is given");
        M2_REQUIRE(aligned16(p->x) && aligned16(p->d_out) && aligned16(p->dx) && p->x_stride_row % V == 0 && p->d_out_stride_row % V == 0 &&
                       p->dx_stride_row % V == 0 && (!p->z || (aligned16(p->dz) && p->dz_stride_row % V == 0)) &&
                       (!p->z || any_z || (aligned16(p->z) && p->z_stride_row % V == 0)),
                   M2_ERR_ALIGN, "rmsnorm_gated_bwd: pointers must be 16-byte aligned and row strides multiples of %d elements", V);
        const size_t need = m2_rmsnorm_gated_bwd_workspace_bytes(p->rows, p->channels, p->n_groups, p->dtype);
        M2_REQUIRE(p->workspace && p->workspace_bytes >= need, M2_ERR_WORKSPACE, "rmsnorm_gated_bwd: workspace %zu bytes < %zu needed",
                   p->workspace_bytes, need);
        M2_REQUIRE((reinterpret_cast<uintptr_t>(p->workspace) & 15u) == 0, M2_ERR_ALIGN, "rmsnorm_gated_bwd: workspace must be 16-byte aligned");
        NormArgs a{};
        a.x = p->x; a.x_sr = p->x_stride_row; a.z = p->z; a.z_sr = p->z_stride_row; a.w = p->weight;
        a.g = p->d_out; a.g_sr = p->d_out_stride_row; a.dx = p->dx; a.dx_sr = p->dx_stride_row; a.dz = p->dz; a.dz_sr = p->dz_stride_row;
        a.partial = static_cast<float*>(p->workspace);
        a.rows = p->rows; a.d = p->channels; a.gw = p->channels / p->n_groups; a.groups = p->n_groups; a.eps = p->eps;
        a.rows_per_block = norm_rows_per_workgroup(p->rows, p->n_groups, a.gw / V, V, true);
        int wpg = 0, nv = 0;
        if (!norm_shape(a.gw / V, V, &wpg, &nv))
            return fail(M2_ERR_SHAPE, "rmsnorm_gated_bwd: %lld channels per group exceed the supported 8192", (long long)a.gw);
        prows = ceil_div(p->rows, a.rows_per_block);
        M2_DISPATCH_DTYPE(p->dtype, T, rc = (launch_norm<T, true>(a, p->n_groups, st)));
        if (rc) return rc;
    }
    *rows = prows;
    return M2_OK;
}

}  // namespace
}  // namespace m2

extern "C" int m2_softplus_bias_fwd(const void* dt, int64_t dt_stride_row, const float* dt_bias, void* out, int64_t out_stride_row,
                                    int64_t rows, int64_t nheads, int32_t dtype, void* stream) {
    using namespace m2;
    M2_REQUIRE(rows >= 0 && nheads > 0, M2_ERR_SHAPE, "softplus_bias_fwd: rows %lld, heads %lld", (long long)rows, (long long)nheads);
    if (rows == 0) return M2_OK;
    M2_REQUIRE(dt && dt_bias && out, M2_ERR_NULL, "softplus_bias_fwd: dt, dt_bias and out are required");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const unsigned blocks = (unsigned)ceil_div(rows * nheads, (int64_t)256);
    M2_DISPATCH_DTYPE(dtype, T, (softplus_fwd_kernel<T><<<blocks, 256, 0, st>>>(static_cast<const T*>(dt), dt_stride_row, dt_bias,
                                                                                 static_cast<T*>(out), out_stride_row, rows, nheads)));
    return check_launch("softplus_fwd_kernel");
}

extern "C" size_t m2_softplus_bias_bwd_workspace_bytes(int64_t rows, int64_t nheads) {
    if (rows <= 0 || nheads <= 0) return 256;
    return m2::align_up((size_t)m2::ceil_div(rows, (int64_t)m2::kSpRows) * (size_t)nheads * sizeof(float), 256);
}

extern "C" int m2_softplus_bias_bwd(const void* dt, int64_t dt_stride_row, const float* dt_bias, const void* d_out, int64_t d_out_stride_row,
                                    void* d_in, int64_t d_in_stride_row, float* d_bias, void* workspace, size_t workspace_bytes,
                                    int64_t rows, int64_t nheads, int32_t dtype, void* stream) {
    using namespace m2;
    M2_REQUIRE(rows >= 0 && nheads > 0, M2_ERR_SHAPE, "softplus_bias_bwd: rows %lld, heads %lld", (long long)rows, (long long)nheads);
    M2_REQUIRE(d_bias, M2_ERR_NULL, "softplus_bias_bwd: d_bias is required");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t nblk = ceil_div(rows, (int64_t)kSpRows);
    if (rows > 0) {
        M2_REQUIRE(dt && dt_bias && d_out && d_in, M2_ERR_NULL, "softplus_bias_bwd: dt, dt_bias, d_out and d_in are required");
        M2_REQUIRE(workspace && workspace_bytes >= m2_softplus_bias_bwd_workspace_bytes(rows, nheads), M2_ERR_WORKSPACE,
                   "softplus_bias_bwd: workspace %zu bytes < %zu needed", workspace_bytes, m2_softplus_bias_bwd_workspace_bytes(rows, nheads));
        float* partial = static_cast<float*>(workspace);
        M2_DISPATCH_DTYPE(dtype, T, (softplus_bwd_kernel<T><<<(unsigned)nblk, 256, 0, st>>>(
                                         static_cast<const T*>(dt), dt_stride_row, dt_bias, static_cast<const T*>(d_out), d_out_stride_row,
                                         static_cast<T*>(d_in), d_in_stride_row, partial, rows, nheads)));
        int rc = check_launch("softplus_bwd_kernel");
        if (rc) return rc;
    }
    // with no rows the sum is empty: column_sum_kernel writes zeros
    return launch_column_sum(static_cast<const float*>(workspace), d_bias, nblk, nheads, st);
}

extern "C" int m2_rmsnorm_gated_fwd_check(const m2_rmsnorm_params* p) { return m2::check_norm_fwd(p, false); }
extern "C" int m2_rmsnorm_gated_fwd(const m2_rmsnorm_params* p, void* stream) { return m2::norm_fwd(p, false, stream); }
extern "C" int m2_core_norm_fwd_check(const m2_rmsnorm_params* p) { return m2::check_norm_fwd(p, true); }
extern "C" int m2_core_norm_fwd(const m2_rmsnorm_params* p, void* stream) { return m2::norm_fwd(p, true, stream); }

extern "C" size_t m2_rmsnorm_gated_bwd_workspace_bytes(int64_t rows, int64_t channels, int32_t n_groups, int32_t dtype) {
    if (rows <= 0 || channels <= 0 || n_groups <= 0) return 256;
    // A partial row per workgroup.  The rule gives a column of the grid at most 512 of them on 256 compute units, and room for as many is
    // asked for whatever it gives here: a size that followed the units would depend on the device that is current when it is asked
    // for, and a caller may size its scratch without one.
    const int V = dtype == M2_F32 ? 4 : 8;
    const int64_t nvec = channels / n_groups / V, per_column = m2::ceil_div((int64_t)512, m2::norm_columns(nvec, n_groups));
    const int64_t used = m2::ceil_div(rows, m2::norm_rows_per_workgroup(rows, n_groups, nvec, V, true));
    const int64_t most = rows < per_column ? rows : per_column;
    return m2::align_up((size_t)(used > most ? used : most) * (size_t)channels * sizeof(float), 256);
}

extern "C" int m2_rmsnorm_gated_bwd_partial(const m2_rmsnorm_params* p, int64_t* rows, void* stream) {
    return m2::norm_bwd_partial(p, false, rows, stream);
}
extern "C" int m2_core_norm_bwd_partial(const m2_rmsnorm_params* p, int64_t* rows, void* stream) { return m2::norm_bwd_partial(p, true, rows, stream); }

extern "C" int m2_rmsnorm_gated_bwd(const m2_rmsnorm_params* p, void* stream) {
    using namespace m2;
    int rc = check_norm_common(p, "rmsnorm_gated_bwd");
    if (rc) return rc;
    M2_REQUIRE(p->d_weight, M2_ERR_NULL, "rmsnorm_gated_bwd: d_weight is required");
    int64_t prows = 0;
    if ((rc = m2_rmsnorm_gated_bwd_partial(p, &prows, stream))) return rc;
    return launch_column_sum(static_cast<const float*>(p->workspace), p->d_weight, prows, p->channels, static_cast<hipStream_t>(stream));
}

extern "C" int m2_add_rmsnorm(float* residual, int64_t residual_stride_row, const void* delta, int64_t delta_stride_row,
                              const float* weight, void* out, int64_t out_stride_row, int64_t rows, int64_t channels, float eps,
                              int32_t dtype, void* stream) {
    using namespace m2;
    M2_REQUIRE(rows >= 0 && channels > 0, M2_ERR_SHAPE, "add_rmsnorm: rows %lld, channels %lld", (long long)rows, (long long)channels);
    M2_REQUIRE(channels % 4 == 0 && channels <= 8192, M2_ERR_SHAPE, "add_rmsnorm: channels %lld must be a multiple of 4, at most 8192",
               (long long)channels);
    M2_REQUIRE(dtype == M2_F32 || dtype == M2_BF16, M2_ERR_DTYPE, "add_rmsnorm: unsupported dtype %d", (int)dtype);
    if (rows == 0) return M2_OK;
    M2_REQUIRE(residual && weight && out, M2_ERR_NULL, "add_rmsnorm: residual, weight and out are required");
    const size_t es = dtype == M2_F32 ? 4 : 2;
    M2_REQUIRE(aligned16(residual) && aligned16(weight) && residual_stride_row % 4 == 0 && (uintptr_t)out % (4 * es) == 0 &&
                   out_stride_row % 4 == 0 && (!delta || ((uintptr_t)delta % (4 * es) == 0 && delta_stride_row % 4 == 0)),
               M2_ERR_ALIGN, "add_rmsnorm: rows must start on 4-element boundaries (residual and weight on 16 bytes)");
    M2_REQUIRE(rows <= 0x7fffffff, M2_ERR_SHAPE, "add_rmsnorm: too many rows");
    hipStream_t st = static_cast<hipStream_t>(stream);
    M2_DISPATCH_DTYPE(dtype, T, (add_rmsnorm_kernel<T><<<(unsigned)rows, 256, 0, st>>>(residual, residual_stride_row, static_cast<const T*>(delta),
                                                                                     delta_stride_row, weight, static_cast<T*>(out),
                                                                                     out_stride_row, (int)channels, eps)));
    return check_launch("add_rmsnorm_kernel");
}

extern "C" int m2_mixer_params(const void* A_log, int32_t A_dtype, const void* D, int32_t D_dtype, const void* dt_bias, int32_t dt_bias_dtype,
                               const void* norm_weight, int32_t norm_dtype, float* out, int64_t nheads, int64_t channels, void* stream) {
    using namespace m2;
    M2_REQUIRE(nheads > 0 && channels > 0, M2_ERR_SHAPE, "mixer_params: heads %lld, channels %lld", (long long)nheads, (long long)channels);
    M2_REQUIRE(A_log && dt_bias && norm_weight && out, M2_ERR_NULL, "mixer_params: A_log, dt_bias, norm_weight and out are required");
    for (const int32_t dt : {A_dtype, D_dtype, dt_bias_dtype, norm_dtype})
        M2_REQUIRE(dt == M2_F32 || dt == M2_BF16, M2_ERR_DTYPE, "mixer_params: unsupported dtype %d", (int)dt);
    const int64_t n = nheads > channels ? nheads : channels;
    mixer_params_kernel<<<(unsigned)ceil_div(n, (int64_t)256), 256, 0, static_cast<hipStream_t>(stream)>>>(
        MixerParams{A_log, D, dt_bias, norm_weight, A_dtype, D_dtype, dt_bias_dtype, norm_dtype}, out, nheads, channels);
    return check_launch("mixer_params_kernel");
}

extern "C" int m2_param_sums(const float* norm_partial, int64_t norm_rows, int64_t channels, void* d_norm, int32_t norm_dtype, const float* conv_partial,
                             int64_t conv_slots, int64_t conv_channels, void* dw, void* db, int32_t conv_dtype, int64_t nheads, const float* A,
                             const float* dA, const float* dD, const float* d_dt_bias, void* dA_out, int32_t A_dtype, void* dD_out, int32_t D_dtype,
                             void* d_dt_bias_out, int32_t dt_bias_dtype, void* stream) {
    using namespace m2;
    M2_REQUIRE(norm_rows >= 0 && channels >= 0 && conv_slots >= 0 && conv_channels >= 0 && nheads >= 0, M2_ERR_SHAPE, "param_sums: negative size");
    M2_REQUIRE(channels == 0 || (d_norm && (norm_partial || norm_rows == 0)), M2_ERR_NULL, "param_sums: the norm's partial rows and gradient are required");
    M2_REQUIRE(conv_slots == 0 || conv_channels == 0 || (conv_partial && dw), M2_ERR_NULL, "param_sums: the conv's partials and gradient are required");
    M2_REQUIRE(nheads == 0 || (dA && d_dt_bias && dA_out && d_dt_bias_out && (!dD_out || dD)), M2_ERR_NULL, "param_sums: a gradient or its destination is missing");
    for (const int32_t dt : {norm_dtype, conv_dtype, A_dtype, D_dtype, dt_bias_dtype})
        M2_REQUIRE(dt == M2_F32 || dt == M2_BF16, M2_ERR_DTYPE, "param_sums: unsupported dtype %d", (int)dt);
    ParamSums p{norm_partial, norm_rows, channels, d_norm, norm_dtype, conv_partial, conv_slots, conv_channels, dw, db, conv_dtype,
                nheads, A, dA, dD, d_dt_bias, dA_out, dD_out, d_dt_bias_out, A_dtype, D_dtype, dt_bias_dtype, 0, 0};
    const int64_t n_norm = ceil_div(channels, (int64_t)kSumCols), n_conv = conv_slots ? ceil_div(conv_channels * 5 * 4, (int64_t)1024) : 0;
    const int64_t blocks = n_norm + n_conv + ceil_div(nheads, (int64_t)1024);
    M2_REQUIRE(blocks < ((int64_t)1 << 31), M2_ERR_SHAPE, "param_sums: too many workgroups");
    if (blocks == 0) return M2_OK;
    p.n_norm = (unsigned)n_norm; p.n_conv = (unsigned)n_conv;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (channels % 4 == 0 && aligned16(norm_partial)) param_sums_kernel<4><<<(unsigned)blocks, 1024, 0, st>>>(p);
    else param_sums_kernel<1><<<(unsigned)blocks, 1024, 0, st>>>(p);
    return check_launch("param_sums_kernel");
}

extern "C" int m2_mixer_params_grads(const float* A, const float* dA, const float* dD, const float* d_dt_bias, const float* d_norm_weight,
                                     void* dA_log, int32_t A_dtype, void* dD_out, int32_t D_dtype, void* d_dt_bias_out, int32_t dt_bias_dtype,
                                     void* d_norm_out, int32_t norm_dtype, int64_t nheads, int64_t channels, void* stream) {
    using namespace m2;
    M2_REQUIRE(nheads > 0 && channels > 0, M2_ERR_SHAPE, "mixer_params_grads: heads %lld, channels %lld", (long long)nheads, (long long)channels);
    M2_REQUIRE(A && dA && d_dt_bias && d_norm_weight && dA_log && d_dt_bias_out && d_norm_out && (!dD_out || dD), M2_ERR_NULL,
               "mixer_params_grads: a gradient or its destination is missing");
    // the finished gradient of the norm weight is a single partial row
    return m2_param_sums(d_norm_weight, 1, channels, d_norm_out, norm_dtype, nullptr, 0, 0, nullptr, nullptr, M2_F32, nheads, A, dA, dD, d_dt_bias, dA_log,
                         A_dtype, dD_out, D_dtype, d_dt_bias_out, dt_bias_dtype, stream);
}
