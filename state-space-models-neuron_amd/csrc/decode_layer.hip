// One decode step of a whole mixer layer for few sequences: three launches (mamba2/mamba2_mixer.py:243-282 step, and around it
// modeling_mamba2.py:94-103, 133-140, the block's norm and residual add).
//
//   linear_small (in_proj)     [norm of the residual row ->] zxBCdt = W x
//   decode_gated               conv + SiLU of the token, S' = S exp(A dt) + dt x (x) B, h = (S' C + D x) silu(z), sum of h^2 per head
//   linear_small (out_proj)    h scaled to the gated RMSNorm -> W h [+ residual]; shifts the B/C conv states on the side
//
// At this size a step is bound by its launches and by latency: the same layer as separate kernels is seven of 4.6-11 us each
// (two library products, conv, scan, norm, add + norm), most of them idle, and 2.3x the host work.  Folding every row-wise
// operation into the product that reads its result leaves three launches whose time is the weights' and states' way from HBM.
#include "common.hpp"

namespace m2 {
namespace {

// ------------------------------------------------------------------------------------------ small products
// out[m][n] = sum_k X[m][k] W[n][k] for m < M <= 32, bf16 operands, fp32 accumulation.
//
// A workgroup owns 16 rows of W at a time; its NW waves split K, each with v_mfma_f32_16x16x32_bf16 whose A operand is the
// weights (16 bytes per lane straight from HBM, UN loads ahead) and whose B operand is the activations, and the NW partial
// tiles meet in LDS.  16 rows rather than 32 because the narrow products have few of them (1024 outputs: 64 workgroups) and
// what counts is the number of loads in flight over the chip.  X kinds:
//   plain   bf16 rows read where they lie (L2 hits: every workgroup reads all of them)
//   norm    fp32 residual rows -> w x rsqrt(mean(x^2) + eps), formed once per workgroup into LDS as bf16
//   gated   bf16 h rows and per-head sums of squares -> w h rsqrt(group mean + eps), likewise
// The weights of the first tile are on their way before the rows are normalised.
enum { kPlain = 0, kNorm = 1, kGated = 2 };
enum { kOutBf16 = 0, kOutF32 = 1, kOutAdd = 2 };
constexpr int kUN = 8;           // k steps of 32 in flight per wave

struct LinearArgs {
    const bf16_t* w; const bf16_t* bias;
    const void* x; int64_t x_sr;
    const float* norm_w; const float* head_sq;
    void* out; int64_t out_sr;
    int M, N, K, tiles, nheads, norm_groups;
    float eps;
    // conv states of the B and C channels, shifted here because every head of the scan in front of this reads them whole
    bf16_t* conv_state; const bf16_t* conv_in; int64_t conv_in_sb; int conv_c0, conv_cx, conv_W;
};

__device__ __forceinline__ bf16x8 as_frag(uint4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (bf16_t)v[e];
    return __builtin_bit_cast(uint4, r);
}

template <int XK, int NW>
__device__ __forceinline__ void stage_rows(const LinearArgs& a, bf16_t* xs, float (*rs)[8], int ld) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if constexpr (XK == kNorm) {
        for (int m = wave; m < a.M; m += NW) {
            const float* xr = static_cast<const float*>(a.x) + m * a.x_sr;
            float ss = 0.f;
            for (int k = lane * 4; k < a.K; k += 256) {
                const floatx4 v = *reinterpret_cast<const floatx4*>(xr + k);
                ss += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
            }
            const float rinv = rsqrtf(warp_sum(ss) / (float)a.K + a.eps);
            for (int k = lane * 4; k < a.K; k += 256) {
                const floatx4 v = *reinterpret_cast<const floatx4*>(xr + k), w = *reinterpret_cast<const floatx4*>(a.norm_w + k);
                bf16x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (bf16_t)(w[e] * (v[e] * rinv));
                *reinterpret_cast<bf16x4*>(xs + m * ld + k) = o;
            }
        }
        __syncthreads();
    } else if constexpr (XK == kGated) {
        const int hpg = a.nheads / a.norm_groups, gw = a.K / a.norm_groups;
        for (int i = wave; i < a.M * a.norm_groups; i += NW) {
            const int m = i / a.norm_groups, g = i - m * a.norm_groups;
            float ss = 0.f;
            for (int h = lane; h < hpg; h += 64) ss += a.head_sq[(int64_t)m * a.nheads + g * hpg + h];
            ss = warp_sum(ss);
            if (lane == 0) rs[m][g] = rsqrtf(ss / (float)gw + a.eps);
        }
        __syncthreads();
        const int vecs = a.K / 8;
        for (int i = tid; i < a.M * vecs; i += NW * 64) {
            const int m = i / vecs, k = (i - m * vecs) * 8;
            const float r = rs[m][k / gw];
            float h[8], o[8];
            cvt16<bf16_t>(*reinterpret_cast<const uint4*>(static_cast<const bf16_t*>(a.x) + m * a.x_sr + k), h);
            const floatx4 w0 = *reinterpret_cast<const floatx4*>(a.norm_w + k), w1 = *reinterpret_cast<const floatx4*>(a.norm_w + k + 4);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (e < 4 ? w0[e & 3] : w1[e & 3]) * (h[e] * r);
            *reinterpret_cast<uint4*>(xs + m * ld + k) = pack8(o);
        }
        __syncthreads();
    }
}

template <int XK, int OK, int MT, int NW>
__global__ void __launch_bounds__(NW * 64)
linear_small_kernel(const LinearArgs a) {
    extern __shared__ __align__(16) char smem[];
    __shared__ float red[NW][MT][256];
    __shared__ float rs[XK == kGated ? 32 : 1][8];
    bf16_t* xs = reinterpret_cast<bf16_t*>(smem);
    const int ld = a.K + 8;                                  // rows 16 bytes apart in the banks
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, kq = (lane >> 4) * 8;
    const int steps = a.K / 32, s0 = steps * wave / NW, s1 = steps * (wave + 1) / NW;
    const bf16_t* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = t * 16 + r16 < a.M ? t * 16 + r16 : 0;     // columns past M repeat a row and are not stored
        xrow[t] = XK == kPlain ? static_cast<const bf16_t*>(a.x) + m * a.x_sr + kq : xs + m * ld + kq;
    }
    uint4 wa[kUN];
    auto wrow = [&](int tile) {
        const int n = tile * 16 + r16;
        return a.w + (int64_t)(n < a.N ? n : a.N - 1) * a.K + kq;
    };
    const bf16_t* wp = wrow(blockIdx.x);
#pragma unroll
    for (int u = 0; u < kUN; ++u)
        if (s0 + u < s1) wa[u] = *reinterpret_cast<const uint4*>(wp + (s0 + u) * 32);
    stage_rows<XK, NW>(a, xs, rs, ld);

    for (int tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
        floatx4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
        const int next = tile + (int)gridDim.x;
        const bf16_t* np = wrow(next < a.tiles ? next : tile);
        for (int s = s0; s < s1; s += kUN) {
            uint4 cur[kUN];
#pragma unroll
            for (int u = 0; u < kUN; ++u) cur[u] = wa[u];
            // the next kUN steps of this tile, or the first ones of the workgroup's next tile
            const bool more = s + kUN < s1;
            const bf16_t* p = more ? wp : np;
            const int f = more ? s + kUN : s0;
            if (more || next < a.tiles) {
#pragma unroll
                for (int u = 0; u < kUN; ++u)
                    if (f + u < s1) wa[u] = *reinterpret_cast<const uint4*>(p + (f + u) * 32);
            }
#pragma unroll
            for (int u = 0; u < kUN; ++u) {
                if (s + u >= s1) break;
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(cur[u]), as_frag(*reinterpret_cast<const uint4*>(xrow[t] + (s + u) * 32)),
                                                                     acc[t], 0, 0, 0);
            }
        }
        wp = np;
        // lane: column m = lane & 15, rows n = 4 (lane >> 4) + 0..3
#pragma unroll
        for (int t = 0; t < MT; ++t) *reinterpret_cast<floatx4*>(&red[wave][t][r16 * 16 + (lane >> 4) * 4]) = acc[t];
        __syncthreads();
        for (int i = tid; i < MT * 256; i += NW * 64) {
            const int m = i >> 4, n = tile * 16 + (i & 15);
            float v = 0.f;
#pragma unroll
            for (int q = 0; q < NW; ++q) v += red[q][i >> 8][i & 255];
            if (m < a.M && n < a.N) {
                if (a.bias) v += to_f32(a.bias[n]);
                const int64_t o = m * a.out_sr + n;
                if (OK == kOutBf16) static_cast<bf16_t*>(a.out)[o] = (bf16_t)v;
                else if (OK == kOutF32) static_cast<float*>(a.out)[o] = v;
                else static_cast<float*>(a.out)[o] += v;
            }
        }
        __syncthreads();
    }
    if (a.conv_state) {
        const int nch = a.conv_cx - a.conv_c0;
        for (int i = blockIdx.x * NW * 64 + tid; i < a.M * nch; i += gridDim.x * NW * 64) {
            const int b = i / nch, c = a.conv_c0 + i - b * nch;
            bf16_t* cs = a.conv_state + ((int64_t)b * a.conv_cx + c) * a.conv_W;
            for (int j = 0; j + 1 < a.conv_W; ++j) cs[j] = cs[j + 1];
            cs[a.conv_W - 1] = a.conv_in[b * a.conv_in_sb + c];
        }
    }
}

constexpr size_t kLdsRows = 40 * 1024;       // normalised rows that fit beside the partial tiles in the 64 KB a launch may ask for

template <int XK, int OK>
int launch_linear(LinearArgs a, hipStream_t st) {
    a.tiles = (int)ceil_div(a.N, 16);
    // eight waves per tile where the tiles do not fill the chip by themselves, four otherwise; workgroups that normalise
    // rows take several tiles each once there are more than two per CU
    const int64_t cus = device_cus();
    const bool wide = a.tiles < 2 * cus && a.K >= 1024;
    const int64_t most = XK == kPlain ? 4 * cus : 2 * cus;
    const unsigned grid = (unsigned)(a.tiles < most ? a.tiles : most);
    const size_t lds = XK == kPlain ? 0 : (size_t)a.M * (a.K + 8) * sizeof(bf16_t);
    auto go = [&](auto mt) {
        constexpr int MT = decltype(mt)::value;
        if (wide) linear_small_kernel<XK, OK, MT, 8><<<grid, 512, lds, st>>>(a);
        else linear_small_kernel<XK, OK, MT, 4><<<grid, 256, lds, st>>>(a);
    };
    if (a.M <= 16) go(std::integral_constant<int, 1>{}); else go(std::integral_constant<int, 2>{});
    return check_launch("linear_small_kernel");
}

// ------------------------------------------------------------------------------------------ conv + scan + gate
// One workgroup per (head, sequence), its 256 lanes laid over the state as float4s (GL lanes per row, UP rows each, all loads
// issued first).  While they arrive the lanes form the head's conv outputs: its own P channels (whose conv state it shifts)
// and the N + N channels of its group's B and C, which every head of the group forms anew (4 KB from L2 beside a 64 KB state)
// rather than wait for a kernel of their own; their states stay as they are until the product behind this kernel.
struct GatedArgs {
    float* S; const bf16_t* zx; int64_t zx_sb;            // [z | x | B | C | dt] row of a sequence
    bf16_t* conv_state; const void* conv_w; const void* conv_b;
    const float *A, *D, *dt_bias;
    bf16_t* h; float* head_sq;
    int nheads, ngroups, conv_cx, W;
};
template <typename WT, int P, int N>
__global__ void __launch_bounds__(256)
decode_gated_kernel(const GatedArgs a) {
    constexpr int GL = N / 4, ROWS = 256 / GL, UP = P / ROWS < 8 ? P / ROWS : 8, NCH = P + 2 * N;
    static_assert(P % (ROWS * UP) == 0, "whole passes over the state rows");
    __shared__ float xa[P], za[P], Ba[N], Ca[N], ha[P], red[4];
    const int tid = threadIdx.x, h = blockIdx.x, b = blockIdx.y;
    const int g = h / (a.nheads / a.ngroups), d = a.nheads * P;
    const bf16_t* row = a.zx + b * a.zx_sb;
    float* Sp = a.S + ((int64_t)b * a.nheads + h) * (P * N);
    const int sub = tid % GL, rowi = tid / GL;
    floatx4 sv[UP];
#pragma unroll
    for (int u = 0; u < UP; ++u) sv[u] = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(Sp + (u * ROWS + rowi) * N + sub * 4));
    const float dtv = softplus_f(to_f32(row[d + a.conv_cx + h]) + (a.dt_bias ? a.dt_bias[h] : 0.f));
    const float dA = __expf(a.A[h] * dtv), Dh = a.D ? a.D[h] : 0.f;
    for (int i = tid; i < NCH; i += 256) {
        const int c = i < P ? h * P + i : (i < P + N ? d + g * N + (i - P) : d + (a.ngroups + g) * N + (i - P - N));
        bf16_t* cs = a.conv_state + ((int64_t)b * a.conv_cx + c) * a.W;
        const bf16_t in = row[d + c];
        const WT* w = static_cast<const WT*>(a.conv_w) + c * 4;
        const bf16_t o1 = cs[a.W - 3], o2 = cs[a.W - 2], o3 = cs[a.W - 1];
        float z = a.conv_b ? to_f32(static_cast<const WT*>(a.conv_b)[c]) : 0.f;
        z += to_f32(w[0]) * to_f32(o1) + to_f32(w[1]) * to_f32(o2) + to_f32(w[2]) * to_f32(o3) + to_f32(w[3]) * to_f32(in);
        const float v = silu_f(z);
        if (i < P) {
            xa[i] = v;
            za[i] = silu_f(to_f32(row[h * P + i]));
            for (int j = 0; j + 1 < a.W; ++j) cs[j] = cs[j + 1];
            cs[a.W - 1] = in;
        } else if (i < P + N) Ba[i - P] = v;
        else Ca[i - P - N] = v;
    }
    __syncthreads();
    const floatx4 bv = *reinterpret_cast<const floatx4*>(Ba + sub * 4), cv = *reinterpret_cast<const floatx4*>(Ca + sub * 4);
    for (int p0 = 0; p0 < P; p0 += ROWS * UP) {
        if (p0 > 0) {
#pragma unroll
            for (int u = 0; u < UP; ++u)
                sv[u] = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(Sp + (p0 + u * ROWS + rowi) * N + sub * 4));
        }
#pragma unroll
        for (int u = 0; u < UP; ++u) {
            const int pp = p0 + u * ROWS + rowi;
            const float xv = xa[pp], dx = dtv * xv;
            float part = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q) { sv[u][q] = sv[u][q] * dA + dx * bv[q]; part += sv[u][q] * cv[q]; }
            __builtin_nontemporal_store(sv[u], reinterpret_cast<floatx4*>(Sp + pp * N + sub * 4));
            part = lane_xor_add<1>(part); part = lane_xor_add<2>(part); part = lane_xor_add<4>(part); part = lane_xor_add<8>(part);
            if (GL > 16) part = lane_xor_add<16>(part);
            if (sub == 0) ha[pp] = (part + Dh * xv) * za[pp];
        }
    }
    __syncthreads();
    float sq = 0.f;
    if (tid < P) {
        sq = ha[tid] * ha[tid];
        a.h[(int64_t)b * d + h * P + tid] = (bf16_t)ha[tid];
    }
    sq = warp_sum(sq);
    if ((tid & 63) == 0) red[tid >> 6] = sq;
    __syncthreads();
    if (tid == 0) a.head_sq[(int64_t)b * a.nheads + h] = (red[0] + red[1]) + (red[2] + red[3]);
}

int check_linear(const m2_linear_params* p) {
    M2_REQUIRE(p, M2_ERR_NULL, "linear_small: params is NULL");
    M2_REQUIRE(p->M >= 0 && p->N > 0 && p->K > 0, M2_ERR_SHAPE, "linear_small: M %lld, N %lld, K %lld", (long long)p->M, (long long)p->N, (long long)p->K);
    M2_REQUIRE(m2_linear_small_fits(p->M, p->N, p->K, p->x_kind, p->norm_groups), M2_ERR_SHAPE,
               "linear_small: M %lld, N %lld, K %lld, x kind %d: at most 32 rows, K a multiple of 32, normalised rows within 40 KB",
               (long long)p->M, (long long)p->N, (long long)p->K, (int)p->x_kind);
    if (p->M == 0) return M2_OK;
    M2_REQUIRE(p->x && p->w && p->out, M2_ERR_NULL, "linear_small: x, w and out are required");
    M2_REQUIRE(p->x_kind == kPlain || p->norm_weight, M2_ERR_NULL, "linear_small: norm_weight is required");
    M2_REQUIRE(p->x_kind != kGated || (p->head_sq && p->nheads > 0 && p->nheads % p->norm_groups == 0 && p->K % p->norm_groups == 0), M2_ERR_SHAPE,
               "linear_small: gated rows need head_sq and whole heads per norm group");
    const int64_t xv = p->x_kind == kNorm ? 4 : 8;
    M2_REQUIRE(aligned16(p->x) && aligned16(p->w) && p->x_stride_row % xv == 0 && (!p->norm_weight || aligned16(p->norm_weight)), M2_ERR_ALIGN,
               "linear_small: x rows, w and norm_weight must be 16-byte aligned");
    return M2_OK;
}

int launch_linear_params(const m2_linear_params* p, const LinearArgs& conv, hipStream_t st) {
    const int rc = check_linear(p);
    if (rc || p->M == 0) return rc;
    LinearArgs a = conv;
    a.w = static_cast<const bf16_t*>(p->w); a.bias = static_cast<const bf16_t*>(p->bias);
    a.x = p->x; a.x_sr = p->x_stride_row; a.norm_w = p->norm_weight; a.head_sq = p->head_sq;
    a.out = p->out; a.out_sr = p->out_stride_row;
    a.M = (int)p->M; a.N = (int)p->N; a.K = (int)p->K; a.nheads = (int)p->nheads; a.norm_groups = p->norm_groups; a.eps = p->eps;
    auto out = [&](auto xk) {
        constexpr int XK = decltype(xk)::value;
        if (p->out_kind == kOutBf16) return launch_linear<XK, kOutBf16>(a, st);
        if (p->out_kind == kOutF32) return launch_linear<XK, kOutF32>(a, st);
        return launch_linear<XK, kOutAdd>(a, st);
    };
    if (p->x_kind == kPlain) return out(std::integral_constant<int, kPlain>{});
    if (p->x_kind == kNorm) return out(std::integral_constant<int, kNorm>{});
    return out(std::integral_constant<int, kGated>{});
}

}  // namespace
}  // namespace m2

extern "C" int m2_linear_small_fits(int64_t M, int64_t N, int64_t K, int32_t x_kind, int32_t norm_groups) {
    using namespace m2;
    return M >= 0 && M <= 32 && N > 0 && N < (int64_t(1) << 30) && K > 0 && K % 32 == 0 && K <= (1 << 20) && x_kind >= kPlain && x_kind <= kGated &&
           (x_kind == kPlain || (size_t)M * (K + 8) * sizeof(bf16_t) <= kLdsRows) && (x_kind != kGated || (norm_groups >= 1 && norm_groups <= 8 && K / norm_groups % 8 == 0));
}

extern "C" int m2_linear_small(const m2_linear_params* p, void* stream) {
    return m2::launch_linear_params(p, m2::LinearArgs{}, static_cast<hipStream_t>(stream));
}

extern "C" int m2_decode_layer(const m2_linear_params* in, const m2_decode_params* dec, const m2_linear_params* out, void* h, float* head_sq, void* stream) {
    using namespace m2;
    M2_REQUIRE(in && dec && out, M2_ERR_NULL, "decode_layer: params is NULL");
    const int64_t P = dec->headdim, N = dec->dstate, d = dec->nheads * P, cx = d + 2 * dec->ngroups * N;
    M2_REQUIRE((P == 64 || P == 128) && (N == 64 || N == 128) && dec->k == 4 && dec->W >= 3 && dec->W <= 8 && dec->nheads > 0 && dec->ngroups > 0 &&
                   dec->nheads % dec->ngroups == 0, M2_ERR_SHAPE,
               "decode_layer: headdim %lld and dstate %lld must be 64 or 128, the conv 4 wide, the heads whole per group", (long long)P, (long long)N);
    M2_REQUIRE(dec->dtype == M2_BF16 && dec->activation == M2_ACT_SILU && (dec->param_dtype == M2_F32 || dec->param_dtype == M2_BF16), M2_ERR_DTYPE,
               "decode_layer: bf16 activations with SiLU only");
    M2_REQUIRE(in->M == dec->batch && out->M == dec->batch && in->N == d + cx + dec->nheads && out->K == d && out->x_kind == kGated && in->out_kind == kOutBf16,
               M2_ERR_SHAPE, "decode_layer: the projections do not match the layer");
    if (dec->batch == 0) return M2_OK;
    M2_REQUIRE(dec->conv_state && dec->conv_w && dec->S && dec->A && dec->dt_bias && h && head_sq, M2_ERR_NULL,
               "decode_layer: conv_state, conv_w, S, A, dt_bias, h and head_sq are required");
    M2_REQUIRE(aligned16(dec->S), M2_ERR_ALIGN, "decode_layer: S must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    int rc = check_linear(out);
    if (rc) return rc;
    rc = launch_linear_params(in, LinearArgs{}, st);
    if (rc) return rc;
    const bf16_t* zx = static_cast<const bf16_t*>(in->out);
    GatedArgs g{};
    g.S = dec->S; g.zx = zx; g.zx_sb = in->out_stride_row; g.conv_state = static_cast<bf16_t*>(dec->conv_state);
    g.conv_w = dec->conv_w; g.conv_b = dec->conv_b; g.A = dec->A; g.D = dec->D; g.dt_bias = dec->dt_bias;
    g.h = static_cast<bf16_t*>(h); g.head_sq = head_sq;
    g.nheads = (int)dec->nheads; g.ngroups = (int)dec->ngroups; g.conv_cx = (int)cx; g.W = dec->W;
    const dim3 grid((unsigned)dec->nheads, (unsigned)dec->batch);
    auto go = [&](auto wt, auto p, auto n) {
        decode_gated_kernel<decltype(wt), decltype(p)::value, decltype(n)::value><<<grid, 256, 0, st>>>(g);
    };
    auto dims = [&](auto wt) {
        using c64 = std::integral_constant<int, 64>;
        using c128 = std::integral_constant<int, 128>;
        if (P == 64) { if (N == 64) go(wt, c64{}, c64{}); else go(wt, c64{}, c128{}); }
        else { if (N == 64) go(wt, c128{}, c64{}); else go(wt, c128{}, c128{}); }
    };
    if (dec->param_dtype == M2_F32) dims(float{}); else dims(bf16_t{});
    rc = check_launch("decode_gated_kernel");
    if (rc) return rc;
    LinearArgs conv{};
    conv.conv_state = g.conv_state; conv.conv_in = zx + d; conv.conv_in_sb = in->out_stride_row;
    conv.conv_c0 = (int)d; conv.conv_cx = (int)cx; conv.conv_W = dec->W;
    return launch_linear_params(out, conv, st);
}
