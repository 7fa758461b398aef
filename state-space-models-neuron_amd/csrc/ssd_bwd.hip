// SSD chunked-scan backward for gfx950.
//
// Replaces the reference's NKI kernel mamba_kernel_bwd_ (mamba2/mamba2_kernel.py:277-485): same
// gradients (ddt, dA, dX, dB, dC, dD), forward recomputed per chunk instead of storing the decay
// matrix L, any batch size (the reference is batch-1 only, :315-317), optional gradient of the
// final state and of the initial state.
//
// Per head and chunk, with l the in-chunk cumulative sum of A*dt, Lam = l_{Q-1}, xd = dt*x,
// dS the gradient w.r.t. the state LEAVING the chunk and S_prev the state ENTERING it:
//   dxd_j = sum_{i>=j} e^{l_i-l_j} G[i][j] dy_i + e^{Lam-l_j} dS B_j          dx = dt dxd + D dy
//   dG[i][j] = sum_h e^{l_i-l_j} dt_j (dy_i . x_j)           (i >= j, summed over the heads of a group)
//   dC_i = sum_j dG[i][j] B_j + sum_h e^{l_i} dy_i^T S_prev
//   dB_j = sum_i dG[i][j] C_i + sum_h dt_j e^{Lam-l_j} x_j^T dS
//   dl_i = sum_n (C_i o dC_i^h - B_i o dB_i^h)               (row role minus column role of l_i, per head;
//                                                             the reference's C o dC - B o dB, :401,456)
//        = rowsum_i(dG^h o G) - colsum_i(dG^h o G) + C_i . dCoff_i^h - B_i . dBoff_i^h
//   da_j = sum_{i>=j, same chunk} dl_i + <dS, S_new>         ddt_j = A da_j + dxd_j . x_j
//   dA   = sum_j da_j dt_j                                   dD = sum dy . x
// Row sums and column sums are taken from the SAME fp32 tile dG^h o G, so pairs (i, j) that both lie
// in a suffix cancel exactly and only pairs straddling the position contribute, as in exact
// arithmetic.  (Forming dl from dy . (y - D x) with the stored bf16 y loses everything to
// cancellation once D x dominates y.)  The state term is evaluated in the equivalent form
//   <dS, S_new> - sum_{i>=j} (B_i . dBoff_i^h)  =  e^{Lam} <dS, S_prev> + sum_{i<j} (B_i . dBoff_i^h)
// (a prefix instead of a suffix of the per-token terms), which avoids subtracting two large numbers that were
// rounded differently.  Everything is exact per chunk, so rounding does not accumulate along the sequence as it
// would with a global reverse cumulative sum (:459-461).
//
// Launch sequence (16-bit operands; fp32 operands take the kernels named in brackets):
//   prep_kernel, state_pass16_kernel [chunk_state + state_scan]   recompute G, tables, S_prev (skipped if the caller kept them)
//   state_pass16_kernel<REVERSE> [chunk_state32<DSTATE> + state_scan<REVERSE>]
//                                                              dS per chunk, d initial state
//   dg16_kernel               per (b, chunk, group, head slice)  partial dG (heads reduced in registers), dl_diag per head
//   ssd_bwd16_kernel          per (b, chunk, group, head slice)  dx, per-token decay-gradient terms, dD and e^{Lam} <dS, S_prev> partials,
//                                                                partial state parts of dB / dC
//   [ssd_bwd32_kernel         what those two do in one pass; dB and dC too where a workgroup has all heads of its group]
//   tail1_kernel              da_body: ddt, dA partials per (b, head, chunk);  slice_sum_body: partials over the head slices
//   tail2_kernel              group_finish16_body per (b, chunk, group, token block) [bc_final32_body per (b, chunk, group, side)], unless done
//                             already: dC = dG B + dCoff, dB = dG^T C + dBoff;  ad_reduce_body per head: dA, dD (fixed order, no atomics)
#include "ssd_host.hpp"

namespace m2 {
namespace {

// Sum of the per-slice partials (fixed order) of up to three arrays in one launch.  One thread per float4;
// `tile` floats per (group, slice) tile; segment k covers threads [first_k, first_{k+1}).
struct SliceSumSeg { const float* part; float* out; int64_t nslices, tile, first; int lower; };      // lower: kQ x kQ, blocks above the diagonal unused
struct SliceSumArgs { SliceSumSeg seg[3]; int nseg; int64_t total; };
template <int THREADS>
__device__ __forceinline__ void slice_sum_body(const SliceSumArgs& a, int64_t blk) {
    const int64_t idx = blk * THREADS + threadIdx.x;
    if (idx >= a.total) return;
    int k = 0;
    if (a.nseg > 1 && idx >= a.seg[1].first) k = 1;
    if (a.nseg > 2 && idx >= a.seg[2].first) k = 2;
    const SliceSumSeg sg = a.seg[k];
    const int64_t per = sg.tile / 4, loc = idx - sg.first;
    const int64_t grp = loc / per, e = (loc % per) * 4;
    if (sg.lower && ((e % kQ) >> 5) > e / (32 * kQ)) return;
    floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int64_t sl = 0; sl < sg.nslices; ++sl) s += *reinterpret_cast<const floatx4*>(sg.part + (grp * sg.nslices + sl) * sg.tile + e);
    *reinterpret_cast<floatx4*>(sg.out + grp * sg.tile + e) = s;
}
// The slice sums and the per-chunk decay-gradient scan (da_body) in one launch: they are independent, and both are short.
template <typename T>
__global__ void __launch_bounds__(kDaHeads * 64)
tail1_kernel(const DaArgs d, const int64_t n_da, const SliceSumArgs a) {
    const int64_t blk = blockIdx.x;
    if (blk < n_da) da_body<T>(d, blk);
    else slice_sum_body<kDaHeads * 64>(a, blk - n_da);
}

// ------------------------------------------------------------------------------------------
// Group-level finish for 16-bit operands whose heads are cut into slices, from the summed partials:
//   dC[i][n] = sum_{j<=i} dG[i][j] B[j][n] + dCoff[i][n],      dB[j][n] = sum_{i>=j} dG[i][j] C[i][n] + dBoff[j][n]
// One workgroup of 8 waves per (batch, chunk, group) and block of 32 tokens, wave w the column block w & 3 of dC (w < 4) or dB.  The
// token block meets four 32x32 blocks of dG, (rb, 0 .. rb) for dC and (rb .. 3, rb) for dB: they come through LDS, fp32, 16-byte slots
// swizzled by the row, and a fragment is split into value and remainder in registers, so the contractions see dG at ~2^-17 relative.
// The accumulators start from the summed state parts (16-byte loads), B^T / C^T fragments are contiguous KiB of the operand-order
// tiles; everything is asked for in front of the one barrier, and a lane owns one token: 16-byte stores after one lane-pair swap per
// 4-column group.
// What bounds it is latency: hence the quarter of a triple per workgroup.  As one workgroup per side, which put all of dG through LDS in
// two 16-bit tiles, the launch took 8.8 us at 27 triples, 8.6 at 4 and 10.4 at 64 (b4 l2048 h80); 6.7, 6.5 and 9.1 so.
struct GroupFinishArgs {
    const float* dG; const float* dCoff; const float* dBoff; const void* Bt; const void* Ct; void* dB; void* dC;
    int64_t dBsb, dBsl, dBsg, dCsb, dCsl, dCsg, seqlen, ngroups, nchunks, n;      // n: workgroups
};
template <typename T, int N>
__device__ __forceinline__ void group_finish16_body(const GroupFinishArgs& a, int64_t blk) {
    static_assert(sizeof(T) == 2, "16-bit operands only");
    __shared__ __align__(16) float sG[4][32 * 32];      // block q: (rb, q) up to the diagonal, (q, rb) behind it
    const int tid = threadIdx.x, wave = (int)uniform(tid >> 6), lane = tid & 63, r = lane & 31, half = lane >> 5;
    const int rb = (int)(blk & 3), tok = rb * 32 + r;
    const int64_t grp = blk >> 2, g = grp % a.ngroups, c = grp / a.ngroups % a.nchunks, b = grp / (a.ngroups * a.nchunks), t0 = c * kQ;
    const int valid = (int)((a.seqlen - t0) < kQ ? (a.seqlen - t0) : kQ);
    const bool side_b = wave >= 4;
    const int nb = wave & 3, row = (tid & 255) >> 3, slot = tid & 7;
    const bool active = nb < N / 32;                    // with 64 state columns half of the waves only help to fetch dG
    floatx4 v[2];
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int q = it * 2 + (wave >> 2), bi = q <= rb ? rb : q, bj = q <= rb ? q : rb;
        v[it] = *reinterpret_cast<const floatx4*>(a.dG + grp * (int64_t)(kQ * kQ) + (bi * 32 + row) * kQ + bj * 32 + slot * 4);
    }
    floatx16 acc;
    Frag<T> xf[8];
    const int ks0 = side_b ? 2 * rb : 0, ks1 = side_b ? 8 : 2 * rb + 2;      // 16-wide k blocks of this wave
    if (active) {
        const float* op = (side_b ? a.dBoff : a.dCoff) + grp * (int64_t)(kQ * N) + (int64_t)tok * N + nb * 32 + 4 * half;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const floatx4 o = *reinterpret_cast<const floatx4*>(op + 8 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * q + e] = o[e];
        }
        const char* tile = static_cast<const char*>(side_b ? a.Ct : a.Bt) + grp * (int64_t)(N * kQ * 2) + nb * 8 * 1024;      // see mt_offset
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
            if (ks >= ks0 && ks < ks1) xf[ks].v = *reinterpret_cast<const bf16x8*>(tile + ((uint32_t)lane * 16u + (uint32_t)(ks * 1024)));
    }
#pragma unroll
    for (int it = 0; it < 2; ++it) *reinterpret_cast<floatx4*>(&sG[it * 2 + (wave >> 2)][row * 32 + ((slot ^ (row & 7)) * 4)]) = v[it];
    __syncthreads();
    if (!active) return;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        if (ks < ks0 || ks >= ks1) continue;      // wave-uniform
        const float* blk_g = sG[ks >> 1];
        const int k0 = (ks & 1) * 16 + 8 * half;
        float f[8];
        if (side_b) {
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = blk_g[(k0 + e) * 32 + (((r >> 2) ^ e) * 4) + (r & 3)];
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const floatx4 o = *reinterpret_cast<const floatx4*>(blk_g + r * 32 + (((k0 >> 2) + q) ^ (r & 7)) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) f[4 * q + e] = o[e];
            }
        }
        Frag<T> yh, yl;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            yh.v[e] = from_f32<T>(f[e]);
            yl.v[e] = from_f32<T>(f[e] - to_f32((T)yh.v[e]));
        }
        mma_frag(acc, xf[ks], yh);
        mma_frag(acc, xf[ks], yl);
    }
    T* out = side_b ? static_cast<T*>(a.dB) + b * a.dBsb + (t0 + tok) * a.dBsl + g * a.dBsg : static_cast<T*>(a.dC) + b * a.dCsb + (t0 + tok) * a.dCsl + g * a.dCsg;
#pragma unroll
    for (int qp = 0; qp < 2; ++qp) {
        float g8[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) pair_swap(acc[8 * qp + e], acc[8 * qp + 4 + e], g8[e], g8[4 + e]);
        const uint4 o = {pack2<T>(g8[0], g8[1]), pack2<T>(g8[2], g8[3]), pack2<T>(g8[4], g8[5]), pack2<T>(g8[6], g8[7])};
        if (tok < valid) *reinterpret_cast<uint4*>(out + nb * 32 + 8 * (2 * qp + half)) = o;
    }
}

// dA[h] = sum_{b,c} dAp[b][h][c], dD likewise (fixed order, no atomics).  One workgroup of 512 threads per head.
__device__ __forceinline__ void ad_reduce_body(const float* __restrict__ dAp, const float* __restrict__ dDp, const float* __restrict__ dbp,
                                               float* __restrict__ dA, float* __restrict__ dD, float* __restrict__ dbias,
                                               int64_t nb, int64_t nheads, int64_t nchunks, int64_t h) {
    __shared__ float red[3][8];
    float sa = 0.f, sd = 0.f, sb = 0.f;
    for (int64_t e = threadIdx.x; e < nb * nchunks; e += 512) {
        const int64_t b = e / nchunks, c = e % nchunks;
        sa += dAp[(b * nheads + h) * nchunks + c];
        sd += dDp[(b * nheads + h) * nchunks + c];
        if (dbias) sb += dbp[(b * nheads + h) * nchunks + c];
    }
    sa = warp_sum(sa); sd = warp_sum(sd); sb = warp_sum(sb);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { red[0][wave] = sa; red[1][wave] = sd; red[2][wave] = sb; }
    __syncthreads();
    if (threadIdx.x == 0) {
        float ta = 0.f, td = 0.f, tb = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) { ta += red[0][q]; td += red[1][q]; tb += red[2][q]; }
        dA[h] = ta;
        if (dD) dD[h] = td;
        if (dbias) dbias[h] = tb;
    }
}

// The group-level finish, where the main kernel has not done it, and behind its workgroups the per-head reductions, one workgroup each,
// in one launch.
struct Tail2Args {
    const float* dAp; const float* dDp; const float* dbp; float* dA; float* dD; float* dbias;
    int64_t seqlen, ngroups, nchunks, batch, nheads;
};
struct Tail2Args32 : Tail2Args {
    const float* dGp; const float* dCp; const float* dBp; const void* B; const void* C; void* dB; void* dC;
    int64_t dBsb, dBsl, dBsg, dCsb, dCsl, dCsg, Bsb, Bsl, Bsg, Csb, Csl, Csg, n_bc;
};
template <typename T, int N>
__global__ void __launch_bounds__(512)
tail2_kernel(const Tail2Args a, const GroupFinishArgs f) {
    const int64_t blk = blockIdx.x;
    if (blk < f.n) group_finish16_body<T, N>(f, blk);
    else ad_reduce_body(a.dAp, a.dDp, a.dbp, a.dA, a.dD, a.dbias, a.batch, a.nheads, a.nchunks, blk - f.n);
}
template <int N>
__global__ void __launch_bounds__(512)
tail2_32_kernel(const Tail2Args32 a) {
    const int64_t blk = blockIdx.x;
    if (blk < a.n_bc) {
        const int64_t grp = blk >> 1, c = grp % a.nchunks, g = (grp / a.nchunks) % a.ngroups, b = grp / (a.nchunks * a.ngroups);
        auto finish = [&](auto side) {
            bc_final32_body<N, decltype(side)::value>(a.dGp, a.dCp, a.dBp, static_cast<const float*>(a.B), a.Bsb, a.Bsl, a.Bsg, static_cast<const float*>(a.C), a.Csb,
                                                      a.Csl, a.Csg, static_cast<float*>(a.dB), a.dBsb, a.dBsl, a.dBsg, static_cast<float*>(a.dC), a.dCsb, a.dCsl, a.dCsg,
                                                      a.seqlen, a.ngroups, a.nchunks, c, g, b);
        };
        if (blk & 1) finish(std::integral_constant<int, 2>{});
        else finish(std::integral_constant<int, 1>{});
    } else {
        ad_reduce_body(a.dAp, a.dDp, a.dbp, a.dA, a.dD, a.dbias, a.batch, a.nheads, a.nchunks, blk - a.n_bc);
    }
}

__global__ void zero_f32_kernel(float* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}
__global__ void copy_f32_kernel(const float* __restrict__ src, float* __restrict__ dst, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src ? src[i] : 0.f;
}

template <typename T, int P, int N, int HS>
int ssd_bwd_impl(const SsdCall* p, hipStream_t st) {
    const int64_t nc = ceil_div(p->seqlen, (int64_t)kQ);
    const SsdWorkspace w = ssd_carve(p, p->workspace, true);
    const int dt_f32 = p->dt_dtype == M2_F32;
    const T* x = static_cast<const T*>(p->x);
    const T* dy = static_cast<const T*>(p->dy);
    const dim3 grid_g((unsigned)nc, (unsigned)(p->ngroups * w.ns_g), (unsigned)p->batch);
    const dim3 grid_b((unsigned)nc, (unsigned)(p->ngroups * w.ns_b), (unsigned)p->batch);
    M2_REQUIRE(p->nheads <= 65535, M2_ERR_SHAPE, "ssd_bwd: too many group slices");
    int rc;
    // decay tables, G (+ operand tiles) and the state entering each chunk, unless the caller kept the forward's
    if (!p->chunk_states && (rc = ssd_launch_states<T, P, N, HS>(p, w, nullptr, false, true, st))) return rc;
    // gradient of the state leaving each chunk (reverse recurrence over the chunks' own contributions)
    if constexpr (sizeof(T) == 2) {
        StatePassArgs sa{};
        sa.X = dy; sa.X_sb = p->dy_stride_b; sa.X_sl = p->dy_stride_l; sa.X_sh = p->dy_stride_h;
        sa.ldtab = w.ldtab; sa.Mt = w.Ct; sa.init = p->d_final_state; sa.prev = w.dprev; sa.final_out = p->d_initial_state;
        sa.seqlen = p->seqlen; sa.nheads = p->nheads; sa.ngroups = p->ngroups; sa.nchunks = nc;
        if ((rc = launch_state_pass16<T, P, N, true, HS, false>(sa, w, p->batch, kSegOneTile, st))) return rc;
        if ((rc = check_launch("ssd state_pass16_kernel<reverse>"))) return rc;
    } else
    {   // fp32: local dS contributions (reuses the `local` region), then the reverse recurrence
        if ((rc = launch_chunk_state32<N, true, HS>(p, w, dy, p->dy_stride_b, p->dy_stride_l, p->dy_stride_h, p->C, p->C_stride_b, p->C_stride_l, p->C_stride_g, st))) return rc;
        state_scan_kernel<P * N, true><<<dim3((unsigned)p->nheads, (unsigned)p->batch, kScanSplit), 256, 0, st>>>(
            w.local, w.lam, p->d_final_state, static_cast<float*>(w.dprev), p->d_initial_state, p->nheads, nc);
        if ((rc = check_launch("ssd state_scan_kernel<reverse>"))) return rc;
    }
    if constexpr (sizeof(T) == 2) {
        {
            auto k = dg16_kernel<T, P, HS>;
            const size_t sm = dg16_smem<P>();
            if ((rc = allow_smem(k, sm))) return rc;
            k<<<grid_g, kDgWaves * 64, sm, st>>>(x, w.ldtab, dy, w.G, w.dGp, w.dl,
                                       p->seqlen, p->nheads, p->ngroups, nc, w.ns_g, w.hps_g,
                                       p->x_stride_b, p->x_stride_l, p->x_stride_h,
                                       p->dy_stride_b, p->dy_stride_l, p->dy_stride_h);
            if ((rc = check_launch("ssd dg16_kernel"))) return rc;
        }
        Bwd16Args m{};
        m.ldtab = w.ldtab; m.D = p->D;
        m.Bm = p->B; m.B_sb = p->B_stride_b; m.B_sl = p->B_stride_l; m.B_sg = p->B_stride_g;
        m.Cm = p->C; m.C_sb = p->C_stride_b; m.C_sl = p->C_stride_l; m.C_sg = p->C_stride_g;
        m.Gmt = w.Gmt; m.dS = w.dprev; m.Sprev = w.prev;
        m.dy = p->dy; m.dy_sb = p->dy_stride_b; m.dy_sl = p->dy_stride_l; m.dy_sh = p->dy_stride_h;
        m.x = p->x; m.x_sb = p->x_stride_b; m.x_sl = p->x_stride_l; m.x_sh = p->x_stride_h;
        m.dx = p->dx; m.dx_sb = p->dx_stride_b; m.dx_sl = p->dx_stride_l; m.dx_sh = p->dx_stride_h;
        m.dirp = w.dirp; m.rbp = w.rbp; m.dlc = w.dlc; m.dDp8 = w.dDp8; m.dlam = w.dlam; m.dBp = w.dBp; m.dCp = w.dCp;
        m.seqlen = p->seqlen; m.nheads = p->nheads; m.ngroups = p->ngroups; m.nchunks = nc;
        m.nslices = w.ns_b; m.hps = w.hps_b;
        m.dG = w.dGp; m.Bt = w.Bt; m.Ct = w.Ct;
        m.dB = p->dB; m.dB_sb = p->dB_stride_b; m.dB_sl = p->dB_stride_l; m.dB_sg = p->dB_stride_g;
        m.dC = p->dC; m.dC_sb = p->dC_stride_b; m.dC_sl = p->dC_stride_l; m.dC_sg = p->dC_stride_g;
        auto k = w.finished ? ssd_bwd16_kernel<T, P, N, HS, true> : ssd_bwd16_kernel<T, P, N, HS, false>;
        const size_t sm = bwd16_smem<P, N>();
        if ((rc = allow_smem(k, sm))) return rc;
        k<<<grid_b, 512, sm, st>>>(m);
        if ((rc = check_launch("ssd_bwd16_kernel"))) return rc;
    } else {
        Bwd32Args m{};
        m.ldtab = w.ldtab; m.D = p->D;
        m.Bm = static_cast<const float*>(p->B); m.B_sb = p->B_stride_b; m.B_sl = p->B_stride_l; m.B_sg = p->B_stride_g;
        m.Cm = static_cast<const float*>(p->C); m.C_sb = p->C_stride_b; m.C_sl = p->C_stride_l; m.C_sg = p->C_stride_g;
        m.Bt = static_cast<const float*>(w.Bt); m.Gm = static_cast<const float*>(w.Gm); m.Gmt = static_cast<const float*>(w.Gmt);
        m.dS = static_cast<const float*>(w.dprev); m.Sprev = static_cast<const float*>(w.prev);
        m.dy = dy; m.dy_sb = p->dy_stride_b; m.dy_sl = p->dy_stride_l; m.dy_sh = p->dy_stride_h;
        m.x = x; m.x_sb = p->x_stride_b; m.x_sl = p->x_stride_l; m.x_sh = p->x_stride_h;
        m.dx = static_cast<float*>(p->dx); m.dx_sb = p->dx_stride_b; m.dx_sl = p->dx_stride_l; m.dx_sh = p->dx_stride_h;
        m.dB = static_cast<float*>(p->dB); m.dB_sb = p->dB_stride_b; m.dB_sl = p->dB_stride_l; m.dB_sg = p->dB_stride_g;
        m.dC = static_cast<float*>(p->dC); m.dC_sb = p->dC_stride_b; m.dC_sl = p->dC_stride_l; m.dC_sg = p->dC_stride_g;
        m.dGp = w.dGp; m.dBp = w.dBp; m.dCp = w.dCp; m.dirp = w.dirp; m.rbp = w.rbp; m.dl = w.dl; m.dlc = w.dlc; m.dDp8 = w.dDp8; m.dlam = w.dlam;
        m.seqlen = p->seqlen; m.nheads = p->nheads; m.ngroups = p->ngroups; m.nchunks = nc; m.nslices = w.ns_b; m.hps = w.hps_b;
        auto k = ssd_bwd32_kernel<N, HS>;
        const size_t sm = bwd32_smem<N>();
        if ((rc = allow_smem(k, sm))) return rc;
        k<<<grid_b, 512, sm, st>>>(m);
        if ((rc = check_launch("ssd_bwd32_kernel"))) return rc;
    }
    // the per-chunk scan that turns the per-token terms into ddt and dA partials runs with the slice sums below
    DaArgs da{};
    da.ldtab = w.ldtab; da.A = p->A; da.dl_diag = w.dl; da.dl_c = w.dlc; da.dlam = w.dlam;
    da.dirp = w.dirp; da.rbp = w.rbp; da.dDp8 = w.dDp8;
    da.ddt = p->ddt; da.dt_f32 = dt_f32; da.ddt_sb = p->ddt_stride_b; da.ddt_sl = p->ddt_stride_l; da.dAp = w.dAp; da.dDp = w.dDp;
    da.dbp = p->dt_bias ? w.dbp : nullptr;
    da.seqlen = p->seqlen; da.nheads = p->true_heads; da.nchunks = nc; da.batch = p->batch; da.hs = p->hs;
    {
        const int64_t ngrp = p->batch * nc * p->ngroups;
        const float *gs = w.dGp, *cs = w.dCp, *bs = w.dBp;
        {
            SliceSumArgs sa{};
            int64_t first = 0;
            auto add = [&](const float* part, float* out, int64_t ns, int64_t tile, int lower, const float** use) {
                if (ns <= 1) return;
                sa.seg[sa.nseg++] = SliceSumSeg{part, out, ns, tile, first, lower};
                first += ngrp * tile / 4;
                *use = out;
            };
            add(w.dGp, w.dGs, w.ns_g, (int64_t)kQ * kQ, 1, &gs);
            add(w.dCp, w.dCs, w.ns_b, (int64_t)kQ * N, 0, &cs);
            add(w.dBp, w.dBs, w.ns_b, (int64_t)kQ * N, 0, &bs);
            sa.total = first;
            const int64_t n_da = da_blocks(da), n_ss = ceil_div(first, (int64_t)(kDaHeads * 64));
            tail1_kernel<T><<<(unsigned)(n_da + n_ss), kDaHeads * 64, 0, st>>>(da, n_da, sa);
        }
        if ((rc = check_launch("ssd tail1_kernel"))) return rc;
        const int64_t n_bc = w.finished ? 0 : ngrp;
        Tail2Args32 ta{};
        ta.dAp = w.dAp; ta.dDp = w.dDp; ta.dbp = w.dbp; ta.dA = p->dA; ta.dD = p->D ? p->dD : nullptr;
        ta.dbias = p->dt_bias ? p->d_dt_bias : nullptr;
        ta.seqlen = p->seqlen; ta.ngroups = p->ngroups; ta.nchunks = nc; ta.batch = p->batch; ta.nheads = p->true_heads;
        if constexpr (sizeof(T) == 2) {
            GroupFinishArgs f{};
            f.dG = gs; f.dCoff = cs; f.dBoff = bs; f.Bt = w.Bt; f.Ct = w.Ct; f.dB = p->dB; f.dC = p->dC;
            f.dBsb = p->dB_stride_b; f.dBsl = p->dB_stride_l; f.dBsg = p->dB_stride_g;
            f.dCsb = p->dC_stride_b; f.dCsl = p->dC_stride_l; f.dCsg = p->dC_stride_g;
            f.seqlen = p->seqlen; f.ngroups = p->ngroups; f.nchunks = nc; f.n = 4 * n_bc;
            tail2_kernel<T, N><<<(unsigned)(f.n + p->true_heads), 512, 0, st>>>(ta, f);
        } else {
            ta.dGp = gs; ta.dCp = cs; ta.dBp = bs; ta.B = p->B; ta.C = p->C; ta.dB = p->dB; ta.dC = p->dC;
            ta.Bsb = p->B_stride_b; ta.Bsl = p->B_stride_l; ta.Bsg = p->B_stride_g; ta.Csb = p->C_stride_b; ta.Csl = p->C_stride_l; ta.Csg = p->C_stride_g;
            ta.dBsb = p->dB_stride_b; ta.dBsl = p->dB_stride_l; ta.dBsg = p->dB_stride_g;
            ta.dCsb = p->dC_stride_b; ta.dCsl = p->dC_stride_l; ta.dCsg = p->dC_stride_g;
            ta.n_bc = 2 * n_bc;
            auto k = tail2_32_kernel<N>;
            if ((rc = allow_smem(k, finish32_smem<N>()))) return rc;
            k<<<(unsigned)(2 * n_bc + p->true_heads), 512, n_bc ? finish32_smem<N>() : 0, st>>>(ta);
        }
        if ((rc = check_launch("ssd tail2_kernel"))) return rc;
    }
    return M2_OK;
}

}  // namespace
}  // namespace m2

extern "C" size_t m2_ssd_bwd_workspace_bytes(const m2_ssd_params* p) {
    if (!p || p->batch <= 0 || p->seqlen <= 0 || p->nheads <= 0 || p->ngroups <= 0) return 256;
    const m2::SsdCall q(p);
    return m2::ssd_carve(&q, nullptr, true).bytes;
}

extern "C" int m2_ssd_bwd(const m2_ssd_params* p, void* stream) {
    using namespace m2;
    int rc = ssd_check(p, "ssd_bwd");
    if (rc) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (p->nheads == 0) return M2_OK;
    M2_REQUIRE(p->dA, M2_ERR_NULL, "ssd_bwd: dA is required");
    M2_REQUIRE(!p->D || p->dD, M2_ERR_NULL, "ssd_bwd: dD is required when D is given");
    M2_REQUIRE(!p->dt_bias || p->d_dt_bias, M2_ERR_NULL, "ssd_bwd: d_dt_bias is required when dt_bias is given");
    if (p->batch == 0 || p->seqlen == 0) {
        // empty reductions: parameter gradients are zero; the state gradient passes straight through
        zero_f32_kernel<<<(unsigned)ceil_div(p->nheads, (int64_t)256), 256, 0, st>>>(p->dA, p->nheads);
        if (p->dD) zero_f32_kernel<<<(unsigned)ceil_div(p->nheads, (int64_t)256), 256, 0, st>>>(p->dD, p->nheads);
        if (p->dt_bias) zero_f32_kernel<<<(unsigned)ceil_div(p->nheads, (int64_t)256), 256, 0, st>>>(p->d_dt_bias, p->nheads);
        if (p->d_initial_state && p->batch > 0) {
            const int64_t n = p->batch * p->nheads * p->headdim * p->dstate;
            copy_f32_kernel<<<(unsigned)ceil_div(n, (int64_t)256), 256, 0, st>>>(p->d_final_state, p->d_initial_state, n);
        }
        return check_launch("ssd_bwd (empty)");
    }
    M2_REQUIRE(p->x && p->dt && p->A && p->B && p->C && p->dy, M2_ERR_NULL, "ssd_bwd: x, dt, A, B, C, dy are required");
    M2_REQUIRE(p->dx && p->ddt && p->dB && p->dC, M2_ERR_NULL, "ssd_bwd: dx, ddt, dB, dC are required");
    const int V = p->dtype == M2_F32 ? 4 : 8;
    M2_REQUIRE(p->dy_stride_b % V == 0 && p->dy_stride_l % V == 0 && p->dy_stride_h % V == 0 && aligned16(p->dy), M2_ERR_ALIGN,
               "ssd_bwd: dy must be 16-byte aligned with strides that are multiples of %d elements", V);
    // the gradients leave as 16-byte row stores
    M2_REQUIRE(p->dx_stride_b % V == 0 && p->dx_stride_l % V == 0 && p->dx_stride_h % V == 0 && aligned16(p->dx) &&
               p->dB_stride_b % V == 0 && p->dB_stride_l % V == 0 && p->dB_stride_g % V == 0 && aligned16(p->dB) &&
               p->dC_stride_b % V == 0 && p->dC_stride_l % V == 0 && p->dC_stride_g % V == 0 && aligned16(p->dC), M2_ERR_ALIGN,
               "ssd_bwd: dx, dB, dC must be 16-byte aligned with strides that are multiples of %d elements", V);
    const size_t need = m2_ssd_bwd_workspace_bytes(p);
    M2_REQUIRE(p->workspace && p->workspace_bytes >= need, M2_ERR_WORKSPACE, "ssd_bwd: workspace %zu bytes < %zu needed",
               p->workspace_bytes, need);
    M2_REQUIRE((reinterpret_cast<uintptr_t>(p->workspace) & 255u) == 0, M2_ERR_ALIGN, "ssd_bwd: workspace must be 256-byte aligned");
    const SsdCall q(p);
    M2_DISPATCH_DTYPE(p->dtype, T, M2_DISPATCH_N_HS(&q, N, HS, return (ssd_bwd_impl<T, kP, N, HS>(&q, st))));
    return M2_OK;
}
