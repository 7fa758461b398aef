// SSD chunked-scan building blocks shared by the forward and the backward (gfx950).
//
// Notation (one head, one chunk of kQ = 128 tokens, local indices i, j):
//   a_j = A * dt_j,  l_i = sum_{j<=i} a_j (inclusive, fp32),  Lam = l_{Q-1}
//   G[i][j]  = C_i . B_j                         (per group)
//   y_i      = sum_{j<=i} e^{l_i-l_j} dt_j G[i][j] x_j  +  e^{l_i} C_i . S_prev  +  D x_i
//   S_new    = e^{Lam} S_prev + sum_j e^{Lam-l_j} dt_j x_j (x) B_j          (S is [p][n])
// The decay is always evaluated on the DIFFERENCE l_i - l_j <= 0 (the factorised form
// overflows fp32: with A = -16, dt = 0.1 the cumulative sum reaches -204.8 in one chunk),
// as the reference does (mamba2/mamba2_kernel.py:32-33).
//
// Kernels here (all launched with the chunk index in blockIdx.x so consecutive workgroups,
// which the hardware deals round-robin to the 8 XCDs, still share B/C/G tiles of one batch
// row through the MALL, and each XCD's L2 sees whole (head, chunk) tiles):
//   prep_kernel        decay tables per (batch, head, chunk); G = C B^T and the operand tiles per (batch, chunk, group)
//   state_scan_kernel  sequential-in-chunks, parallel-in-(b,h,p,n) fp32 recurrence over the chunks' own contributions
//                      (chunk_state32_kernel); writes the state ENTERING each chunk, and the final state
//                      (REVERSE variant: the gradient recurrence).  fp32 operands only; for 16-bit operands
//                      ssd_states16.hpp forms the contributions and the recurrence in one pass.
#pragma once
#include <type_traits>

#include "mma.hpp"

namespace m2 {


// ------------------------------------------------------------------------------------------
// Per (batch, chunk, group): G = C B^T and the head-independent operand tiles every other kernel reuses.
//   Gf  [kQ][kQ] fp32            G[i][j] (all blocks with block-row >= block-col)
//   Gm  [kQ][kQ] T               causal G:  G[i][j] for i >= j, else 0         (forward diagonal term, rows i)
//   Gmt [kQ][kQ] T               its transpose: Gmt[j][i] = G[i][j] for i >= j (backward dx term, rows j)
//   (each of Gf, Gm, Gmt and Ct only where it is not null: the forward alone reads Gm and Bt)
//   Bt, Ct N x kQ T              (16-bit) B and C transposed, laid out by mt_offset: MFMA operands of the chunk-state products
// fp32 operands: Gm and Gmt (and, where the backward will run, a copy of B in Bt) in the order in which a wave takes its operand
// rows, op32_offset; no Gf, Ct.
// kCbParts workgroups of 256 threads per (chunk, group, batch), see cb_body.  The upper-right 64x64 quadrant of G is
// never consumed and is neither computed nor written.
// Element offset of the 8 tokens s0 .. s0 + 7 (s0 a multiple of 8) of state column n inside a transposed B / C tile: MFMA operand
// order [N / 32][kQ / 16][64 lanes][8], so that the B-operand fragment of a wave for column block n / 32 and k-step s0 / 16 is one
// contiguous KiB, lane = 32 ((s0 / 8) & 1) + n % 32 (read by state_pass16_kernel straight into registers, eight full cache lines
// per load instruction).
__device__ __forceinline__ int64_t mt_offset(int n, int s0) {
    return ((int64_t)((n >> 5) * (kQ / 16) + (s0 >> 4)) * 64 + ((s0 >> 3) & 1) * 32 + (n & 31)) * 8;
}

// The four elements k = 16 (u / 2) + 8 half + 4 (u % 2) + 0..3 of operand row 32 rb + r, fp32: step u of row block rb is one contiguous
// KiB, lane 32 half + r (a step straight from rows touches 32 of them, 2 x 16 bytes each: the loads of B and of C B^T then held the
// phase of ssd_bwd32_kernel that needs them for 23.5 k cycles instead of 21.5).
template <int STEPS>
__device__ __forceinline__ int op32_offset(int rb, int u, int lane) { return ((rb * STEPS + u) * 64 + lane) * 4; }

// Workgroups per (chunk, group, batch): three for the 64x64 quadrants of G on and below the diagonal, four for the
// transposed tiles or the copy of B (32 tokens each; none without Bt) -- seven short independent pieces rather than two long ones.
constexpr int kCbParts = 7, kCbGParts = 3;
constexpr int kXcds = 8;
__host__ __device__ inline int64_t cb_blocks(int64_t n_cb, int parts) { return (n_cb + kXcds - 1) / kXcds * kXcds * parts; }
// Contraction length staged at once: all of it (one staging phase, one barrier), but fp32 rows of 128 in two halves, so that
// four workgroups fit a CU and not two (66 -> 51 us at b3 l2048 h32 g8 with transposed tiles of B and C, 33 since B is copied as it lies).
template <typename T> __host__ __device__ constexpr int cb_kh(int n) { return sizeof(T) == 4 && n > 64 ? n / 2 : n; }
template <typename T, int N>
__device__ __forceinline__ void
cb_body(const T* __restrict__ Bm, const T* __restrict__ Cm, float* __restrict__ Gf, T* __restrict__ Gm, T* __restrict__ Gmt,
        T* __restrict__ Bt, T* __restrict__ Ct,
        int64_t seqlen, int64_t ngroups, int64_t nchunks,
        int64_t Bsb, int64_t Bsl, int64_t Bsg, int64_t Csb, int64_t Csl, int64_t Csg, int64_t c, int64_t g, int64_t b,
        const int part) {
    constexpr int KH = cb_kh<T>(N), LD = lds_ld<T>(KH);
    constexpr int V = VecTraits<T>::kVec;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* sC = reinterpret_cast<T*>(smem_raw);      // [64][LD]
    T* sB = sC + 64 * LD;                        // [64][LD], the transposing parts: behind [32][LDT]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t t0 = c * kQ;
    const int valid = (int)((seqlen - t0) < kQ ? (seqlen - t0) : kQ);
    const T* Bp = Bm + b * Bsb + t0 * Bsl + g * Bsg;
    const T* Cp = Cm + b * Csb + t0 * Csl + g * Csg;
    const int64_t grp = (b * nchunks + c) * ngroups + g;
    if constexpr (sizeof(T) == 4) {
        if (part >= kCbGParts) {
            const int rb = part - kCbGParts, r = lane & 31, row = rb * 32 + r;
            const T* src = Bp + (int64_t)(row < valid ? row : valid - 1) * Bsl + 8 * (lane >> 5);
#pragma unroll
            for (int it = 0; it < N / 32; ++it) {
                const int u = it * 4 + wave;
                *reinterpret_cast<floatx4*>(Bt + grp * (int64_t)(N * kQ) + op32_offset<N / 8>(rb, u, lane)) =
                    *reinterpret_cast<const floatx4*>(src + (u >> 1) * 16 + 4 * (u & 1));
            }
            return;
        }
    }
    if (sizeof(T) == 2 && part >= kCbGParts) {
        // transposed copies of tokens [tk0, tk0 + 32): thread -> (state column n, group of V tokens)
        const int tk0 = (part - kCbGParts) * 32;
        constexpr int LDT = lds_ld<T>(N);
        T* sBt = sC + 32 * LDT;
        T* Btp = Bt + grp * (int64_t)(N * kQ);
        T* Ctp = Ct ? Ct + grp * (int64_t)(N * kQ) : nullptr;
        StagedRows<T, 32, N, 256> rc, rb;
        rb.load(Bp + (int64_t)tk0 * Bsl, Bsl, valid - tk0, tid);
        if (Ct) rc.load(Cp + (int64_t)tk0 * Csl, Csl, valid - tk0, tid);
        rb.put(sBt, LDT, valid - tk0, tid);
        if (Ct) rc.put(sC, LDT, valid - tk0, tid);
        __syncthreads();
        for (int e = tid; e < N * (32 / V); e += 256) {
            const int n = e % N, s0 = (e / N) * V;
            T v[V];
#pragma unroll
            for (int q = 0; q < V; ++q) v[q] = sBt[(s0 + q) * LDT + n];
            *reinterpret_cast<uint4*>(Btp + mt_offset(n, tk0 + s0)) = *reinterpret_cast<const uint4*>(v);
            if (Ct) {
#pragma unroll
                for (int q = 0; q < V; ++q) v[q] = sC[(s0 + q) * LDT + n];
                *reinterpret_cast<uint4*>(Ctp + mt_offset(n, tk0 + s0)) = *reinterpret_cast<const uint4*>(v);
            }
        }
        return;
    }
    // quadrant (wm, wn) of G = C B^T; wave (wi, wj) takes one 32x32 block of it
    const int wm = part == 0 ? 0 : 1, wn = part == 2 ? 1 : 0;
    const int wi = wave >> 1, wj = wave & 1;
    const bool live = wm * 2 + wi >= wn * 2 + wj;   // else a block above the diagonal
    floatx16 acc[1][1];
    acc_zero(acc);
#pragma unroll
    for (int n0 = 0; n0 < N; n0 += KH) {
        if (n0) __syncthreads();
        StagedRows<T, 64, KH, 256> rc, rb;
        rc.load(Cp + (int64_t)(wm * 64) * Csl + n0, Csl, valid - wm * 64, tid);
        rb.load(Bp + (int64_t)(wn * 64) * Bsl + n0, Bsl, valid - wn * 64, tid);
        rc.put(sC, LD, valid - wm * 64, tid);
        rb.put(sB, LD, valid - wn * 64, tid);
        __syncthreads();
        if (live) wave_mma<1, 1>(acc, sC + wi * 32 * LD, LD, sB + wj * 32 * LD, LD, 0, KH);
    }
    __syncthreads();                                // the operand tiles give way to the four waves' blocks
    if (!live) return;
    // The block leaves through LDS: eight lanes store a row (of G, or of its transpose) of 32 elements, where accumulator
    // registers would go out one element (or four of a column) at a time -- 36 store instructions per wave instead of 12.
    constexpr int LDG = 36;                         // 4 rows on: 16 banks on
    float* blk = reinterpret_cast<float*>(smem_raw) + wave * (32 * LDG);
#pragma unroll
    for (int v = 0; v < 16; ++v) blk[acc_row(lane, v) * LDG + acc_col(lane)] = acc[0][0][v];
    wave_lds_sync();
    const int i0 = wm * 64 + wi * 32, j0 = wn * 64 + wj * 32;      // first row, first column of the block
    if constexpr (sizeof(T) == 4) {
        const int r = lane & 31, k8 = 8 * (lane >> 5), I = i0 / 32, J = j0 / 32;
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int k = 16 * (it >> 1) + k8 + 4 * (it & 1);
            if (Gm) {
                floatx4 v = *reinterpret_cast<const floatx4*>(blk + r * LDG + k);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = i0 + r >= j0 + k + e ? v[e] : 0.f;
                *reinterpret_cast<floatx4*>(Gm + grp * (int64_t)(kQ * kQ) + op32_offset<16>(I, 4 * J + it, lane)) = v;
            }
            if (Gmt) {
                floatx4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = blk[(k + e) * LDG + r];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = i0 + k + e >= j0 + r ? v[e] : 0.f;
                *reinterpret_cast<floatx4*>(Gmt + grp * (int64_t)(kQ * kQ) + op32_offset<16>(J, 4 * I + it, lane)) = v;
            }
        }
        return;
    }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
        const int a = it * 8 + (lane >> 3), k0 = (lane & 7) * 4;   // row of the output, first of its four elements
        const floatx4 v = *reinterpret_cast<const floatx4*>(blk + a * LDG + k0);
        if (Gf) *reinterpret_cast<floatx4*>(Gf + grp * (int64_t)(kQ * kQ) + (i0 + a) * kQ + j0 + k0) = v;
        if (Gm) {
            T o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = from_f32<T>(i0 + a >= j0 + k0 + e ? v[e] : 0.f);
            *reinterpret_cast<RawVec<T, 4>*>(Gm + grp * (int64_t)(kQ * kQ) + (i0 + a) * kQ + j0 + k0) = *reinterpret_cast<const RawVec<T, 4>*>(o);
        }
        if (Gmt) {
            float t[4];
            T o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] = blk[(k0 + e) * LDG + a];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = from_f32<T>(i0 + k0 + e >= j0 + a ? t[e] : 0.f);
            *reinterpret_cast<RawVec<T, 4>*>(Gmt + grp * (int64_t)(kQ * kQ) + (j0 + a) * kQ + i0 + k0) = *reinterpret_cast<const RawVec<T, 4>*>(o);
        }
    }
}

// ------------------------------------------------------------------------------------------
// Cumulative log-decay table per (batch, head, chunk): ldtab[bhc] = [ l[0..kQ) | dt[0..kQ) ] in fp32,
// l = inclusive cumsum of A_h dt within the chunk, lam[bhc] = l[kQ-1]; tokens past the end of the sequence hold dt = 0 and the last
// l.  Every other kernel reads this table instead
// of gathering dt (stride = nheads elements) and scanning it again per head.  A workgroup takes eight consecutive heads of
// one (batch, chunk), two per wave: dt is [b][l][h], so two threads per token fetch 8 (fp32: 16) bytes each and hand them
// to the waves through LDS.  These workgroups are chains of latencies that hold the shared memory of a cb_body workgroup, so
// fewer of them with interleaved scans beat more with one (alone, four / eight / sixteen heads: 14.8 / 12.4 / 12.8 us at b2
// l4096 h128; b1 l200 h80, where a handful of workgroups take the softplus of everything: 5.7 / 6.2 / 8.9).
constexpr int kLdHeads = 8;
inline int64_t ld_table_blocks(int64_t batch, int64_t nheads, int64_t nchunks) { return batch * nchunks * ((nheads + kLdHeads - 1) / kLdHeads); }
template <typename T>
__device__ __forceinline__ void
ld_table_body(const void* __restrict__ dt, int dt_f32, const float* __restrict__ dt_bias, const float* __restrict__ A, float* __restrict__ ldtab,
              float* __restrict__ lam, int64_t seqlen, int64_t nheads, int64_t nchunks,
              int64_t dtsb, int64_t dtsl, int hs, int64_t blk) {
    constexpr int kPer = kLdHeads / 2, kHW = kLdHeads / 4;      // heads per loading thread, per wave
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float (*sdt)[kQ] = reinterpret_cast<float (*)[kQ]>(smem_raw);      // [kLdHeads][kQ], in what cb_body would use
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t hgroups = (nheads + kLdHeads - 1) / kLdHeads;
    const int64_t hg = blk % hgroups, c = (blk / hgroups) % nchunks, b = blk / (hgroups * nchunks);
    const int64_t h0 = hg * kLdHeads;
    const int64_t t0 = c * kQ;
    const int valid = (int)((seqlen - t0) < kQ ? (seqlen - t0) : kQ);
    float Ah[kHW], bh[kHW];      // fetched along with dt: one latency, not one per head
#pragma unroll
    for (int k = 0; k < kHW; ++k) {
        const int64_t h = h0 + wave * kHW + k < nheads ? h0 + wave * kHW + k : nheads - 1;
        Ah[k] = A[h];
        bh[k] = dt_bias ? dt_bias[h] : 0.f;
    }
    {
        const int t = threadIdx.x & (kQ - 1), k0 = (threadIdx.x >> 7) * kPer;
        const int64_t left = nheads - h0 - k0;
        const int hc = (int)(left < kPer ? left : kPer);
        float v[kPer];      // tokens past the end of the sequence behave as dt = 0
#pragma unroll
        for (int k = 0; k < kPer; ++k) v[k] = 0.f;
        auto fetch = [&](auto* p) {
            using E = std::remove_const_t<std::remove_pointer_t<decltype(p)>>;
            if (hc == kPer && (reinterpret_cast<uintptr_t>(p) & (kPer * sizeof(E) - 1)) == 0) {
                const RawVec<E, kPer> raw = *reinterpret_cast<const RawVec<E, kPer>*>(p);
                const E* e = reinterpret_cast<const E*>(&raw);
#pragma unroll
                for (int k = 0; k < kPer; ++k) v[k] = to_f32(e[k]);
            } else {
#pragma unroll
                for (int k = 0; k < kPer; ++k)
                    if (k < hc) v[k] = to_f32(p[k]);
            }
        };
        if (t < valid) {
            const int64_t off = b * dtsb + (t0 + t) * dtsl + h0 + k0;
            if (dt_f32) fetch(static_cast<const float*>(dt) + off);
            else fetch(static_cast<const T*>(dt) + off);
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) sdt[k0 + k][t] = v[k];
    }
    __syncthreads();
    float l0[kHW], l1[kHW], d0[kHW], d1[kHW];
#pragma unroll
    for (int k = 0; k < kHW; ++k) {      // past the last head: its values once more, not stored
        d0[k] = sdt[wave * kHW + k][lane]; d1[k] = sdt[wave * kHW + k][lane + 64];
        if (dt_bias) {
            // dt holds the raw projection: the step size is softplus(dt + dt_bias) (0 stays 0 past the end of the sequence)
            d0[k] = lane < valid ? softplus_f(d0[k] + bh[k]) : 0.f;
            d1[k] = lane + 64 < valid ? softplus_f(d1[k] + bh[k]) : 0.f;
        }
        wave_cumsum_from(Ah[k], d0[k], d1[k], l0[k], l1[k]);
    }
#pragma unroll
    for (int k = 0; k < kHW; ++k) {
        const int64_t h = h0 + wave * kHW + k;
        if (h >= nheads) return;
        for (int v = 0; v < (1 << hs); ++v) {      // one table per kernel head
            const int64_t bhc = (((b * nheads + h) << hs) + v) * nchunks + c;
            float* p = ldtab + bhc * (2 * kQ);
            p[lane] = l0[k]; p[lane + 64] = l1[k]; p[kQ + lane] = d0[k]; p[kQ + lane + 64] = d1[k];
            if (lane == 63) lam[bhc] = l1[k];
        }
    }
}

// Both preparations in one launch (they are independent, and either alone leaves most of the GPU idle): the first
// cb_blocks workgroups run cb_body, the others ld_table_body.
struct PrepArgs {
    const void* Bm; const void* Cm; float* Gf; void* Gm; void* Gmt; void* Bt; void* Ct;
    int64_t Bsb, Bsl, Bsg, Csb, Csl, Csg;
    const void* dt; int dt_f32; const float* dt_bias; const float* A; float* ldtab; float* lam; int64_t dtsb, dtsl;
    int64_t seqlen, nheads, ngroups, nchunks, n_cb;      // nheads: true heads
    int hs, parts;                                       // parts: kCbParts, or kCbGParts without Bt
};
template <typename T, int N>
__global__ void __launch_bounds__(256)
prep_kernel(const PrepArgs a) {
    const int64_t blk = blockIdx.x;
    const int parts = sizeof(T) == 2 ? kCbParts : a.parts;
    if (blk < cb_blocks(a.n_cb, parts)) {
        // The parts of one (chunk, group, batch) read the same rows.  Workgroups are dealt round-robin to the XCDs, so the
        // parts are kXcds apart: one L2 then fetches those rows once, where seven neighbours would each fetch their own.
        const uint32_t u = (uint32_t)blk / kXcds;
        const int64_t q = (int64_t)(u / parts) * kXcds + blk % kXcds;
        if (q >= a.n_cb) return;
        const int64_t c = q % a.nchunks, g = (q / a.nchunks) % a.ngroups, b = q / (a.nchunks * a.ngroups);
        cb_body<T, N>(static_cast<const T*>(a.Bm), static_cast<const T*>(a.Cm), a.Gf, static_cast<T*>(a.Gm), static_cast<T*>(a.Gmt),
                      static_cast<T*>(a.Bt), static_cast<T*>(a.Ct), a.seqlen, a.ngroups, a.nchunks,
                      a.Bsb, a.Bsl, a.Bsg, a.Csb, a.Csl, a.Csg, c, g, b, (int)(u % parts));
    } else {
        ld_table_body<T>(a.dt, a.dt_f32, a.dt_bias, a.A, a.ldtab, a.lam, a.seqlen, a.nheads, a.nchunks, a.dtsb, a.dtsl, a.hs, blk - cb_blocks(a.n_cb, parts));
    }
}

// ------------------------------------------------------------------------------------------
// Inter-chunk recurrence, fp32 operands.  grid (nheads, batch, kScanSplit), 256 threads; a workgroup owns 1/kScanSplit of the
// [p][n] state of one (batch, head), each thread EPT float4 slices of it, and walks the chunks with the running
// state in registers.  The split only exists to put enough waves on the GPU to hide memory latency.
//
// forward (REVERSE == false):
//     run = init;  for c = 0..nc-1:  prev[c] = run;  run = e^{lam_c} run + local[c];  final = run
// reverse (REVERSE == true), the gradient recurrence:
//     run = dfinal;  for c = nc-1..0:  prev[c] = run   (= dL/dS_new(c));  run = e^{lam_c} run + local[c];  dinit = run.
constexpr int kScanSplit = 4;
constexpr int kDlamParts = 8;     // partial sums of dlam per (batch, head, chunk), one per wave of the main backward kernel

template <int PN, bool REVERSE>
__global__ void __launch_bounds__(256)
state_scan_kernel(const float* __restrict__ local, const float* __restrict__ lam, const float* __restrict__ init,
                  float* __restrict__ prev, float* __restrict__ final_out, int64_t nheads, int64_t nchunks) {
    constexpr int EPT = PN / 4 / 256 / kScanSplit;
    static_assert(PN % (1024 * kScanSplit) == 0, "state size must be a multiple of 4096 elements");
    const int part0 = blockIdx.z * (PN / kScanSplit);      // first element of this workgroup's part
    const int tid = threadIdx.x;
    const int64_t h = blockIdx.x, b = blockIdx.y;
    const int64_t bh = b * nheads + h;
    floatx4 run[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
        if (init) run[e] = *reinterpret_cast<const floatx4*>(init + bh * PN + part0 + (e * 256 + tid) * 4);
        else run[e] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll 1
    for (int64_t cc = 0; cc < nchunks; ++cc) {
        const int64_t c = REVERSE ? nchunks - 1 - cc : cc;
        const int64_t tile = ((b * nchunks + c) * nheads + h) * (int64_t)PN;
        const float dec = __expf(lam[bh * nchunks + c]);
#pragma unroll
        for (int e = 0; e < EPT; ++e) {
            const int off = part0 + (e * 256 + tid) * 4;
            const floatx4 loc = *reinterpret_cast<const floatx4*>(local + tile + off);
            *reinterpret_cast<floatx4*>(prev + tile + off) = run[e];
#pragma unroll
            for (int q = 0; q < 4; ++q) run[e][q] = dec * run[e][q] + loc[q];
        }
    }
    if (final_out) {
#pragma unroll
        for (int e = 0; e < EPT; ++e)
            *reinterpret_cast<floatx4*>(final_out + bh * PN + part0 + (e * 256 + tid) * 4) = run[e];
    }
}

}  // namespace m2
