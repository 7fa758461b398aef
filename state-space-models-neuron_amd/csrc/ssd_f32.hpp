// The SSD kernels for fp32 operands (v_mfma_f32_32x32x2_f32, 64 cycles each on a SIMD: a sixteenth of the 16-bit rate).
//
// What bounds them is the matrix pipe, so everything else has to run behind it: tiles come global -> LDS by asynchronous copies
// in their natural layout (16-byte slots XOR-swizzled by the row), both operand orientations are read from that one copy -- with
// 4-byte elements a transposed fragment is eight ds_read_b32 of 32 neighbouring columns, no slower per byte than a row read --,
// the block work is dealt so that the four SIMDs of a CU carry the same number of products, and the four products of the backward
// share one pass over dy, x, S_prev and dS.  The kernels before these staged every tile through registers (the transposed ones by
// 4-byte LDS writes), waited for it between two barriers, and ran the backward as four kernels that each staged their own.
// b3 l2048 h16 p128 n128 g8, forward and backward with their gaps: 705 -> 496 us (its products alone 173 at the rate of a large one).
//
// MFMAs are issued with swapped operands, as in ssd_y.hpp: a lane's accumulators belong to one token (or state row), decay scales
// are one scalar per lane, and results leave in 16-byte stores.  Decay factors: see ssd_y.hpp.
#pragma once
#include "ssd_y.hpp"

namespace m2 {

// ------------------------------------------------------------------------------------------ LDS tiles of fp32
// Rows of COLS floats, 16-byte slot s of row `row` at slot s ^ (row & 15).  Row reads: 16 consecutive rows, one slot each, spread over
// all 64 banks; transposed reads: the lanes of the two halves read rows 8 apart, whose slots then differ in bit 3: 32 + 32 banks.
// An operand moves in steps of 8 k: step u of a lane is four values, k = 16 (u / 2) + 8 half + 4 (u % 2) + 0..3.
template <int COLS>
__device__ __forceinline__ floatx4 row_step32(const float* t, int row, int half, int u) {      // row `row` of the tile, k along it
    return *reinterpret_cast<const floatx4*>(t + row * COLS + (((u * 2 - (u & 1) + 2 * half) ^ (row & 15)) * 4));
}
template <int COLS>
__device__ __forceinline__ floatx4 col_step32(const float* t, int col, int half, int u) {      // column `col`, k down the rows
    floatx4 f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int k = 8 * half + 4 * (u & 1) + e;      // row & 15
        f[e] = t[((u >> 1) * 16 + k) * COLS + (((col >> 2) ^ k) * 4) + (col & 3)];
    }
    return f;
}
__device__ __forceinline__ floatx4 mem_step32(const float* row, int half, int u) { return *reinterpret_cast<const floatx4*>(row + (u >> 1) * 16 + 8 * half + 4 * (u & 1)); }
// columns col .. col + 3 (col a multiple of 4) of a row
template <int COLS>
__device__ __forceinline__ floatx4 row_quad32(const float* t, int row, int col) {
    return *reinterpret_cast<const floatx4*>(t + row * COLS + (((col >> 2) ^ (row & 15)) * 4));
}

// A value (the lane; the thread) unknown to the optimiser from here on: the addresses formed of it are then formed where they are used
// (a few vector instructions behind products of 256 cycles), where a loop would keep dozens of them in registers.
__device__ __forceinline__ int here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int lane_here() { return here(threadIdx.x & 63); }

// acc[q] += b(u, q) x a(u) [scaled along k by f(u)] for the steps u in [u0, u1).  Operands are asked for ahead of the products that
// take them, a by DA steps and b and f by one (the compiler would put each LDS read right in front of its product: a round trip of 130
// cycles beside 64 of work, 45 % of the matrix pipe in all); `last` runs in front of the last step's products.
// (products32_ring: the first DA steps of a are in av already.)
template <int NB, bool SCALED, int DA, typename A, typename F, typename B, typename L>
__device__ __forceinline__ void products32_ring(floatx16 (&acc)[NB], int u0, int u1, floatx4 (&av)[DA + 1], A a, F f, B b, L last) {
    floatx4 fv[2], bv[2][NB];
    if (SCALED) fv[0] = f(u0);
#pragma unroll
    for (int q = 0; q < NB; ++q) bv[0][q] = b(u0, q);
#pragma unroll
    for (int u = u0; u < u1; ++u) {
        const int ca = (u - u0) % (DA + 1), c = (u - u0) & 1;
        if (u + DA < u1) av[(u - u0 + DA) % (DA + 1)] = a(u + DA);
        if (u + 1 < u1) {
            if (SCALED) fv[c ^ 1] = f(u + 1);
#pragma unroll
            for (int q = 0; q < NB; ++q) bv[c ^ 1][q] = b(u + 1, q);
        } else last();
        __builtin_amdgcn_sched_barrier(0);
        if (SCALED) av[ca] *= fv[c];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int q = 0; q < NB; ++q) acc[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(bv[c][q][s], av[ca][s], acc[q], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <int NB, bool SCALED, int DA, typename A, typename F, typename B, typename L>
__device__ __forceinline__ void products32(floatx16 (&acc)[NB], int u0, int u1, A a, F f, B b, L last) {
    floatx4 av[DA + 1];
#pragma unroll
    for (int d = 0; d < DA; ++d)
        if (u0 + d < u1) av[d] = a(u0 + d);
    products32_ring<NB, SCALED, DA>(acc, u0, u1, av, a, f, b, last);
}
__device__ __forceinline__ void step32(floatx16& acc, const floatx4& b, const floatx4& a) {
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[s], a[s], acc, 0, 0, 0);
}
// f(k) with the row block as a constant: the lengths of the causal products are known, and what they index stays in registers
template <typename F>
__device__ __forceinline__ void by_row_block(int rb, F f) {
    if (rb == 0) f(std::integral_constant<int, 0>{});
    else if (rb == 1) f(std::integral_constant<int, 1>{});
    else if (rb == 2) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 3>{});
}
constexpr int kFar32 = 5;
struct NoScale32 { __device__ floatx4 operator()(int) const { return {}; } };
struct NoLast32 { __device__ void operator()() const {} };

// Asynchronous copy of a [ROWS][COLS] tile by WAVES waves; `set` fixes the lanes' source offsets (rows from `valid` on re-read row
// valid - 1: every use meets them with a factor of zero), `issue` sends the wave's share.
template <int ROWS, int COLS, int WAVES>
struct TileCopy32 {
    static constexpr int SPR = COLS / 4, PER = ROWS * SPR / 64 / WAVES;
    static_assert(PER * 64 * WAVES == ROWS * SPR, "whole wave-wide copies");
    uint32_t off[PER];
    __device__ __forceinline__ void set(int wave, int64_t stride, int valid) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int it = 0; it < PER; ++it) {
            const int s = (wave * PER + it) * 64 + lane, row = s / SPR, cs = (s % SPR) ^ (row & 15);
            off[it] = (uint32_t)((row < valid ? row : valid - 1) * stride + cs * 4) * 4u;
        }
    }
    __device__ __forceinline__ void issue(const float* g, uint32_t wave, uint32_t lds) const {
#pragma unroll
        for (int it = 0; it < PER; ++it) async_copy16(g, off[it], lds + (wave * PER + it) * 1024u);
    }
};

// ------------------------------------------------------------------------------------------ local chunk states
// out[p][n] = sum_t scale_t X[t][p] M[t][n],  X = x, M = B, scale_t = dt_t e^{Lam - l_t};  DSTATE: X = dy, M = C, scale_t = e^{l_t}.
// A wave owns one 32x32 block of [P][N] and keeps its columns of M (all 128 tokens) as fragments for the whole head loop; the X tile of
// the next head is under way while the products of this one run.  b3 l2048 h16 p128 n128 g8: 47 (x) and 51 (dy) -> 46.5 us each, 54 % of
// the busy cycles in the matrix pipe (what waits in the rest was not found: stores left in flight across the wait change nothing).
template <int N> constexpr int chunk_state32_threads() { return N * 4; }
template <int N> constexpr size_t chunk_state32_smem() { return (size_t)(2 * kQ * kP + 2 * 2 * kQ + N / 16 * kQ) * sizeof(float); }
struct ChunkState32Args {
    const float* X; int64_t X_sb, X_sl, X_sh;
    const float* M; int64_t M_sb, M_sl, M_sg;
    const float* ldtab; float* out;
    int64_t seqlen, nheads, ngroups, nchunks, nslices, hps;
};
template <int N, bool DSTATE, int HS>
__global__ void __launch_bounds__(chunk_state32_threads<N>(), N == 128 ? 4 : 2)
chunk_state32_kernel(const ChunkState32Args a) {
    constexpr int WAVES = N / 16, P = kP;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float* sX = reinterpret_cast<float*>(smem_raw);      // [2][kQ][P]
    float* sLD = sX + 2 * kQ * P;                        // [2][ l kQ | dt kQ ]
    float* wsc = sLD + 2 * 2 * kQ + (threadIdx.x >> 6) * kQ;      // this wave's scales
    const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5;
    const int wave = (int)uniform(threadIdx.x >> 6), pb = wave & 1, nb = wave >> 1;
    const int64_t c = blockIdx.x, b = blockIdx.z, g = blockIdx.y / a.nslices, slice = blockIdx.y % a.nslices;
    const int64_t t0 = c * kQ, hpg = a.nheads / a.ngroups, h0 = g * hpg + slice * a.hps, hps = slice_heads(hpg, slice, a.hps);
    const int valid = (int)(a.seqlen - t0 < kQ ? a.seqlen - t0 : kQ);
    TileCopy32<kQ, P, WAVES> cp;
    cp.set(wave, a.X_sl, valid);
    const uint32_t lds_X = uniform(lds_addr_of(sX)), lds_LD = uniform(lds_addr_of(sLD));
    auto issue = [&](int64_t h, int buf) {
        cp.issue(a.X + b * a.X_sb + t0 * a.X_sl + head_off<HS>(h, a.X_sh), wave, lds_X + (uint32_t)(buf * kQ * P * 4));
        async_copy_ldtab(a.ldtab, (b * a.nheads + h) * a.nchunks + c, lds_LD + (uint32_t)(buf * 2 * kQ * 4));
    };
    floatx4 fm[16];
    {
        const float* Mp = a.M + b * a.M_sb + t0 * a.M_sl + g * a.M_sg + nb * 32 + r;
#pragma unroll
        for (int u = 0; u < 16; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = (u >> 1) * 16 + 8 * half + 4 * (u & 1) + e;
                fm[u][e] = Mp[(t < valid ? t : valid - 1) * a.M_sl];
            }
    }
    issue(h0, 0);
    for (int64_t hh = 0; hh < hps; ++hh) {
        const int buf = (int)(hh & 1);
        wait_vmem_all();
        {
            const float* sl = sLD + buf * 2 * kQ;
            const float Lam = sl[kQ - 1], la = sl[lane], lb = sl[lane + 64];
            wsc[lane] = DSTATE ? (lane < valid ? __expf(la) : 0.f) : sl[kQ + lane] * __expf(Lam - la);
            wsc[lane + 64] = DSTATE ? (lane + 64 < valid ? __expf(lb) : 0.f) : sl[kQ + lane + 64] * __expf(Lam - lb);
        }
        __syncthreads();      // the tile is whole, and everyone is done with the other buffer
        if (hh + 1 < hps) issue(h0 + hh + 1, buf ^ 1);
        const float* tx = sX + buf * kQ * P;
        const int lane = lane_here(), r = lane & 31, half = lane >> 5;
        floatx16 acc[1][1];
        acc_zero(acc);
        products32<1, true, 1>(acc[0], 0, 16, [&](int u) { return col_step32<P>(tx, pb * 32 + r, half, u); }, [&](int u) { return mem_step32(wsc, half, u); },
                               [&](int u, int) { return fm[u]; }, NoLast32{});
        float* op = a.out + ((b * a.nchunks + c) * a.nheads + h0 + hh) * (int64_t)(P * N) + (pb * 32 + r) * N + nb * 32 + 4 * half;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<floatx4*>(op + 8 * q) = floatx4{acc[0][0][4 * q], acc[0][0][4 * q + 1], acc[0][0][4 * q + 2], acc[0][0][4 * q + 3]};
    }
}

// ------------------------------------------------------------------------------------------ forward output
// y[i][p] = u_i ( e^{l_ref} sum_n C[i][n] S_prev[p][n] + sum_{j<=i} (G[i][j] v_j) x[j][p] ) + D x[i][p], factors as in ssd_y.hpp.
// Wave w owns row block w (w < 4) or 7 - w, and channel block w >> 2: the two waves of a SIMD then have row blocks w and 3 - w,
// whose causal parts add up to the same on all four.  The C rows and the causal C B^T rows stay in registers.
// b3 l2048 h16 p128 n128 g8: 110 -> 79 us, of which the products are 31 at the rate of a large one.
template <int N> constexpr size_t y32_smem() { return (size_t)(2 * (kP * N + kQ * kP + 2 * kQ) + 8 * kQ) * sizeof(float); }
template <int N, int HS>
__global__ void __launch_bounds__(512, 2)
ssd_y32_kernel(const YArgs a) {
    constexpr int P = kP, KSN = N / 16;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float* sS = reinterpret_cast<float*>(smem_raw);      // [2][P][N]
    float* sX = sS + 2 * P * N;                          // [2][kQ][P]
    float* sLD = sX + 2 * kQ * P;                        // [2][ l kQ | dt kQ ]
    const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5;
    const int wave = (int)uniform(threadIdx.x >> 6), rb = wave < 4 ? wave : 7 - wave, pb = wave >> 2, row0 = rb * 32, tok = row0 + r;
    float* wv = sLD + 2 * 2 * kQ + wave * kQ;            // this wave's v
    const int64_t c = blockIdx.x, b = blockIdx.z, g = blockIdx.y / a.nslices, slice = blockIdx.y % a.nslices;
    const int64_t t0 = c * kQ, hpg = a.nheads / a.ngroups, h0 = g * hpg + slice * a.hps, hps = slice_heads(hpg, slice, a.hps);
    const int valid = (int)(a.seqlen - t0 < kQ ? a.seqlen - t0 : kQ);
    TileCopy32<P, N, 8> cs;
    TileCopy32<kQ, P, 8> cx;
    cs.set(wave, N, P);
    cx.set(wave, a.Z_sl, valid);
    const uint32_t lds_S = uniform(lds_addr_of(sS)), lds_X = uniform(lds_addr_of(sX)), lds_LD = uniform(lds_addr_of(sLD));
    auto issue = [&](int64_t h, int buf) {
        cs.issue(static_cast<const float*>(a.S) + ((b * a.nchunks + c) * a.nheads + h) * (int64_t)(P * N), wave, lds_S + (uint32_t)(buf * P * N * 4));
        cx.issue(static_cast<const float*>(a.Z) + b * a.Z_sb + t0 * a.Z_sl + head_off<HS>(h, a.Z_sh), wave, lds_X + (uint32_t)(buf * kQ * P * 4));
        async_copy_ldtab(a.ldtab, (b * a.nheads + h) * a.nchunks + c, lds_LD + (uint32_t)(buf * 2 * kQ * 4));
    };
    floatx4 fd[16], fo[2 * KSN];
    const float* Gp = static_cast<const float*>(a.Gd) + ((b * a.nchunks + c) * a.ngroups + g) * (int64_t)(kQ * kQ);
    {
        const float* Cp = static_cast<const float*>(a.Aoff) + b * a.Ao_sb + (t0 + (tok < valid ? tok : valid - 1)) * a.Ao_sl + g * a.Ao_sg;
#pragma unroll
        for (int u = 0; u < 2 * KSN; ++u) fo[u] = mem_step32(Cp, half, u);
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (u < 4 * rb + 4) fd[u] = *reinterpret_cast<const floatx4*>(Gp + op32_offset<16>(rb, u, lane));
    }
    issue(h0, 0);
    for (int64_t hh = 0; hh < hps; ++hh) {
        const int64_t h = h0 + hh;
        const int buf = (int)(hh & 1);
        const float Dh = a.D ? load_uniform_f32(a.D + (h >> HS)) : 0.f;
        wait_vmem_all();
        const float* sl = sLD + buf * 2 * kQ;
        const float* sd = sl + kQ;
        const float lref = sl[row0], l_row = sl[tok];
        const bool fast = lref - sl[row0 + 31] < kMaxRange;
        wv[lane] = lane < row0 + 32 ? __expf(lref - sl[lane]) * sd[lane] : 0.f;
        wv[lane + 64] = lane + 64 < row0 + 32 ? __expf(lref - sl[lane + 64]) * sd[lane + 64] : 0.f;
        __syncthreads();      // the tiles are whole, and everyone is done with the other buffers
        if (hh + 1 < hps) issue(h + 1, buf ^ 1);
        const float* tS = sS + buf * P * N;
        const float* tX = sX + buf * kQ * P;
        const int lane = lane_here(), r = lane & 31, half = lane >> 5, tok = row0 + r;
        floatx16 acc[1][1];
        acc_zero(acc);
        products32<1, false, 1>(acc[0], 0, 2 * KSN, [&](int u) { return fo[u]; }, NoScale32{}, [&](int u, int) { return row_step32<N>(tS, pb * 32 + r, half, u); }, NoLast32{});
        const float off = __expf(fast ? lref : l_row), fin = fast ? __expf(fminf(l_row - lref, 0.f)) : 1.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[0][0][v] *= off;
        if (fast)
            by_row_block(rb, [&](auto k) {
                products32<1, true, 1>(acc[0], 0, 4 * decltype(k)::value + 4, [&](int u) { return fd[u]; }, [&](int u) { return mem_step32(wv, half, u); },
                                       [&](int u, int) { return col_step32<P>(tX, pb * 32 + r, half, u); }, NoLast32{});
            });
        else
#pragma unroll 1
            for (int u = 0; u < 4 * rb + 4; ++u) {
                floatx4 f = *reinterpret_cast<const floatx4*>(Gp + op32_offset<16>(rb, u, lane));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = (u >> 1) * 16 + 8 * half + 4 * (u & 1) + e;
                    f[e] *= k <= tok ? __expf(l_row - sl[k]) * sd[k] : 0.f;
                }
                step32(acc[0][0], col_step32<P>(tX, pb * 32 + r, half, u), f);
            }
        float* Yp = static_cast<float*>(a.Y) + b * a.Y_sb + (t0 + tok) * a.Y_sl + head_off<HS>(h, a.Y_sh);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int col = pb * 32 + 8 * q + 4 * half;
            const floatx4 x4 = row_quad32<P>(tX, tok, col);
            floatx4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = acc[0][0][4 * q + e] * fin + Dh * x4[e];
            if (tok < valid) *reinterpret_cast<floatx4*>(Yp + col) = o;
        }
    }
}

// ------------------------------------------------------------------------------------------ backward
// One pass over dy, x, S_prev and dS per (batch, chunk, group, head slice); per head four phases of products, a barrier between any
// two, each of which frees the tile that the phase was the last to read for the copy of the next head's:
//   1  dB_off[j][n] += dt_j e^{Lam-l_j} sum_p x[j][p] dS[p][n]
//   2  dxd[j][p] = u_j ( e^{Lam-l_ref} sum_n B[j][n] dS[p][n] + sum_{i>=j} (G[i][j] v_i) dy[i][p] ),  l_ref: last token of the row block
//      dx = dt_j dxd + D dy,  dir_j = dxd . x,  rb_j = dt_j (state part of dxd) . x,  dD partial = dy . x,  dlam = e^{Lam} <dS, S_prev>;   dS is free
//   3  dG^h[i][j] = e^{l_i-l_j} dt_j dy_i . x_j (i >= j);   dG += dG^h,   and from the row and column sums of dG^h o G what the
//      diagonal term gives to da;                                                                                                      x is free
//   4  t = e^{l_i} sum_p dy[i][p] S_prev[p][n];   dC_off += t,   dl_c[i] = sum_n C[i][n] t[i][n];                                 dy, S_prev are free
// Phases 1, 2, 4: row blocks as in ssd_y32_kernel, the column blocks dealt by w >> 2; phase 3: the ten lower blocks of dG over the eight
// waves.  Per head and SIMD 66 to 70 products of 512 cycles, against 2 x 2 waves that wait for each other at the barriers only.
// Where one workgroup has all heads of the group, it finishes dB and dC too (finish32), and no partial sum leaves the chip.
// b3 l2048 h16 p128 n128 g8: 334 us as four kernels (dG, the two state parts, the rest), 258 as this one, and the group finish 58 -> 5.
// A head takes 61 k cycles, 35 k of them products, a workgroup 25 us beside its heads; 384 workgroups leave half of the CUs idle in
// the second round.
struct Bwd32Args {
    const float* ldtab; const float* D;
    const float* Bm; int64_t B_sb, B_sl, B_sg;
    const float* Cm; int64_t C_sb, C_sl, C_sg;
    const float* Bt; const float* Gm; const float* Gmt;   // B, causal C B^T and its transpose: [b][c][g][kQ][N | kQ | kQ] in operand order
    const float* dS; const float* Sprev;                  // [b][c][h][P][N]
    const float* dy; int64_t dy_sb, dy_sl, dy_sh;
    const float* x; int64_t x_sb, x_sl, x_sh;
    float* dx; int64_t dx_sb, dx_sl, dx_sh;
    float* dB; int64_t dB_sb, dB_sl, dB_sg;               // nslices == 1
    float* dC; int64_t dC_sb, dC_sl, dC_sg;
    float* dGp; float* dBp; float* dCp;                   // nslices > 1: [b][c][g][slice][kQ][kQ | N]
    float* dirp; float* rbp; float* dl; float* dlc;       // [b][h][c][kQ]; dl: the diagonal term's share of da (16-bit kernels leave per-token terms that are still to be scanned)
    float* dDp8; float* dlam;                             // [b][h][c][8]
    int64_t seqlen, nheads, ngroups, nchunks, nslices, hps;
};
template <int N> constexpr size_t bwd32_smem() { return (size_t)(2 * kQ * kP + 2 * kP * N + 2 * 2 * kQ + 8 * (kQ + 64) + 6 * kQ + 2 * 10 * 32 + 2 * 1024) * sizeof(float); }

// The group-level finish of one (batch, chunk, group):  dC[i] += sum_{j<=i} dG[i][j] B[j],  dB[j] += sum_{i>=j} dG[i][j] C[i].
// dG lies in sG ([kQ][kQ], swizzled; blocks above the diagonal are not read), sM takes B and then C.  Wave: row block rb, column
// blocks nb0 .. nb0 + NBW - 1, a token per lane.  SIDES: 1 dC, 2 dB, 3 both, one behind the other.
template <int N, int NBW, int SIDES = 3>
__device__ __forceinline__ void finish32(const float* sG, float* sM, floatx16 (&accB)[NBW], floatx16 (&accC)[NBW], const float* Bp, int64_t B_sl, const float* Cp,
                                         int64_t C_sl, float* dB, int64_t dB_sl, float* dC, int64_t dC_sl, int valid, int wave, int rb, int nb0) {
    const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5, tok = rb * 32 + r;
    const uint32_t lds_M = uniform(lds_addr_of(sM));
    TileCopy32<kQ, N, 8> cp;
    auto m = [&](int u, int q) { return col_step32<N>(sM, (nb0 + q) * 32 + r, half, u); };
    if constexpr (SIDES & 1) {
        cp.set(wave, B_sl, valid);
        cp.issue(Bp, wave, lds_M);
        wait_vmem_all();
        __syncthreads();      // dG and B are there
        by_row_block(rb, [&](auto k) {
            products32<NBW, false, 1>(accC, 0, 4 * decltype(k)::value + 4, [&](int u) { return row_step32<kQ>(sG, tok, half, u); }, NoScale32{}, m, NoLast32{});
        });
        if (SIDES & 2) __syncthreads();      // everyone is done with B
    }
    if constexpr (SIDES & 2) {
        cp.set(wave, C_sl, valid);
        cp.issue(Cp, wave, lds_M);
    }
    if ((SIDES & 1) && tok < valid) {
        float* o = dC + tok * dC_sl + nb0 * 32 + 4 * half;
#pragma unroll
        for (int q = 0; q < NBW; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                *reinterpret_cast<floatx4*>(o + q * 32 + 8 * v) = floatx4{accC[q][4 * v], accC[q][4 * v + 1], accC[q][4 * v + 2], accC[q][4 * v + 3]};
    }
    if constexpr (!(SIDES & 2)) return;
    wait_vmem_all();
    __syncthreads();
    by_row_block(rb, [&](auto k) {
        products32<NBW, false, 1>(accB, 4 * decltype(k)::value, 16, [&](int u) { return col_step32<kQ>(sG, tok, half, u); }, NoScale32{}, m, NoLast32{});
    });
    if (tok < valid) {
        float* o = dB + tok * dB_sl + nb0 * 32 + 4 * half;
#pragma unroll
        for (int q = 0; q < NBW; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                *reinterpret_cast<floatx4*>(o + q * 32 + 8 * v) = floatx4{accB[q][4 * v], accB[q][4 * v + 1], accB[q][4 * v + 2], accB[q][4 * v + 3]};
    }
}

template <int N, int HS>
__global__ void __launch_bounds__(512, 2)
ssd_bwd32_kernel(const Bwd32Args a) {
    constexpr int P = kP, KSN = N / 16, KSP = P / 16, NBW = N / 64;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float* sX = reinterpret_cast<float*>(smem_raw);      // [kQ][P]
    float* sY = sX + kQ * P;                             // [kQ][P]   dy
    float* sP = sY + kQ * P;                             // [P][N]    S_prev
    float* sD = sP + P * N;                              // [P][N]    dS
    float* sLD = sD + P * N;                             // [2][ l kQ | dt kQ ]
    float* tabs = sLD + 2 * 2 * kQ;                      // [8 waves][ v of phase 2, kQ | v of phase 3, 2 x 32 ]
    float* s_dir = tabs + 8 * (kQ + 64);                 // [2][kQ] each: the halves of the channels, of the state columns
    float* s_rb = s_dir + 2 * kQ;
    float* s_c = s_rb + 2 * kQ;
    float* s_rs = s_c + 2 * kQ;                          // [10 blocks][32] row sums, column sums
    float* s_cs = s_rs + 10 * 32;
    float* s_dG = s_cs + 10 * 32;                        // [2][4][64 lanes][4] the second blocks of dG of the last two waves (in registers all waves would pay for them)
    const int tid = threadIdx.x, wave = (int)uniform(tid >> 6), rb = wave < 4 ? wave : 7 - wave, sec = wave >> 2, row0 = rb * 32;
    const int nb0 = sec * NBW;
    float* wv = tabs + wave * (kQ + 64);
    float* wg = wv + kQ;
    const int64_t c = blockIdx.x, b = blockIdx.z, g = blockIdx.y / a.nslices, slice = blockIdx.y % a.nslices;
    const int64_t t0 = c * kQ, hpg = a.nheads / a.ngroups, h0 = g * hpg + slice * a.hps, hps = slice_heads(hpg, slice, a.hps), grp = (b * a.nchunks + c) * a.ngroups + g;
    const int valid = (int)(a.seqlen - t0 < kQ ? a.seqlen - t0 : kQ);

    TileCopy32<P, N, 8> cs;
    TileCopy32<kQ, P, 8> cx, cy;
    cs.set(wave, N, P);
    cx.set(wave, a.x_sl, valid);
    cy.set(wave, a.dy_sl, valid);
    const uint32_t lds_X = uniform(lds_addr_of(sX)), lds_Y = uniform(lds_addr_of(sY)), lds_P = uniform(lds_addr_of(sP)), lds_D = uniform(lds_addr_of(sD)),
                   lds_LD = uniform(lds_addr_of(sLD));
    auto state = [&](int64_t h) { return ((b * a.nchunks + c) * a.nheads + h) * (int64_t)(P * N); };
    auto issue_dS = [&](int64_t h) { cs.issue(a.dS + state(h), wave, lds_D); };
    auto issue_x = [&](int64_t h, int buf) {
        cx.issue(a.x + b * a.x_sb + t0 * a.x_sl + head_off<HS>(h, a.x_sh), wave, lds_X);
        async_copy_ldtab(a.ldtab, (b * a.nheads + h) * a.nchunks + c, lds_LD + (uint32_t)(buf * 2 * kQ * 4));
    };
    auto issue_dy_Sp = [&](int64_t h) {
        cy.issue(a.dy + b * a.dy_sb + t0 * a.dy_sl + head_off<HS>(h, a.dy_sh), wave, lds_Y);
        cs.issue(a.Sprev + state(h), wave, lds_P);
    };
    issue_dS(h0);
    issue_x(h0, 0);
    issue_dy_Sp(h0);

    // phase 3: block `wave` of the lower triangle in row order; the last two waves, whose blocks lie in the last row, take the one two columns on as well
    const int gi = wave < 1 ? 0 : wave < 3 ? 1 : wave < 6 ? 2 : 3, gj = wave - gi * (gi + 1) / 2, ngb = wave >= 6 ? 2 : 1;
    floatx16 accB[NBW], accC[NBW], dG;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
#pragma unroll
        for (int q = 0; q < NBW; ++q) accB[q][v] = accC[q][v] = 0.f;
        dG[v] = 0.f;
    }
    float* dG2 = s_dG + (wave & 1) * 1024;
    if (ngb > 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<floatx4*>(dG2 + (q * 64 + (tid & 63)) * 4) = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    const float* Gg = a.Gm + grp * (int64_t)(kQ * kQ);
    const float* Gt = a.Gmt + grp * (int64_t)(kQ * kQ);
    const float* Bg = a.Bt + grp * (int64_t)(kQ * N);
    const float* Cg = a.Cm + b * a.C_sb + t0 * a.C_sl + g * a.C_sg;

    wait_vmem_all();
    __syncthreads();
    for (int64_t hh = 0; hh < hps; ++hh) {
        const int64_t h = h0 + hh, bhc = (b * a.nheads + h) * a.nchunks + c;
        const bool more = hh + 1 < hps;
        const float Dh = a.D ? load_uniform_f32(a.D + (h >> HS)) : 0.f;
        const float* sl = sLD + (hh & 1) * 2 * kQ;
        const float* sd = sl + kQ;
        const float Lam = sl[kQ - 1], lref = sl[row0 + 31];
        const bool fast = sl[row0] - lref < kMaxRange;
        // ---- 1: state part of dB
        {
            const int lane = lane_here(), r = lane & 31, half = lane >> 5, tok = row0 + r;
            const float sc = sd[tok] * __expf(Lam - sl[tok]);
            products32<NBW, true, 1>(accB, 0, 2 * KSP, [&](int u) { return row_step32<P>(sX, tok, half, u); }, [&](int) { return floatx4{sc, sc, sc, sc}; },
                                     [&](int u, int q) { return col_step32<N>(sD, (nb0 + q) * 32 + r, half, u); }, NoLast32{});
        }
        if (hh > 0) {
            wait_vmem_all();
            __syncthreads();      // dy and S_prev are there; dl_c of the head before is complete
            if (wave < 2) { const int t = here(tid); a.dlc[(bhc - a.nchunks) * kQ + t] = s_c[t] + s_c[kQ + t]; }
        }
        // ---- 2: dx and the sums over its rows
        {
            const int lane = lane_here(), r = lane & 31, half = lane >> 5, tok = row0 + r;
            const bool tok_ok = tok < valid;
            const float l_row = sl[tok], dt_row = sd[tok];
            wv[lane] = lane >= row0 && lane < valid ? __expf(sl[lane] - lref) : 0.f;
            wv[lane + 64] = lane + 64 >= row0 && lane + 64 < valid ? __expf(sl[lane + 64] - lref) : 0.f;
            floatx16 acc[1][1];
            acc_zero(acc);
            // B and C B^T come from behind the L2 (every workgroup of an XCD has its own, 192 KB): asked for early
            products32<1, false, kFar32>(acc[0], 0, 2 * KSN, [&](int u) { return *reinterpret_cast<const floatx4*>(Bg + op32_offset<N / 8>(rb, u, lane)); }, NoScale32{},
                                         [&](int u, int) { return row_step32<N>(sD, sec * 32 + r, half, u); }, NoLast32{});
            floatx4 gv[5];
            auto g_step = [&](int u) { return *reinterpret_cast<const floatx4*>(Gt + op32_offset<16>(rb, u, lane)); };
#pragma unroll
            for (int d = 0; d < 4; ++d) gv[d] = g_step(4 * rb + d < 16 ? 4 * rb + d : 15);
            const float off = __expf(Lam - (fast ? lref : l_row)), fin = fast ? __expf(fminf(lref - l_row, 0.f)) : 1.f;
            float rbs = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const floatx4 x4 = row_quad32<P>(sX, tok, sec * 32 + 8 * q + 4 * half);
#pragma unroll
                for (int e = 0; e < 4; ++e) { acc[0][0][4 * q + e] *= off; rbs += acc[0][0][4 * q + e] * x4[e]; }
            }
            wave_lds_sync();
            if (fast)
                by_row_block(rb, [&](auto k) {
                    products32_ring<1, true, 4>(acc[0], 4 * decltype(k)::value, 16, gv, g_step, [&](int u) { return mem_step32(wv, half, u); },
                                                     [&](int u, int) { return col_step32<P>(sY, sec * 32 + r, half, u); }, NoLast32{});
                });
            else
#pragma unroll 1
                for (int u = 4 * rb; u < 16; ++u) {
                    floatx4 f = g_step(u);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int k = (u >> 1) * 16 + 8 * half + 4 * (u & 1) + e;
                        f[e] *= k >= tok && k < valid ? __expf(sl[k] - l_row) : 0.f;
                    }
                    step32(acc[0][0], col_step32<P>(sY, sec * 32 + r, half, u), f);
                }
            float* dXp = a.dx + b * a.dx_sb + (t0 + tok) * a.dx_sl + head_off<HS>(h, a.dx_sh);
            float dir = 0.f, dDs = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int col = sec * 32 + 8 * q + 4 * half;
                const floatx4 x4 = row_quad32<P>(sX, tok, col), g4 = row_quad32<P>(sY, tok, col);
                floatx4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float dxd = acc[0][0][4 * q + e] * fin;
                    o[e] = dt_row * dxd + Dh * g4[e];
                    dir += dxd * x4[e];
                    dDs += g4[e] * x4[e];
                }
                if (tok_ok) *reinterpret_cast<floatx4*>(dXp + col) = o;
            }
            dir = lane_xor_add<32>(dir);
            rbs = lane_xor_add<32>(rbs * fin);
            if (lane < 32) { s_dir[sec * kQ + tok] = dir; s_rb[sec * kQ + tok] = rbs * dt_row; }
            dDs = warp_sum(tok_ok ? dDs : 0.f);
            float dot = 0.f;      // this wave's eighth of <dS, S_prev>
#pragma unroll
            for (int it = 0; it < P * N / 4 / 512; ++it) {
                const int e = ((wave * (P * N / 4 / 512) + it) * 64 + lane) * 4;
                const floatx4 u = *reinterpret_cast<const floatx4*>(sD + e), w = *reinterpret_cast<const floatx4*>(sP + e);
#pragma unroll
                for (int k = 0; k < 4; ++k) dot += u[k] * w[k];
            }
            dot = warp_sum(dot) * __expf(Lam);
            if (lane == 0) { a.dDp8[bhc * 8 + wave] = dDs; a.dlam[bhc * kDlamParts + wave] = dot; }
        }
        // ---- 3: dG and the row and column sums of dG^h o G
        const int lane = lane_here(), r = lane & 31, half = lane >> 5, ti = gi * 32 + r;
        floatx4 Gv[4];            // G at this lane's places of a block
        auto fetch_G = [&](int cb) {
#pragma unroll
            for (int q = 0; q < 4; ++q) Gv[q] = *reinterpret_cast<const floatx4*>(Gg + op32_offset<16>(gi, 4 * cb + 2 * (q >> 1) + half, (q & 1) * 32 + r));
        };
        fetch_G(gj);
        __syncthreads();          // everyone is done with dS
        // here before the copies are under way: its wait, once they are, would be one for them as well
#pragma unroll
        for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(Gv[q]));
        if (more && sec == 0) issue_dS(h + 1);
        if (wave < 2) { const int t = here(tid); a.dirp[bhc * kQ + t] = s_dir[t] + s_dir[kQ + t]; a.rbp[bhc * kQ + t] = s_rb[t] + s_rb[kQ + t]; }
        {
            const float l_first = sl[gi * 32], l_i = sl[ti];
            const bool gfast = l_first - sl[gi * 32 + 31] < kMaxRange;
            if (lane < 32 * ngb) {
                const int j = (gj + 2 * (lane >> 5)) * 32 + r;
                wg[lane] = __expf(fminf(l_first - sl[j], kMaxRange)) * sd[j];
            }
            const float live = ti < valid ? 1.f : 0.f, u_i = live * __expf(l_i - l_first);
            auto block = [&](auto kc, auto last) {
                constexpr int k = decltype(kc)::value;
                const int cb = gj + 2 * k, j0 = cb * 32;
                floatx16 pa[1][1];
                acc_zero(pa);
                products32<1, false, 1>(pa[0], 0, 2 * KSP, [&](int u) { return row_step32<P>(sY, ti, half, u); }, NoScale32{},
                                        [&](int u, int) { return row_step32<P>(sX, j0 + r, half, u); }, last);
                wave_lds_sync();
                float rs4[4] = {0.f, 0.f, 0.f, 0.f}, cs16[16];
                auto sums = [&](auto factored) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        floatx4 w;
                        if constexpr (decltype(factored)::value) w = u_i * *reinterpret_cast<const floatx4*>(wg + k * 32 + 8 * q + 4 * half);
                        else {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int j = j0 + 8 * q + 4 * half + e;
                                w[e] = live * (__expf(fminf(l_i - sl[j], 0.f)) * sd[j]);
                            }
                        }
                        floatx4 dh;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int j = j0 + 8 * q + 4 * half + e;
                            const float d = ti >= j ? w[e] * pa[0][0][4 * q + e] : 0.f;
                            dh[e] = d;
                            // i == j is part of its row's sum and of its column's: left out of both, so that it cancels without a rounding
                            const float pr = ti == j ? 0.f : d * Gv[q][e];
                            rs4[e] += pr;
                            cs16[4 * q + e] = pr;
                        }
                        if constexpr (k == 0) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) dG[4 * q + e] += dh[e];
                        } else *reinterpret_cast<floatx4*>(dG2 + (q * 64 + lane) * 4) += dh;
                    }
                };
                if (gfast) sums(std::true_type{}); else sums(std::false_type{});
                const float rsum = lane_xor_add<32>((rs4[0] + rs4[1]) + (rs4[2] + rs4[3]));
                int ri;
                const float csum = half_wave_reduce16(cs16, &ri);
                const int blk = wave + 2 * k;
                if (lane < 32) s_rs[blk * 32 + lane] = rsum;
                if ((lane & 1) == 0) s_cs[blk * 32 + acc_row(lane, ri)] = csum;
            };
            block(std::integral_constant<int, 0>{}, [&] { if (more && sec == 1) issue_dS(h + 1); });
            if (ngb > 1) {
                fetch_G(gj + 2);
                block(std::integral_constant<int, 1>{}, NoLast32{});
            }
        }
        // ---- 4: state part of dC
        const int tok = row0 + r;
        const bool tok_ok = tok < valid;
        const float* Cp = Cg + (tok_ok ? tok : valid - 1) * a.C_sl + nb0 * 32 + 4 * half;
        __syncthreads();          // everyone is done with x
        if (more) issue_x(h + 1, (int)((hh + 1) & 1));
        if (wave < 2) {
            // What da needs of these is, per token t,  sum_{i>=t} sum_{j<t} pr[i][j]:  for t in block T the rows of T from t on (less
            // their columns inside T), the columns of T in front of t over the blocks below, and the blocks that lie below T and left of
            // it.  Pairs on one side of the whole block are never summed, where a scan over all 128 row sums minus column sums adds them
            // twice and relies on the two to cancel (6 times the error of dA with step sizes around 10).
            const int t = here(tid), T = t >> 5, k = t & 31;
            const int back = 31 - k;      // the row sums in reverse, so that their suffix is a prefix too
            float rv[4], fv[4];
#pragma unroll
            for (int J = 0; J < 4; ++J) {
                rv[J] = s_rs[(T * (T + 1) / 2 + (J < T ? J : T)) * 32 + back];
                fv[J] = s_cs[((J > T ? J * (J + 1) / 2 : T * (T + 1) / 2) + T) * 32 + k];
            }
            const float own = s_cs[(T * (T + 1) / 2 + T) * 32 + back];
            const float w1 = s_rs[(T == 1 ? 3 : 6) * 32 + k], w2 = s_rs[(T == 1 ? 6 : 7) * 32 + k];      // blocks (2, 0) and (3, 0), or (3, 0) and (3, 1)
            float e = rv[3] - own, f = 0.f, w = T == 1 || T == 2 ? w1 + w2 : 0.f;      // rv[3]: (T, T) whatever T
#pragma unroll
            for (int J = 0; J < 3; ++J) {
                if (J < T) e += rv[J];
                if (J + 1 > T) f += fv[J + 1];
            }
            w = lane_xor_add<1>(w); w = lane_xor_add<2>(w); w = lane_xor_add<4>(w); w = lane_xor_add<8>(w); w = lane_xor_add<16>(w);
            e = half_wave_scan(e);
            const float f_in = half_wave_scan(f);
            e = __shfl(e, back, 32);
            const float f_up = __shfl_up(f_in, 1, 32), f_ex = k ? f_up : 0.f;      // every lane takes part in the exchange
            a.dl[bhc * kQ + t] = e + f_ex + w;
        }
        {
            const float sc = tok_ok ? __expf(sl[tok]) : 0.f;
            float dot = 0.f;
#pragma unroll
            for (int q = 0; q < NBW; ++q) {
                floatx16 t[1][1];
                acc_zero(t);
                floatx4 Cv[4];
                products32<1, false, 1>(t[0], 0, 2 * KSP, [&](int u) { return row_step32<P>(sY, tok, half, u); }, NoScale32{},
                                        [&](int u, int) { return col_step32<N>(sP, (nb0 + q) * 32 + r, half, u); },
                                        [&] {
#pragma unroll
                                            for (int v = 0; v < 4; ++v) Cv[v] = *reinterpret_cast<const floatx4*>(Cp + q * 32 + v * 8);
                                        });
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float s = sc * t[0][0][v];
                    accC[q][v] += s;
                    dot += s * Cv[v >> 2][v & 3];
                }
            }
            dot = lane_xor_add<32>(dot);
            if (lane < 32) s_c[sec * kQ + tok] = dot;
        }
        wait_vmem_all();
        __syncthreads();          // everyone is done with dy and S_prev; x and dS of the next head are there
        if (more) issue_dy_Sp(h + 1);
        else if (wave < 2) { const int t = here(tid); a.dlc[bhc * kQ + t] = s_c[t] + s_c[kQ + t]; }
    }

    const int lane = lane_here(), r = lane & 31, half = lane >> 5, ti = gi * 32 + r, tok = row0 + r;
    auto dG_quad = [&](int k, int q) { return k ? *reinterpret_cast<const floatx4*>(dG2 + (q * 64 + lane) * 4) : floatx4{dG[4 * q], dG[4 * q + 1], dG[4 * q + 2], dG[4 * q + 3]}; };
    if (a.nslices == 1) {
        float* sG = sX;           // [kQ][kQ] over the tiles of x and dy
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (k < ngb) {
                    const int slot = ((gj + 2 * k) * 32 + 8 * q + 4 * half) >> 2;
                    *reinterpret_cast<floatx4*>(sG + ti * kQ + ((slot ^ (ti & 15)) * 4)) = dG_quad(k, q);
                }
        finish32<N, NBW>(sG, sP, accB, accC, a.Bm + b * a.B_sb + t0 * a.B_sl + g * a.B_sg, a.B_sl, a.Cm + b * a.C_sb + t0 * a.C_sl + g * a.C_sg, a.C_sl,
                         a.dB + b * a.dB_sb + t0 * a.dB_sl + g * a.dB_sg, a.dB_sl, a.dC + b * a.dC_sb + t0 * a.dC_sl + g * a.dC_sg, a.dC_sl, valid, wave, rb, nb0);
        return;
    }
    const int64_t part = grp * a.nslices + slice;
    float* op = a.dGp + part * (kQ * kQ) + ti * kQ + gj * 32 + 4 * half;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (k < ngb) *reinterpret_cast<floatx4*>(op + k * 64 + 8 * q) = dG_quad(k, q);
    const int64_t o = part * (kQ * N) + tok * N + nb0 * 32 + 4 * half;
#pragma unroll
    for (int q = 0; q < NBW; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            *reinterpret_cast<floatx4*>(a.dBp + o + q * 32 + 8 * v) = floatx4{accB[q][4 * v], accB[q][4 * v + 1], accB[q][4 * v + 2], accB[q][4 * v + 3]};
            *reinterpret_cast<floatx4*>(a.dCp + o + q * 32 + 8 * v) = floatx4{accC[q][4 * v], accC[q][4 * v + 1], accC[q][4 * v + 2], accC[q][4 * v + 3]};
        }
}

// The finish from partials that are already summed over the head slices: a workgroup of 512 threads per (batch, chunk, group) and side.
// It is one chain of memory latencies, a CU to itself (128 KiB of LDS): both sides in one workgroup took 22.5 us at b1 l785 g2 and
// at b1 l347 g1, 12.5 a side (and 12.5 for both, side by side).
template <int N> constexpr size_t finish32_smem() { return (size_t)(kQ * kQ + kQ * N) * sizeof(float); }
template <int N, int SIDE>
__device__ __forceinline__ void bc_final32_body(const float* dGs, const float* dCs, const float* dBs, const float* Bm, int64_t B_sb, int64_t B_sl, int64_t B_sg,
                                                const float* Cm, int64_t C_sb, int64_t C_sl, int64_t C_sg, float* dB, int64_t dB_sb, int64_t dB_sl, int64_t dB_sg,
                                                float* dC, int64_t dC_sb, int64_t dC_sl, int64_t dC_sg, int64_t seqlen, int64_t ngroups, int64_t nchunks,
                                                int64_t c, int64_t g, int64_t b) {
    constexpr int NBW = N / 64;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float* sG = reinterpret_cast<float*>(smem_raw);
    float* sM = sG + kQ * kQ;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, half = lane >> 5;
    const int wave = (int)uniform(tid >> 6), rb = wave < 4 ? wave : 7 - wave, nb0 = (wave >> 2) * NBW, tok = rb * 32 + r;
    const int64_t t0 = c * kQ, grp = (b * nchunks + c) * ngroups + g;
    const int valid = (int)(seqlen - t0 < kQ ? seqlen - t0 : kQ);
    const float* gp = dGs + grp * (int64_t)(kQ * kQ);
    // every load out before the first is waited for; pieces above the diagonal: the row's first in their place
    constexpr int PIECES = kQ * kQ / 4 / 512;
    floatx4 gv[PIECES];
#pragma unroll
    for (int it = 0; it < PIECES; ++it) {
        const int e = it * 512 + tid, i = e / (kQ / 4), s = e % (kQ / 4);
        gv[it] = *reinterpret_cast<const floatx4*>(gp + i * kQ + ((s >> 3) <= (i >> 5) ? s : 0) * 4);
    }
    floatx16 acc[NBW];
    const int64_t o = grp * (int64_t)(kQ * N) + tok * N + nb0 * 32 + 4 * half;
    const float* part = (SIDE == 1 ? dCs : dBs) + o;
#pragma unroll
    for (int q = 0; q < NBW; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const floatx4 p = *reinterpret_cast<const floatx4*>(part + q * 32 + 8 * v);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[q][4 * v + e] = p[e];
        }
#pragma unroll
    for (int it = 0; it < PIECES; ++it) {
        const int e = it * 512 + tid, i = e / (kQ / 4), s = e % (kQ / 4);
        if ((s >> 3) <= (i >> 5)) *reinterpret_cast<floatx4*>(sG + i * kQ + ((s ^ (i & 15)) * 4)) = gv[it];
    }
    finish32<N, NBW, SIDE>(sG, sM, acc, acc, Bm + b * B_sb + t0 * B_sl + g * B_sg, B_sl, Cm + b * C_sb + t0 * C_sl + g * C_sg, C_sl,
                     dB + b * dB_sb + t0 * dB_sl + g * dB_sg, dB_sl, dC + b * dC_sb + t0 * dC_sl + g * dC_sg, dC_sl, valid, wave, rb, nb0);
}

}  // namespace m2
