// Chunk states for 16-bit operands in ONE pass: the per-chunk contributions and the recurrence over the chunks fused,
// with the running state in registers (fp32), so that no per-chunk contribution is ever written to memory.
//
//   forward:  S = init;   for c = 0 .. nc-1:   prev[c] = T(S);   S = e^{Lam_c} S + sum_j (dt_j e^{Lam_c - l_j}) x_j (x) B_j;   final = S
//   reverse:  R = dfinal; for c = nc-1 .. 0:   prev[c] = T(R);   R = e^{Lam_c} R + sum_i e^{l_i} dy_i (x) C_i;   dinit = R
//
// grid (nheads * SPLIT, batch, segments), N / 32 waves.  Segments: one, the walk over all chunks (PHASE 0); or, of few heads' long walks, two
// launches over all segments but one (PHASE 1 walks the first, storing the states, and forms the sums of the middle ones from zero, storing nothing
// else; PHASE 2 walks the second to the last from the sums in front of each).  A workgroup owns 1 / SPLIT of the ROWS of the [P][N] state (head
// channels; all N columns), wave w the columns [32 w, +32) of them, as 32x32 MFMA accumulator blocks: only that part of the x / dy columns
// is loaded, scaled and staged, so the workgroups of a head share no work.  Per chunk the MFMA computes
// X_scaled^T [P/2 x kQ] * M [kQ x N]:
//   * M (B or C of the group) comes from the transposed tiles that prep_kernel wrote in MFMA operand order: a wave's
//     B-operand fragment is one contiguous KiB of global memory, loaded straight into registers at the top of the
//     chunk's iteration (the tile is shared by all heads of the group and stays in L2);
//   * x / dy rows are loaded two chunks ahead into registers, scaled per token in fp32, rounded once and written
//     row-major into one of two LDS buffers (one barrier per chunk); the A-operand fragments (k = token contiguous)
//     come out of it through LDS transpose reads.
// The state leaves through an LDS tile of the workgroup's whole slab (one per chunk parity), written before the chunk's barrier
// and read behind it, so that a wave stores whole state rows: its share of the slab is one contiguous piece of memory.
#pragma once
#include <type_traits>

#include "ssd_y.hpp"

namespace m2 {

struct StatePassArgs {
    const void* X; int64_t X_sb, X_sl, X_sh;      // x (forward) / dy (reverse): [b][l][h][P]
    const float* ldtab;                            // [b][h][c][ l kQ | dt kQ ]
    const void* Mt;                                // B^T (forward) / C^T (reverse) tiles: [b][c][g][N x kQ in operand order]
    const float* init;                             // fp32 [b][h][P][N]: initial state / gradient of the final state, or null
    void* prev;                                    // out [b][c][h][P][N], operand type
    float* final_out;                              // out fp32 [b][h][P][N]: final state / gradient of the initial state, or null
    int64_t seqlen, nheads, ngroups, nchunks;
    floatx4* seg; float* seg_lam;                  // in segments: a segment's state [segment][b][h] in accumulator order, and the sum of its Lam
    int64_t seg_chunks;                            // chunks per segment
};

// What bounds the pass: a CU's vector-memory path.  Its loads retire in order, so the operand fragments (which come from L2)
// queue behind the x rows (which come from HBM), and the bytes that one step takes through it decide the step's time: x and
// dy 8 KiB, fragments 32 KiB and states 8 KiB for half a head, whose stores and loads each cost their own time at b4 l2048
// h80 (57 us; 42 without the stores, 41 without the x rows, 46 without the fragments, 16 without any).
// SPLIT = 2, half a head per workgroup, spreads few heads over more CUs and fills the last round of many better.  SPLIT = 1
// feeds two products from each fragment, 48 KiB a step for a whole head where two halves take 80, and reads whole 128-byte
// lines of x: state_pass_split says where that wins.
constexpr int kStatePassSplit = 2;
// SPLIT = 1 only with 128 state columns (with 64 there are two waves of 256 registers, and they spill), only for the one-tile
// form, and only where whole heads fill the CUs in nearly whole rounds (the last one idle by a fifth at most).  Forward at
// l 4096 (b h up to 256) or 2048: b h 192 136 -> 132 us, 224 162 -> 152, 256 177 -> 163, 448 157 -> 150, 512 178 -> 163,
// 768 252 -> 247, 1024 367 -> 355; below the line 80 63 -> 79, 160 98 -> 100, 288 88 -> 91, 320 98 -> 101, 384 124 -> 126.
inline int state_pass_split(int64_t heads, int n) {
    const int64_t cus = device_cus(), rounds = ceil_div(heads, cus);
    return n == 128 && heads * 5 >= rounds * cus * 4 ? 1 : kStatePassSplit;
}
// Chunks per segment, or 0: one pass over the whole sequence.  Half heads that leave half the CUs idle walk a long sequence as a chain
// of steps of about 1.05 us each; in segments the chain is as long as two of them: the first launch walks the first segment and forms
// the sums of the others but the last from zero, all side by side, and the second starts each of the others from the sums in front of
// it, decayed (the decay is one number per head, so this costs a product per element and segment).
// A launch more and the filling of two chains cost about 3 us on the device: below a line they are not earned.  The launch also costs 2.5 us
// of the host, which a prompt's forward does not wait for and training few heads does: lines of their own for a forward that keeps its states
// for the backward (with the final state, forward and backward: b1 l2600 h8 g8 112.9 -> 115.5 us, l3000 h4 111 -> 114.5, l4000 h8 g8 120 -> 114, l4000
// h16 126 -> 114) and for the passes that leave no final state, where the operands of one tile walk faster (l4000 h8 g8 98 -> 104, l7519 h16 g8
// 243 -> 170).  Whole forward scan alone, us, whole pass ->
// segments, for 16, 48, 64, 84 and 128 half heads (16, 5, 4, 3 and 2 sets), 128 state columns:
//   8 chunks    22.9 -> 23.8   24.3 -> 25.5   24.9 -> 26.0   28.1 -> 30.8   30.2 -> 33.0
//   12 chunks   25.7 -> 24.7   29.8 -> 29.2   30.8 -> 30.7   31.4 -> 33.2   35.6 -> 37.8
//   16 chunks   28.4 -> 25.5   33.6 -> 31.9   34.6 -> 35.4   36.5 -> 37.6   39.3 -> 41.4
//   24 chunks   34.0 -> 27.4   41.8 -> 37.5   43.1 -> 38.9   43.0 -> 42.3   51.1 -> 51.1
//   64 chunks   65.8 -> 38.2   74.9 -> 53.5   80.3 -> 60.9   81.6 -> 74.5   96.8 -> 88.5
constexpr int64_t kSegPrompt = 20, kSegKept = 28, kSegOneTile = 48;      // chunks from which a walk goes in segments
inline int64_t state_pass_seg_chunks(int64_t heads, int64_t nchunks, int64_t least) {
    const int64_t sets = heads > 0 ? device_cus() / (heads * kStatePassSplit) : 0;      // of workgroups that the CUs hold, one each
    if (sets < 2 || nchunks < least || nchunks * sets < 96) return 0;
    const int64_t chunks = ceil_div(nchunks, sets + 1);
    return chunks < 2 ? 2 : chunks;
}
// Lane by lane, an instruction that reads the initial state touches 32 rows for 32 bytes each.  STAGED takes whole rows through LDS, but its
// loop comes out of the compiler about 20 ns a chunk slower.  Whole prefill core with 80 heads of 64 x 128 states behind a cached prefix, us, as
// lanes -> staged: 8 x 1 chunk 57.4 -> 50.1, 8 x 3 91.1 -> 83.5, 1 x 8 48.3 -> 47.6, 1 x 32 115.2 -> 115.0, 4 x 32 380.0 -> 377.1, 1 x 64 221.9 ->
// 222.9, 1 x 128 424.8 -> 426.8.
inline bool state_pass_staged(bool init, int64_t nchunks) { return init && nchunks <= 32; }
// one wave per 32 state columns
template <int N> constexpr int state_pass_threads() { return (N / 32) * 64; }
template <int P, int N, bool HILO = false, int SPLIT = kStatePassSplit>
constexpr size_t state_pass_smem() {
    return (size_t)(HILO ? 2 : 1) * 2 * kQ * (P / SPLIT) * 2 + (size_t)2 * (P / SPLIT) * (N + 8) * 2;
}

// HILO: the scaled rows are staged as TWO 16-bit tiles, the rounded value and the rounded remainder, and each k step takes
// two products, so that the fp32 scale dt e^{Lam - l} reaches the accumulators with 16 significand bits instead of 8 (the
// final state is an fp32 output; with one tile its error is that of the operand rounding, 2^-9 of every term).
// STAGED: the initial state comes as whole rows through the slab tiles (see state_pass_staged).
// PHASE 0: the whole sequence.  1: segment z, up to the last but one, from the initial state (the first, whose states are stored) or from
// zero, to `seg` and `seg_lam`.  2: segment z + 1 from what `seg` holds for those in front of it.  Segments count in the order of the walk.
// The initial state is read in the first launch only and the final one written in the second: they may be the same tensor.
template <typename T, int P, int N, bool REVERSE, int HS, bool HILO = false, int SPLIT = kStatePassSplit, int PHASE = 0, bool STAGED = false>
__global__ void __launch_bounds__(state_pass_threads<N>(), SPLIT == 1 ? 2 : 3)
state_pass16_kernel(const StatePassArgs a) {
    static_assert(sizeof(T) == 2, "16-bit operands only");
    constexpr int NWAVES = N / 32, THREADS = state_pass_threads<N>();
    constexpr int PH = P / SPLIT;                      // state rows (head channels) of this workgroup
    constexpr int NW = 32;                             // state columns per wave
    constexpr int PBW = PH / 32, NBW = 1;              // 32x32 blocks per wave
    constexpr int SPR_X = PH / 8;                      // 16-byte slots per staged x row
    constexpr int NXR = kQ * SPR_X / THREADS;              // x pieces per thread per chunk
    constexpr int LDO = N + 8;
    constexpr int LPR = N / 8;                         // lanes per state row (8 elements each)
    constexpr int RPP = 64 / LPR;                      // rows per store pass
    constexpr int RW = PH / NWAVES;                    // rows a wave stores: the workgroup's slab leaves as whole rows
    constexpr int NSP = RW / RPP;                      // store passes
    static_assert(RW % RPP == 0, "whole store passes");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int XT = HILO ? 2 : 1;                   // staged tiles per chunk
    T* sX = reinterpret_cast<T*>(smem_raw);                                 // [2][XT][kQ][P / 2], slots swizzled inside each row
    T* sO = sX + 2 * XT * kQ * PH;                                          // [2][P / 2][LDO]

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r = lane & 31, half = lane >> 5;
    const int pw = (int)(blockIdx.x / a.nheads);       // which part of the rows
    // the workgroups of one head are nheads apart in the grid: with a head count that is a multiple of 8 they land on the
    // same XCD and share the head's rows in its L2
    const int64_t h = blockIdx.x % a.nheads, b = blockIdx.y;
    const int wave_u = (int)uniform((uint32_t)wave), n0 = wave_u * NW;      // first state column of this wave
    const int64_t g = h / (a.nheads / a.ngroups);
    const int64_t bh = b * a.nheads + h;
    const int64_t nc = a.nchunks;
    const int tr_tok = 8 * half + ((lane >> 2) & 3);
    const int tr_col = ((lane >> 4) & 1) * 16 + 4 * (lane & 3);
    typedef T tvec4 __attribute__((ext_vector_type(4)));
    // element offsets of this lane's transpose reads of k step 0 (a step is 16 rows, and tile_swz looks at the row modulo 16)
    const int tr_lo = (tr_tok * SPR_X + ((tr_col >> 3) ^ tile_swz<SPR_X>(tr_tok))) * 8 + (tr_col & 7);
    const int tr_hi = ((tr_tok + 4) * SPR_X + ((tr_col >> 3) ^ tile_swz<SPR_X>(tr_tok + 4))) * 8 + (tr_col & 7);

    // The MFMAs are issued with swapped operands: acc[i][j][v] is the state at row pw P/2 + 32 i + r, column
    // n0 + 32 j + acc_row(lane, v), i.e. a lane holds groups of 4 consecutive columns of ONE row (8-byte staging writes).
    floatx16 acc[PBW][NBW];
    const int64_t seg = PHASE == 0 ? 0 : (int64_t)blockIdx.z + (PHASE == 2 ? 1 : 0);
    const int64_t seg_pitch = (int64_t)gridDim.y * a.nheads * (P * N / 4);
    floatx4* const seg_q = PHASE == 0 ? nullptr : a.seg + ((bh * SPLIT + pw) * NWAVES + wave_u) * (PBW * NBW * 4 * 64) + lane;
    const float* init = PHASE == 0 || (PHASE == 1 && seg == 0) ? a.init : nullptr;
    static_assert(!STAGED || PHASE == 0, "a whole walk");
    constexpr int NI = PH * N / 4 / THREADS, CV = N / 4;
    typedef float AnyFloat4 __attribute__((ext_vector_type(4), aligned(4)));      // a caller's tensor: any element
    [[maybe_unused]] floatx4 first[NI];
    if constexpr (STAGED) {
#pragma unroll
        for (int it = 0; it < NI; ++it) first[it] = *reinterpret_cast<const AnyFloat4*>(init + bh * (P * N) + pw * (PH * N) + (it * THREADS + tid) * 4);
    } else {
#pragma unroll
        for (int i = 0; i < PBW; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int row = pw * PH + i * 32 + r, col = n0 + j * 32 + acc_row(lane, v);
                    acc[i][j][v] = init ? init[bh * (P * N) + row * N + col] : 0.f;
                }
    }
    auto take_init = [&] {      // behind the first rows' loads
        float* const sI = reinterpret_cast<float*>(sO);      // [PH][LDO]: the slab tiles are as large as the workgroup's rows in fp32
#pragma unroll
        for (int it = 0; it < NI; ++it) {
            const int e = it * THREADS + tid;
            *reinterpret_cast<floatx4*>(sI + e / CV * LDO + e % CV * 4) = first[it];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PBW; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const floatx4 v = *reinterpret_cast<const floatx4*>(sI + (i * 32 + r) * LDO + n0 + j * 32 + 8 * q + 4 * half);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] = v[e];
                }
        __syncthreads();      // the first state's tile is written over it
    };
    if constexpr (PHASE == 2) {
        // A segment's e^Lam can overflow where no chunk's does (dt A > 0).  Then it is taken in factors that fp32 holds, so that a state of zeros stays
        // zero (not 0 inf) and a tiny one grows as it did chunk by chunk; three of them take any other to inf.  (Found out behind the loop: a branch
        // in it stands in front of the next segment's loads, 1.5 us at 24 segments.)
        float most = 0.f;
        auto in_front = [&](auto safe) {
            for (int64_t t = 0; t < seg; ++t) {
                float lam = t ? a.seg_lam[t * (int64_t)gridDim.y * a.nheads + bh] : 0.f;      // nothing in front of the first
                if constexpr (decltype(safe)::value) {
                    for (int k = 0; k < 3 && lam > 80.f; ++k) {
                        const float f = __expf(80.f);
                        lam -= 80.f;
#pragma unroll
                        for (int i = 0; i < PBW; ++i)
#pragma unroll
                            for (int j = 0; j < NBW; ++j)
#pragma unroll
                                for (int v = 0; v < 16; ++v) acc[i][j][v] *= f;
                    }
                    lam = lam > 80.f ? 80.f : lam;      // (NaN stays)
                } else {
                    most = fmaxf(most, lam);
                }
                const float dec = t ? __expf(lam) : 0.f;
#pragma unroll
                for (int i = 0; i < PBW; ++i)
#pragma unroll
                    for (int j = 0; j < NBW; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const floatx4 v = seg_q[t * seg_pitch + ((i * NBW + j) * 4 + q) * 64];
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] = acc[i][j][4 * q + e] * dec + v[e];
                        }
            }
        };
        in_front(std::false_type{});
        if (__builtin_expect(most > 80.f, false)) {
            acc_zero(acc);
            in_front(std::true_type{});
        }
    }

    // two chunks ahead in registers, in two sets used alternately: the x / dy pieces with their token's l and dt, and
    // the chunk's Lam.  The values of chunk cc are consumed before the barrier of its iteration; behind it the same set
    // is loaded with chunk cc + 2, so that a load has two iterations to land.
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    struct Ahead { u32x4 x[NXR]; float l[NXR], d[NXR], lam; };
    // Addresses are a wave-uniform base (scalar registers) plus a 32-bit per-lane byte offset, recomputed from the thread
    // index where it is cheap: 64-bit per-lane pointers kept alive across the chunk loop cost more registers than the data.
    const uint32_t row_t = (uint32_t)tid / SPR_X, slot_t = (uint32_t)tid % SPR_X;      // piece `it` of this thread: row_t + it * RSTEP
    constexpr int RSTEP = THREADS / SPR_X;
    const uint32_t x_row_bytes = (uint32_t)(a.X_sl * 2);
    // The bases walk from chunk to chunk by constant steps: formed anew for each chunk out of 64-bit products (and the issue
    // priority below out of a 64-bit quotient) they were 150 of the 200 scalar instructions of an iteration, which on a chip
    // holding few workgroups stand between one chunk's products and the next: 181 -> 169 us at b1 l16384 h80.
    const int nci = (int)nc, c0 = PHASE == 0 ? 0 : (int)(seg * a.seg_chunks);      // c0: chunks in front of the segment
    const bool last_seg = PHASE == 0 || (PHASE == 2 && blockIdx.z + 1 == gridDim.z);
    const int cfirst = REVERSE ? nci - 1 - c0 : c0, tail_at = (REVERSE ? 0 : nci - 1) - c0;
    const int count = last_seg ? nci - c0 : (int)a.seg_chunks;
    // Steps of the recurrence: what the last chunk adds reaches only the state behind it, so without a reader of that the last
    // chunk's state is stored and nothing of it is loaded or multiplied (forward and backward at b4 l2048 h80 335.5 -> 332.5 us; fp32
    // operands, whose chunks are workgroups of part-filled rounds, gained nothing by the same).
    const bool ends = PHASE == 1 || (last_seg && (HILO || a.final_out));      // (two-tile operands are for a final state)
    const int nsteps = ends ? count : count - 1;
    const int tail_rows = (int)(a.seqlen - (nc - 1) * kQ);      // valid rows of the last chunk
    constexpr int DIR = REVERSE ? -1 : 1;
    const char* xq = reinterpret_cast<const char*>(static_cast<const T*>(a.X) + b * a.X_sb + (int64_t)cfirst * kQ * a.X_sl + head_off<HS>(h, a.X_sh) + pw * PH);
    const float* tq = a.ldtab + (bh * nc + cfirst) * (2 * kQ);
    const char* mp = reinterpret_cast<const char*>(static_cast<const T*>(a.Mt) + ((b * nc + cfirst) * a.ngroups + g) * (int64_t)(N * kQ) + wave_u * (8 * 512));
    char* op = reinterpret_cast<char*>(static_cast<T*>(a.prev) + ((b * nc + cfirst) * a.nheads + h) * (int64_t)(P * N) + (pw * PH + wave_u * RW) * N);
    const int64_t x_step = DIR * (int64_t)kQ * a.X_sl * 2, m_step = DIR * a.ngroups * (int64_t)(N * kQ * 2), o_step = DIR * a.nheads * (int64_t)(P * N * 2);
    int kload = 0;                                      // processing index of the chunk xq and tq stand at
    auto load_ahead = [&](Ahead& s) {
        const uint32_t last = (uint32_t)((kload == tail_at ? tail_rows : kQ) - 1);      // last valid row
        const uint32_t last_off = last * x_row_bytes;
        const char* xp = xq;
        const float* tab = tq;
        s.lam = tab[kQ - 1];
#pragma unroll
        for (int it = 0; it < NXR; ++it) {
            const uint32_t row = row_t + it * RSTEP;
            // rows past the end: finite stand-ins, scaled by zero (minimum of products, not product of the minimum: hipcc
            // multiplies and adds in a 64-bit instruction whose unused high half it puts into a load's target register)
            const uint32_t off = row * x_row_bytes < last_off ? row * x_row_bytes : last_off;
            s.x[it] = *reinterpret_cast<const u32x4*>(xp + (off + slot_t * 16u));
            s.l[it] = tab[row];
            s.d[it] = REVERSE ? (row <= last ? 1.f : 0.f) : tab[kQ + row];      // dt is 0 past the end of the sequence
        }
        if (kload < nsteps - 1) { ++kload; xq += x_step; tq += DIR * 2 * kQ; }      // past the end: the last step's chunk once more
    };
    // loaded at the top of the iteration that consumes them (so that the wait in front of their use can be counted
    // exactly and leaves the next chunk's rows, issued behind them, in flight): the group's B^T / C^T fragments (L2)
    Frag<T> bf[NBW][8];
    const uint32_t st_off = (uint32_t)((lane / LPR * N + (lane % LPR) * 8) * 2);      // pass ps: + ps * RPP * N * 2
    auto load_same = [&] {
#pragma unroll
        for (int j = 0; j < NBW; ++j)
#pragma unroll
            for (int ks = 0; ks < 8; ++ks)      // see mt_offset
                bf[j][ks].v = *reinterpret_cast<const bf16x8*>((mp + ((j * 8 + ks) & ~3) * 1024) + ((uint32_t)lane * 16u + (uint32_t)((ks & 3) * 1024)));
        mp += m_step;
    };

    const int q1 = (nsteps + 3) / 4, q2 = (2 * nsteps + 3) / 4, q3 = (3 * nsteps + 3) / 4;      // first chunk of each quarter
    auto put_state = [&](T* cO) {
#pragma unroll
        for (int i = 0; i < PBW; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int qp = 0; qp < 2; ++qp) {
                    // a lane and its partner (lane ^ 32) hold the two halves of every 8-column group: one exchange of the packed
                    // words leaves each with a whole group, written as 16 bytes (8-byte writes of 32 rows at this pitch would
                    // meet pairwise in the same banks)
                    const int q0 = 2 * qp, q1 = q0 + 1;
                    uint32_t o0, o1, o2, o3;
                    pair_swap(pack2<T>(acc[i][j][4 * q0], acc[i][j][4 * q0 + 1]), pack2<T>(acc[i][j][4 * q1], acc[i][j][4 * q1 + 1]), o0, o2);
                    pair_swap(pack2<T>(acc[i][j][4 * q0 + 2], acc[i][j][4 * q0 + 3]), pack2<T>(acc[i][j][4 * q1 + 2], acc[i][j][4 * q1 + 3]), o1, o3);
                    *reinterpret_cast<u32x4*>(cO + (i * 32 + r) * LDO + n0 + j * 32 + 8 * (q0 + half)) = u32x4{o0, o1, o2, o3};
                }
    };
    auto store_rows = [&](const T* cO) {      // whole rows of the workgroup's slab
#pragma unroll
        for (int ps = 0; ps < NSP; ++ps) {
            const int rl = wave * RW + ps * RPP + lane / LPR, cv = lane % LPR;
            const u32x4 o = *reinterpret_cast<const u32x4*>(cO + rl * LDO + cv * 8);
            *reinterpret_cast<u32x4*>((op + ps * RPP * N * 2) + st_off) = o;
        }
        op += o_step;
    };
    int next_drop = q1;
    float lam_sum = 0.f;
    __builtin_amdgcn_s_setprio(3);
    auto walk = [&](auto keeps) {      // keeps: the states leave
    constexpr bool KEEPS = decltype(keeps)::value;
    auto step = [&](int cc, Ahead& s) {
        const int buf = cc & 1;
        // Issue priority falls as the workgroup advances, so that of the workgroups sharing a CU the one furthest behind
        // goes first: the hardware otherwise prefers the oldest waves, and the last workgroup placed on a CU that holds
        // one more than its neighbours finishes long after everybody else.
        if (cc == next_drop) {
            if (cc == q1) __builtin_amdgcn_s_setprio(2);
            else if (cc == q2) __builtin_amdgcn_s_setprio(1);
            else __builtin_amdgcn_s_setprio(0);
            next_drop = cc < q2 ? q2 : q3;
        }
        T* cX = sX + buf * (XT * kQ * PH);
        __builtin_amdgcn_sched_barrier(0);      // keep this chunk's loads out of the previous chunk's MFMA phase (registers)
        load_same();
        // the values loaded one chunk ahead become visible to the optimiser here and no earlier: otherwise their
        // unpacking is scheduled right behind the loads, which then wait for the data a whole chunk too early
#pragma unroll
        for (int it = 0; it < NXR; ++it)
            asm volatile("" : "+v"(s.x[it]), "+v"(s.l[it]), "+v"(s.d[it]));      // whole 128-bit vectors: no re-packing
        asm volatile("" : "+v"(s.lam));
        // ---- scaled rows into LDS
#pragma unroll
        for (int it = 0; it < NXR; ++it) {
            const int row = (int)row_t + it * RSTEP, slot = (int)slot_t;
            const float sc = REVERSE ? s.d[it] * __expf(s.l[it]) : s.d[it] * __expf(s.lam - s.l[it]);
            // word-wise (two elements per 32-bit word), so that the loaded vectors stay four whole registers until here
            u32x4 o;
            if constexpr (HILO) {
                u32x4 o2;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float v0 = unpack_lo<T>(s.x[it][q]) * sc, v1 = unpack_hi<T>(s.x[it][q]) * sc;
                    o[q] = pack2<T>(v0, v1);
                    o2[q] = pack2<T>(v0 - unpack_lo<T>(o[q]), v1 - unpack_hi<T>(o[q]));
                }
                *reinterpret_cast<u32x4*>(cX + kQ * PH + (row * SPR_X + (slot ^ tile_swz<SPR_X>(row))) * 8) = o2;
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) o[q] = pack2<T>(unpack_lo<T>(s.x[it][q]) * sc, unpack_hi<T>(s.x[it][q]) * sc);
            }
            *reinterpret_cast<u32x4*>(cX + (row * SPR_X + (slot ^ tile_swz<SPR_X>(row))) * 8) = o;
        }
        const float dec = __expf(s.lam);
        if (PHASE == 1) lam_sum += s.lam;
        // the state as it enters this chunk goes into the slab tile of this parity (the other one may still be read by a
        // wave that is behind: it was filled one barrier ago)
        if (KEEPS) put_state(sO + buf * (PH * LDO));
        __syncthreads();          // both tiles are complete; every wave is done with the other buffers
        load_ahead(s);            // the rows two chunks on

        // ---- the state entering (forward) / the gradient leaving (reverse) this chunk
        if (KEEPS) store_rows(sO + buf * (PH * LDO));

        // ---- S = e^{Lam} S + X_scaled^T M  (accumulated as its transpose M^T X_scaled)
#pragma unroll
        for (int i = 0; i < PBW; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] *= dec;
        // all A-operand fragments of the chunk are read from LDS first: the eight products form one dependent chain, and a
        // read issued next to its product would put an LDS round trip between any two of them
#pragma unroll
        for (int xt = 0; xt < XT; ++xt) {
            const T* tX = cX + xt * (kQ * PH);
            Frag<T> af[PBW][8];
#pragma unroll
            for (int ks = 0; ks < 8; ++ks)
#pragma unroll
                for (int i = 0; i < PBW; ++i) {
                    const tvec4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((M2_LDS tvec4*)(tX + (tr_lo ^ (i * 32)) + ks * 16 * PH));
                    const tvec4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((M2_LDS tvec4*)(tX + (tr_hi ^ (i * 32)) + ks * 16 * PH));
#pragma unroll
                    for (int e = 0; e < 4; ++e) { af[i][ks].v[e] = lo[e]; af[i][ks].v[4 + e] = hi[e]; }
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < 8; ++ks)
#pragma unroll
                for (int i = 0; i < PBW; ++i)
#pragma unroll
                    for (int j = 0; j < NBW; ++j) mma_frag(acc[i][j], bf[j][ks], af[i][ks]);
            if (XT > 1) __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Chunks are taken two per loop iteration (one per register set); an odd first chunk is peeled off in front so that
    // the loop body is free of conditionals (a branch around loads costs register copies, and with them early waits).
    Ahead s0, s1;
    int cc = 0;
    if (nsteps & 1) {
        load_ahead(s1);
        load_ahead(s0);
        if constexpr (STAGED) take_init();
        step(0, s1);
        cc = 1;
    } else {
        if (nsteps > 0) {
            load_ahead(s0);
            load_ahead(s1);
        }
        if constexpr (STAGED) take_init();
    }
#pragma unroll 1
    for (; cc < nsteps; cc += 2) {
        step(cc, s0);
        step(cc + 1, s1);
    }
    };
    if (PHASE == 1 && seg > 0) walk(std::false_type{});
    else walk(std::true_type{});
    if (PHASE == 1) {
#pragma unroll
        for (int i = 0; i < PBW; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    seg_q[seg * seg_pitch + ((i * NBW + j) * 4 + q) * 64] =
                        floatx4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        if (tid == 0 && pw == 0) a.seg_lam[seg * (int64_t)gridDim.y * a.nheads + bh] = lam_sum;
    } else if (ends) {
#pragma unroll
        for (int i = 0; i < PBW; ++i)
#pragma unroll
            for (int j = 0; j < NBW; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int row = pw * PH + i * 32 + r, col = n0 + j * 32 + acc_row(lane, v);
                    a.final_out[bh * (P * N) + row * N + col] = acc[i][j][v];
                }
    } else {
        T* cO = sO + (nsteps & 1) * (PH * LDO);
        put_state(cO);
        __syncthreads();
        store_rows(cO);
    }
}

}  // namespace m2
