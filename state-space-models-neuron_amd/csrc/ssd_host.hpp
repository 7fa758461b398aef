// Host-side helpers shared by the SSD forward and backward launchers.
#pragma once
#include "ssd_kernels.hpp"
#include "ssd_bwd_main.hpp"
#include "ssd_dg.hpp"
#include "ssd_states16.hpp"
#include "ssd_f32.hpp"

namespace m2 {

// A call as the kernels see it: heads of kP channels, hs = 1 where a true head is two of them (see head_off; the HS of the kernels).
struct SsdCall : m2_ssd_params {
    int hs;
    int64_t true_heads;
    explicit SsdCall(const m2_ssd_params* p) : m2_ssd_params(*p), hs(p->headdim > kP ? 1 : 0), true_heads(p->nheads) {
        nheads <<= hs;
        headdim = kP;
    }
};

// Workspace regions.  Forward uses G, local, prev, lam.  Backward additionally uses
// dprev (gradient w.r.t. the state leaving each chunk, operand type), dlam, dl (per-token gradient of the in-chunk cumulative
// sum, per head), per-(b,h,chunk) partials of dA and dD, and
// per-(b,chunk,group,head-slice) fp32 partials of dB and dC.
struct SsdWorkspace {
    float* G = nullptr; float* local = nullptr; void* prev = nullptr; float* lam = nullptr;
    void* Gm = nullptr; void* Gmt = nullptr; void* Bt = nullptr; void* Ct = nullptr;
    float* ldtab = nullptr;             // [b][h][c][ l kQ | dt kQ ]
    void* dprev = nullptr; float* dlam = nullptr;
    float* dbp = nullptr;                                               // per (b, h, chunk) partials of d_dt_bias
    float* dAp = nullptr; float* dDp = nullptr; float* dBp = nullptr; float* dCp = nullptr; float* dl = nullptr; float* dlc = nullptr; float* dGp = nullptr;
    float* dGs = nullptr; float* dBs = nullptr; float* dCs = nullptr;   // partials summed over the head slices, where there are several
    float* dirp = nullptr; float* rbp = nullptr; float* dDp8 = nullptr; // per token, per wave: what the main kernel leaves for ddt and dD
    int64_t ns_g = 1, hps_g = 1, ns_b = 1, hps_b = 1;   // head slicing of dg16 and of the main backward kernel
    void* seg = nullptr; float* seg_lam = nullptr;      // the state pass in segments
    bool finished = false;              // the main kernel's workgroups have whole groups and leave dB and dC: no partials of those
    size_t bytes = 0;
    size_t kept_bytes = 0;              // size of the forward -> backward carry-over (chunk_states buffer)
};

// f(slices, heads of all of them but the last) for every division of hpg heads into equal slices and a rest, fewest slices first: the largest count that a
// slice can have below the one before, and the fewest slices of it (22 of 128 counts: looking at each of them cost a call 0.96 us).
template <typename F> void each_slicing(int64_t hpg, F&& f) {
    for (int64_t s = 1;;) {
        const int64_t heads = ceil_div(hpg, s);
        f(s, heads);
        if (heads <= 1) break;
        s = ceil_div(hpg, heads - 1);
    }
}

// A workgroup owns one chunk of one group and loops over a slice of that group's heads (operands shared by the
// group stay on chip, group-level reductions happen in registers).  The slices have equal numbers of heads but the last, which has
// what is left (with divisors of the heads per group only, a prime count had one head a slice or all of them: forward and backward at
// b3 l1111 h31 166 -> 102 us, b1 l2130 h106 406 -> 266, fp32 b4 l416 h83 346 -> 258).  Their count is the one with the least of:
// workgroups on the busiest CU times heads per slice -- a CU that could hold two (`wgs_per_cu`) and has one takes three
// quarters of two's time, and with few tokens, where a head is latency, all of it (y at b9 l1 h58 p128 13.1 -> 9.9 us, b11 l9 h96 whole forward
// 34.5 -> 32.2) --, 1.5 heads' worth for filling and draining each of them (of the longer fp32 heads half of that with few tokens: forward at b33 l6
// h31 102 -> 98, b38 l4 h13 62 -> 58; with whole chunks b9 l903 h15 102 | 106), and, `partials`, what the slices' partial
// sums cost on their way out and back (128 KiB each: a head's worth per 110 workgroups).  Taking whatever first filled the chip
// instead left a nearly empty last round and twice the partials at b3 l1111 h32: main backward kernel 41 -> 31 us, dG 17.7 ->
// 14.2, slice sums 17.9 -> 10.1, y 17.4 -> 15.4; y at b8 l333 h80 25.9 -> 22.1.
inline void ssd_slicing(const SsdCall* p, int wgs_per_cu, bool partials, int64_t* nslices, int64_t* hps) {
    const int64_t nc = ceil_div(p->seqlen, (int64_t)kQ);
    const int64_t hpg = p->nheads / p->ngroups;
    const int64_t base = p->batch * nc * p->ngroups;
    const int64_t cus = device_cus();
    const float whole = (float)(p->seqlen < kQ ? p->seqlen : kQ) / (float)kQ;      // how much of a chunk there is
    const float alone = 1.f - 0.25f * whole, fill = p->dtype == M2_F32 ? 0.75f + 0.75f * whole : 1.5f;
    int64_t best = 1;
    float least = 1e30f;
    each_slicing(hpg, [&](int64_t s, int64_t heads) {
        const float n = (float)ceil_div(base * s, cus), busy = n < (float)wgs_per_cu ? alone * (float)wgs_per_cu : n;
        const float cost = busy * (float)heads + fill * n + (partials ? 0.009f * (float)(base * s) : 0.f);
        if (cost <= least) { least = cost; best = s; }      // (of equals the shorter slices: forward at b1 l1525 h87 n64 39.7 us with the longer ones, 37.6)
    });
    *nslices = best;
    *hps = ceil_div(hpg, best);
}
constexpr int kWgsChunkState32 = 2, kWgsY = 2, kWgsY32 = 1, kWgsDx = 1, kWgsDg = 1;

// The same for the backward of fp32 operands, whose heads take 61 k cycles: in heads, rounds of workgroups x (heads
// per slice + one for the way in and the finish), and for more than one slice the partials' way out, back and through kernels of
// their own.
inline void ssd_slicing32(const SsdCall* p, int64_t* nslices, int64_t* hps) {
    const int64_t hpg = p->nheads / p->ngroups, base = p->batch * ceil_div(p->seqlen, (int64_t)kQ) * p->ngroups;
    int64_t best = 1;
    float least = 1e30f;
    each_slicing(hpg, [&](int64_t s, int64_t heads) {
        const float cost = (float)ceil_div(base * s, device_cus()) * ((float)heads + 1.f) + (s > 1 ? 1.f + 0.007f * (float)(base * s) : 0.f);
        if (cost < least) { least = cost; best = s; }
    });
    *nslices = best;
    *hps = ceil_div(hpg, best);
}

inline SsdWorkspace ssd_carve(const SsdCall* p, void* base, bool bwd, bool kept_only = false) {
    const int64_t nc = ceil_div(p->seqlen, (int64_t)kQ);
    const size_t esz = p->dtype == M2_F32 ? 4 : 2;
    const size_t tiles = (size_t)p->batch * nc * p->nheads * p->headdim * p->dstate;
    const size_t bhc = (size_t)p->batch * p->nheads * nc;
    size_t off = 0;
    SsdWorkspace w;
    unsigned char* b8 = static_cast<unsigned char*>(base);
    auto take = [&](size_t n) { unsigned char* r = b8 ? b8 + off : nullptr; off += align_up(n, 256); return r; };
    // per-chunk state contributions: only the fp32 path materialises them (16-bit operands take the fused state pass)
    if (p->dtype == M2_F32) w.local = reinterpret_cast<float*>(take(tiles * 4));
    // What the backward reuses from the forward: the state entering each chunk, the decay tables and the
    // per-(chunk, group) operand tiles.  They live in the caller's chunk_states buffer when one is given
    // (forward writes, backward reads), otherwise in the workspace (backward recomputes them).
    {
        size_t koff = 0;
        unsigned char* k8 = static_cast<unsigned char*>(p->chunk_states);
        auto keep = [&](size_t n) -> unsigned char* {
            if (!p->chunk_states && !kept_only) return take(n);
            unsigned char* r = k8 ? k8 + koff : nullptr;
            koff += align_up(n, 256);
            return r;
        };
        const size_t grp = (size_t)p->batch * nc * p->ngroups;
        w.prev = keep(tiles * esz);
        w.lam = reinterpret_cast<float*>(keep(bhc * 4));
        w.ldtab = reinterpret_cast<float*>(keep(bhc * 2 * kQ * 4));
        if (p->dtype != M2_F32) w.G = reinterpret_cast<float*>(keep(grp * kQ * kQ * 4));      // fp32 operands: Gm is G already
        w.Gm = keep(grp * kQ * kQ * esz);
        w.Gmt = keep(grp * kQ * kQ * esz);
        w.Bt = keep(grp * p->dstate * kQ * esz);
        if (p->dtype != M2_F32) w.Ct = keep(grp * p->dstate * kQ * esz);
        w.kept_bytes = koff;
    }
    // (a forward's size does not look at final_state: a caller may ask for it before there is one)
    if (p->dtype != M2_F32)
        if (const int64_t m = state_pass_seg_chunks(p->batch * p->nheads, nc, bwd ? kSegOneTile : p->chunk_states ? kSegKept : kSegPrompt)) {
            const size_t sums = (size_t)((ceil_div(nc, m) - 1) * p->batch * p->nheads);
            w.seg = take(sums * p->headdim * p->dstate * 4);
            w.seg_lam = reinterpret_cast<float*>(take(sums * 4));
        }
    if (bwd) {
        ssd_slicing(p, kWgsDg, true, &w.ns_g, &w.hps_g);
        ssd_slicing(p, kWgsDx, true, &w.ns_b, &w.hps_b);
        if (p->dtype == M2_F32) { ssd_slicing32(p, &w.ns_b, &w.hps_b); w.ns_g = w.ns_b; w.hps_g = w.hps_b; }      // one kernel for all three
        w.dprev = take(tiles * esz);
        // Only what a kernel writes: the 16-bit main kernel reads a single slice's dG where dg16_kernel left it, the fp32 one keeps it on
        // chip, and of one slice there is no sum (the 7B core, b2 l4096 h128 g8, had 100 MB for sums that nobody forms).
        const size_t groups = (size_t)p->batch * nc * p->ngroups, g_tile = groups * kQ * kQ * 4, n_tile = groups * kQ * p->dstate * 4;
        w.finished = w.ns_b == 1 && w.ns_g == 1;
        auto part = [&](bool need, size_t n) { return need ? reinterpret_cast<float*>(take(n)) : nullptr; };
        w.dGp = part(!w.finished || p->dtype != M2_F32, g_tile * w.ns_g);
        w.dBp = part(!w.finished, n_tile * w.ns_b);
        w.dCp = part(!w.finished, n_tile * w.ns_b);
        w.dGs = part(w.ns_g > 1, g_tile);
        w.dBs = part(w.ns_b > 1, n_tile);
        w.dCs = part(w.ns_b > 1, n_tile);
        w.dlam = reinterpret_cast<float*>(take(bhc * 4 * kDlamParts));
        w.dAp = reinterpret_cast<float*>(take(bhc * 4));
        w.dDp = reinterpret_cast<float*>(take(bhc * 4));
        w.dbp = reinterpret_cast<float*>(take(bhc * 4));
        w.dl = reinterpret_cast<float*>(take(bhc * kQ * 4));
        w.dlc = reinterpret_cast<float*>(take(bhc * kQ * 4));
        w.dirp = reinterpret_cast<float*>(take(bhc * kQ * 4));
        w.rbp = reinterpret_cast<float*>(take(bhc * kQ * 4));
        w.dDp8 = reinterpret_cast<float*>(take(bhc * 8 * 4));
    }
    w.bytes = off + 256;
    return w;
}

inline int ssd_check(const m2_ssd_params* p, const char* who) {
    M2_REQUIRE(p, M2_ERR_NULL, "%s: params is NULL", who);
    M2_REQUIRE(p->dtype == M2_F32 || p->dtype == M2_BF16, M2_ERR_DTYPE, "%s: bad dtype %d", who, p->dtype);
    M2_REQUIRE(p->dt_dtype == M2_F32 || p->dt_dtype == p->dtype, M2_ERR_DTYPE,
               "%s: dt dtype %d must be fp32 or the activation dtype", who, p->dt_dtype);
    M2_REQUIRE(p->batch >= 0 && p->seqlen >= 0 && p->nheads >= 0, M2_ERR_SHAPE, "%s: negative dimension", who);
    M2_REQUIRE(p->headdim == 64 || p->headdim == 128, M2_ERR_SHAPE, "%s: headdim %lld not in {64,128}", who, (long long)p->headdim);
    M2_REQUIRE(p->dstate == 64 || p->dstate == 128, M2_ERR_SHAPE, "%s: dstate %lld not in {64,128}", who, (long long)p->dstate);
    M2_REQUIRE(p->ngroups >= 1 && p->nheads % p->ngroups == 0, M2_ERR_SHAPE, "%s: nheads %lld not divisible by ngroups %lld", who,
               (long long)p->nheads, (long long)p->ngroups);
    M2_REQUIRE(p->batch <= 65535 && p->nheads <= 65535, M2_ERR_SHAPE, "%s: batch/nheads exceed the grid limit 65535", who);
    const int V = p->dtype == M2_F32 ? 4 : 8;
    M2_REQUIRE(p->x_stride_b % V == 0 && p->x_stride_l % V == 0 && p->x_stride_h % V == 0 &&
               p->B_stride_b % V == 0 && p->B_stride_l % V == 0 && p->B_stride_g % V == 0 &&
               p->C_stride_b % V == 0 && p->C_stride_l % V == 0 && p->C_stride_g % V == 0,
               M2_ERR_ALIGN, "%s: x/B/C strides must be multiples of %d elements (16 bytes)", who, V);
    M2_REQUIRE(aligned16(p->x) && aligned16(p->B) && aligned16(p->C), M2_ERR_ALIGN, "%s: x/B/C must be 16-byte aligned", who);
    {
        // the kernels address the rows of a chunk with 32-bit byte offsets formed by 24-bit multiplies
        const int64_t lim = (int64_t)1 << 21;
        auto ok = [&](int64_t s) { return s >= 0 && s < lim; };
        M2_REQUIRE(ok(p->x_stride_l) && ok(p->B_stride_l) && ok(p->C_stride_l) && ok(p->dt_stride_l) && (!p->y || ok(p->y_stride_l)),
                   M2_ERR_SHAPE, "%s: token strides must lie in [0, 2^21) elements", who);
        M2_REQUIRE(!p->dy || (ok(p->dy_stride_l) && ok(p->dx_stride_l) && ok(p->dB_stride_l) && ok(p->dC_stride_l) && ok(p->ddt_stride_l)),
                   M2_ERR_SHAPE, "%s: token strides of the gradients must lie in [0, 2^21) elements", who);
    }
    M2_REQUIRE(aligned16(p->chunk_states), M2_ERR_ALIGN, "%s: chunk_states must be 16-byte aligned", who);
    return M2_OK;
}

template <typename T>
inline size_t cb_smem(int n) {      // operand rows; 32 tokens of both to transpose; the waves' blocks on their way out
    const size_t a = (size_t)2 * 64 * lds_ld<T>(cb_kh<T>(n)) * sizeof(T), b = (size_t)2 * 32 * lds_ld<T>(n) * sizeof(T), o = (size_t)4 * 32 * 36 * 4;
    return a > b ? (a > o ? a : o) : (b > o ? b : o);
}

template <typename T, int P, int N, bool REVERSE, int HS, bool HILO>
inline int launch_state_pass16(StatePassArgs a, const SsdWorkspace& w, int64_t batch, int64_t seg_least, hipStream_t st) {
    auto launch = [&](auto k, size_t sm, int split, int64_t segs = 1) -> int {
        if (const int rc = allow_smem(k, sm)) return rc;
        k<<<dim3((unsigned)(a.nheads * split), (unsigned)batch, (unsigned)segs), state_pass_threads<N>(), sm, st>>>(a);
        return M2_OK;
    };
    const bool staged = state_pass_staged(a.init != nullptr, a.nchunks);
    if constexpr (N == 128 && !HILO)
        if (state_pass_split(batch * a.nheads, N) == 1)
            return staged ? launch(state_pass16_kernel<T, P, N, REVERSE, HS, HILO, 1, 0, true>, state_pass_smem<P, N, HILO, 1>(), 1) :
                            launch(state_pass16_kernel<T, P, N, REVERSE, HS, HILO, 1>, state_pass_smem<P, N, HILO, 1>(), 1);
    constexpr int SPLIT = kStatePassSplit;
    if (const int64_t m = state_pass_seg_chunks(batch * a.nheads, a.nchunks, seg_least)) {
        a.seg = static_cast<floatx4*>(w.seg); a.seg_lam = w.seg_lam; a.seg_chunks = m;
        const int64_t sums = ceil_div(a.nchunks, m) - 1;
        int rc = launch(state_pass16_kernel<T, P, N, REVERSE, HS, HILO, SPLIT, 1>, state_pass_smem<P, N, HILO, SPLIT>(), SPLIT, sums);
        if (!rc) rc = check_launch("ssd state_pass16_kernel, sums of segments");
        return rc ? rc : launch(state_pass16_kernel<T, P, N, REVERSE, HS, HILO, SPLIT, 2>, state_pass_smem<P, N, HILO, SPLIT>(), SPLIT, sums);
    }
    return staged ? launch(state_pass16_kernel<T, P, N, REVERSE, HS, HILO, SPLIT, 0, true>, state_pass_smem<P, N, HILO, SPLIT>(), SPLIT) :
                    launch(state_pass16_kernel<T, P, N, REVERSE, HS, HILO, SPLIT>, state_pass_smem<P, N, HILO, SPLIT>(), SPLIT);
}

// Local chunk states of fp32 operands: X = x, M = B, or (DSTATE) dy and C.
template <int N, bool DSTATE, int HS>
inline int launch_chunk_state32(const SsdCall* p, const SsdWorkspace& w, const void* X, int64_t X_sb, int64_t X_sl, int64_t X_sh, const void* M, int64_t M_sb,
                                int64_t M_sl, int64_t M_sg, hipStream_t st) {
    auto k = chunk_state32_kernel<N, DSTATE, HS>;
    if (const int rc = allow_smem(k, chunk_state32_smem<N>())) return rc;
    ChunkState32Args a;
    a.X = static_cast<const float*>(X); a.X_sb = X_sb; a.X_sl = X_sl; a.X_sh = X_sh;
    a.M = static_cast<const float*>(M); a.M_sb = M_sb; a.M_sl = M_sl; a.M_sg = M_sg;
    a.ldtab = w.ldtab; a.out = w.local;
    a.seqlen = p->seqlen; a.nheads = p->nheads; a.ngroups = p->ngroups; a.nchunks = ceil_div(p->seqlen, (int64_t)kQ);
    ssd_slicing(p, kWgsChunkState32, false, &a.nslices, &a.hps);
    M2_REQUIRE(p->ngroups * a.nslices <= 65535, M2_ERR_SHAPE, "ssd: too many group slices");
    k<<<dim3((unsigned)a.nchunks, (unsigned)(p->ngroups * a.nslices), (unsigned)p->batch), chunk_state32_threads<N>(), chunk_state32_smem<N>(), st>>>(a);
    return check_launch("ssd chunk_state32_kernel");
}

// Decay tables, G = C B^T (+ operand tiles), local chunk states, forward state scan.  Used by the forward and, when the
// caller did not keep the forward's chunk_states buffer, by the backward (recompute).  for_fwd, for_bwd: which of the operand
// tiles will be read.
template <typename T, int P, int N, int HS>
inline int ssd_launch_states(const SsdCall* p, const SsdWorkspace& w, float* final_out, bool for_fwd, bool for_bwd, hipStream_t st) {
    const int64_t nc = ceil_div(p->seqlen, (int64_t)kQ);
    const T* x = static_cast<const T*>(p->x);
    const T* Bm = static_cast<const T*>(p->B);
    const T* Cm = static_cast<const T*>(p->C);
    const int dt_f32 = p->dt_dtype == M2_F32;
    int rc;
    {
        // decay tables and G = C B^T (+ operand tiles), one launch
        auto k = prep_kernel<T, N>;
        const size_t sm = cb_smem<T>(N);
        if ((rc = allow_smem(k, sm))) return rc;
        PrepArgs pa;
        pa.Bm = Bm; pa.Cm = Cm; pa.Bt = sizeof(T) == 2 || for_bwd ? w.Bt : nullptr; pa.parts = pa.Bt ? kCbParts : kCbGParts;
        pa.Gf = for_bwd ? w.G : nullptr; pa.Gmt = for_bwd ? w.Gmt : nullptr; pa.Ct = for_bwd && sizeof(T) == 2 ? w.Ct : nullptr;
        pa.Gm = for_fwd || sizeof(T) == 4 ? w.Gm : nullptr;
        pa.Bsb = p->B_stride_b; pa.Bsl = p->B_stride_l; pa.Bsg = p->B_stride_g;
        pa.Csb = p->C_stride_b; pa.Csl = p->C_stride_l; pa.Csg = p->C_stride_g;
        pa.dt = p->dt; pa.dt_f32 = dt_f32; pa.dt_bias = p->dt_bias; pa.A = p->A; pa.ldtab = w.ldtab; pa.lam = w.lam;
        pa.dtsb = p->dt_stride_b; pa.dtsl = p->dt_stride_l;
        pa.seqlen = p->seqlen; pa.nheads = p->true_heads; pa.hs = p->hs; pa.ngroups = p->ngroups; pa.nchunks = nc;
        pa.n_cb = nc * p->ngroups * p->batch;
        const int64_t blocks = cb_blocks(pa.n_cb, pa.parts) + ld_table_blocks(p->batch, p->true_heads, nc);
        M2_REQUIRE(blocks < ((int64_t)1 << 31), M2_ERR_SHAPE, "ssd: too many workgroups");
        k<<<(unsigned)blocks, 256, sm, st>>>(pa);
        if ((rc = check_launch("ssd prep_kernel"))) return rc;
    }
    if constexpr (sizeof(T) == 2) {
        // 16-bit operands: contributions and recurrence in one pass, running state in registers
        // a caller that wants the final state (an fp32 output) gets the two-tile form, whose operand rounding is 2^-17
        // (3.7 us more per pass at b4 l2048 h80; the states entering the chunks come out of the same accumulators, so y
        // differs from the one-tile form in the last bit here and there)
        const bool hilo = final_out != nullptr;
        StatePassArgs sa{};
        sa.X = x; sa.X_sb = p->x_stride_b; sa.X_sl = p->x_stride_l; sa.X_sh = p->x_stride_h;
        sa.ldtab = w.ldtab; sa.Mt = w.Bt; sa.init = p->initial_state; sa.prev = w.prev; sa.final_out = final_out;
        sa.seqlen = p->seqlen; sa.nheads = p->nheads; sa.ngroups = p->ngroups; sa.nchunks = nc;
        rc = hilo ? launch_state_pass16<T, P, N, false, HS, true>(sa, w, p->batch, p->chunk_states ? kSegKept : kSegPrompt, st) :
                    launch_state_pass16<T, P, N, false, HS, false>(sa, w, p->batch, kSegOneTile, st);
        if (rc) return rc;
        return check_launch("ssd state_pass16_kernel");
    } else {
        // fp32 operands: per-chunk contributions (workspace), then the recurrence over the chunks
        if ((rc = launch_chunk_state32<N, false, HS>(p, w, p->x, p->x_stride_b, p->x_stride_l, p->x_stride_h, Bm, p->B_stride_b, p->B_stride_l, p->B_stride_g, st))) return rc;
        state_scan_kernel<P * N, false><<<dim3((unsigned)p->nheads, (unsigned)p->batch, kScanSplit), 256, 0, st>>>(
            w.local, w.lam, p->initial_state, static_cast<float*>(w.prev), final_out, p->nheads, nc);
        if ((rc = check_launch("ssd state_scan_kernel"))) return rc;
        return M2_OK;
    }
}

#define M2_DISPATCH_N_HS(p, N, HS, ...)                                                                                   \
    do {                                                                                                                  \
        if ((p)->dstate == 64 && (p)->hs == 0) { constexpr int N = 64, HS = 0; __VA_ARGS__; }                             \
        else if ((p)->dstate == 64) { constexpr int N = 64, HS = 1; __VA_ARGS__; }                                        \
        else if ((p)->hs == 0) { constexpr int N = 128, HS = 0; __VA_ARGS__; }                                            \
        else { constexpr int N = 128, HS = 1; __VA_ARGS__; }                                                              \
    } while (0)

}  // namespace m2
