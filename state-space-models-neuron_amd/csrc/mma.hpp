// MFMA tile helpers for gfx950 (CDNA4, 64-lane wavefronts).
//
// All SSD contractions are expressed as  OUT[m][n] += sum_k A[m][k] * Bt[n][k]  with BOTH
// operands staged in LDS with k contiguous, so every lane fetches its MFMA fragment with one
// 16-byte ds_read (bf16) and the two operands use the same code path.
//
//   bf16: v_mfma_f32_32x32x16_bf16   lane -> row (lane & 31), k = 8 * (lane >> 5) + 0..7
//   fp32: v_mfma_f32_32x32x2_f32     eight steps per 16 k, same lane -> (row, k) assignment (see Frag)
//   accumulator (both): 16 floats per lane; register v of lane holds
//        column  (lane & 31),   row  8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)
#pragma once
#include "common.hpp"

namespace m2 {

constexpr int kQ = M2_CHUNK;   // 128 tokens per chunk
constexpr int kP = 64;         // channels of a head as the SSD kernels see it

// A head of 128 channels is two kernel heads of 64 (HS = 1): they share dt, A, D, B and C, their states and channels lie one
// behind the other, and every per-head sum is linear in the channels, so only the final sums (da_body) know of the pair.
// Element offset of kernel head h in a tensor whose true heads are `sh` elements apart.  (A template argument, not a value:
// one more scalar per tensor in the head loops sends kernel arguments back to memory, and their reloads wait for the LDS
// traffic around them: 340 -> 347 us for forward + backward at b4 l2048 h80.)
template <int HS>
__device__ __forceinline__ int64_t head_off(int64_t h, int64_t sh) { return HS ? (h >> 1) * sh + (h & 1) * kP : h * sh; }

// Heads of a slice of a group's: `most`, and in the last slice what is left of them.
__device__ __forceinline__ int64_t slice_heads(int64_t hpg, int64_t slice, int64_t most) {
    const int64_t left = hpg - slice * most;
    return left < most ? left : most;
}

template <typename T> struct MmaTraits;
template <> struct MmaTraits<bf16_t> { static constexpr int kPad = 8; };
template <> struct MmaTraits<float> { static constexpr int kPad = 4; };

// leading dimension (elements) of an LDS tile with `k` contiguous columns; the pad keeps
// 16-byte alignment of every row and spreads rows over banks.
template <typename T> __host__ __device__ constexpr int lds_ld(int k) { return k + MmaTraits<T>::kPad; }

__device__ __forceinline__ int acc_row(int lane, int v) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }
__device__ __forceinline__ int acc_col(int lane) { return lane & 31; }

template <int BM, int BN>
__device__ __forceinline__ void acc_zero(floatx16 (&acc)[BM][BN]) {
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
}

// A fragment is the slice of an MFMA operand one lane owns for a 16-wide k step: 8 CONSECUTIVE k values,
// k = k0 + 8 * (lane >> 5) + 0..7, of row (lane & 31).  For bf16 this is the register layout of
// v_mfma_f32_32x32x16_bf16.  For fp32 the same 8 values are fed to eight v_mfma_f32_32x32x2_f32 (element s of
// both operands in step s); the hardware would pair k = 2s + (lane >> 5), but a contraction does not care in
// which order k is visited as long as A and B agree, and the contiguous form needs two 16-byte reads
// instead of eight scalar ones.
template <typename T> struct Frag;
template <> struct Frag<bf16_t> { bf16x8 v; };
template <> struct Frag<float> { float v[8]; };

__device__ __forceinline__ Frag<bf16_t> load_frag(const bf16_t* __restrict__ p) {
    Frag<bf16_t> f;
    f.v = *reinterpret_cast<const bf16x8*>(p);
    return f;
}
__device__ __forceinline__ Frag<float> load_frag(const float* __restrict__ p) {
    Frag<float> f;
    const floatx4 a = *reinterpret_cast<const floatx4*>(p), b = *reinterpret_cast<const floatx4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { f.v[i] = a[i]; f.v[4 + i] = b[i]; }
    return f;
}
__device__ __forceinline__ void mma_frag(floatx16& acc, const Frag<bf16_t>& a, const Frag<bf16_t>& b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, b.v, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma_frag(floatx16& acc, const Frag<float>& a, const Frag<float>& b) {
#pragma unroll
    for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[s], b.v[s], acc, 0, 0, 0);
}
// element-wise scale of a fragment by 8 fp32 factors (one per k), result rounded to the operand type
__device__ __forceinline__ Frag<bf16_t> scale_frag(const Frag<bf16_t>& a, const float (&f)[8]) {
    Frag<bf16_t> r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r.v[i] = (bf16_t)((float)a.v[i] * f[i]);
    return r;
}

// the two 16-bit elements of a 32-bit word as fp32, and back (round to nearest even)
template <typename T> __device__ __forceinline__ float unpack_lo(uint32_t w);
template <typename T> __device__ __forceinline__ float unpack_hi(uint32_t w);
template <> __device__ __forceinline__ float unpack_lo<bf16_t>(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
template <> __device__ __forceinline__ float unpack_hi<bf16_t>(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
// c + a.lo * b.lo + a.hi * b.hi for two words of 16-bit pairs in one instruction (v_dot2c_f32_bf16): the products of two
// 8-bit significands are exact in fp32, so this is the same sum as two FMAs on unpacked values, without the four unpacks
template <typename T> __device__ __forceinline__ float dot2_acc(uint32_t a, uint32_t b, float c);
template <> __device__ __forceinline__ float dot2_acc<bf16_t>(uint32_t a, uint32_t b, float c) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, a), __builtin_bit_cast(bf2, b), c, false);
}
template <typename T> __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef T tvec2 __attribute__((ext_vector_type(2)));
    const tvec2 v = {from_f32<T>(lo), from_f32<T>(hi)};
    return __builtin_bit_cast(uint32_t, v);
}

// Lane-pair exchange (lanes l and l + 32): lo = { own a | partner's b }, hi = { partner's a | own b } for the lower | upper
// half of the wave (v_permlane32_swap).  With the transposed 32x32 accumulator layout (a lane and its partner hold the two
// halves of each 8-element group of one row) this leaves every lane with whole groups of 8 consecutive elements.
// (The scalars are passed by value on purpose: a bit cast applied directly to a vector element reads element 0.)
__device__ __forceinline__ void pair_swap(uint32_t a, uint32_t b, uint32_t& lo, uint32_t& hi) {
    const auto sw = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    lo = sw[0];
    hi = sw[1];
}
__device__ __forceinline__ void pair_swap(float a, float b, float& lo, float& hi) {
    const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
    const auto sw = __builtin_amdgcn_permlane32_swap(ua, ub, false, false);
    const uint32_t r0 = sw[0], r1 = sw[1];
    lo = __builtin_bit_cast(float, r0);
    hi = __builtin_bit_cast(float, r1);
}

// Makes a fragment opaque to the optimiser at this point (no instruction is emitted).  Used on loop-invariant
// fragments that are re-scaled inside a loop: without it the bf16 -> fp32 unpacking of the fragment is hoisted out of
// the loop and the fragment then occupies eight fp32 registers instead of four packed ones for the whole loop.
__device__ __forceinline__ void keep_packed(Frag<bf16_t>& f) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 raw = __builtin_bit_cast(u32x4, f.v);
    asm volatile("" : "+v"(raw));
    f.v = __builtin_bit_cast(bf16x8, raw);
}

// One wave: acc[i][j] (32x32 blocks) += A[rows i*32.., k0:k1] * Bt[rows j*32.., k0:k1]^T, operands in LDS.
// A points at the first of this wave's BM*32 rows, Bt at the first of its BN*32 rows.  k0, k1 multiples of 16.
template <int BM, int BN, typename T>
__device__ __forceinline__ void wave_mma(floatx16 (&acc)[BM][BN], const T* __restrict__ A, int lda,
                                         const T* __restrict__ Bt, int ldb, int k0, int k1) {
    const int lane = threadIdx.x & 63;
    const int r = lane & 31, kh = (lane >> 5) * 8;
    for (int k = k0; k < k1; k += 16) {
        Frag<T> a[BM], b[BN];
#pragma unroll
        for (int i = 0; i < BM; ++i) a[i] = load_frag(A + (i * 32 + r) * lda + k + kh);
#pragma unroll
        for (int j = 0; j < BN; ++j) b[j] = load_frag(Bt + (j * 32 + r) * ldb + k + kh);
#pragma unroll
        for (int i = 0; i < BM; ++i)
#pragma unroll
            for (int j = 0; j < BN; ++j) mma_frag(acc[i][j], a[i], b[j]);
    }
}

// ------------------------------------------------------------------------------------------
// Cooperative staging, global -> LDS.  NT threads; `tid` in [0, NT).
//
// StagedRows: global tile [ROWS][COLS] (COLS contiguous, row stride gstride) -> LDS [ROWS][ld], rows >= valid zero-filled: load() and
// put(), so that the loads of several tiles are under way together.  Rows past the end read the last one there is (valid may be
// negative: that row then lies in front of the tile), so that no branch stands in front of a load: with one, each of a thread's eight
// loads of two tiles waited for the one before it.
template <typename T, int ROWS, int COLS, int NT>
struct StagedRows {
    static constexpr int V = VecTraits<T>::kVec, VPR = COLS / V, PER = ROWS * VPR / NT;
    static_assert(COLS % V == 0 && ROWS * VPR % NT == 0, "whole vectors, the same many per thread");
    uint4 raw[PER];
    __device__ __forceinline__ void load(const T* __restrict__ g, int64_t gstride, int valid, int tid) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = i * NT + tid, r = e / VPR, cv = e % VPR;
            raw[i] = *reinterpret_cast<const uint4*>(g + (int64_t)(r < valid ? r : valid - 1) * gstride + cv * V);
        }
    }
    __device__ __forceinline__ void put(T* __restrict__ s, int ld, int valid, int tid) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = i * NT + tid, r = e / VPR, cv = e % VPR;
            *reinterpret_cast<uint4*>(s + r * ld + cv * V) = r < valid ? raw[i] : uint4{0u, 0u, 0u, 0u};
        }
    }
};

// Sum of v over the 32 lanes that share (lane >> 5), for 16 values at once (the 16 accumulator rows of a lane),
// by a butterfly reduce-scatter: 16 cross-lane moves instead of 80 (the widest step selects and adds with one row swap, the
// single-move DPP steps fold into their additions: 45 instructions, not 85, in kernels bound by their vector instructions).  On return every lane holds ONE total:
// that of register index  r = 8*b4 + 4*b3 + 2*b2 + b1  (b_k = bit k of lane), i.e. of accumulator row
// acc_row(lane, r); lanes differing only in bit 0 hold the same total.
__device__ __forceinline__ float half_wave_reduce16(float (&v)[16], int* reg_index) {
    const int lane = threadIdx.x & 63;
    const bool b4 = lane & 16, b3 = lane & 8, b2 = lane & 4, b1 = lane & 2;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        // the row swap leaves the pair's two halves of v[k] in the lanes with b4 = 0, of v[k + 8] in the others
        const auto sw = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v[k]), __builtin_bit_cast(uint32_t, v[k + 8]), false, false);
        const uint32_t r0 = sw[0], r1 = sw[1];
        v[k] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float keep = b3 ? v[k + 4] : v[k], send = b3 ? v[k] : v[k + 4];
        v[k] = keep + lane_xor<8>(send);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float keep = b2 ? v[k + 2] : v[k], send = b2 ? v[k] : v[k + 2];
        v[k] = keep + lane_xor<4>(send);
    }
    {
        const float keep = b1 ? v[1] : v[0], send = b1 ? v[0] : v[1];
        v[0] = keep + lane_xor<2>(send);
    }
    v[0] = lane_xor_add<1>(v[0]);
    *reg_index = (b4 ? 8 : 0) + (b3 ? 4 : 0) + (b2 ? 2 : 0) + (b1 ? 1 : 0);
    return v[0];
}

// Inclusive sum over the lanes of a wave in six DPP additions: row shifts inside the rows of 16 lanes, then the last lane of
// row 0 (2) broadcast to row 1 (3), and lane 31 to the upper half.  All 64 lanes must be active.
__device__ __forceinline__ float wave_scan(float x) {
    x += dpp_from<0x111, 0xF>(x); x += dpp_from<0x112, 0xF>(x); x += dpp_from<0x114, 0xF>(x); x += dpp_from<0x118, 0xF>(x);      // row_shr
    x += dpp_from<0x142, 0xA>(x);      // row_bcast:15
    x += dpp_from<0x143, 0xC>(x);      // row_bcast:31
    return x;
}
// The same over each half of a wave
__device__ __forceinline__ float half_wave_scan(float x) {
    x += dpp_from<0x111, 0xF>(x); x += dpp_from<0x112, 0xF>(x); x += dpp_from<0x114, 0xF>(x); x += dpp_from<0x118, 0xF>(x);      // row_shr
    x += dpp_from<0x142, 0xA>(x);      // row_bcast:15
    return x;
}
// l[t] = sum_{s <= t} A d[s] over a chunk, lane holding tokens `lane` and `lane + 64`
__device__ __forceinline__ void wave_cumsum_from(float A, float d0, float d1, float& l0, float& l1) {
    l0 = wave_scan(A * d0); l1 = wave_scan(A * d1);
    l1 += __shfl(l0, 63, 64);
}

// Orders this wave's LDS writes before its later LDS reads of what OTHER lanes of the same wave wrote
// (wave-private staging buffers).  The hardware executes one wave's LDS operations in order; the fences
// keep the compiler from reordering them.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace m2
