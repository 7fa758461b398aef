// Matrix products of a layer's projections on few tokens (bf16 operands, fp32 accumulation), in the three forms that a linear
// layer's forward and backward need:
//   out[m][n] = sum_k A(m, k) B(n, k) (+ bias[n]),   A stored [M][K] (k contiguous) or [K][M], B stored [N][K] or [K][N]
//
// What bounds them at a few hundred tokens is not the matrix cores: it is how many bytes are in flight (the weights are read
// once, by few workgroups with short k loops) and, on the host, the call itself.  Hence small tiles -- 64 x 64, so that 500
// tokens make a few hundred workgroups --, a ring of four k tiles that asynchronous copies fill three ahead, and one barrier
// per tile of 64 k.
//
// A workgroup's four waves split each k tile (wave w takes its k step w): a wave then feeds four products from two fragments of
// either operand, where a quarter of the tile per wave would read each fragment for a single product and be bound by LDS
// reads (256 bytes a clock needed, 128 there).  The four partial tiles meet once, in LDS, at the end; the rows leave in
// 16-byte stores.  Fragments of an operand with k contiguous are row reads, of one with k strided LDS transpose reads: both
// operands stay in LDS as they lie in memory.
// Where the tiles are too few for the chip, k is split over workgroups too: fp32 partials, and a second kernel sums them.
#include <type_traits>

#include "ssd_y.hpp"

namespace m2 {
namespace {

constexpr int kK = 64, kRing = 4;      // k tile, tiles in the ring

struct ProductArgs {
    const bf16_t* A; const bf16_t* B; const bf16_t* bias; bf16_t* out; float* part;
    int64_t lda, ldb, ldo;
    int M, N, K, tiles_m, tiles_n, splits, ksteps;      // ksteps: k tiles per split
};

// Source of one wave-wide copy of an operand tile of R rows or columns: the 16-byte piece of lane s % 64 of 1 KiB chunk s / 64.
template <bool KC, int R>
struct Piece {
    static constexpr int SPR = KC ? 8 : R / 8;      // slots per tile row: 64 k, or R columns
    uint32_t a, b;       // KC: row offset, piece offset inside the row's 128 bytes; otherwise: k row, column offset (bytes)
    __device__ void set(int s, int r0, int rows, int64_t ld) {
        const int row = s / SPR, cs = (s % SPR) ^ tile_swz<SPR>(row);
        if (KC) { a = (uint32_t)((int64_t)(r0 + row < rows ? r0 + row : rows - 1) * ld * 2); b = (uint32_t)cs * 16u; }
        else { a = (uint32_t)row; b = (uint32_t)(r0 + cs * 8 < rows - 8 ? r0 + cs * 8 : rows - 8) * 2u; }
    }
    // byte offset from the k tile's base with `left` k's left; past the end the last ones again (they meet zeros, see below)
    __device__ uint32_t at(int left, uint32_t ld2) const {
        if (KC) { const uint32_t last = (uint32_t)(left * 2 - 16); return a + (left < kK && b > last ? last : b); }
        return (left < kK && a > (uint32_t)(left - 1) ? (uint32_t)(left - 1) : a) * ld2 + b;
    }
};

// k step ks (16 k) of rows or columns r0 .. r0 + 31 of an operand tile
template <bool KC, int R>
__device__ __forceinline__ Frag<bf16_t> tile_frag(const bf16_t* t, int r0, int ks) {
    const int lane = threadIdx.x & 63, half = lane >> 5;
    if (KC) {
        const int row = r0 + (lane & 31);
        return load_frag(t + (row * 8 + ((ks * 2 + half) ^ tile_swz<8>(row))) * 8);
    }
    constexpr int SPR = R / 8;
    typedef bf16_t tvec4 __attribute__((ext_vector_type(4)));
    const int k = ks * 16 + 8 * half + ((lane >> 2) & 3), col = r0 + ((lane >> 4) & 1) * 16 + 4 * (lane & 3);
    const tvec4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((M2_LDS tvec4*)(t + (k * SPR + ((col >> 3) ^ tile_swz<SPR>(k))) * 8 + (col & 7)));
    const tvec4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((M2_LDS tvec4*)(t + ((k + 4) * SPR + ((col >> 3) ^ tile_swz<SPR>(k + 4))) * 8 + (col & 7)));
    Frag<bf16_t> f;
#pragma unroll
    for (int e = 0; e < 4; ++e) { f.v[e] = lo[e]; f.v[4 + e] = hi[e]; }
    return f;
}

// Workgroup `block` of `blocks` (a multiple of 8, and block 0 on the first XCD) of a product.
template <bool AK, bool BK, int R>
__device__ __forceinline__ void product_body(const ProductArgs& p, unsigned block, unsigned blocks) {
    static_assert(R == 64 || R == 128, "tiles of 64 x 64 or 128 x 128");
    constexpr bool KSPLIT = R == 64;                               // the waves split k, else the tile
    constexpr int kElems = R * kK, NP = R / 32, PER = 2 * NP;      // an operand tile; copies per wave of one operand, of both
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    bf16_t* ring = reinterpret_cast<bf16_t*>(smem_raw);            // [kRing][ A tile | B tile ]
    float* red = reinterpret_cast<float*>(smem_raw);               // [KSPLIT ? 4 : 1][R][R], after the last k tile
    const int lane = threadIdx.x & 63, wave = (int)uniform(threadIdx.x >> 6), half = lane >> 5;
    // Each XCD gets an eighth of the (split, column of tiles, row tile) triples in that order: the row tiles of one column follow one
    // another on it, and its L2 hands them the same rows of B.  Whole columns dealt round the XCDs instead left some with half as much
    // again as others, and two rounds where one would do (20 columns of 3 tiles, four splits: 36 workgroups on the 32 CUs of half of
    // them): 257 x 2560 x 10576 63 -> 39 us, 737 x 1792 x 7480 65 -> 40, 1326 x 2560 x 10576 216 -> 120.
    const int tiles = p.tiles_m * p.tiles_n, at = (int)((block & 7) * (blocks >> 3) + (block >> 3));
    if (at >= tiles * p.splits) return;
    const int split = at / tiles, tn = (at - split * tiles) / p.tiles_m, tm = (at - split * tiles) % p.tiles_m;
    const int m0 = tm * R, n0 = tn * R;
    const int k_first = split * p.ksteps * kK;
    const int steps = min(p.ksteps, (p.K - k_first + kK - 1) / kK);

    Piece<AK, R> pa[NP];
    Piece<BK, R> pb[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        pa[i].set((wave * NP + i) * 64 + lane, m0, p.M, p.lda);
        pb[i].set((wave * NP + i) * 64 + lane, n0, p.N, p.ldb);
    }
    const uint32_t lds = uniform(lds_addr_of(ring)), lda2 = (uint32_t)(p.lda * 2), ldb2 = (uint32_t)(p.ldb * 2);
    auto issue = [&](int t) {
        const int k = k_first + t * kK, left = p.K - k;
        const bf16_t* ga = p.A + (AK ? (int64_t)k : k * p.lda);
        const bf16_t* gb = p.B + (BK ? (int64_t)k : k * p.ldb);
        const uint32_t dst = lds + (uint32_t)((t % kRing) * 2 * kElems * 2) + (uint32_t)(wave * NP) * 1024u;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            async_copy16(ga, pa[i].at(left, lda2), dst + i * 1024u);
            async_copy16(gb, pb[i].at(left, ldb2), dst + kElems * 2u + i * 1024u);
        }
    };
#pragma unroll
    for (int t = 0; t < kRing - 1; ++t)
        if (t < steps) issue(t);

    const int wm = KSPLIT ? 0 : (wave >> 1) * 64, wn = KSPLIT ? 0 : (wave & 1) * 64;      // this wave's 64 x 64 part
    floatx16 acc[2][2];      // the transposed blocks: lane holds row m = lane & 31, register v column n = acc_row(lane, v)
    acc_zero(acc);
    for (int t = 0; t < steps; ++t) {
        wait_vmem_keep<PER>(min(steps - 1 - t, kRing - 2));
        __syncthreads();          // the tile is there, and everyone is done with the one before it
        if (t + kRing - 1 < steps) issue(t + kRing - 1);
        const bf16_t* ta = ring + (t % kRing) * 2 * kElems;
        const bf16_t* tb = ta + kElems;
        // all fragments of the k tile first: a read issued next to its products would put an LDS round trip between any two groups
        constexpr int NK = KSPLIT ? 1 : 4;
        Frag<bf16_t> a[NK][2], b[NK][2];
#pragma unroll
        for (int kk = 0; kk < NK; ++kk)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[kk][i] = tile_frag<AK, R>(ta, wm + i * 32, KSPLIT ? wave : kk);
                b[kk][i] = tile_frag<BK, R>(tb, wn + i * 32, KSPLIT ? wave : kk);
            }
        if (k_first + (t + 1) * kK > p.K) {      // the last k tile: nothing past the end
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) {
                const int k0 = k_first + t * kK + (KSPLIT ? wave : kk) * 16 + 8 * half;
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        a[kk][i].v[e] = k0 + e < p.K ? a[kk][i].v[e] : (bf16_t)0.f;
                        b[kk][i].v[e] = k0 + e < p.K ? b[kk][i].v[e] : (bf16_t)0.f;
                    }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < NK; ++kk)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) mma_frag(acc[i][j], b[kk][j], a[kk][i]);
    }
    __syncthreads();
    // the tile (or its four partial ones); groups of four columns swizzled by the row, so that rows spread over the banks
    float* mine = red + (KSPLIT ? wave * R * R : 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int m = wm + i * 32 + (lane & 31), g4 = wn / 4 + j * 8 + 2 * q + half;
                const floatx4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                *reinterpret_cast<floatx4*>(mine + m * R + ((g4 ^ (m & 15)) * 4)) = v;
            }
    __syncthreads();
    constexpr int LPR = R / 8, RPI = 64 / LPR;      // lanes per row of 8-column pieces, rows per iteration
#pragma unroll 2
    for (int it = 0; it < R / 4 / RPI; ++it) {
        const int m = wave * (R / 4) + it * RPI + lane / LPR, c = lane % LPR;
        floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int w = 0; w < (KSPLIT ? 4 : 1); ++w) {
            s0 += *reinterpret_cast<const floatx4*>(red + w * R * R + m * R + (((2 * c) ^ (m & 15)) * 4));
            s1 += *reinterpret_cast<const floatx4*>(red + w * R * R + m * R + (((2 * c + 1) ^ (m & 15)) * 4));
        }
        const int row = m0 + m, col = n0 + c * 8;
        if (row >= p.M || col >= p.N) continue;
        if (p.part) {
            float* o = p.part + ((int64_t)split * p.M + row) * p.N + col;
            *reinterpret_cast<floatx4*>(o) = s0;
            *reinterpret_cast<floatx4*>(o + 4) = s1;
        } else {
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[e] = s0[e]; v[4 + e] = s1[e]; }
            if (p.bias) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += to_f32(p.bias[col + e]);
            }
            store16(p.out + row * p.ldo + col, v);
        }
    }
}

template <bool AK, bool BK, int R>
__global__ void __launch_bounds__(256, R == 64 ? 2 : 1)
product_kernel(const ProductArgs p) { product_body<AK, BK, R>(p, blockIdx.x, gridDim.x); }

// Both products of a linear layer's backward in one launch: dx = dy W (x) and dW = dy^T x (w), in tiles of 64.  On a few hundred tokens
// either alone leaves half of the chip to wait through its prologue and its last tile (4.6 us of the 7 to 15 that it takes).  The
// workgroups with the longer sums go first.  500 tokens,
// 768 channels: out_proj's 13.8 -> 8.4 us, in_proj's (dx split in two) 24.8 -> 18.6.
__global__ void __launch_bounds__(256, 2)
product_pair_kernel(const ProductArgs x, const ProductArgs w, unsigned x_blocks, unsigned w_blocks, int x_first) {
    const unsigned first = x_first ? x_blocks : w_blocks;
    const bool is_x = (blockIdx.x < first) == (x_first != 0);
    const unsigned block = blockIdx.x < first ? blockIdx.x : blockIdx.x - first;
    if (is_x) product_body<true, false, 64>(x, block, x_blocks);
    else product_body<false, false, 64>(w, block, w_blocks);
}

__global__ void __launch_bounds__(256)
product_sum_kernel(const float* __restrict__ part, const bf16_t* __restrict__ bias, bf16_t* __restrict__ out, int64_t ldo, int M, int N, int splits) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x, n8 = N / 8;
    if (idx >= M * n8) return;
    const int64_t row = idx / n8, col = idx % n8 * 8;
    floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
    for (int s = 0; s < splits; ++s) {
        const float* q = part + ((int64_t)s * M + row) * N + col;
        s0 += *reinterpret_cast<const floatx4*>(q);
        s1 += *reinterpret_cast<const floatx4*>(q + 4);
    }
    float v[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[e] = s0[e]; v[4 + e] = s1[e]; }
    if (bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += to_f32(bias[col + e]);
    }
    store16(out + row * ldo + col, v);
}

// Tile size and number of k splits: the cheapest of a count of k steps on the busiest CU (of the XCDs' equal shares), in microseconds as
// fitted to 144 products of layers of 256 to 3072 channels over 33 to 2048 tokens, in all forms (the choice is within 1 % of the best of
// tiles and one to six splits there on average, within 20 % for all).  Two workgroups of the small tile share a CU and hide each
// other's waits; a split costs its second launch and the partials' way out and back.
struct ProductPlan { int r, splits, ksteps; float us; };
ProductPlan product_plan(int64_t M, int64_t N, int64_t K) {
    const int64_t cus = device_cus() / 8, ktiles = ceil_div(K, (int64_t)kK);
    ProductPlan best{64, 1, (int)ktiles, 1e30f};
    for (const int r : {64, 128}) {
        const int64_t tiles = ceil_div(M, (int64_t)r) * ceil_div(N, (int64_t)r);
        for (int64_t want = 1; want <= 6 && (want == 1 || ktiles / want >= 4); ++want) {
            const int64_t ks = ceil_div(ktiles, want), s = ceil_div(ktiles, ks), busiest = ceil_div(ceil_div(tiles * s, (int64_t)8), cus);
            float us = r == 64 ? (float)ks * 0.3f * (1.6f * (busiest / 2) + busiest % 2) + 1.2f * ceil_div(busiest, (int64_t)2)
                               : (float)busiest * (ks * 0.54f + 1.8f);
            if (s > 1) us += 1.6f + 3e-6f * s * M * N;
            if (us < best.us) best = {r, (int)s, (int)ks, us};
        }
    }
    return best;
}

// Both products of a linear layer's backward in one launch, in the same count: the longer chain of k steps (0.36 us each beside the other
// product's), or all of them at the rate of CUs with two workgroups each.  Only dx's sum, over the layer's outputs, is split.
struct PairPlan { int splits, ksteps; float us, work, dw_chain; };      // work: k steps per CU; dw_chain: us of dW's sum over the tokens
PairPlan pair_plan(const m2_product_params& x, const m2_product_params& w) {
    const int64_t kx = ceil_div(x.K, (int64_t)kK), kw = ceil_div(w.K, (int64_t)kK);
    const int64_t tx = ceil_div(x.M, (int64_t)64) * ceil_div(x.N, (int64_t)64), tw = ceil_div(w.M, (int64_t)64) * ceil_div(w.N, (int64_t)64);
    const float work = (float)(tx * kx + tw * kw) / (float)device_cus();
    const float dw_chain = 0.36f * (float)kw;
    PairPlan best{1, (int)kx, 1e30f, work, dw_chain};
    for (int64_t want = 1; want <= 6 && (want == 1 || kx / want >= 4); ++want) {
        const int64_t ks = ceil_div(kx, want), n = ceil_div(kx, ks);
        const float dx_chain = 0.36f * (float)ks, chain = dx_chain > dw_chain ? dx_chain : dw_chain;
        const float us = (chain > 0.24f * work ? chain : 0.24f * work) + 1.2f + (n > 1 ? 1.6f + 3e-6f * (float)(n * x.M * x.N) : 0.f);
        if (us < best.us) best = {(int)n, (int)ks, us, work, dw_chain};
    }
    return best;
}

}  // namespace
}  // namespace m2

extern "C" int m2_product_fits(int64_t M, int64_t N, int64_t K, int32_t a_k, int32_t b_k) {
    if (M < 1 || N < 8 || K < 1 || N % 8 || M > (1 << 24) || N > (1 << 24) || K > (1 << 24)) return 0;
    if ((a_k || b_k) && K % 8) return 0;
    if (!a_k && M % 8) return 0;
    return 1;
}

// Where these kernels are ahead of the general library's product with its default solution (bf16, by size; its call also costs the
// host 18 us to their 4).  Solutions chosen by timing are another matter: at 128 rows of a 2560-channel layer they are ahead, so a
// program that has them chosen keeps its products there (library_is_tuned in binding.cpp).
//   weight gradients (k = tokens) with few outputs -- 768 x 3352 x 768: 13.7 -> 12.9 us, 1024 x 2048 x 1536: 16.5 -> 14.0; with ten
//   million outputs the stores bound both and the library's are better (200 tokens, 10576 x 2560: 35 us to 46);
//   other products up to 4e9 multiply-adds -- 200 x 2560 x 5120: 25.6 -> 20.1 us, 360 x 4384 x 1024: 11.4 -> 9.5; beyond, its larger
//   tiles reuse more (512 x 10576 x 2560: 39 us to 57);
//   long sums for few outputs, where it does not split k -- 512 x 2560 x 10576: 108 -> 52 us, 200 tokens: 69 -> 32.
extern "C" int m2_product_pays(int64_t M, int64_t N, int64_t K, int32_t a_k, int32_t b_k) {
    if (!m2_product_fits(M, N, K, a_k, b_k)) return 0;
    const int64_t outputs = M * N, macs = outputs * K;
    if (!a_k) return outputs <= 4000000 && macs <= 8000000000ll;
    return macs <= 4000000000ll || (outputs <= 4000000 && K >= 4 * N && M <= 4096);
}

extern "C" size_t m2_product_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    const int s = m2::product_plan(M, N, K).splits;
    return s > 1 ? (size_t)s * M * N * sizeof(float) : 0;
}

namespace m2 {
namespace {

int check_product(const m2_product_params* p) {
    M2_REQUIRE(p && p->a && p->b && p->out, M2_ERR_NULL, "product: a, b and out are required");
    M2_REQUIRE(m2_product_fits(p->M, p->N, p->K, p->a_k, p->b_k), M2_ERR_SHAPE, "product: shape %lld x %lld x %lld is not taken",
               (long long)p->M, (long long)p->N, (long long)p->K);
    M2_REQUIRE(aligned16(p->a) && aligned16(p->b) && aligned16(p->out) && p->lda % 8 == 0 && p->ldb % 8 == 0 && p->ldo % 8 == 0, M2_ERR_ALIGN,
               "product: operands and rows must be 16-byte aligned");
    M2_REQUIRE(p->lda >= (p->a_k ? p->K : p->M) && p->ldb >= (p->b_k ? p->K : p->N) && p->ldo >= p->N, M2_ERR_SHAPE, "product: row strides too short");
    M2_REQUIRE((p->a_k ? p->M : 64) * p->lda < ((int64_t)1 << 31) && (p->b_k ? p->N : 64) * p->ldb < ((int64_t)1 << 31), M2_ERR_SHAPE,
               "product: operand too large for 32-bit offsets");
    return M2_OK;
}

ProductArgs product_args(const m2_product_params* p, int r, int splits, int ksteps) {
    ProductArgs a{};
    a.A = static_cast<const bf16_t*>(p->a); a.B = static_cast<const bf16_t*>(p->b); a.bias = static_cast<const bf16_t*>(p->bias);
    a.out = static_cast<bf16_t*>(p->out); a.lda = p->lda; a.ldb = p->ldb; a.ldo = p->ldo;
    a.M = (int)p->M; a.N = (int)p->N; a.K = (int)p->K;
    a.tiles_m = (int)ceil_div(p->M, (int64_t)r); a.tiles_n = (int)ceil_div(p->N, (int64_t)r);
    a.splits = splits; a.ksteps = ksteps;
    return a;
}
int launch_sum(const ProductArgs& a, hipStream_t st) {
    product_sum_kernel<<<(unsigned)ceil_div((int64_t)a.M * (a.N / 8), (int64_t)256), 256, 0, st>>>(a.part, a.bias, a.out, a.ldo, a.M, a.N, a.splits);
    return check_launch("product_sum_kernel");
}
unsigned product_blocks(const ProductArgs& a) { return (unsigned)(ceil_div((int64_t)a.tiles_m * a.tiles_n * a.splits, (int64_t)8) * 8); }

}  // namespace
}  // namespace m2

extern "C" int m2_product(const m2_product_params* p, void* stream) {
    using namespace m2;
    if (const int bad = check_product(p)) return bad;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const ProductPlan plan = product_plan(p->M, p->N, p->K);
    const int splits = plan.splits;
    ProductArgs a = product_args(p, plan.r, splits, plan.ksteps);
    if (splits > 1) {
        M2_REQUIRE(p->workspace && p->workspace_bytes >= (size_t)splits * p->M * p->N * 4, M2_ERR_WORKSPACE, "product: workspace too small");
        a.part = static_cast<float*>(p->workspace);
    }
    const unsigned grid = product_blocks(a);
    const size_t sm = (size_t)kRing * 2 * plan.r * kK * 2;
    auto launch = [&](auto k) -> int {
        if (const int rc = allow_smem(k, sm)) return rc;
        k<<<grid, 256, sm, st>>>(a);
        return check_launch("product_kernel");
    };
    auto form = [&](auto r) -> int {
        constexpr int R = decltype(r)::value;
        return p->a_k ? (p->b_k ? launch(product_kernel<true, true, R>) : launch(product_kernel<true, false, R>))
                      : (p->b_k ? launch(product_kernel<false, true, R>) : launch(product_kernel<false, false, R>));
    };
    const int rc = plan.r == 64 ? form(std::integral_constant<int, 64>{}) : form(std::integral_constant<int, 128>{});
    if (rc || splits == 1) return rc;
    return launch_sum(a, st);
}

// Against two products of this file their own count decides (3 us for the launch more): 1.1 to 1.8 times as fast over 40 such pairs
// of layers of 256 to 1024 channels on 40 to 2000 tokens and 230 of 32 to 3000 channels on 8 to 60000.  Where either would go to the
// general library: up to 150 k steps per CU.  Below it 40 tokens, 1024 channels 24.5 -> 14.1 us, 1000 tokens 54 -> 40, 500 tokens, 1536
// channels, out_proj 30 -> 23.6, in_proj 48.5 -> 46.9; above it 1000 tokens, 1280 channels, in_proj 59 -> 67, 2048 channels, out_proj 54 -> 65.
// And not where dW's sum over many tokens, which nothing splits here, outlasts the rest: 15785 tokens, 736 x 368 63 -> 87 us.
extern "C" int m2_product_pair_pays(const m2_product_params* x, const m2_product_params* w) {
    using namespace m2;
    if (!x || !w || !x->a_k || x->b_k || w->a_k || w->b_k || x->bias || w->bias) return 0;
    if (!m2_product_fits(x->M, x->N, x->K, 1, 0) || !m2_product_fits(w->M, w->N, w->K, 0, 0)) return 0;
    const PairPlan plan = pair_plan(*x, *w);
    if (!m2_product_pays(x->M, x->N, x->K, 1, 0) || !m2_product_pays(w->M, w->N, w->K, 0, 0)) return plan.work <= 150.f && (plan.dw_chain <= 12.f || plan.dw_chain <= 0.24f * plan.work);
    return plan.us < product_plan(x->M, x->N, x->K).us + product_plan(w->M, w->N, w->K).us + 3.f;
}

extern "C" size_t m2_product_pair_workspace_bytes(const m2_product_params* x, const m2_product_params* w) {
    const int n = x && w ? m2::pair_plan(*x, *w).splits : 1;
    return n > 1 ? (size_t)n * x->M * x->N * sizeof(float) : 0;
}

extern "C" int m2_product_pair(const m2_product_params* x, const m2_product_params* w, void* stream) {
    using namespace m2;
    int rc = check_product(x);
    if (!rc) rc = check_product(w);
    if (rc) return rc;
    M2_REQUIRE(x->a_k && !x->b_k && !w->a_k && !w->b_k && !x->bias && !w->bias, M2_ERR_SHAPE, "product_pair: dy W and dy^T x, without a bias");
    M2_REQUIRE(ceil_div(x->M, (int64_t)64) * ceil_div(x->N, (int64_t)64) + ceil_div(w->M, (int64_t)64) * ceil_div(w->N, (int64_t)64) < (1 << 30), M2_ERR_SHAPE,
               "product_pair: too many tiles");
    const PairPlan plan = pair_plan(*x, *w);
    ProductArgs ax = product_args(x, 64, plan.splits, plan.ksteps);
    const ProductArgs aw = product_args(w, 64, 1, (int)ceil_div(w->K, (int64_t)kK));
    if (plan.splits > 1) {
        M2_REQUIRE(x->workspace && x->workspace_bytes >= m2_product_pair_workspace_bytes(x, w), M2_ERR_WORKSPACE, "product_pair: workspace too small");
        ax.part = static_cast<float*>(x->workspace);
    }
    const unsigned bx = product_blocks(ax), bw = product_blocks(aw);
    const size_t sm = (size_t)kRing * 2 * 64 * kK * 2;
    if ((rc = allow_smem(product_pair_kernel, sm))) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    product_pair_kernel<<<bx + bw, 256, sm, st>>>(ax, aw, bx, bw, ax.ksteps >= aw.ksteps);
    if ((rc = check_launch("product_pair_kernel")) || plan.splits == 1) return rc;
    return launch_sum(ax, st);
}
