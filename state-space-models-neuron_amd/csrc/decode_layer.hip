// One decode step of a whole mixer layer for few sequences: three launches (mamba2/mamba2_mixer.py:243-282 step, and around it
// modeling_mamba2.py:94-103, 133-140, the block's norm and residual add).
//
//   linear_small (in_proj)     zxBCdt = W x, scaled by the row's 1 / rms when x comes from the residual stream
//   decode_gated               conv + SiLU of the token, S' = S exp(A dt) + dt x (x) B, h = (S' C + D x) silu(z): w h and sum of h^2 per head
//   linear_small (out_proj)    W (w h), scaled by the groups' 1 / rms [+ residual: the new residual times the next norm's weight
//                              and its sums of squares]; shifts the B/C conv states on the side
//
// At this size a step is bound by its launches and by latency: the same layer as separate kernels is seven of 4.6-11 us each
// (two library products, conv, scan, norm, add + norm), most of them idle, and 2.3x the host work.  An RMS norm in front of a
// product costs nothing when it is taken apart: the weight is applied by whoever writes the row, the sum of squares is left
// beside it, and 1 / rms scales the finished product (a common factor of the row, or of the K range of one wave for grouped
// norms).  Normalising the rows inside the product instead (once per workgroup, through LDS) made it 7.9 us where the plain
// product takes 5.3 (8 rows of 1024, 4384 outputs), and a kernel of its own is 4.7 us.
#include <initializer_list>

#include "ssd_host.hpp"
#include "ssd_y.hpp"

namespace m2 {
namespace {

// ------------------------------------------------------------------------------------------ small products
// out[m][n] = scale[m] * sum_k X[m][k] W[n][k] for m < M <= 32, bf16 operands, fp32 accumulation.
//
// A workgroup owns 16 rows of W at a time; its NW waves split K, each with v_mfma_f32_16x16x32_bf16 (A = weights, B = x), and
// the NW partial tiles meet in LDS.  16 rows rather than 32 because the narrow products have few of them (1024 outputs: 64
// workgroups) and what counts is the number of loads in flight over the chip.
// Both operands come through LDS by asynchronous copies of whole 128-byte lines (8 rows x 128 bytes per wave-wide copy), each
// wave in a ring of its own that runs D - 1 steps ahead, also into the workgroup's next tile: no barrier but the one around a
// tile's sum.  Loading the fragments straight into registers touches 16 rows, 64 bytes each, per instruction, and the L1 then
// delivers 12 bytes per clock: 18 us for 10576 x 2560 at 16 rows and 26 at 32 with the weights in the memory-side cache.
// Slots of 16 bytes are swizzled by the row so that the 16 rows of a fragment read spread over all banks.
// What bounds the larger products is a CU's path to memory (10576 x 2560 with the weights in the memory-side cache: 10.6 us of the
// 12.1 with cold ones), and of the ring's three copies per step one is x, however few its rows.  Up to four rows (XM < 8, padded to
// 1, 2 or 4) therefore come ahead of the ring and stay, 8 rows-times-steps per copy, where they fit beside it: 10576 x 2560 and
// 2560 x 5120 at 4 rows 12.9 + 9.5 -> 12.1 + 8.5 us, at 1 row 12.0 + 8.7 -> 11.9 + 8.4.  The LDS they free is not for a deeper
// ring: 6 or 8 steps give nothing there and 5.7 -> 6.3 / 6.4 us at 4384 x 1024.
// The small products wait for memory once.  The ring's copies go out first and everything else that a workgroup will need (sums,
// old values, the conv states it shifts) right behind them: shifted behind the last tile the states were a second wait, and with
// the sums in front the weights came 0.5 us later (24 layers of 1024 channels, 8 rows: 487 -> 476 us a step; 1 row 436 -> 399).
enum { kOutBf16 = 0, kOutF32 = 1, kOutAdd = 2 };

struct LinearArgs {
    const bf16_t* w; const bf16_t* bias;
    const bf16_t* x; int64_t x_sr;
    const float* sq;                        // (M, nsq) sums of squares of the unscaled rows, or null: no scale
    void* out; int64_t out_sr;
    const float* next_w; bf16_t* next_x; float* next_sq;      // kOutAdd: next norm's weight -> rows (M, N) and sums (M, tiles)
    int M, N, K, tiles, nsq, groups;
    float eps;
    // conv states of the B and C channels, shifted here because every head of the scan in front of this reads them whole
    bf16_t* conv_state; const bf16_t* conv_in; int64_t conv_in_sb; int conv_c0, conv_cx, conv_W;
};

// Every LDS read that this wave has issued has returned its data.
__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// Barrier for LDS traffic alone: the copies in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
    lds_reads_done();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Bytes of a wave's share of the resident rows
template <int XM>
__host__ __device__ constexpr int linear_resident(int steps, int nw) { return XM < 8 ? ((steps + nw - 1) / nw * XM + 7) / 8 * 1024 : 0; }

template <int OK, int XM, int NW, int D>
__global__ void __launch_bounds__(NW * 64)
linear_small_kernel(const LinearArgs a) {
    constexpr bool RESIDENT = XM < 8;
    constexpr int MT = (XM + 15) / 16, PER = 2 + (RESIDENT ? 0 : XM / 8), SLOT = PER * 1024;     // column tiles; copies and bytes of a step of 64 k
    extern __shared__ __align__(1024) char ring_mem[];
    __shared__ __align__(16) float red[NW][MT][256];
    __shared__ float rs[32][8];
    const int tid = threadIdx.x, wave = (int)uniform(tid >> 6), lane = tid & 63, r16 = lane & 15, q4 = lane >> 4;
    const int steps = a.K / 64, s0 = steps * wave / NW, mine = steps * (wave + 1) / NW - s0;
    const char* ring = ring_mem + wave * (D * SLOT + linear_resident<XM>(steps, NW));
    const uint32_t ring_addr = uniform(lds_addr_of(ring));
    // copies: lane i fills slot i & 7 of row i >> 3 with the row's chunk (slot ^ swizzle)
    const int crow = lane >> 3;
    auto chunk_off = [&](int row) { return (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16); };
    constexpr int XR = RESIDENT ? 1 : XM / 8;
    uint32_t xoff[XR];
#pragma unroll
    for (int j = 0; j < XR; ++j) {
        const int row = j * 8 + crow;
        xoff[j] = (uint32_t)((row < a.M ? row : a.M - 1) * a.x_sr * 2) + chunk_off(row);
    }
    int itile = blockIdx.x, is = 0, islot = 0;               // the next step to issue
    uint32_t woff[2];
    auto tile_rows = [&](int tile) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = j * 8 + crow, n = tile * 16 + row;
            woff[j] = (uint32_t)((n < a.N ? row : a.N - 1 - tile * 16) * (int64_t)a.K * 2) + chunk_off(row);
        }
    };
    tile_rows(itile);
    auto issue = [&] {
        const int64_t k0 = (int64_t)(s0 + is) * 64;
        const bf16_t* wp = a.w + (int64_t)itile * 16 * a.K + k0;
        const uint32_t dst = ring_addr + islot * SLOT;
#pragma unroll
        for (int j = 0; j < 2; ++j) async_copy16(wp, woff[j], dst + j * 1024);
        if constexpr (!RESIDENT) {
#pragma unroll
            for (int j = 0; j < XR; ++j) async_copy16(a.x + k0, xoff[j], dst + (2 + j) * 1024);
        }
        islot = islot + 1 == D ? 0 : islot + 1;
        if (++is == mine) {
            is = 0;
            itile += gridDim.x;
            if (itile < a.tiles) tile_rows(itile);
        }
    };
    if constexpr (RESIDENT) {
        for (int j = 0; j * 8 < mine * XM; ++j) {            // 8 rows of 64 k, row % XM of step row / XM
            const int row = j * 8 + crow, m = row % XM, step = row / XM < mine ? row / XM : mine - 1;
            async_copy16(a.x + (int64_t)s0 * 64, (uint32_t)((m < a.M ? m : a.M - 1) * a.x_sr * 2) + (uint32_t)(step * 128) + chunk_off(m),
                         ring_addr + D * SLOT + j * 1024);
        }
    }
    const int total = mine * ((a.tiles - 1 - (int)blockIdx.x) / (int)gridDim.x + 1);
    for (int j = 0; j < D - 1 && j < total; ++j) issue();
    // the row scales: this wave's rows, their partial sums asked for ahead of everything and added up behind the first tile
    constexpr int RU = 4, RV = 3;
    const int per = a.sq ? a.nsq / a.groups : 0, nrs = a.sq ? a.M * a.groups : 0;
    const bool early = nrs <= RU * NW && per <= RV * 64;
    float part[RU][RV];
#pragma unroll
    for (int u = 0; u < RU; ++u)
#pragma unroll
        for (int v = 0; v < RV; ++v) {
            const int i = wave + u * NW, q = v * 64 + lane;
            part[u][v] = early && i < nrs && q < per ? a.sq[(int64_t)i * per + q] : 0.f;
        }
    // old values of the outputs that a thread adds to
    constexpr int NO = (MT * 256 + NW * 64 - 1) / (NW * 64);
    float old[NO], nw[NO];
    auto fetch_old = [&](int tile) {
        if constexpr (OK == kOutAdd) {
#pragma unroll
            for (int j = 0; j < NO; ++j) {
                const int i = j * NW * 64 + tid, m = i >> 4, n = tile * 16 + (i & 15);
                const bool own = i < MT * 256 && m < a.M && n < a.N;
                old[j] = own ? static_cast<const float*>(a.out)[m * a.out_sr + n] : 0.f;
                nw[j] = own && a.next_w ? a.next_w[n] : 0.f;
            }
        }
    };
    fetch_old(blockIdx.x);
    // the first conv state that this thread shifts
    constexpr int CW = 8;                                    // widest
    const int nch = a.conv_cx - a.conv_c0, conv_n = a.conv_state ? a.M * nch : 0, conv_i = blockIdx.x * NW * 64 + tid;
    bf16_t* conv_at = nullptr;
    bf16_t conv_v[CW];
    auto conv_fetch = [&](int i) {
        const int b = i / nch, c = a.conv_c0 + i - b * nch;
        conv_at = a.conv_state + ((int64_t)b * a.conv_cx + c) * a.conv_W;
#pragma unroll
        for (int j = 1; j < CW; ++j) if (j < a.conv_W) conv_v[j - 1] = conv_at[j];
        conv_v[CW - 1] = a.conv_in[b * a.conv_in_sb + c];
    };
    auto conv_store = [&] {
#pragma unroll
        for (int j = 0; j < CW - 1; ++j) if (j + 1 < a.conv_W) conv_at[j] = conv_v[j];
        conv_at[a.conv_W - 1] = conv_v[CW - 1];
    };
    if (conv_i < conv_n) conv_fetch(conv_i);
    int done = 0, slot = 0;
    for (int tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
        floatx4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < mine; ++s, ++done) {
            // The slot that is filled now was read in the step before.  Those reads have to have returned before a copy is issued on
            // top of them: nothing orders an LDS read against the LDS write of a copy but this wait (the step's products wait for
            // most of them anyway; asked for here, it holds however the compiler schedules them).
            if (done + D - 1 < total) {
                lds_reads_done();
                issue();
            }
            wait_vmem_keep<PER>(total - 1 - done < D - 1 ? total - 1 - done : D - 1);
            const char* base = ring + slot * SLOT;
            const char* xbase = RESIDENT ? ring + D * SLOT + s * (XM * 128) : base + 2048;
            slot = slot + 1 == D ? 0 : slot + 1;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const int c = kk * 4 + q4;
                const bf16x8 wf = *reinterpret_cast<const bf16x8*>(base + r16 * 128 + ((c ^ ((r16 >> 1) & 7)) * 16));
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int m = XM <= 8 ? r16 & (XM - 1) : t * 16 + r16;
                    const bf16x8 xf = *reinterpret_cast<const bf16x8*>(xbase + m * 128 + ((c ^ ((m >> 1) & 7)) * 16));
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf, acc[t], 0, 0, 0);
                }
            }
        }
        const int next = tile + (int)gridDim.x;
        // lane: column m = lane & 15, rows n = 4 (lane >> 4) + 0..3
#pragma unroll
        for (int t = 0; t < MT; ++t) *reinterpret_cast<floatx4*>(&red[wave][t][r16 * 16 + q4 * 4]) = acc[t];
        if (a.sq && tile == (int)blockIdx.x) {
#pragma unroll
            for (int u = 0; u < RU; ++u) {
                const int i = wave + u * NW;
                if (early && i < nrs) {
                    const float v = warp_sum(part[u][0] + part[u][1] + part[u][2]);
                    if (lane == 0) rs[i / a.groups][i % a.groups] = rsqrtf(v * (float)a.groups / (float)a.K + a.eps);
                }
            }
            if (!early)
                for (int i = wave; i < nrs; i += NW) {
                    float v = 0.f;
                    for (int q = lane; q < per; q += 64) v += a.sq[(int64_t)i * per + q];
                    v = warp_sum(v);
                    if (lane == 0) rs[i / a.groups][i % a.groups] = rsqrtf(v * (float)a.groups / (float)a.K + a.eps);
                }
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const int i = j * NW * 64 + tid, m = i >> 4, n = tile * 16 + (i & 15);
            if (i >= MT * 256) break;                        // whole waves
            const bool own = m < a.M && n < a.N;
            float v = 0.f;
            if (a.sq) {
                const int wpg = NW / a.groups;               // waves per norm group: their K ranges lie inside one
#pragma unroll
                for (int q = 0; q < NW; ++q) v += red[q][i >> 8][i & 255] * rs[m][a.groups == 1 ? 0 : q / wpg];
            } else {
#pragma unroll
                for (int q = 0; q < NW; ++q) v += red[q][i >> 8][i & 255];
            }
            const int64_t o = m * a.out_sr + n;
            if (own && a.bias) v += to_f32(a.bias[n]);
            if (OK == kOutBf16) {
                if (own) static_cast<bf16_t*>(a.out)[o] = (bf16_t)v;
            } else if (OK == kOutF32) {
                if (own) static_cast<float*>(a.out)[o] = v;
            } else {
                v = own ? v + old[j] : 0.f;
                if (own) static_cast<float*>(a.out)[o] = v;
                if (a.next_w) {
                    if (own) a.next_x[(int64_t)m * a.N + n] = (bf16_t)(v * nw[j]);
                    float s = v * v;
                    s = lane_xor_add<1>(s); s = lane_xor_add<2>(s); s = lane_xor_add<4>(s); s = lane_xor_add<8>(s);
                    if ((i & 15) == 0 && m < a.M) a.next_sq[(int64_t)m * a.tiles + tile] = s;
                }
            }
        }
        if (next < a.tiles) {
            fetch_old(next);
            lds_barrier();
        }
    }
    if (conv_i < conv_n) {
        conv_store();
        for (int i = conv_i + (int)gridDim.x * NW * 64; i < conv_n; i += gridDim.x * NW * 64) { conv_fetch(i); conv_store(); }
    }
}

// Waves per tile: eight where the tiles do not fill the chip by themselves, and for more than 16 rows, whose ring leaves room
// for one workgroup per CU; else four.  A grouped norm needs every wave's share of K inside one group (0: no such split).
int linear_waves(int64_t M, int64_t N, int64_t K, int64_t groups) {
    const int64_t steps = K / 64;
    const int want = (ceil_div(N, (int64_t)16) <= device_cus() || M > 16) && steps >= 8 ? 8 : 4;
    if (groups == 1) return steps >= want ? want : (steps >= 4 ? 4 : 1);
    for (const int nw : {want, 8, 4})
        if (nw % groups == 0 && steps % nw == 0) return nw;
    return 0;
}

template <int OK>
int launch_linear(LinearArgs a, hipStream_t st) {
    a.tiles = (int)ceil_div(a.N, 16);
    const int nw = linear_waves(a.M, a.N, a.K, a.sq ? a.groups : 1);
    int rc = M2_OK;
    auto go = [&](auto xm, auto waves) {
        constexpr int XM = decltype(xm)::value, NW = decltype(waves)::value, D = XM == 32 && NW == 8 ? 2 : 4;
        constexpr size_t ring = (size_t)NW * D * (XM < 8 ? 2 : 2 + XM / 8) * 1024, room = (NW == 8 ? 160 : 80) * 1024 - NW * ((XM + 15) / 16) * 1024 - 1024;
        static_assert(ring <= room || (XM == 32 && NW == 4), "ring and partial tiles within a workgroup's share of the LDS of a CU");
        const size_t lds = ring + (size_t)NW * linear_resident<XM>(a.K / 64, NW);
        if (XM < 8 && lds > room) return false;
        // Two workgroups of four waves, or one of eight, per CU; each goes on to its next tile without draining its ring.
        // (10576 x 2560, 1 / 8 / 16 rows, four waves: 12.1 / 12.9 / 14.8 us with 512 workgroups, 13.7 / 14.5 / 16.6 with one per
        // tile; 32 rows, eight waves: 20.4 with 256, 23.8 with one per tile.)
        const int64_t most = (NW == 8 ? 1 : 2) * device_cus();
        const unsigned grid = (unsigned)(a.tiles < most ? a.tiles : most);
        rc = allow_smem(linear_small_kernel<OK, XM, NW, D>, lds > 48 * 1024 && XM < 8 ? room : lds);      // one value per kernel: threads may launch side by side
        if (rc == M2_OK) linear_small_kernel<OK, XM, NW, D><<<grid, NW * 64, lds, st>>>(a);
        return true;
    };
    auto rows = [&](auto waves) {
        if (a.M <= 1 && go(std::integral_constant<int, 1>{}, waves)) return;
        if (a.M <= 2 && go(std::integral_constant<int, 2>{}, waves)) return;
        if (a.M <= 4 && go(std::integral_constant<int, 4>{}, waves)) return;
        if (a.M <= 8) go(std::integral_constant<int, 8>{}, waves);
        else if (a.M <= 16) go(std::integral_constant<int, 16>{}, waves);
        else go(std::integral_constant<int, 32>{}, waves);
    };
    if (nw == 8) rows(std::integral_constant<int, 8>{});
    else if (nw == 4) rows(std::integral_constant<int, 4>{});
    else rows(std::integral_constant<int, 1>{});
    return rc ? rc : check_launch("linear_small_kernel");
}

// The head of the chain: residual [+= delta], and the rows (residual times the norm's weight) with their sums of squares, as
// linear_small leaves them behind a layer.  One workgroup per row.  With ids the row is set from row ids[row] of a table of `vocab`
// rows, the embedding (NaN for an id outside it): what bounds a few rows is the launch and one trip to memory after the other, here
// the id and then everything else at once, V elements a lane
// (24 layers of 1024 channels, 8 sequences, captured: 474 -> 465.5 us a step; the library's lookup had taken 8.5 and this kernel 4.3).
template <typename T, int V>
__global__ void __launch_bounds__(256)
decode_rows_kernel(float* __restrict__ res, const T* __restrict__ add, const int64_t* __restrict__ ids, int64_t vocab, int set,
                   const float* __restrict__ w, bf16_t* __restrict__ x, float* __restrict__ sq, int64_t K) {
    typedef T avec __attribute__((ext_vector_type(V)));
    typedef float fvec __attribute__((ext_vector_type(V)));
    typedef bf16_t xvec __attribute__((ext_vector_type(V)));
    __shared__ float red[4];
    const int64_t row = (int64_t)blockIdx.x * K, id = ids ? ids[blockIdx.x] : (int64_t)blockIdx.x;
    const bool known = !ids || (id >= 0 && id < vocab);
    float s = 0.f;
    for (int64_t k = threadIdx.x * V; k < K; k += 256 * V) {
        fvec wv = 0.f, v = 0.f;
        if (w) wv = *reinterpret_cast<const fvec*>(w + k);
        if (!set) v = *reinterpret_cast<const fvec*>(res + row + k);
        if (!known) v = __builtin_nanf("");
        else if (add) {
            const avec av = *reinterpret_cast<const avec*>(add + id * K + k);
#pragma unroll
            for (int e = 0; e < V; ++e) v[e] += to_f32(av[e]);
        }
        *reinterpret_cast<fvec*>(res + row + k) = v;
        if (!w) continue;
        xvec xv;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            xv[e] = (bf16_t)(v[e] * wv[e]);
            s += v[e] * v[e];
        }
        *reinterpret_cast<xvec*>(x + row + k) = xv;
    }
    if (!w) return;
    s = warp_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) sq[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// ------------------------------------------------------------------------------------------ conv + scan + gate
// One workgroup per (head, sequence), its 256 lanes laid over the state as float4s (GL lanes per row, UP rows each, all loads
// issued first).  While they arrive the lanes form the head's conv outputs: its own P channels (whose conv state it shifts)
// and the N + N channels of its group's B and C, which every head of the group forms anew (4 KB from L2 beside a 64 KB state)
// rather than wait for a kernel of their own; their states stay as they are until the product behind this kernel.
struct GatedArgs {
    float* S; const bf16_t* zx; int64_t zx_sb;            // [z | x | B | C | dt] row of a sequence
    bf16_t* conv_state; const void* conv_w; const void* conv_b;
    const float *A, *D, *dt_bias, *norm_w;
    bf16_t* h; float* head_sq;                            // w h (batch, heads * P) and sum of h^2 (batch, heads)
    int nheads, ngroups, conv_cx, W;
};
// STATES_FIRST: which loads go out first, the states' or the conv's dozen small ones per lane.  With more workgroups than CUs the
// memory has to be kept busy: 8 sequences of 80 heads 10.3 -> 8.9 us, 4 of 128 8.7 -> 7.8, 32 of 32 13.3 -> 12.7 (a whole layer, 12 of
// 32: 20.2 -> 19.3, 4 of 80: 28.5 -> 27.4).  Below that a workgroup's own chain counts too, and the conv is at its head: a layer of 8
// of 32 17.5 us, 17.6 with the states first; 1 and 4 the same.
template <typename WT, int P, int N, bool STATES_FIRST>
__global__ void __launch_bounds__(256)
decode_gated_kernel(const GatedArgs a) {
    constexpr int GL = N / 4, ROWS = 256 / GL, UP = P / ROWS < 8 ? P / ROWS : 8, NCH = P + 2 * N;
    static_assert(P % (ROWS * UP) == 0, "whole passes over the state rows");
    constexpr int NI = (NCH + 255) / 256;
    __shared__ __align__(16) float xa[P], za[P], Ba[N], Ca[N], ha[P], red[4];
    const int tid = threadIdx.x, h = blockIdx.x, b = blockIdx.y;
    const int g = h / (a.nheads / a.ngroups), d = a.nheads * P;
    const bf16_t* row = a.zx + b * a.zx_sb;
    float* Sp = a.S + ((int64_t)b * a.nheads + h) * (P * N);
    const int sub = tid % GL, rowi = tid / GL;
    floatx4 sv[UP];
    auto load_states = [&] {
#pragma unroll
        for (int u = 0; u < UP; ++u) sv[u] = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(Sp + (u * ROWS + rowi) * N + sub * 4));
    };
    if constexpr (STATES_FIRST) load_states();
    // Every load goes out before any value is looked at.  With the taps converted, and so waited for, in a branch per 256 channels, the
    // states asked for behind them and the cache's columns waited for behind the states, a layer of 8 sequences of 32 heads took 0.9 us
    // more.  Where the chip has idle CUs, without a branch at all: lanes past the last channel read it once more (a model of 24 such
    // layers 445 us, with branches of whole waves 460); else in branches of whole waves (P and N are multiples of 64): 8 sequences of
    // 80 heads 27.3 us a layer, 27.8 without.
    const int w64 = __builtin_amdgcn_readfirstlane(tid >> 6) * 64;
    bf16_t hist[NI][3], in[NI];
    RawVec<WT, 4> taps[NI];
    WT bias[NI];
    auto channel = [&](int i) { return i < P ? h * P + i : (i < P + N ? d + g * N + (i - P) : d + (a.ngroups + g) * N + (i - P - N)); };
    const WT* cb = static_cast<const WT*>(a.conv_b ? a.conv_b : a.conv_w);      // (read and dropped without a bias)
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        if (STATES_FIRST && q * 256 + w64 >= NCH) continue;
        const int i = q * 256 + tid, c = channel(i < NCH ? i : NCH - 1);
        const bf16_t* cs = a.conv_state + ((int64_t)b * a.conv_cx + c) * a.W + a.W - 3;
#pragma unroll
        for (int j = 0; j < 3; ++j) hist[q][j] = cs[j];
        in[q] = row[d + c];
        taps[q] = loadv_raw<WT, 4>(static_cast<const WT*>(a.conv_w) + c * 4);
        bias[q] = cb[c];
    }
    bf16_t zin = (bf16_t)0.f;
    float nw = 0.f;
    if (!STATES_FIRST || w64 < P) {
        const int c = h * P + (tid < P ? tid : P - 1);
        zin = row[c];
        nw = a.norm_w[c];
    }
    const bf16_t dt_in = row[d + a.conv_cx + h];
    const float db = a.dt_bias ? a.dt_bias[h] : 0.f, Ah = a.A[h], Dh = a.D ? a.D[h] : 0.f;
    if constexpr (!STATES_FIRST) load_states();
    __builtin_amdgcn_sched_barrier(0);
    const float dtr = to_f32(dt_in) + db;
    const float dtv = softplus_f(dtr), dA = __expf(Ah * dtv);
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int i = q * 256 + tid;
        if (i < NCH) {
            float w[4];
            cvtv<WT, 4>(taps[q], w);
            const float z = (a.conv_b ? to_f32(bias[q]) : 0.f) + w[0] * to_f32(hist[q][0]) + w[1] * to_f32(hist[q][1]) + w[2] * to_f32(hist[q][2]) + w[3] * to_f32(in[q]);
            const float v = silu_f(z);
            if (i < P) {
                xa[i] = v;
                za[i] = silu_f(to_f32(zin));
                bf16_t* cs = a.conv_state + ((int64_t)b * a.conv_cx + h * P + i) * a.W;
                for (int j = 0; j < a.W - 4; ++j) cs[j] = cs[j + 1];
                if (a.W > 3) cs[a.W - 4] = hist[q][0];      // (read above: a load here would wait for the states)
                cs[a.W - 3] = hist[q][1]; cs[a.W - 2] = hist[q][2]; cs[a.W - 1] = in[q];
            } else if (i < P + N) Ba[i - P] = v;
            else Ca[i - P - N] = v;
        }
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
        a.h[(int64_t)b * d + h * P + tid] = (bf16_t)(ha[tid] * nw);
    }
    sq = warp_sum(sq);
    if ((tid & 63) == 0) red[tid >> 6] = sq;
    __syncthreads();
    if (tid == 0) a.head_sq[(int64_t)b * a.nheads + h] = (red[0] + red[1]) + (red[2] + red[3]);
}

int check_linear(const m2_linear_params* p) {
    M2_REQUIRE(p, M2_ERR_NULL, "linear_small: params is NULL");
    M2_REQUIRE(p->M >= 0 && p->N > 0 && p->K > 0, M2_ERR_SHAPE, "linear_small: M %lld, N %lld, K %lld", (long long)p->M, (long long)p->N, (long long)p->K);
    M2_REQUIRE(m2_linear_small_fits(p->M, p->N, p->K, p->sq ? p->groups : 1), M2_ERR_SHAPE,
               "linear_small: M %lld, N %lld, K %lld, %d groups: at most 32 rows, K a multiple of 64, whole K ranges per group",
               (long long)p->M, (long long)p->N, (long long)p->K, (int)p->groups);
    if (p->M == 0) return M2_OK;
    M2_REQUIRE(p->x && p->w && p->out, M2_ERR_NULL, "linear_small: x, w and out are required");
    M2_REQUIRE(!p->sq || (p->nsq > 0 && p->nsq % p->groups == 0), M2_ERR_SHAPE, "linear_small: %lld sums do not divide into %d groups", (long long)p->nsq, (int)p->groups);
    M2_REQUIRE(p->out_kind >= kOutBf16 && p->out_kind <= kOutAdd && (!p->next_weight || (p->out_kind == kOutAdd && p->next_x && p->next_sq)), M2_ERR_NULL,
               "linear_small: next_weight goes with out_kind 2, next_x and next_sq");
    M2_REQUIRE(aligned16(p->x) && aligned16(p->w) && p->x_stride_row % 8 == 0, M2_ERR_ALIGN, "linear_small: x rows and w must be 16-byte aligned");
    M2_REQUIRE(p->x_stride_row >= 0 && p->M * p->x_stride_row < ((int64_t)1 << 31), M2_ERR_SHAPE,
               "linear_small: %lld rows %lld elements apart are out of reach of 32-bit byte offsets", (long long)p->M, (long long)p->x_stride_row);
    return M2_OK;
}

int launch_linear_params(const m2_linear_params* p, const LinearArgs& conv, hipStream_t st) {
    const int rc = check_linear(p);
    if (rc || p->M == 0) return rc;
    LinearArgs a = conv;
    a.w = static_cast<const bf16_t*>(p->w); a.bias = static_cast<const bf16_t*>(p->bias);
    a.x = static_cast<const bf16_t*>(p->x); a.x_sr = p->x_stride_row; a.sq = p->sq; a.nsq = (int)p->nsq; a.groups = p->groups; a.eps = p->eps;
    a.out = p->out; a.out_sr = p->out_stride_row;
    a.next_w = p->next_weight; a.next_x = static_cast<bf16_t*>(p->next_x); a.next_sq = p->next_sq;
    a.M = (int)p->M; a.N = (int)p->N; a.K = (int)p->K;
    if (p->out_kind == kOutBf16) return launch_linear<kOutBf16>(a, st);
    if (p->out_kind == kOutF32) return launch_linear<kOutF32>(a, st);
    return launch_linear<kOutAdd>(a, st);
}

// Four elements a lane where every row starts on a vector of each of the arrays.
template <typename T>
int launch_decode_rows(float* res, const T* add, const int64_t* ids, int64_t vocab, int set, const float* w, bf16_t* x, float* sq, int64_t rows, int64_t K,
                       hipStream_t st) {
    const bool whole = K % 4 == 0 && aligned16(res) && aligned16(w) && reinterpret_cast<uintptr_t>(x) % 8 == 0 && reinterpret_cast<uintptr_t>(add) % (4 * sizeof(T)) == 0;
    if (whole) decode_rows_kernel<T, 4><<<(unsigned)rows, 256, 0, st>>>(res, add, ids, vocab, set, w, x, sq, K);
    else decode_rows_kernel<T, 1><<<(unsigned)rows, 256, 0, st>>>(res, add, ids, vocab, set, w, x, sq, K);
    return check_launch("decode_rows_kernel");
}

}  // namespace
}  // namespace m2

extern "C" int m2_linear_small_fits(int64_t M, int64_t N, int64_t K, int32_t groups) {
    using namespace m2;
    return M >= 0 && M <= 32 && N > 0 && N < (int64_t(1) << 30) && K > 0 && K % 64 == 0 && K <= (1 << 20) && groups >= 1 && groups <= 8 &&
           linear_waves(M, N, K, groups) > 0;
}

extern "C" int m2_linear_small(const m2_linear_params* p, void* stream) {
    return m2::launch_linear_params(p, m2::LinearArgs{}, static_cast<hipStream_t>(stream));
}

extern "C" int m2_decode_rows(float* residual, const void* delta, int32_t delta_dtype, int32_t set, const float* weight, void* x, float* sq, int64_t rows,
                              int64_t channels, void* stream) {
    using namespace m2;
    M2_REQUIRE(rows >= 0 && rows <= 65535 && channels > 0, M2_ERR_SHAPE, "decode_rows: rows %lld, channels %lld", (long long)rows, (long long)channels);
    if (rows == 0) return M2_OK;
    M2_REQUIRE(residual && weight && x && sq && (delta || !set), M2_ERR_NULL, "decode_rows: residual, weight, x and sq are required");
    M2_DISPATCH_DTYPE(delta_dtype, T, return launch_decode_rows<T>(residual, static_cast<const T*>(delta), nullptr, 0, set, weight, static_cast<bf16_t*>(x), sq,
                                                                   rows, channels, static_cast<hipStream_t>(stream)));
    return M2_OK;
}

extern "C" int m2_embed_rows(const void* table, int32_t table_dtype, int64_t vocab, const int64_t* ids, float* residual, const float* weight, void* x, float* sq,
                             int64_t rows, int64_t channels, void* stream) {
    using namespace m2;
    M2_REQUIRE(rows >= 0 && rows <= INT32_MAX && channels > 0 && vocab >= 0, M2_ERR_SHAPE, "embed_rows: rows %lld, channels %lld, vocab %lld", (long long)rows,
               (long long)channels, (long long)vocab);
    if (rows == 0) return M2_OK;
    M2_REQUIRE(table && ids && residual && !weight == !x && !weight == !sq, M2_ERR_NULL, "embed_rows: table, ids and residual are required, and weight, x and sq together or not at all");
    M2_DISPATCH_DTYPE(table_dtype, T, return launch_decode_rows<T>(residual, static_cast<const T*>(table), ids, vocab, 1, weight, static_cast<bf16_t*>(x), sq, rows,
                                                                   channels, static_cast<hipStream_t>(stream)));
    return M2_OK;
}

extern "C" int m2_decode_layer(const m2_linear_params* in, const m2_decode_params* dec, const float* norm_weight, const m2_linear_params* out, void* stream) {
    using namespace m2;
    M2_REQUIRE(in && dec && out, M2_ERR_NULL, "decode_layer: params is NULL");
    const int64_t P = dec->headdim, N = dec->dstate, d = dec->nheads * P, cx = d + 2 * dec->ngroups * N;
    M2_REQUIRE((P == 64 || P == 128) && (N == 64 || N == 128) && dec->k == 4 && dec->W >= 3 && dec->W <= 8 && dec->nheads > 0 && dec->ngroups > 0 &&
                   dec->nheads % dec->ngroups == 0, M2_ERR_SHAPE,
               "decode_layer: headdim %lld and dstate %lld must be 64 or 128, the conv 4 wide, the heads whole per group", (long long)P, (long long)N);
    M2_REQUIRE(dec->dtype == M2_BF16 && dec->activation == M2_ACT_SILU && (dec->param_dtype == M2_F32 || dec->param_dtype == M2_BF16), M2_ERR_DTYPE,
               "decode_layer: bf16 activations with SiLU only");
    M2_REQUIRE(in->M == dec->batch && out->M == dec->batch && in->N == d + cx + dec->nheads && out->K == d && in->out_kind == kOutBf16 && out->nsq == dec->nheads &&
                   dec->batch <= 65535, M2_ERR_SHAPE, "decode_layer: the projections do not match the layer");
    if (dec->batch == 0) return M2_OK;
    M2_REQUIRE(dec->conv_state && dec->conv_w && dec->S && dec->A && dec->dt_bias && norm_weight && out->sq && out->x, M2_ERR_NULL,
               "decode_layer: conv_state, conv_w, S, A, dt_bias, norm_weight, and the scratch behind out->x and out->sq are required");
    M2_REQUIRE(aligned16(dec->S) && (uintptr_t)dec->conv_w % (dec->param_dtype == M2_F32 ? 16 : 8) == 0, M2_ERR_ALIGN,
               "decode_layer: S must be 16-byte aligned, the conv weight on four of its elements");
    hipStream_t st = static_cast<hipStream_t>(stream);
    int rc = check_linear(out);
    if (rc) return rc;
    rc = launch_linear_params(in, LinearArgs{}, st);
    if (rc) return rc;
    const bf16_t* zx = static_cast<const bf16_t*>(in->out);
    GatedArgs g{};
    g.S = dec->S; g.zx = zx; g.zx_sb = in->out_stride_row; g.conv_state = static_cast<bf16_t*>(dec->conv_state);
    g.conv_w = dec->conv_w; g.conv_b = dec->conv_b; g.A = dec->A; g.D = dec->D; g.dt_bias = dec->dt_bias; g.norm_w = norm_weight;
    g.h = static_cast<bf16_t*>(const_cast<void*>(out->x)); g.head_sq = const_cast<float*>(out->sq);
    g.nheads = (int)dec->nheads; g.ngroups = (int)dec->ngroups; g.conv_cx = (int)cx; g.W = dec->W;
    const dim3 grid((unsigned)dec->nheads, (unsigned)dec->batch);
    auto go = [&](auto wt, auto p, auto n) {
        if ((int64_t)grid.x * grid.y > device_cus()) decode_gated_kernel<decltype(wt), decltype(p)::value, decltype(n)::value, true><<<grid, 256, 0, st>>>(g);
        else decode_gated_kernel<decltype(wt), decltype(p)::value, decltype(n)::value, false><<<grid, 256, 0, st>>>(g);
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
