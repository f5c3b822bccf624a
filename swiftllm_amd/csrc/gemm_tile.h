// gemm_tile.h — products of prompt-sized steps on the matrix cores: out[M, N] = act(x[M, K] w[N, K]^T), 16-bit operands, fp32 sums; of dense
// layers (gemm_tile.hip) and of experts, each with rows of its own (moe_grouped.hip).
//
// What bounds it: large products run the card at its power limit (8192^3 at 1.75 GHz: 1426 TFLOP/s, the library's 1338 on the same card),
// whatever the tile; small ones wait for their first columns (5000 cycles from a cold start) and for their results to leave (128 KiB a CU at
// the 32 bytes a cycle that an XCD's L2 takes of each of its CUs), and leave CUs idle in their last turn. So: one workgroup a CU that
// takes tile after tile (two of 128 x 128 and less), the next tile's first columns asked for while one ends, and tiles of eleven sizes of
// which a model of turns and steps picks (gemm_tile_shape).
//   * Four waves tile the result two by two. A step of 64 columns is four parts, the halves of the waves' rows of x and of w, four phases
//     multiply half by half, in the order X0 W0, X0 W1, X1 W1, X1 W0 and then X0 W1, X0 W0, X1 W0, X1 W1: every phase needs one part
//     more, read from LDS into the registers of a part that is done with while the phase before it multiplies. Nothing waits for LDS.
//   * A part's place in LDS is asked for again as soon as everyone has read it, eight parts ahead: LDS holds two steps and all of it is on
//     its way. One barrier for two phases; what it waits for is counted (vmcnt).
//   * Fetches go through buffer descriptors of the tile's own rows: rows beyond the matrix are zeros without a memory access.
//   * Results leave as whole lines through 4 KiB of LDS a wave, without a barrier, as stores that nobody waits for.
// Measured (us, bf16, operands from a pool of 1.5 GB; in brackets the library, in one call and in the blocks of rows that it was called with
// before): 7691 tokens: 1024 x 1024 17.3 (20.7, 27.1), 8192 x 1024 106 (104, 104), 1024 x 4096 55 (62, 74), 2576 x 1024 40 (60, 63); 4498: 2048 x 2048 33
// (38, 45), 2048 x 8192 117 (131, 141), 8192 x 2048 112 (125, 118), 3072 x 2048 45 (47, 59); 3657: 2048 x 8192 97 (105), 7440 x 2048 87 (104); 2029: 5696 x 1024 22
// (34), 1024 x 1024 8.6 (11); 1828: 28672 x 4096 347 with its gated unit (342 to 430 by card, and 32 for the unit), 4096 x 14336 177 (185); 5112: 6144 x
// 4096 182 (180, 207), 4096 x 4096 128 (135, 128). 270 products of 260 to 8192 tokens: 0.8 of the library's time where its calls are in blocks. From
// 16384 tokens on the library's rate is 5 % to 10 % higher (1.55 PFLOP/s).
#pragma once

#include "swl_common.h"

#include <type_traits>

namespace swl {

template <int N>
using Ic = std::integral_constant<int, N>;
typedef int int4v __attribute__((ext_vector_type(4)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

// acc += w x, or acc = w x (FIRST). (Tied in and out, in the accumulation registers where ACC: left to the builtin, the compiler moves
// accumulators between registers in every turn of the loop.)
#define SWL_TILE_MFMA(V, T, NAME)                                                                                            \
    template <bool ACC, bool FIRST>                                                                                          \
    __device__ __forceinline__ void tile_mfma_to(V &c, vec8_t<T> w, vec8_t<T> x) {                                           \
        if constexpr (ACC && FIRST) asm("v_mfma_f32_" NAME " %0, %1, %2, 0" : "=a"(c) : "v"(w), "v"(x));                     \
        else if constexpr (ACC) asm("v_mfma_f32_" NAME " %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));                        \
        else if constexpr (FIRST) asm("v_mfma_f32_" NAME " %0, %1, %2, 0" : "=&v"(c) : "v"(w), "v"(x));                      \
        else asm("v_mfma_f32_" NAME " %0, %1, %2, %0" : "+v"(c) : "v"(w), "v"(x));                                           \
    }
SWL_TILE_MFMA(float4_t, bf16, "16x16x32_bf16")
SWL_TILE_MFMA(float4_t, f16, "16x16x32_f16")
SWL_TILE_MFMA(float16_t, bf16, "32x32x16_bf16")
SWL_TILE_MFMA(float16_t, f16, "32x32x16_f16")
#undef SWL_TILE_MFMA

// 1 KiB, 16 bytes a lane (or four), to the LDS address `to`; lanes behind the descriptor's end get zeros
template <int BYTES = 16>
__device__ __forceinline__ void tile_fetch(int4v rsrc, unsigned off, unsigned soff, unsigned to) {
    unsigned keep;
    if constexpr (BYTES == 4) {
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep) : "v"(off), "s"(rsrc), "s"(soff), "s"(to) : "memory");
        return;
    }
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(off), "s"(rsrc), "s"(soff), "s"(to) : "memory");
}
__device__ __forceinline__ int4v tile_rsrc(const char *base, unsigned bytes) {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    return int4v{static_cast<int>(b), static_cast<int>((b >> 32) & 0xffff), static_cast<int>(bytes), 0x00020000};
}

// Division by a number known on the host: its 2^32 over it, the quotient at most one too small.
struct Divisor {
    unsigned by, inverse;
    static Divisor of(unsigned n) { return {n, n > 1 ? static_cast<unsigned>((1ULL << 32) / n) : 0xffffffffu}; }
};
__device__ __forceinline__ unsigned divide(unsigned n, Divisor d) {
    const unsigned q = __umulhi(n, d.inverse);
    return n - q * d.by >= d.by ? q + 1 : q;
}

// num / (1 + e^y) of the gated units below, with the error of the library's exponential and division (3.1 units of 2^-24 at most, 0.64 rms, from y = -87
// to 88; infinities and NaN come out as theirs) for less of the time in which no matrix step runs. 2^t of t = y log2 e, rounded, lacks a factor e^low, low = y - t
// ln 2: it goes into the quotient's one correction. That is made on a quarter of both, whose reciprocal is a normal number up to the largest. Results and
// products of 16 bits are the same ones for every 16-bit y. us of 1828 tokens x 28672 x 4096, 3657 x 16384 x 2048, 7691 x 8192 x 1024: the library's two 353, 207, 134;
// so 345, 197, 120; with the transcendental unit's as they are (its reciprocal and 2^(1.4427 y): 18 units at y = 20, 65 at 80, zero beyond 87.3) 342, 187, 112.
__device__ __forceinline__ float over_one_plus_exp(float num, float y) {
    y = fmaxf(y, -200.f);
    const float t = y * 0x1.715476p+0f, low = fmaf(t, 0x1.05c61p-29f, fmaf(t, -0x1.62e43p-1f, y));      // (ln 2 in two parts)
    const float e = fast_exp2(t) * 0.25f, d = e + 0.25f, a = num * 0.25f, r = __builtin_amdgcn_rcpf(d), q = a * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, e * low, fmaf(-d, q, a)), r, q), d, a);
}
// silu(z), and z sigmoid(1.702 z)
__device__ __forceinline__ float tile_silu(float z) { return over_one_plus_exp(z, -z); }
__device__ __forceinline__ float tile_silu_1702(float z) { return z * over_one_plus_exp(1.0f, -1.702f * z); }

struct GemmTileParams {
    void *out;
    const void *x, *w;
    int M, N, K;
    int64_t ldx, ldo;       // elements
    int m_tiles, n_tiles;
    int x_cols, act_cols;       // columns of out that share a matrix x (0: all), that the activation applies to
    int64_t x_next;             // bytes from one matrix x to the next
    // experts: sorted position -> assignment, the experts' first positions, weights by assignment (NULL: 1), how many experts, assignments a
    // token, bytes of x and of the weights
    const int32_t *order, *offsets;
    const float *in_w;
    int experts;
    Divisor top;
    unsigned x_bytes, in_w_bytes;
    Divisor group, wide, rest;      // tiles of a group, row tiles of one, of the last one
    int splits;             // shares of K, each with an fp32 slab of out (one behind the other) of its own
    Divisor share;          // tiles of a row of tiles in one of them
    float limit;
};

constexpr int kTileGroup = 8;       // row tiles that an XCD takes with all their column tiles
constexpr int kTileExperts = 512;   // at most
constexpr int kTileSlabs = -1;      // (for ACT)
enum TileRows { kTileDense = 0, kTileExpert = 1, kTileGather = 2 };     // rows of x: all alike, an expert's a tile, and gathered through `order`

// ACT kTileSlabs: fp32 sums over shares of K; 0: the product; 1: relu(.)^2 of the first act_cols columns; 2 + a: w rows [N first | N second], out = a gated unit of the two (a = 0 .. 2:
// gated_unit, 3: round(silu(second)) first, rounded). Activations are of the rounded products.
template <typename T, int U, int X0, int X1, int W0, int W1, int ACT, int ROWS = kTileDense>
__global__ __launch_bounds__(256, U * U * (X0 + X1) * (W0 + W1) <= 4096 ? 2 : 1) void gemm_tile_kernel(GemmTileParams p) {
    constexpr int X = X0 + X1, W = W0 + W1, E = U == 32 ? 4 : 2;        // blocks of U rows a wave; matrix steps of 64 columns
    constexpr bool GATED = ACT >= 2, SLABS = ACT == kTileSlabs;
    constexpr int xn[2] = {X0, X1}, wn_[2] = {W0, W1};
    constexpr int BLOCK = 2 * U * 128, ASKS = U / 16;       // bytes of a block of both waves in LDS, fetches of a wave for it
    constexpr int STEP = (X + W) * BLOCK, PAIR = 2 * STEP;
    constexpr int BM = 2 * U * X, OUTW = GATED ? U * W0 : U * W, BN = 2 * OUTW;     // rows, columns of a wave, of the tile
    constexpr int SIZE = SLABS ? 4 : 2;         // bytes of a result
    constexpr int CB = 128 / SIZE / U, PITCH = 128;     // blocks of columns that leave at once; a row of theirs in LDS
    constexpr bool ACC = U * U * X * W > 4096;
    using acc_t = std::conditional_t<U == 32, float16_t, float4_t>;
    static_assert(!GATED || W0 == W1, "");
    constexpr bool GATHER = ROWS == kTileGather, EXPERT = ROWS != kTileDense;
    // the next tile's row of `order` and both tiles' weights; first positions of the experts, first row tiles behind them
    constexpr int LISTS = PAIR + 4 * U * PITCH, TABLES = LISTS + (GATHER ? 3 * 1024 : 0);
    static_assert(!EXPERT || BM <= 256, "");
    __shared__ __attribute__((aligned(16))) char smem[TABLES + (EXPERT ? (2 * kTileExperts + 1) * 4 : 0)];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lu = lane & (U - 1), lg = lane / U, wn = wave & 1, wm = wave >> 1;

    // ---- the tiles of this workgroup: an XCD (workgroup id % 8) takes an equal run of them ------------------------------------------
    int m_tiles = p.m_tiles;
    int32_t *const first_of = reinterpret_cast<int32_t *>(smem + TABLES), *const tiles_to = first_of + kTileExperts + 1;
    if constexpr (EXPERT) {     // the first wave counts the experts' row tiles
        if (wave == 0) {
            int before = 0;
            for (int e0 = 0; e0 < p.experts; e0 += 64) {
                const int e = min(e0 + lane, p.experts - 1), lo = p.offsets[e], hi = e0 + lane < p.experts ? p.offsets[e + 1] : lo;
                int scan = (hi - lo + BM - 1) / BM;
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(scan, o, 64);
                    if (lane >= o) scan += v;
                }
                if (e0 + lane < p.experts) {
                    first_of[e] = lo;
                    tiles_to[e] = before + scan;
                    if (e == p.experts - 1) first_of[p.experts] = hi;
                }
                before += __builtin_amdgcn_readlane(scan, 63);
            }
        }
        __syncthreads();
        m_tiles = __builtin_amdgcn_readfirstlane(tiles_to[p.experts - 1]);
    }
    const int64_t all = static_cast<int64_t>(m_tiles) * p.n_tiles;
    const int xcd = blockIdx.x & 7, stride = gridDim.x >> 3;
    const int last = static_cast<int>((xcd + 1) * all / 8);
    int at = static_cast<int>(xcd * all / 8) + (blockIdx.x >> 3);
    if (at >= last) return;
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    const int64_t xb = p.ldx * 2, wb = static_cast<int64_t>(p.K) * 2, ob = p.ldo * SIZE;
    const int steps = p.K / 64 / (SLABS ? p.splits : 1);
    struct Place {
        int row0, rows, col0, expert;       // (of slabs: the share of K in the expert's place)
    };
    auto place = [&](int t) {
        const unsigned group = divide(t, p.group), in_group = t - group * p.group.by;
        Place to;
        int m_tile;
        if constexpr (EXPERT) {
            const unsigned wide = min(kTileGroup, m_tiles - static_cast<int>(group) * kTileGroup);
            const unsigned n = wide == kTileGroup ? in_group / kTileGroup : in_group / wide;
            m_tile = group * kTileGroup + in_group - n * wide;
            to.col0 = n * BN;
            for (int e0 = 0;; e0 += 64) {       // (a tile of some expert: found)
                const unsigned long long past = __ballot(e0 + lane >= p.experts || tiles_to[min(e0 + lane, p.experts - 1)] > m_tile);
                if (past) {
                    to.expert = e0 + __builtin_ctzll(past);
                    break;
                }
            }
            const int before = to.expert > 0 ? __builtin_amdgcn_readfirstlane(tiles_to[to.expert - 1]) : 0;
            const int lo = __builtin_amdgcn_readfirstlane(first_of[to.expert]), hi = __builtin_amdgcn_readfirstlane(first_of[to.expert + 1]);
            to.row0 = lo + (m_tile - before) * BM;
            to.rows = min(BM, hi - to.row0);
        } else {
            const Divisor wide = (group + 1) * p.wide.by > static_cast<unsigned>(p.m_tiles) ? p.rest : p.wide;
            const unsigned n = divide(in_group, wide), share = SLABS ? divide(n, p.share) : 0;
            to.row0 = (group * p.wide.by + in_group - n * wide.by) * BM;
            to.rows = min(BM, p.M - to.row0);
            to.col0 = (SLABS ? n - share * p.share.by : n) * BN;
            to.expert = share;
        }
        return to;
    };
    auto x_rsrc = [&](const Place &to) {
        if constexpr (GATHER) return tile_rsrc(static_cast<const char *>(p.x), p.x_bytes);
        const char *x = static_cast<const char *>(p.x) + (!EXPERT && p.x_cols ? to.col0 / p.x_cols * p.x_next : 0);
        const int k0 = SLABS ? to.expert * steps * 128 : 0;
        return tile_rsrc(x + to.row0 * xb + k0, static_cast<unsigned>(to.rows * xb - k0));
    };
    auto w_rsrc = [&](const Place &to) {
        const int64_t left = (GATED ? 2LL * p.N : static_cast<int64_t>(p.N)) - to.col0;
        const char *w = static_cast<const char *>(p.w) + (EXPERT ? static_cast<int64_t>(to.expert) * (GATED ? 2 : 1) * p.N * wb : 0);
        const int k0 = SLABS ? to.expert * steps * 128 : 0;
        return tile_rsrc(w + to.col0 * wb + k0, static_cast<unsigned>((GATED ? left : min(static_cast<int64_t>(BN), left)) * wb - k0));
    };

    // ---- staging: a step of 64 columns is four parts, the halves of the waves' rows of x and of w. A fetch is eight rows of 128 bytes, a
    // row's 16-byte units exchanged by bits 1 .. 3 of the row's number ------------------------------------------------------------------
    // Waves 0 and 1 bring the rows that are worked with by the waves of wm = 0, or wn = 0, 2 and 3 the others'.
    unsigned xo[X * ASKS], wo[W * ASKS];        // [half 0's, half 1's]
    const unsigned unit0 = ((lane & 7) ^ (lane >> 4)) * 16;
    // (GATHER: by the list that fetch_list left, and the weights of its assignments to one of two places)
    const unsigned *const list = reinterpret_cast<const unsigned *>(smem + LISTS);
    auto x_offsets = [&](int rows, int slot) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int count = xn[h] * ASKS, odd = wave & count & 1, row = wm * U * X + h * U * X0 + (wave & 1) * count * 8 + (lane >> 3);
#pragma unroll
            for (int i = 0; i < count; ++i) {
                unsigned off;
                if constexpr (GATHER) off = static_cast<unsigned>(divide(list[min(row + i * 8, rows - 1)], p.top) * xb);
                else off = static_cast<unsigned>(row * xb) + static_cast<unsigned>(i * 8 * xb);
                xo[h * X0 * ASKS + i] = off + (unit0 ^ (((i & 1) ^ odd) * 64));
            }
        }
        if constexpr (GATHER) {
            if (p.in_w) tile_fetch<4>(tile_rsrc(reinterpret_cast<const char *>(p.in_w), p.in_w_bytes), list[min(tid, rows - 1)] * 4, 0, lds0 + LISTS + 1024 + slot * 1024 + wave * 256);
        }
    };
    auto fetch_list = [&](const Place &to) { tile_fetch<4>(tile_rsrc(reinterpret_cast<const char *>(p.order + to.row0), to.rows * 4), tid * 4, 0, lds0 + LISTS + wave * 256); };
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int count = wn_[h] * ASKS, odd = wave & count & 1;
        const int64_t first = GATED ? wm * U * W0 + static_cast<int64_t>(h) * p.N : wm * U * W + h * U * W0;
        const unsigned from = static_cast<unsigned>((first + (wave & 1) * count * 8 + (lane >> 3)) * wb);
#pragma unroll
        for (int i = 0; i < count; ++i) wo[h * W0 * ASKS + i] = from + static_cast<unsigned>(i * 8 * wb) + (unit0 ^ (((i & 1) ^ odd) * 64));
    }
    Place here = place(at);
    if constexpr (GATHER) {
        fetch_list(here);
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        __syncthreads();
    }
    x_offsets(here.rows, 0);
    int4v ask_x = x_rsrc(here), ask_w = w_rsrc(here);       // the step that is asked for: its tile, its first column
    unsigned ask_k = 0;

    // Parts in the order of their use, eight for two steps: X0 W0 W1 X1, X0 W1 W0 X1
    auto fetch = [&](auto jc, int i) {
        constexpr int J = decltype(jc)::value & 7, odd = J >> 2, k = J & 3;
        constexpr bool of_x = k == 0 || k == 3;
        constexpr int h = k == 0 ? 0 : k == 3 ? 1 : ((k == 2) ^ odd);
        if constexpr (of_x) tile_fetch(ask_x, xo[h * X0 * ASKS + i], ask_k, lds0 + odd * STEP + h * X0 * BLOCK + (wave * xn[h] * ASKS + i) * 1024);
        else tile_fetch(ask_w, wo[h * W0 * ASKS + i], ask_k, lds0 + odd * STEP + (X + h * W0) * BLOCK + (wave * wn_[h] * ASKS + i) * 1024);
    };
    constexpr auto blocks = [](int j) { const int k = j & 3, odd = (j >> 2) & 1; return k == 0 ? X0 : k == 3 ? X1 : ((k == 2) ^ odd) ? W1 : W0; };
    constexpr auto fetches = [=](int from, int to) { int n = 0; for (int j = from; j < to; ++j) n += blocks(j); return n * ASKS; };

    // ---- fragments: row lu of a block, 16-byte unit (64 / U) e + lg ---------------------------------------------------------------------
    unsigned frag[E];
#pragma unroll
    for (int e = 0; e < E; ++e) frag[e] = static_cast<unsigned>(lu * 128 + ((((64 / U) * e + lg) ^ ((lu >> 1) & 7)) * 16));
    vec8_t<T> xf[X][E], wf[W][E];
    acc_t acc[X][W];
    auto read = [&](auto jc, int i) {
        constexpr int J = decltype(jc)::value & 7, odd = J >> 2, k = J & 3;
        constexpr bool of_x = k == 0 || k == 3;
        constexpr int h = k == 0 ? 0 : k == 3 ? 1 : ((k == 2) ^ odd), n = of_x ? xn[h] : wn_[h];
        const int e = i / n, a = i % n;
        if constexpr (of_x) xf[h * X0 + a][e] = *reinterpret_cast<const vec8_t<T> *>(smem + odd * STEP + (h * X0 * 2 + wm * xn[h] + a) * U * 128 + frag[e]);
        else wf[h * W0 + a][e] = *reinterpret_cast<const vec8_t<T> *>(smem + odd * STEP + ((X + h * W0) * 2 + wn * wn_[h] + a) * U * 128 + frag[e]);
    };
    constexpr int OW = GATED ? W0 : W;
    constexpr auto leaving = [](int left) { return left >= CB ? CB : left >= 2 ? 2 : 1; };     // blocks of columns at once, of those that are left
    constexpr auto lines = [](int nb) { return U * U * nb * SIZE >= 1024 ? U * U * nb * SIZE / 1024 : 1; };     // stores of a wave for them
    constexpr int STORES = [=] { int n = 0; for (int b = 0; b < OW; b += leaving(OW - b)) n += lines(leaving(OW - b)); return X * n; }();   // for a tile
    // Phase P of eight: products of a half of x with a half of w. It reads part P + 2 and asks for part P + 8, whose place part P has left.
    // In front of every second phase: parts P + 2 and P + 3 have landed, everyone has read P and P + 1. (`stored`: the last tile's results, asked
    // to be written behind the parts P + 2 .. 7, need not be.)
    auto phase = [&](auto pc, auto first_pair, int stored) {
        constexpr bool FIRST = decltype(first_pair)::value && decltype(pc)::value < 4;      // (its results are the first of its sums)
        constexpr int P = decltype(pc)::value, odd = P >> 2, k = P & 3;
        constexpr int xh = k >> 1, wh = ((k == 1 || k == 2) ? 1 : 0) ^ odd;
        if constexpr ((P & 1) == 0) {
            constexpr int OUT = fetches(P + 4, P + 8), LATE = decltype(first_pair)::value && P + 3 < 8 ? (OUT + STORES < 63 ? OUT + STORES : 63) : OUT;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (LATE > OUT)
                asm volatile("s_cmp_eq_u32 %0, 0\n\ts_cbranch_scc1 .Lplain%=\n\ts_waitcnt vmcnt(%2) lgkmcnt(0)\n\ts_branch .Lgo%=\n"
                             ".Lplain%=:\n\ts_waitcnt vmcnt(%1) lgkmcnt(0)\n.Lgo%=:" : : "s"(stored), "n"(OUT), "n"(LATE) : "memory", "scc");
            else
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(OUT) : "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        // reads and requests spread between the matrix steps
        constexpr int READS = E * blocks(P + 2), FETCHES = ASKS * blocks(P), NX = xn[xh], NW = wn_[wh], STEPS = E * NX * NW;
        constexpr int RUN = U == 32 ? 2 : 4, RUNS = (STEPS + RUN - 1) / RUN;
        int r = 0, f = 0;
#pragma unroll
        for (int run = 0; run < RUNS; ++run) {
            // (a pair of phases ends with a wait for the reads: those of the second are asked for early)
            const int r_to = min(READS, ((run + 1) * READS * (P & 1 ? 4 : 3) / 3 + RUNS - 1) / RUNS), f_to = (run + 1) * FETCHES / RUNS;
#pragma unroll
            for (int i = 0; i < READS; ++i)
                if (i >= r && i < r_to) read(Ic<P + 2>{}, i);
            r = r_to;
#pragma unroll
            for (int i = 0; i < FETCHES; ++i)
                if (i >= f && i < f_to) fetch(Ic<P>{}, i);
            f = f_to;
#pragma unroll
            for (int i = run * RUN; i < (run + 1) * RUN; ++i) {
                const int e = i / (NX * NW), a = xh * X0 + i % (NX * NW) / NW, b = wh * W0 + i % NW;
                if (FIRST && i < NX * NW) tile_mfma_to<ACC, true>(acc[a][b], wf[b][e], xf[a][e]);
                else if (i < STEPS) tile_mfma_to<ACC, false>(acc[a][b], wf[b][e], xf[a][e]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- the first pair of steps of the first tile ------------------------------------------------------------------------------------
    auto fetch_part = [&](auto jc) {
#pragma unroll
        for (int i = 0; i < ASKS * blocks(decltype(jc)::value); ++i) fetch(jc, i);
    };
    fetch_part(Ic<0>{}); fetch_part(Ic<1>{}); fetch_part(Ic<2>{}); fetch_part(Ic<3>{});
    ask_k = 128;
    fetch_part(Ic<4>{}); fetch_part(Ic<5>{}); fetch_part(Ic<6>{}); fetch_part(Ic<7>{});
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(fetches(2, 8)) : "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < E * X0; ++i) read(Ic<0>{}, i);
#pragma unroll
    for (int i = 0; i < E * W0; ++i) read(Ic<1>{}, i);

    for (int stored = 0, slot = 0;; stored = 1, slot ^= 1) {
        const int next = at + stride;
        Place then = {0, 0, 0, 0};
        if (next < last) then = place(next);
        int4v next_x = x_rsrc(then), next_w = w_rsrc(then);
        if (next >= last) next_x[2] = next_w[2] = 0;        // (no tile: nothing is fetched)
        else if constexpr (GATHER) fetch_list(then);
        auto ask_for = [&](int step) {
            const bool over = step >= steps;
            ask_k = static_cast<unsigned>(over ? step - steps : step) * 128;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                ask_x[i] = over ? next_x[i] : ask_x[i];
                ask_w[i] = over ? next_w[i] : ask_w[i];
            }
        };
        auto pair = [&](int s, auto first_pair) {
            ask_for(s + 2);
            if constexpr (GATHER && !decltype(first_pair)::value) {      // the next tile's first step: its rows, whose list came before this tile's second pair
                if (s + 2 == steps && next < last) x_offsets(then.rows, slot ^ 1);
            }
            phase(Ic<0>{}, first_pair, stored); phase(Ic<1>{}, first_pair, stored); phase(Ic<2>{}, first_pair, stored); phase(Ic<3>{}, first_pair, stored);
            ask_for(s + 3);
            phase(Ic<4>{}, first_pair, stored); phase(Ic<5>{}, first_pair, stored); phase(Ic<6>{}, first_pair, stored); phase(Ic<7>{}, first_pair, stored);
        };
        pair(0, std::true_type{});
#pragma nounroll
        for (int s = 2; s < steps; s += 2) pair(s, std::false_type{});
        // the last matrix steps have written their registers
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < X; ++a)
#pragma unroll
            for (int b = 0; b < W; ++b) {
                if constexpr (ACC) asm volatile("" : "+a"(acc[a][b]));
                else asm volatile("" : "+v"(acc[a][b]));
            }
        if constexpr (ACC) asm volatile("s_nop 15" : "+a"(acc[X - 1][W - 1]));
        else asm volatile("s_nop 15" : "+v"(acc[X - 1][W - 1]));

        // ---- results: U rows of 64 columns at a time through the wave's own piece of LDS, whole lines to memory. acc[a][b][4 q + k]: row U a
        // + lu, column U b + (256 / U) q + 4 lg + k. Stores beyond the rows or columns are dropped by the descriptor ----------------------
        char *mine = smem + PAIR + wave * U * PITCH;
        char *base = static_cast<char *>(p.out) + ((SLABS ? static_cast<int64_t>(here.expert) * p.M : 0) + here.row0) * ob + static_cast<int64_t>(here.col0) * SIZE;
        const int bytes = static_cast<int>(here.rows * ob - static_cast<int64_t>(here.col0) * SIZE), cols = p.N - here.col0;
        unsigned first = static_cast<unsigned>(wm * U * X * ob + wn * OUTW * SIZE);
        asm volatile("" : "+s"(first));     // (addresses made anew for every tile: kept, they cost the loop its registers)
#pragma unroll
        for (int a = 0; a < X; ++a) {
            float weight = 1.f;
            if constexpr (GATHER) {
                if (p.in_w) weight = reinterpret_cast<const float *>(smem + LISTS + 1024 + slot * 1024)[wm * U * X + a * U + lu];
            }
#pragma unroll
            for (int b0 = 0; b0 < OW; b0 += leaving(OW - b0)) {
                const int nb = leaving(OW - b0), pieces = nb * U * SIZE / 16;       // 16-byte pieces of a row
#pragma unroll
                for (int b = b0; b < b0 + nb; ++b)
#pragma unroll
                    for (int q = 0; q < U * U / 256; ++q) {
                        if constexpr (GATED) __builtin_amdgcn_sched_barrier(0);     // (one unit after the other: registers)
                        const int col = (b - b0) * U + q * (256 / U) + 4 * lg;
                        if constexpr (SLABS) {
                            const float4_t v = {acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
                            *reinterpret_cast<float4_t *>(mine + lu * PITCH + ((col >> 2) ^ (lu & 7)) * 16) = v;
                            continue;
                        }
                        vec4_t<T> v;
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const T y = to_t<T>(acc[a][b][4 * q + k]);
                            if constexpr (EXPERT && ACT > 0) {      // (of the fp32 products)
                                const float f = acc[a][b][4 * q + k] * weight, g = GATED ? acc[a][(W0 + b) % W][4 * q + k] * weight : 0.f;
                                if constexpr (ACT == 1) v[k] = to_t<T>(fmaxf(f, 0.f) * fmaxf(f, 0.f));
                                else if constexpr (ACT == 2) v[k] = to_t<T>(tile_silu_1702(fminf(f, p.limit)) * (fminf(fmaxf(g, -p.limit), p.limit) + 1.0f));
                                else v[k] = to_t<T>(tile_silu(f) * g);
                            } else if constexpr (GATED) {
                                const float f = to_f(y), g = to_f(to_t<T>(acc[a][W0 + b][4 * q + k]));
                                if constexpr (ACT == 2) {
                                    v[k] = to_t<T>(tile_silu_1702(fminf(f, p.limit)) * (fminf(fmaxf(g, -p.limit), p.limit) + 1.0f));
                                } else if constexpr (ACT == 3) {
                                    v[k] = to_t<T>(tile_silu(f) * g);
                                } else if constexpr (ACT == 4) {
                                    v[k] = to_t<T>(tile_silu(g) * f);
                                } else {
                                    v[k] = mul_t<T>(y, to_t<T>(tile_silu(g)));
                                }
                            } else if constexpr (ACT == 1) {
                                const float f = fmaxf(to_f(y), 0.f);
                                v[k] = here.col0 + wn * OUTW + b * U + q * (256 / U) + 4 * lg < p.act_cols ? to_t<T>(f * f) : y;
                            } else {
                                v[k] = y;
                            }
                        }
                        *reinterpret_cast<vec4_t<T> *>(mine + lu * PITCH + (((col >> 3) ^ (lu & 7)) * 16 + (col & 4) * 2)) = v;
                    }
                const int c = lane & (pieces - 1), r0 = lane / pieces;
                unsigned off = static_cast<unsigned>(r0 * ob + c * 16) + first;
                if (c * (16 / SIZE) >= cols - wn * OUTW - b0 * U || r0 >= U) off = 0x80000000u;
                vec8_t<T> line[lines(CB)];
#pragma unroll
                for (int i = 0; i < lines(nb); ++i) {
                    const int r = (i * (64 / pieces) + r0) & (U - 1);
                    line[i] = *reinterpret_cast<const vec8_t<T> *>(mine + r * PITCH + ((c ^ (r & 7)) * 16));
                }
                const __amdgpu_buffer_rsrc_t rsrc =
                    __builtin_amdgcn_make_buffer_rsrc(base + a * U * ob + b0 * U * SIZE, 0, max(0, bytes - static_cast<int>(a * U * ob) - b0 * U * SIZE), 0x00020000);
#pragma unroll
                for (int i = 0; i < lines(nb); ++i)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, line[i]), rsrc, static_cast<int>(off + i * static_cast<unsigned>(64 / pieces * ob)), 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (next >= last) break;
        at = next, here = then;
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
}

template <typename T, int U, int X0, int X1, int W0, int W1, int ACT, int ROWS = kTileDense>
int gemm_tile_launch(GemmTileParams p, hipStream_t s) {
    constexpr int BM = 2 * U * (X0 + X1), BN = 2 * U * (W0 + W1) / (ACT >= 2 ? 2 : 1), A_CU = U * U * (X0 + X1) * (W0 + W1) <= 4096 ? 2 : 1;
    p.n_tiles = (p.N + BN - 1) / BN;
    if constexpr (ACT == kTileSlabs) p.share = Divisor::of(p.n_tiles), p.n_tiles *= p.splits;
    // (experts: as many row tiles as there can be, each of theirs may end in a part of one; how many there are is on the device)
    p.m_tiles = (p.M + BM - 1) / BM + (ROWS == kTileDense ? 0 : min(p.experts, p.M));
    const int64_t tiles = static_cast<int64_t>(p.m_tiles) * p.n_tiles;
    if (tiles > (1 << 27)) return SWL_ERR_UNSUPPORTED;
    const unsigned rest = p.m_tiles % kTileGroup;
    p.group = Divisor::of(kTileGroup * p.n_tiles);
    p.wide = Divisor::of(kTileGroup);
    p.rest = Divisor::of(rest ? rest : kTileGroup);
    const unsigned grid = static_cast<unsigned>(tiles < 256 * A_CU ? (tiles + 7) / 8 * 8 : 256 * A_CU);
    hipLaunchKernelGGL((gemm_tile_kernel<T, U, X0, X1, W0, W1, ACT, ROWS>), dim3(grid), dim3(256), 0, s, p);
    return check_launch();
}

// The tiles that there are: rows and rows of w in 32s. The last two share a CU, the others take one each.
struct TileShape {
    int x, w;
};
constexpr TileShape kTileShapes[] = {{8, 8}, {6, 8}, {6, 6}, {5, 8}, {7, 8}, {8, 6}, {5, 4}, {5, 6}, {7, 6}, {4, 4}, {2, 4}};
constexpr int kTileShapeCount = 11;
constexpr unsigned kTilesPlain = 0x7ff, kTilesAct = 0x63f;      // with an activation: not 160 x 128, 160 x 192 and 224 x 192

// Which tile of the set: the one whose time a model of turns and steps has as the least, us = 1.86 + turns (steps of 128 columns (0.0134 x w + 0.0667 (x +
// w)) + 0.0666 x w) + 0.0123 x w steps tiles / 256, for two tiles a CU by turns of whole and of half filled CUs: fitted to 270 products (260 to 8192
// tokens, 1024 to 28672 rows of w, 1024 to 14336 columns; bf16), 4 % to 8 % off; what it picks takes 1.004 times the best one's time.
// tiles(rows, rows of w): how many. (Six tiles instead of eleven: 1.05 of the time, 1.08 to 1.14 for 1828 of 28672 x 4096, 4498 of 2048 x 2048, 3657 of
// 2048 x 8192, 5112 of 4096 x 4096.)
template <typename Tiles>
int gemm_tile_shape(Tiles &&tiles, int64_t k, unsigned set, double *us_out = nullptr) {
    const double p = static_cast<double>(k) / 128;
    auto one = [&](const TileShape &s) {
        const int64_t t = tiles(32 * s.x, 32 * s.w), turns = ((t + 7) / 8 + 31) / 32;
        const double area = s.x * s.w;
        return 1.86 + turns * (p * (0.0134 * area + 0.0667 * (s.x + s.w)) + 0.0666 * area) + 0.0123 * area * p * t / 256;
    };
    auto two = [&](const TileShape &s, double start, double a, double b, double half, double c) {
        const int64_t t = tiles(32 * s.x, 32 * s.w), each = (t + 7) / 8, rest = each % 64, full = each / 64 + (rest > 32), part = rest > 0 && rest <= 32;
        return start + full * p * a + (full + part) * b + part * p * half + p * t / 256 * c;
    };
    int best = -1;
    double least = 0;
    for (int i = 0; i < kTileShapeCount; ++i) {
        if (!(set >> i & 1)) continue;
        const TileShape &s = kTileShapes[i];
        const double us = i == 9 ? two(s, 1.81, 1.03, 0.78, 0.63, 0.42) : i == 10 ? two(s, 2.29, 0.85, 0.0, 0.55, 0.20) : one(s);
        if (best < 0 || us < least) best = i, least = us;
    }
    if (us_out) *us_out = least;
    return best + 1;
}

} // namespace swl
