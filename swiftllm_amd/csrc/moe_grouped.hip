// moe_grouped.hip — the expert products of prompt-sized steps: assignments sorted by expert on the device, then ONE matrix-core
// launch per product for all experts (16-bit storage, fp32 accumulation).
//
// A library product per expert leaves most of the chip idle at these sizes (2048 x 1024 x 1024: 128 tiles for 256 CUs) and needs the experts' row
// counts on the host: a read-back and the launches' gaps behind it in every layer. Here the tiles of all experts are one list. Token rows are
// gathered by the staging itself (no sorted copy of the inputs), the gated unit or the squared ReLU runs on the fp32 products in the
// epilogue, and results leave as whole lines through LDS.
//   * Reductions of whole steps of 128 columns, up to 512 experts: the tiles of gemm_tile.h, which says what bounds them. Every workgroup counts the
//     experts' tiles from the sorted assignments; a tile's assignments come to LDS while the tile before it is multiplied.
//   * Others: a tile of 128 assignments of one expert x 128 weight rows a workgroup of four waves, each a 64 x 64 piece (mfma 32x32x16, 2 x 2
//     accumulators), operands in 64-deep slices (tile_product.h). Bound by what a CU takes from L2 (32 KiB per 64 columns) beside the matrix steps.
// Measured (us, bf16, by the second / by the first, gate/up with the unit, then down): 9000 assignments over 8 experts, width and ff 2048: 193 / 165, 89 / 73;
// 7314: 147 / 113, 69 / 54; 15252, width and ff 1024: 75 / 60, 37 / 31; 1400, 2048: 40 / 33, 26 / 19; 200: 32 / 24, 22 / 16; 64000 over 64, width 2048, ff 1024: 637 /
// 475, 320 / 255. (Before the exponential and the quotient of gemm_tile.h's units were as exact as the second's: with rows spread evenly over cold weights gate/up then
// and now 151 / 156 at the first of these sizes, 113 / 115, 60 / 64, 46 / 47, 39 / 40, 474 / 483.) Passes of 3 x 1500, 11 x 333 and 4 x 2000 tokens with experts in two of four layers or in all: 1.05, 1.04, 1.06.
#include "gemm_tile.h"
#include "tile_product.h"

namespace swl {

constexpr int kSortThreads = 1024;

// One workgroup per expert: how many assignments go to lower experts, then a stable list of its own. Bound by latency: a thread asks for its
// I consecutive ids at once (16 bytes a load) and counts, scans and places from registers, one barrier for 1024 I assignments.
// Measured (us, launches back to back, ids read twice and one at a time -> now, I = 4 up to 4096 assignments, else 16): 4096 over 8 experts 4.6 ->
// 4.3, 9000 7.8 -> 5.5, 16000 11.2 -> 6.6, 16384 over 64 10.8 -> 5.4, 40000 over 128 22.3 -> 10.3.
template <int I>
__global__ __launch_bounds__(kSortThreads) void moe_sort_kernel(int32_t *order, int64_t *where, int32_t *offsets, const int32_t *idx,
                                                                int n, int experts) {
    constexpr int kWaves = kSortThreads / 64, kPiece = I * kSortThreads;
    __shared__ int part[2][kWaves], low[kWaves];
    const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool whole = (reinterpret_cast<uintptr_t>(idx) & 15u) == 0;
    int id[I];      // (past the end: no expert)
    auto load = [&](int i0) {
        const int at = i0 + I * tid;
        if (whole && at + I <= n) {
#pragma unroll
            for (int k = 0; k < I; k += 4) {
                const int4 v = *reinterpret_cast<const int4 *>(idx + at + k);
                id[k] = v.x, id[k + 1] = v.y, id[k + 2] = v.z, id[k + 3] = v.w;
            }
#pragma unroll
            for (int k = 0; k < I; ++k) id[k] = min(max(id[k], 0), experts - 1);
        } else {
#pragma unroll
            for (int k = 0; k < I; ++k) id[k] = at + k < n ? min(max(idx[at + k], 0), experts - 1) : experts;
        }
    };
    int lower = 0;
    auto count_lower = [&] {
#pragma unroll
        for (int k = 0; k < I; ++k) lower += id[k] < e;
    };
    for (int i0 = kPiece; i0 < n; i0 += kPiece) {
        load(i0);
        count_lower();
    }
    load(0);
    count_lower();
    for (int o = 32; o > 0; o >>= 1) lower += __shfl_xor(lower, o, 64);
    if (lane == 0) low[wave] = lower;       // (read behind the first piece's barrier)
    int base = 0;
    for (int i0 = 0, turn = 0; turn == 0 || i0 < n; i0 += kPiece, ++turn) {
        if (turn > 0) load(i0);
        int mine = 0;
#pragma unroll
        for (int k = 0; k < I; ++k) mine += id[k] == e;
        int scan = mine;
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(scan, o, 64);
            if (lane >= o) scan += v;
        }
        if (lane == 63) part[turn & 1][wave] = scan;
        __syncthreads();
        if (turn == 0) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) base += low[w];
            if (tid == 0) {
                offsets[e] = base;
                if (e == experts - 1) offsets[experts] = n;
            }
        }
        int before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int v = part[turn & 1][w];
            before += w < wave ? v : 0;
            all += v;
        }
        int pos = base + before + scan - mine;
        const int at = i0 + I * tid;
#pragma unroll
        for (int k = 0; k < I; ++k)
            if (id[k] == e) {
                order[pos] = at + k;
                where[at + k] = pos++;
            }
        base += all;
    }
}

struct MoeGemmParams {
    void *out;
    const void *x, *w;
    const int32_t *order, *offsets;     // order NULL: row i of x belongs to sorted position i
    const float *in_w;
    int top, experts, K, N, act, n_tiles;
    float limit;
};

// The tile of this workgroup: every XCD (workgroup id % 8) takes an equal run of the tiles that there are, row tiles eight at a time with
// all their column tiles, the row tile fastest: what an XCD works on at once is about as many rows as columns of weights.
struct MgTile {
    int expert, row0, rows, n_tile;     // expert < 0: no tile
};
__device__ __forceinline__ MgTile mg_tile(const MoeGemmParams &p) {
    constexpr int GROUP = 8;
    const int lane = threadIdx.x & 63;
    int a = 0, b = 0;
    // row tiles of 64 experts, counted by a scan over the wave
    auto tiles_to = [&](int e0) {
        const int e = min(e0 + lane, p.experts - 1);
        a = p.offsets[e];
        b = e0 + lane < p.experts ? p.offsets[e + 1] : a;
        int scan = (b - a + kTile - 1) / kTile;
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(scan, o, 64);
            if (lane >= o) scan += v;
        }
        return scan;
    };
    int total = 0;
    for (int e0 = 64; e0 < p.experts; e0 += 64) total += __builtin_amdgcn_readlane(tiles_to(e0), 63);
    int scan = tiles_to(0);
    total += __builtin_amdgcn_readlane(scan, 63);
    const int64_t all = static_cast<int64_t>(total) * p.n_tiles;
    const int xcd = blockIdx.x & 7;
    const int64_t at = xcd * all / 8 + (blockIdx.x >> 3);
    MgTile t = {-1, 0, 0, 0};
    if (at >= (xcd + 1) * all / 8) return t;
    const int group = static_cast<int>(at / (GROUP * static_cast<int64_t>(p.n_tiles)));
    const int in_group = static_cast<int>(at - group * (GROUP * static_cast<int64_t>(p.n_tiles)));
    const int wide = min(GROUP, total - GROUP * group);
    t.n_tile = in_group / wide;
    int m_tile = GROUP * group + in_group - t.n_tile * wide;
    for (int e0 = 0; e0 < p.experts; e0 += 64) {
        if (e0 > 0) scan = tiles_to(e0);
        const unsigned long long past = __ballot(scan > m_tile);
        if (past) {
            const int l = __builtin_ctzll(past);
            const int lo = __builtin_amdgcn_readlane(a, l), hi = __builtin_amdgcn_readlane(b, l);
            t.expert = e0 + l;
            t.row0 = lo + (m_tile - __builtin_amdgcn_readlane(scan, l) + (hi - lo + kTile - 1) / kTile) * kTile;
            t.rows = min(kTile, hi - t.row0);
            break;
        }
        m_tile -= __builtin_amdgcn_readlane(scan, 63);
    }
    return t;
}

// MODE 0: out[pos][N] = x w^T; 1: w rows [N gate | N up], out = gated unit; 2: out = relu(x w^T)^2
// BUFS staged slices: 2 with two workgroups a CU, a slice on its way while one is multiplied; 1 with four workgroups a CU, which hide
// each other's waits, first and last slices too.
template <typename T, int MODE, int BUFS>
__global__ __launch_bounds__(256, BUFS == 1 ? 4 : 2) void moe_gemm_kernel(MoeGemmParams p) {
    constexpr int OUTC = MODE == 1 ? 64 : 128, PITCH = OUTC + 8;          // output columns of a tile, elements between its rows in LDS
    constexpr int STAGED = BUFS * 2 * kTileSliceB, RESULT = kTile * PITCH * 2;
    __shared__ __attribute__((aligned(16))) char smem[STAGED > RESULT ? STAGED : RESULT];      // [buffer][weights, tokens]; then the output tile
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hf = lane >> 5, wn = wave & 1, wm = wave >> 1;
    const MgTile t = mg_tile(p);
    if (t.expert < 0) return;
    const int row0 = t.row0, rows = t.rows, n_tile = t.n_tile;

    // ---- staging --------------------------------------------------------------------------------------------------------------------
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    unsigned w_off[4], x_off[4];
    const int64_t kb = static_cast<int64_t>(p.K) * 2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = tile_row(wave, i, lane), unit = tile_unit(r, lane);
        int wr;
        if (MODE == 1) {        // a wave's 64 weight rows: 32 gate rows, then the up rows of the same columns
            const int c = min(n_tile * 64 + (r >> 6) * 32 + (r & 31), p.N - 1);
            wr = (r & 32) ? p.N + c : c;
        } else {
            wr = min(n_tile * 128 + r, p.N - 1);
        }
        w_off[i] = static_cast<unsigned>(wr * kb + unit * 16);
        const int pos = row0 + min(r, rows - 1);
        const int xr = p.order ? p.order[pos] / p.top : pos;
        x_off[i] = static_cast<unsigned>(xr * kb + unit * 16);
    }
    const char *wb = static_cast<const char *>(p.w) + static_cast<int64_t>(t.expert) * (MODE == 1 ? 2 : 1) * p.N * kb;
    const char *xb = static_cast<const char *>(p.x);
    float16_t acc[2][2];        // [weight piece][token piece]
    tile_product<T, BUFS, false>(smem, p.K / kTileDepth, wn, wm, lane, acc, [&](int st) {
        const char *ws = wb + static_cast<int64_t>(st) * kTileDepth * 2, *xs = xb + static_cast<int64_t>(st) * kTileDepth * 2;
        const unsigned to = lds0 + static_cast<unsigned>((st & (BUFS - 1)) * 2 * kTileSliceB + wave * 4096);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            tile_ask(ws, w_off[i], to + i * 1024);
            tile_ask(xs, x_off[i], to + kTileSliceB + i * 1024);
        }
    });
    // ---- epilogue: acc[a][b][4 q + r] = product (weight row 64 wn + 32 a + 8 q + 4 hf + r, token 64 wm + 32 b + l32) ----------------
    __syncthreads();        // every wave is done with the staged slices
    T *tile = reinterpret_cast<T *>(smem);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int r = wm * 64 + b * 32 + l32;
        float scale = 1.f;
        if (MODE == 1 && p.in_w) scale = p.in_w[p.order[row0 + min(r, rows - 1)]];
#pragma unroll
        for (int a = 0; a < (MODE == 1 ? 1 : 2); ++a)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                vec4_t<T> v;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float y = acc[a][b][4 * q + k];
                    if constexpr (MODE == 1) {
                        float g = y * scale, u = acc[1][b][4 * q + k] * scale;
                        if (p.act == 1) {
                            y = g / (1.0f + expf(-g)) * u;
                        } else {
                            g = fminf(g, p.limit);
                            u = fminf(fmaxf(u, -p.limit), p.limit);
                            y = g * (1.0f / (1.0f + expf(-1.702f * g))) * (u + 1.0f);
                        }
                    } else if constexpr (MODE == 2) {
                        y = fmaxf(y, 0.f);
                        y *= y;
                    }
                    v[k] = to_t<T>(y);
                }
                *reinterpret_cast<vec4_t<T> *>(tile + r * PITCH + wn * (OUTC / 2) + a * 32 + 8 * q + 4 * hf) = v;
            }
    }
    __syncthreads();
    T *out = static_cast<T *>(p.out);
    constexpr int CPR = OUTC / 8;       // 16-byte pieces of a row
    for (int i = tid; i < kTile * CPR; i += 256) {
        const int r = i / CPR, c = (i - r * CPR) * 8;
        if (r < rows && n_tile * OUTC + c < p.N)
            store8(out + static_cast<int64_t>(row0 + r) * p.N + n_tile * OUTC + c, *reinterpret_cast<const vec8_t<T> *>(tile + r * PITCH + c));
    }
}

// An expert's last row tile is taken as half full.
constexpr unsigned kTilesExperts = 1u << 0 | 1u << 1 | 1u << 2 | 1u << 5 | 1u << 9;
template <typename T, int ACT, int ROWS>
int moe_gemm_dispatch(const GemmTileParams &p, int64_t w_rows, hipStream_t s) {
    auto tiles = [&](int rows, int cols) { return (p.M / rows + (min(p.experts, p.M) + 1) / 2) * ((w_rows + cols - 1) / cols); };
    switch (gemm_tile_shape(tiles, p.K, kTilesExperts)) {
    case 1: return gemm_tile_launch<T, 16, 4, 4, 4, 4, ACT, ROWS>(p, s);
    case 2: return gemm_tile_launch<T, 16, 3, 3, 4, 4, ACT, ROWS>(p, s);
    case 3: return gemm_tile_launch<T, 16, 3, 3, 3, 3, ACT, ROWS>(p, s);
    case 6: return gemm_tile_launch<T, 16, 4, 4, 3, 3, ACT, ROWS>(p, s);
    default: return gemm_tile_launch<T, 16, 2, 2, 2, 2, ACT, ROWS>(p, s);
    }
}

} // namespace swl

extern "C" int swl_moe_sort(int32_t *order, int64_t *where, int32_t *offsets, const int32_t *expert_idx, int64_t num_assignments,
                            int32_t experts, swl_stream_t stream) {
    if (num_assignments < 0 || experts <= 0) return SWL_ERR_BAD_ARG;
    if (num_assignments > (1 << 30)) return SWL_ERR_UNSUPPORTED;
    if (!order || !where || !offsets || !expert_idx) return SWL_ERR_BAD_ARG;
    const auto kernel = num_assignments <= 4 * swl::kSortThreads ? swl::moe_sort_kernel<4> : swl::moe_sort_kernel<16>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(experts)), dim3(swl::kSortThreads), 0,
                       static_cast<hipStream_t>(stream), order, where, offsets, expert_idx, static_cast<int>(num_assignments), experts);
    return swl::check_launch();
}

/* 1 when swl_moe_gemm serves products of these sizes: 16-bit, a reduction of whole 64-deep slices, rows of whole 16-byte pieces, and
 * operand rows within 4 GiB of their matrix's start. */
extern "C" int swl_moe_gemm_supported(int64_t x_rows, int32_t K, int32_t N, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    if (x_rows <= 0 || K <= 0 || N <= 0 || K % swl::kTileDepth || N % 8) return 0;
    const int64_t row = static_cast<int64_t>(K) * 2;
    return x_rows * row < (1LL << 32) && 2LL * N * row < (1LL << 32);
}

extern "C" int swl_moe_gemm(void *out, const void *x, const void *w, const int32_t *order, const int32_t *offsets, const float *in_w,
                            int64_t num_assignments, int64_t x_rows, int32_t top, int32_t experts, int32_t K, int32_t N, int32_t mode,
                            int32_t act, float limit, int32_t dtype, swl_stream_t stream) {
    if (num_assignments < 0 || experts <= 0 || top <= 0 || mode < 0 || mode > 2 || act < 0 || act > 1) return SWL_ERR_BAD_ARG;
    if (in_w && (mode != 1 || !order)) return SWL_ERR_BAD_ARG;
    if (num_assignments == 0) return SWL_OK;
    if (!swl_moe_gemm_supported(x_rows, K, N, dtype)) return SWL_ERR_UNSUPPORTED;
    // (rows of x: assignments when sorted, else tokens)
    if (order ? x_rows * top < num_assignments : x_rows < num_assignments) return SWL_ERR_BAD_ARG;
    if (!out || !x || !w || !offsets || !swl::aligned16(out) || !swl::aligned16(x) || !swl::aligned16(w)) return SWL_ERR_BAD_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (K >= 256 && K % 128 == 0 && experts <= swl::kTileExperts && num_assignments <= (1 << 29) && 256LL * K * 2 < (1LL << 31) && 512LL * N < (1LL << 31)) {
        swl::GemmTileParams p = {};
        p.out = out; p.x = x; p.w = w; p.M = static_cast<int>(num_assignments); p.N = N; p.K = K; p.ldx = K; p.ldo = N; p.limit = limit;
        p.order = order; p.offsets = offsets; p.in_w = in_w; p.experts = experts; p.top = swl::Divisor::of(static_cast<unsigned>(top));
        p.x_bytes = static_cast<unsigned>(x_rows * K * 2); p.in_w_bytes = static_cast<unsigned>(num_assignments * 4);
        const int64_t w_rows = mode == 1 ? 2LL * N : N;
        SWL_DISPATCH_DTYPE(dtype, T, {
            if (order) {
                if (mode == 0) return swl::moe_gemm_dispatch<T, 0, swl::kTileGather>(p, w_rows, s);
                if (mode == 2) return swl::moe_gemm_dispatch<T, 1, swl::kTileGather>(p, w_rows, s);
                return act == 0 ? swl::moe_gemm_dispatch<T, 2, swl::kTileGather>(p, w_rows, s) : swl::moe_gemm_dispatch<T, 3, swl::kTileGather>(p, w_rows, s);
            }
            if (mode == 0) return swl::moe_gemm_dispatch<T, 0, swl::kTileExpert>(p, w_rows, s);
        });
    }
    swl::MoeGemmParams p;
    p.out = out; p.x = x; p.w = w; p.order = order; p.offsets = offsets; p.in_w = in_w;
    p.top = top; p.experts = experts; p.K = K; p.N = N; p.act = act; p.limit = limit;
    const int cols = mode == 1 ? 64 : 128;
    p.n_tiles = (N + cols - 1) / cols;
    // as many row tiles as there can be (every expert may end in a part of one); surplus workgroups leave at once
    const int64_t m_tiles = (num_assignments + swl::kTile - 1) / swl::kTile + (experts < num_assignments ? experts : num_assignments);
    const int64_t grid = (m_tiles * p.n_tiles + 7) / 8 * 8;
    if (grid > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    // One staged slice and four workgroups a CU where there are more tiles than two a CU (about: an expert's last row tile half full),
    // else two slices: 31.3 and 35.7 us at 688 tiles (4950 rows, width and ff 1024, gate/up), 39.1 and 36.6 at 512, 20.7 and 19.3 at 344.
    const bool many = (num_assignments + 64LL * experts) / swl::kTile * p.n_tiles > 512;
#define SWL_MG(MODE, BUFS) hipLaunchKernelGGL((swl::moe_gemm_kernel<T, MODE, BUFS>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, s, p)
#define SWL_MG2(MODE) do { if (many) SWL_MG(MODE, 1); else SWL_MG(MODE, 2); } while (0)
    SWL_DISPATCH_DTYPE(dtype, T, {
        if (mode == 0) SWL_MG2(0);
        else if (mode == 1) SWL_MG2(1);
        else SWL_MG2(2);
    });
#undef SWL_MG2
#undef SWL_MG
    return swl::check_launch();
}
