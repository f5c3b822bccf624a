// latent_expand.hip — the cached rows of a latent attention (normed latent | rotated shared key part) expanded to the keys and values of
// every head, as pages that the attention of prompt portions walks (span_attn.hip):
//     key   h, t: [ W_uk,h c_t | rotated part of t ]       value h, t: W_uv,h c_t        (transposed pages, as in the pool)
//
// Why: a prompt's queries folded through W_uk attend to rows of rank + rot columns and sum values of `rank`; expanded, a (query, key, head)
// takes dim + rot + 2 vdim column steps instead of 3 rank + rot (values count twice, in two 16-bit terms): 448 instead of 1600 at 128 + 64,
// 128 and rank 512. The expansion is one product of the cached rows with both matrices, which is what folding the queries in and unfolding
// the values took. Decoded tokens read few queries' worth of keys and stay folded (worker/batch_plan.py, LatentExpansion.pays, has the rule).
// What bounds it: as the expert products (moe_grouped.hip), a CU's share of L2: a workgroup takes 128 cached tokens x 128 columns
// (tile_product.h), 8 pages whose rows the staging picks up one page an instruction; every XCD takes an equal run of the row tiles with all
// their column tiles, so that its L2 holds a few of the rows and the matrices. Results leave as whole lines through LDS.
#include "tile_product.h"

namespace swl {

struct ExpandParams {
    void *out;
    const void *k_cache, *uk, *uv;
    const int32_t *block_table, *page_row, *page_no, *page_dst;
    int pages, max_blocks, H, d, e, dr, rank, k_dim, k_tiles, v_tiles, row_tiles;
    int64_t block_stride;
};

constexpr int kExpandPages = kTile / 16, kExpandPitch = kTile + 8;

template <typename T>
__global__ __launch_bounds__(256, 4) void latent_expand_kernel(ExpandParams p) {
    constexpr int RESULT = kTile * kExpandPitch * 2, STAGED = 2 * kTileSliceB;
    __shared__ __attribute__((aligned(16))) char smem[STAGED > RESULT ? STAGED : RESULT];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hf = lane >> 5, wn = wave & 1, wm = wave >> 1;
    // ---- which tile -----------------------------------------------------------------------------------------------------------------
    const int per_head = p.k_tiles + p.v_tiles, cols = p.H * per_head, all = p.row_tiles * cols, xcd = blockIdx.x & 7;
    const int first = static_cast<int>(static_cast<int64_t>(xcd) * all / 8), last = static_cast<int>(static_cast<int64_t>(xcd + 1) * all / 8);
    const int at = first + static_cast<int>(blockIdx.x >> 3);
    if (at >= last) return;
    const int row_tile = at / cols, col_tile = at - row_tile * cols, head = col_tile / per_head, part = col_tile - head * per_head;
    const bool value = part >= p.k_tiles;
    const int col0 = (value ? part - p.k_tiles : part) * kTile, width = value ? p.e : p.d;
    // this tile's pages (lane l % 8: page l % 8 of it; past the last one, that one again)
    const int entry = min(row_tile * kExpandPages + (lane & 7), p.pages - 1);
    const int blk = p.block_table[static_cast<int64_t>(p.page_row[entry]) * p.max_blocks + p.page_no[entry]];
    const char *kc = static_cast<const char *>(p.k_cache);
    const int64_t bstride = p.block_stride * 2;

    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    unsigned w_off[4], x_off[4];
    const char *xb[2];      // rows of an instruction are of one page: two pages a wave
#pragma unroll
    for (int i = 0; i < 2; ++i) xb[i] = kc + __builtin_amdgcn_readlane(blk, 2 * wave + i) * bstride;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = tile_row(wave, i, lane), unit = tile_unit(r, lane);
        w_off[i] = static_cast<unsigned>((min(col0 + r, width - 1) * p.rank + unit * 8) * 2);
        x_off[i] = static_cast<unsigned>(((r & 15) * p.k_dim + unit * 8) * 2);
    }
    const char *wb = static_cast<const char *>(value ? p.uv : p.uk) + static_cast<int64_t>(head) * width * p.rank * 2;
    auto issue = [&](int st) {
        const int64_t depth = static_cast<int64_t>(st) * kTileDepth * 2;
        const unsigned to = lds0 + static_cast<unsigned>(wave * 4096);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            tile_ask(wb + depth, w_off[i], to + i * 1024);
            tile_ask(xb[i >> 1] + depth, x_off[i], to + kTileSliceB + i * 1024);
        }
    };
    float16_t acc[2][2];
    T *tile = reinterpret_cast<T *>(smem);
    const int stages = p.rank / kTileDepth, kd = p.d + p.dr;
    const int64_t page_elems = static_cast<int64_t>(p.H) * 16 * (kd + p.e);
    T *out = static_cast<T *>(p.out);
    auto put = [&](int a, int b, int row, int col) {        // four results of an accumulator at a time to columns col + 8 q of the tile's row
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            vec4_t<T> v;
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = to_t<T>(acc[a][b][4 * q + k]);
            *reinterpret_cast<vec4_t<T> *>(tile + row * kExpandPitch + col + 8 * q) = v;
        }
    };
    if (value) {        // the tile by columns: what a page's transposed values hold together lies together
        tile_product<T, 1, true>(smem, stages, wn, wm, lane, acc, issue);
        __syncthreads();        // every wave is done with the staged slices
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) put(a, b, wn * 64 + b * 32 + l32, wm * 64 + a * 32 + 4 * hf);
        __syncthreads();
        for (int i = tid; i < kTile * 16; i += 256) {
            const int half = i & 1, c = (i >> 1) & (kTile - 1), slot = i >> 8, at_page = row_tile * kExpandPages + slot;
            if (at_page < p.pages && col0 + c < p.e)
                store8(out + p.page_dst[at_page] * page_elems + static_cast<int64_t>(p.H) * 16 * kd + (static_cast<int64_t>(head) * p.e + col0 + c) * 16 + half * 8,
                       *reinterpret_cast<const vec8_t<T> *>(tile + c * kExpandPitch + slot * 16 + half * 8));
        }
        return;
    }
    tile_product<T, 1, false>(smem, stages, wn, wm, lane, acc, issue);
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) put(a, b, wm * 64 + b * 32 + l32, wn * 64 + a * 32 + 4 * hf);
    __syncthreads();
    for (int i = tid; i < kTile * 16; i += 256) {
        const int r = i >> 4, c = (i & 15) * 8, at_page = row_tile * kExpandPages + (r >> 4);
        if (at_page < p.pages && col0 + c < p.d)
            store8(out + p.page_dst[at_page] * page_elems + static_cast<int64_t>(head) * 16 * kd + (r & 15) * kd + col0 + c,
                   *reinterpret_cast<const vec8_t<T> *>(tile + r * kExpandPitch + c));
    }
    if (col0 > 0) return;
    const int pieces = p.dr / 8;        // the rotated part, the same for every head
    for (int i0 = 0; i0 < kTile * pieces; i0 += 256) {
        const int i = i0 + tid, r = min(i / pieces, kTile - 1), c = (i - i / pieces * pieces) * 8, at_page = row_tile * kExpandPages + (r >> 4);
        const int64_t from = __shfl(blk, r >> 4, 64);       // (every lane of the wave takes part)
        if (i < kTile * pieces && at_page < p.pages)
            store8(out + p.page_dst[at_page] * page_elems + static_cast<int64_t>(head) * 16 * kd + (r & 15) * kd + p.d + c,
                   load8(reinterpret_cast<const T *>(kc + from * bstride) + (r & 15) * p.k_dim + p.rank + c));
    }
}

} // namespace swl

/* 1 when swl_latent_expand serves these sizes: 16-bit, whole 64-deep slices of the latent, 16-byte pieces of everything else. */
extern "C" int swl_latent_expand_supported(int32_t dim, int32_t vdim, int32_t rot_dim, int32_t kv_rank, int32_t k_dim, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    if (dim <= 0 || vdim <= 0 || rot_dim <= 0 || kv_rank <= 0 || k_dim < kv_rank + rot_dim) return 0;
    if (dim > 4096 || vdim > 4096 || kv_rank > 4096 || k_dim > 65536) return 0;
    return kv_rank % swl::kTileDepth == 0 && dim % 8 == 0 && vdim % 8 == 0 && rot_dim % 8 == 0 && k_dim % 8 == 0;
}

extern "C" int swl_latent_expand(void *out, const void *k_cache, const void *uk, const void *uv, const int32_t *block_table,
                                 const int32_t *page_row, const int32_t *page_no, const int32_t *page_dst, int64_t num_pages,
                                 int32_t num_heads, int32_t dim, int32_t vdim, int32_t rot_dim, int32_t kv_rank, int32_t k_dim,
                                 int32_t max_blocks_per_seq, int64_t block_stride, int32_t dtype, swl_stream_t stream) {
    if (num_pages < 0 || num_heads <= 0 || max_blocks_per_seq <= 0) return SWL_ERR_BAD_ARG;
    if (!swl_latent_expand_supported(dim, vdim, rot_dim, kv_rank, k_dim, dtype)) return SWL_ERR_UNSUPPORTED;
    if (num_pages == 0) return SWL_OK;
    if (!out || !k_cache || !uk || !uv || !block_table || !page_row || !page_no || !page_dst) return SWL_ERR_BAD_ARG;
    if (!swl::aligned16(out) || !swl::aligned16(k_cache) || !swl::aligned16(uk) || !swl::aligned16(uv) || (block_stride & 7)) return SWL_ERR_BAD_ARG;
    swl::ExpandParams p;
    p.out = out; p.k_cache = k_cache; p.uk = uk; p.uv = uv;
    p.block_table = block_table; p.page_row = page_row; p.page_no = page_no; p.page_dst = page_dst;
    p.max_blocks = max_blocks_per_seq; p.H = num_heads; p.d = dim; p.e = vdim; p.dr = rot_dim; p.rank = kv_rank; p.k_dim = k_dim;
    p.k_tiles = (dim + swl::kTile - 1) / swl::kTile;
    p.v_tiles = (vdim + swl::kTile - 1) / swl::kTile;
    p.block_stride = block_stride;
    const int64_t row_tiles = (num_pages + swl::kExpandPages - 1) / swl::kExpandPages;
    const int64_t all = row_tiles * num_heads * (p.k_tiles + p.v_tiles), grid = (all + 7) / 8 * 8;
    if (num_pages > (1 << 30) || grid > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    p.pages = static_cast<int>(num_pages);
    p.row_tiles = static_cast<int>(row_tiles);
    SWL_DISPATCH_DTYPE(dtype, T, {
        hipLaunchKernelGGL((swl::latent_expand_kernel<T>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, static_cast<hipStream_t>(stream), p);
    });
    return swl::check_launch();
}
