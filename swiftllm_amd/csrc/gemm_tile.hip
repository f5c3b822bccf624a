// gemm_tile.hip — the dense products of prompt-sized steps: which tile of gemm_tile.h, and the entry points.
#include "gemm_tile.h"

namespace swl {

template <typename T, int ACT>
int gemm_tile_dispatch(const GemmTileParams &p, int shape, hipStream_t s) {     // (in the order of kTileShapes)
    switch (shape) {
    case 1: return gemm_tile_launch<T, 16, 4, 4, 4, 4, ACT>(p, s);
    case 2: return gemm_tile_launch<T, 16, 3, 3, 4, 4, ACT>(p, s);
    case 3: return gemm_tile_launch<T, 16, 3, 3, 3, 3, ACT>(p, s);
    case 4: return gemm_tile_launch<T, 16, 3, 2, 4, 4, ACT>(p, s);
    case 5: return gemm_tile_launch<T, 16, 4, 3, 4, 4, ACT>(p, s);
    case 6: return gemm_tile_launch<T, 16, 4, 4, 3, 3, ACT>(p, s);
    case 10: return gemm_tile_launch<T, 32, 1, 1, 1, 1, ACT>(p, s);
    case 11: return gemm_tile_launch<T, 16, 1, 1, 2, 2, ACT>(p, s);
    default: break;
    }
    if constexpr (ACT <= 0) {
        switch (shape) {
        case 7: return gemm_tile_launch<T, 16, 3, 2, 2, 2, ACT>(p, s);
        case 8: return gemm_tile_launch<T, 16, 3, 2, 3, 3, ACT>(p, s);
        case 9: return gemm_tile_launch<T, 16, 4, 3, 3, 3, ACT>(p, s);
        default: break;
        }
    }
    return SWL_ERR_UNSUPPORTED;
}

} // namespace swl

/* 1 when swl_gemm_tile takes a product of these sizes: 16-bit, whole steps of 128 columns, rows on 16 bytes (out rows with room for whole
 * pieces of eight columns), and a tile's rows within 2 GiB. */
extern "C" int swl_gemm_tile_supported(int64_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldo, int32_t act, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    if (M <= 0 || M > (1 << 30) || N <= 0 || N > (1 << 30) || K < 256 || K % 128 || act < 0 || act > 5) return 0;
    if (ldx < K || ldx % 8 || ldo % 8 || ldo < (static_cast<int64_t>(N) + 7) / 8 * 8) return 0;
    return 256 * ldx * 2 < (1LL << 31) && 256 * ldo * 2 < (1LL << 31) && (act >= 2 ? 2LL * N : 256LL) * K * 2 < (1LL << 32);
}

extern "C" int swl_gemm_tile(void *out, const void *x, const void *w, int64_t M, int32_t N, int32_t K, int64_t ldx, int64_t ldo, int32_t x_cols,
                             int64_t x_next, int32_t act, int32_t act_cols, float limit, int32_t shape, int32_t dtype, swl_stream_t stream) {
    if (M < 0 || act < 0 || act > 5 || shape < 0 || shape > 11 || x_cols < 0) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!swl_gemm_tile_supported(M, N, K, ldx, ldo, act, dtype)) return SWL_ERR_UNSUPPORTED;
    if (x_cols && (x_cols % 256 || act >= 2 || x_next % 8)) return SWL_ERR_UNSUPPORTED;      // (a tile's columns share one matrix x)
    if (act == 1 && act_cols % 4) return SWL_ERR_UNSUPPORTED;
    if (!out || !x || !w || !swl::aligned16(out) || !swl::aligned16(x) || !swl::aligned16(w)) return SWL_ERR_BAD_ARG;
    swl::GemmTileParams p = {};
    p.out = out; p.x = x; p.w = w; p.M = static_cast<int>(M); p.N = N; p.K = K; p.ldx = ldx; p.ldo = ldo;
    p.x_cols = x_cols; p.x_next = x_next * 2; p.act_cols = act_cols; p.limit = limit;
    unsigned set = act ? swl::kTilesAct : swl::kTilesPlain;
    if (x_cols)
        for (int i = 0; i < swl::kTileShapeCount; ++i)
            if (x_cols % (32 * swl::kTileShapes[i].w)) set &= ~(1u << i);
    if (shape == 0) shape = swl::gemm_tile_shape([=](int rows, int cols) { return (M + rows - 1) / rows * (((act >= 2 ? 2LL * N : N) + cols - 1) / cols); }, K, set);
    if (!(set >> (shape - 1) & 1)) return SWL_ERR_UNSUPPORTED;
    hipStream_t s = static_cast<hipStream_t>(stream);
    SWL_DISPATCH_DTYPE(dtype, T, {
        switch (act) {
        case 0: return swl::gemm_tile_dispatch<T, 0>(p, shape, s);
        case 1: return swl::gemm_tile_dispatch<T, 1>(p, shape, s);
        case 2: return swl::gemm_tile_dispatch<T, 2>(p, shape, s);
        case 3: return swl::gemm_tile_dispatch<T, 3>(p, shape, s);
        case 4: return swl::gemm_tile_dispatch<T, 4>(p, shape, s);
        default: return swl::gemm_tile_dispatch<T, 5>(p, shape, s);
        }
    });
}

/* Shares of K for a consumer that adds slabs up. Few tiles of long sums leave CUs idle: by the model of gemm_tile_shape, and what the slabs cost more
 * than 16-bit rows, written and read again (fitted: 2 us, and 0.92 us a share and million results, less 0.85 for the rows). Product and the residual
 * step behind it, 260 to 7800 tokens, us before (the library from 1024 x 4096 and 400 tokens up to the sizes where tiles pay) -> now: 1024 x 2048, 260 tokens 15.8 -> 12.0; 1024 x 4096,
 * 600 21.9 -> 19.2, 1800 31.6 -> 29.0; 1024 x 6144, 260 21.7 -> 16.1, 900 26.7 -> 23.2, 1800 48.4 -> 38.6 to 43, 2500 68.7 -> 45.5 to 48, 3600 71.8 -> 58.5; 2048 x 8192,
 * 260 30.1 -> 22.6, 900 57.0 -> 43.3, 2500 96 -> 89; 2048 x 12288, 600 72 -> 46, 1800 127 -> 95. Two shares where the model says one: 1024 x 1024, 1800 17.7 ->
 * 21.0; 2048 x 2048, 2500 38.4 -> 43.7; 1024 x 4096, 7800 79 -> 82; 2048 x 8192, 5000 156 -> 169. */
extern "C" int swl_gemm_tile_choose_splits(int64_t M, int32_t N, int32_t K) {
    if (!swl_gemm_tile_supported(M, N, K, K, (static_cast<int64_t>(N) + 7) / 8 * 8, 0, SWL_BF16) || N % 8 || 256LL * N * 4 >= (1LL << 31)) return 1;
    const double results = static_cast<double>(M) * N * 1e-6;
    double least = 0;
    int best = 1;
    for (int splits = 1; splits <= 8; ++splits) {
        if (K % (128 * splits) || K / splits < 256) continue;
        double us;
        swl::gemm_tile_shape([=](int rows, int cols) { return (M + rows - 1) / rows * ((N + cols - 1) / cols) * splits; }, K / splits, swl::kTilesPlain, &us);
        us = splits == 1 ? 0.97 * us : us + 2.0 + (0.92 * splits - 0.85) * results;
        if (splits == 1 || us < least) best = splits, least = us;
    }
    return best;
}

/* slabs[splits][M][N] fp32: the sums of x w^T over equal shares of K, for consumers that add them up. */
extern "C" int swl_gemm_tile_partial(float *slabs, size_t slabs_bytes, const void *x, const void *w, int64_t M, int32_t N, int32_t K, int64_t ldx,
                                     int32_t splits, int32_t shape, int32_t dtype, swl_stream_t stream) {
    if (M < 0 || splits < 1 || splits > 16 || shape < 0 || shape > 11) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!swl_gemm_tile_supported(M, N, K, ldx, N, 0, dtype) || K % (128 * splits) || K / splits < 256 || 256LL * N * 4 >= (1LL << 31)) return SWL_ERR_UNSUPPORTED;
    if (!slabs || !x || !w || !swl::aligned16(slabs) || !swl::aligned16(x) || !swl::aligned16(w)) return SWL_ERR_BAD_ARG;
    if (slabs_bytes / 4 / splits / N < static_cast<size_t>(M)) return SWL_ERR_BAD_ARG;
    swl::GemmTileParams p = {};
    p.out = slabs; p.x = x; p.w = w; p.M = static_cast<int>(M); p.N = N; p.K = K; p.ldx = ldx; p.ldo = N; p.splits = splits;
    if (shape == 0) shape = swl::gemm_tile_shape([=](int rows, int cols) { return (M + rows - 1) / rows * ((N + cols - 1) / cols) * splits; }, K / splits, swl::kTilesPlain);
    hipStream_t s = static_cast<hipStream_t>(stream);
    SWL_DISPATCH_DTYPE(dtype, T, { return (swl::gemm_tile_dispatch<T, swl::kTileSlabs>(p, shape, s)); });
}
