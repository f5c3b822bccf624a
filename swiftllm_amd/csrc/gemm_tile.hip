// gemm_tile.hip — the dense products of prompt-sized steps: which tile of gemm_tile.h, and the entry points.
#include "gemm_tile.h"

namespace swl {

template <typename T, int ACT>
int gemm_tile_dispatch(const GemmTileParams &p, int shape, hipStream_t s) {     // (in the order of kTileShapes)
    switch (shape) {
    case 1: return gemm_tile_launch<T, 16, 4, 4, 4, 4, 1, ACT>(p, s);
    case 2: return gemm_tile_launch<T, 16, 3, 3, 4, 4, 1, ACT>(p, s);
    case 3: return gemm_tile_launch<T, 16, 3, 3, 3, 3, 1, ACT>(p, s);
    case 4: return gemm_tile_launch<T, 16, 3, 2, 4, 4, 1, ACT>(p, s);
    case 5: return gemm_tile_launch<T, 16, 4, 3, 4, 4, 1, ACT>(p, s);
    case 6: return gemm_tile_launch<T, 16, 4, 4, 3, 3, 1, ACT>(p, s);
    case 10: return gemm_tile_launch<T, 32, 1, 1, 1, 1, 1, ACT>(p, s);
    case 11: return gemm_tile_launch<T, 16, 1, 1, 2, 2, 1, ACT>(p, s);
    default: break;
    }
    if constexpr (ACT == 0) {
        switch (shape) {
        case 7: return gemm_tile_launch<T, 16, 3, 2, 2, 2, 1, ACT>(p, s);
        case 8: return gemm_tile_launch<T, 16, 3, 2, 3, 3, 1, ACT>(p, s);
        case 9: return gemm_tile_launch<T, 16, 4, 3, 3, 3, 1, ACT>(p, s);
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
