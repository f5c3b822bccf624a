// gemm_f32.hip — projections of a few tokens in true fp32: out[M, N] = x[M, K] w[N, K]^T for up to 16 tokens.
//
// What bounds it: latency, then the weight stream. A library product of 3 rows takes 10 to 13 us whatever its size (1024 x 1024: 4 MiB, which
// HBM delivers in 0.7 us) because a few workgroups walk all of K. Here the whole matrix is asked for at once: a wave takes R rows of w, a lane
// four neighbouring columns of every 256; the sums over lanes go by DPP inside rows of 16 lanes, then through LDS together with those of
// the waves that share K. Every output is the sum of per-lane partial sums, at most K / 64 terms in a row: no further from the exact sum
// than the library's, and the same whatever M is.
// Measured (us, w cycled through 600 MB; library product -> here) at 1 / 3 / 8 / 16 tokens: 1024 x 1024 10.8 -> 2.8 / 11.0 -> 3.1 / 11.0 -> 4.0 /
// 11.0 -> 5.5; 3200 x 1024 11.5 -> 4.4 / 4.9 / 6.4 / 11.8; 1024 x 4096 12.3 -> 5.8 / 6.5 / 10.3 / 12.1; 8192 x 1024 14.4 -> 7.6 / 8.0 / 11.0 / 21;
// 32000 x 1024 36 -> 21.7 / 22.5 / 33.6 / 66. Beyond a few tokens their share of x, read for every four rows, is what costs, and a library that
// shares K over workgroups wins where there are many rows and columns. Library / here, at 4 tokens: 4096 x 4096 16.7 / 16.1, 4096 x 14336 47.9 /
// 46.4, 28672 x 4096 113 / 78; at 8: 1024 x 16384 37.5 / 28.4, 1536 x 8192 22.1 / 20.5, 4096 x 3072 18.4 / 15.1, 2048 x 4096 13.6 / 14.3,
// 4096 x 4096 16.6 / 20.1, 8192 x 2048 17.9 / 21.4; at 16: 1024 x 16384 38.1 / 34.6, 1536 x 2048 11.8 / 9.6, 1280 x 4096 12.8 / 16.1, 2048 x 1536
// 10.0 / 11.2, 2048 x 8192 24 / 34. Hence the lines of swl_gemm_f32_supported. Error against 64 bits 1.0e-7
// (relative, 2-norm) where the library's is 2.9e-7, at K 4096 1.2e-7 and 5.8e-7. Waves that share K (1 / 2 / 4): 4.9 / 3.6 / 3.1 us at
// 1024 x 1024, 5.9 / 4.9 / 4.9 at 3200 rows, 26.1 / 22.5 / 22.4 at 32000.
#include "swl_common.h"

namespace swl {

constexpr int kF32MaxTokens = 16;

// KS waves share the columns of the same rows, 4 / KS groups of rows a workgroup
// GLU: rows [gate; up] of w, a wave takes R / 2 of each; out[c] = gated_unit of the two products. relu2: the first so many columns of out are
// max(0, product)^2.
template <int M, int R, int KS, bool GLU>
__device__ __forceinline__ void gemm_f32_block(float (*part)[4][M * R], int block, float *__restrict__ out, const float *__restrict__ x,
                                               const float *__restrict__ w, int rows, int N, int K, int64_t x_stride, int64_t out_stride,
                                               int relu2, float limit) {
    constexpr int V = M * R, OUT = GLU ? R / 2 : R;
    const int columns = GLU ? N / 2 : N;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = (block * (4 / KS) + wave / KS) * OUT;
    const int chunks = (K + 255) / 256, per = (chunks + KS - 1) / KS;
    const int k_end = min(K, (wave % KS + 1) * per * 256);
    float acc[R][M];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
    const float *wr[R], *xr[M];
#pragma unroll
    for (int r = 0; r < R; ++r) wr[r] = w + static_cast<int64_t>(min(n0 + r % OUT, columns - 1) + r / OUT * columns) * K;
#pragma unroll
    for (int m = 0; m < M; ++m) xr[m] = x + min(m, rows - 1) * x_stride;
    auto slice = [&](int k) {
        float4_t a[R], b[M];
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = __builtin_nontemporal_load(reinterpret_cast<const float4_t *>(wr[r] + k));
#pragma unroll
        for (int m = 0; m < M; ++m) b[m] = *reinterpret_cast<const float4_t *>(xr[m] + k);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r][m] = fmaf(a[r][e], b[m][e], acc[r][m]);
    };
    int k = wave % KS * per * 256 + lane * 4;
    constexpr int U = M <= 4 ? 4 : 2;
    for (; k - lane * 4 + U * 256 <= k_end; k += U * 256) {
#pragma unroll
        for (int u = 0; u < U; ++u) slice(k + u * 256);
    }
    for (; k < k_end; k += 256) slice(k);
    // sums over the lanes of a row of 16; lane i keeps those of value i (and 16 + i)
    float keep[(V + 15) / 16];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int v = r * M + m;
            const float s = group_allreduce_sum<16>(acc[r][m]);
            if (v % 16 == 0) keep[v / 16] = s;
            else keep[v / 16] = (lane & 15) == v % 16 ? s : keep[v / 16];
        }
#pragma unroll
    for (int j = 0; j < (V + 15) / 16; ++j)
        if (16 * j + (lane & 15) < V) part[wave][lane >> 4][16 * j + (lane & 15)] = keep[j];
    __syncthreads();
    auto sum = [&](int g, int v) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) s += part[g * KS + i][q][v];
        return s;
    };
    for (int t = threadIdx.x; t < OUT * M * (4 / KS); t += 256) {
        const int g = t / (OUT * M), v = t - g * OUT * M, r = v / M, m = v - r * M;
        const int n = (block * (4 / KS) + g) * OUT + r;
        float s = sum(g, v);
        if constexpr (GLU) {
            s = gated_unit(s, sum(g, v + OUT * M), limit, 0);
        } else if (n < relu2) {
            s = fmaxf(s, 0.f);
            s *= s;
        }
        if (n < columns && m < rows) out[m * out_stride + n] = s;
    }
}

template <int M, int R, int KS>
__global__ __launch_bounds__(256) void gemm_f32_kernel(float *__restrict__ out, const float *__restrict__ x, const float *__restrict__ w, int rows,
                                                       int N, int K, int64_t x_stride, int64_t out_stride) {
    __shared__ float part[4][4][M * R];         // [wave][16-lane row]
    gemm_f32_block<M, R, KS, false>(part, blockIdx.x, out, x, w, rows, N, K, x_stride, out_stride, 0, 0.f);
}

struct F32Product {
    float *out;
    const float *x, *w;
    int64_t x_stride, out_stride;
    int N;
};

// Two products of the same tokens and columns in one launch, the first in the first `blocks` workgroups (four waves share K in it).
// A decode step is a chain of launches of 3 to 5 us each, and a product of a few MiB does not fill the chip: 3 tokens of width 1024 through 8
// sublayers, the gate's 1024 rows beside the sublayer's first product and its activation in the same launch (12 launches less), 396 -> 363 us
// a step. Every sum is that of a launch of its own.
template <int M, int R, int KS, bool GLU>
__global__ __launch_bounds__(256) void gemm_f32_pair_kernel(F32Product a, F32Product b, int blocks, int rows, int K, int relu2, float limit) {
    __shared__ float part[4][4][M * R];
    if (static_cast<int>(blockIdx.x) < blocks)
        gemm_f32_block<M, R, 4, false>(part, blockIdx.x, a.out, a.x, a.w, rows, a.N, K, a.x_stride, a.out_stride, 0, 0.f);
    else
        gemm_f32_block<M, R, KS, GLU>(part, blockIdx.x - blocks, b.out, b.x, b.w, rows, b.N, K, b.x_stride, b.out_stride, relu2, limit);
}

template <int M, int R>
static void launch_f32(int ks, hipStream_t s, float *out, const float *x, const float *w, int rows, int N, int K, int64_t xs, int64_t os) {
    const int per = R * (4 / ks);
    const dim3 grid(static_cast<unsigned>((N + per - 1) / per));
    if (ks == 4) hipLaunchKernelGGL((gemm_f32_kernel<M, R, 4>), grid, dim3(256), 0, s, out, x, w, rows, N, K, xs, os);
    else if (ks == 2) hipLaunchKernelGGL((gemm_f32_kernel<M, R, 2>), grid, dim3(256), 0, s, out, x, w, rows, N, K, xs, os);
    else hipLaunchKernelGGL((gemm_f32_kernel<M, R, 1>), grid, dim3(256), 0, s, out, x, w, rows, N, K, xs, os);
}

template <int M, int R>
static void launch_f32_pair(int ks, hipStream_t s, const F32Product &a, const F32Product &b, int rows, int K, bool glu, int relu2, float limit) {
    const int first = (a.N + R - 1) / R, per = (glu ? R / 2 : R) * (4 / ks), columns = glu ? b.N / 2 : b.N;
    const dim3 grid(static_cast<unsigned>(first + (columns + per - 1) / per));
#define SWL_F32_PAIR(KS, GLU) hipLaunchKernelGGL((gemm_f32_pair_kernel<M, R, KS, GLU>), grid, dim3(256), 0, s, a, b, first, rows, K, relu2, limit)
    if (ks == 4 && glu) SWL_F32_PAIR(4, true);
    else if (ks == 4) SWL_F32_PAIR(4, false);
    else if (glu) SWL_F32_PAIR(2, true);
    else SWL_F32_PAIR(2, false);
#undef SWL_F32_PAIR
}

// (the rows of w alone decide: a token's bits do not hang on its company)
static int f32_k_waves(int N) { return N <= 4096 ? 4 : 2; }

} // namespace swl

/* 1 when swl_gemm_f32 serves these sizes (up to 16 tokens, rows of whole 16-byte pieces), 2 when it is the faster one beside a library
 * product too. */
extern "C" int swl_gemm_f32_supported(int32_t M, int32_t N, int32_t K) {
    if (M <= 0 || M > swl::kF32MaxTokens || N <= 0 || K <= 0 || K % 4) return 0;
    if (M <= 4) return 2;
    if (M <= 8) return N <= 1536 || K <= 1024 || (N <= 4096 && K <= 3072) ? 2 : 1;
    return N <= 1024 || (N <= 1536 && K <= 2048) || (N <= 2048 && K <= 1024) ? 2 : 1;
}

extern "C" int swl_gemm_f32(float *out, const float *x, const float *w, int32_t M, int32_t N, int32_t K, int64_t x_row_stride,
                            int64_t out_row_stride, int32_t k_waves, swl_stream_t stream) {
    if (M < 0 || N <= 0 || K <= 0) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!out || !x || !w) return SWL_ERR_BAD_ARG;
    if (!swl_gemm_f32_supported(M, N, K)) return SWL_ERR_UNSUPPORTED;
    if (x_row_stride < K || out_row_stride < N || x_row_stride % 4 || !swl::aligned16(x) || !swl::aligned16(w)) return SWL_ERR_BAD_ARG;
    if (!(k_waves == 0 || k_waves == 1 || k_waves == 2 || k_waves == 4)) return SWL_ERR_BAD_ARG;
    const int ks = k_waves ? k_waves : swl::f32_k_waves(N);
    hipStream_t s = static_cast<hipStream_t>(stream);
#define SWL_F32_CASE(MM, R) swl::launch_f32<MM, R>(ks, s, out, x, w, M, N, K, x_row_stride, out_row_stride)
    switch (M) {
        case 1: SWL_F32_CASE(1, 4); break;
        case 2: SWL_F32_CASE(2, 4); break;
        case 3: SWL_F32_CASE(3, 4); break;
        case 4: SWL_F32_CASE(4, 4); break;
        default:
            if (M <= 8) SWL_F32_CASE(8, 4);
            else SWL_F32_CASE(16, 2);
    }
#undef SWL_F32_CASE
    return swl::check_launch();
}

extern "C" int swl_gemm_f32_pair(float *out1, const float *x1, const float *w1, int32_t N1, int64_t x1_row_stride, int64_t out1_row_stride,
                                 float *out2, const float *x2, const float *w2, int32_t N2, int64_t x2_row_stride, int64_t out2_row_stride,
                                 int32_t M, int32_t K, int32_t glu, int32_t relu2_columns, float limit, swl_stream_t stream) {
    if (M < 0 || N1 <= 0 || N2 <= 0 || K <= 0 || relu2_columns < 0 || relu2_columns > N2 || (glu && (relu2_columns || N2 % 2))) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!out1 || !x1 || !w1 || !out2 || !x2 || !w2) return SWL_ERR_BAD_ARG;
    if (!swl_gemm_f32_supported(M, N1, K) || !swl_gemm_f32_supported(M, N2, K) || swl::f32_k_waves(N1) != 4) return SWL_ERR_UNSUPPORTED;
    if (x1_row_stride < K || out1_row_stride < N1 || x1_row_stride % 4 || x2_row_stride < K || out2_row_stride < (glu ? N2 / 2 : N2) ||
        x2_row_stride % 4 || !swl::aligned16(x1) || !swl::aligned16(w1) || !swl::aligned16(x2) || !swl::aligned16(w2))
        return SWL_ERR_BAD_ARG;
    const swl::F32Product a{out1, x1, w1, x1_row_stride, out1_row_stride, N1}, b{out2, x2, w2, x2_row_stride, out2_row_stride, N2};
    const int ks = swl::f32_k_waves(N2);
    hipStream_t s = static_cast<hipStream_t>(stream);
#define SWL_F32_CASE(MM, R) swl::launch_f32_pair<MM, R>(ks, s, a, b, M, K, glu != 0, relu2_columns, limit)
    switch (M) {
        case 1: SWL_F32_CASE(1, 4); break;
        case 2: SWL_F32_CASE(2, 4); break;
        case 3: SWL_F32_CASE(3, 4); break;
        case 4: SWL_F32_CASE(4, 4); break;
        default:
            if (M <= 8) SWL_F32_CASE(8, 4);
            else SWL_F32_CASE(16, 2);
    }
#undef SWL_F32_CASE
    return swl::check_launch();
}
