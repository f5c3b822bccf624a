// layernorm.hip — fp32 residual stream operators: embedding with learned positions, LayerNorm (weight + bias), and the
// fused "normalised sublayer output into the residual, then the next sublayer's input norm" step of sandwich-norm
// models. The residual x is fp32 [tokens, width]; sublayer inputs/outputs are the compute dtype (bf16 / f16 / f32);
// every statistic (mean, mean of squared deviations) is taken in fp32 with two passes over the row.
#include "row_wide.h"
#include "swl_common.h"

namespace swl {

constexpr int kLnThreads = 256;

// Sum over the workgroup; every thread gets the total. `red` holds kLnThreads / 64 floats.
__device__ __forceinline__ float block_sum(float v, float *red) {
    v = wave_allreduce_sum(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();    // (red may still be read from the previous reduction)
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kLnThreads / 64; ++w) t += red[w];
    return t;
}

// Mean and 1/sqrt(var + eps) of row[0..n) held in LDS (fp32).
__device__ __forceinline__ void row_stats(const float *row, int n, float eps, float *red, float &mean, float &rstd) {
    float s = 0.f;
    for (int i = threadIdx.x; i < n; i += kLnThreads) s += row[i];
    mean = block_sum(s, red) / static_cast<float>(n);
    float q = 0.f;
    for (int i = threadIdx.x; i < n; i += kLnThreads) {
        const float d = row[i] - mean;
        q += d * d;
    }
    const float var = block_sum(q, red) / static_cast<float>(n);
    rstd = 1.0f / sqrtf(var + eps);
}

// x[t] = embed[token[t]] * scale + pos[position[t]]  (fp32); x0 (optional) receives a copy. pos NULL: no learned positions.
template <typename T>
__global__ __launch_bounds__(kLnThreads) void embed_pos_kernel(float *x, float *x0, const T *embed, const T *pos,
                                                               const int32_t *tokens, const int32_t *positions,
                                                               float scale, int width) {
    const int64_t t = blockIdx.x;
    const T *e = embed + static_cast<int64_t>(tokens[t]) * width;
    const T *p = pos ? pos + static_cast<int64_t>(positions[t]) * width : nullptr;
    // rows of whole aligned quads: four columns a lane (4500 x 2048, bf16: 33 -> 17 us)
    if (width % 4 == 0 && row_aligned<T>(embed) && row_aligned<T>(pos) && row_aligned<float>(x) && row_aligned<float>(x0)) {
        for (int i = threadIdx.x * 4; i < width; i += kLnThreads * 4) {
            float v[4], q[4] = {0.f, 0.f, 0.f, 0.f};
            row_load<T>(v, e + i);
            if (p) row_load<T>(q, p + i);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = p ? v[j] * scale + q[j] : v[j] * scale;
            row_store<float>(x + t * width + i, v);
            if (x0) row_store<float>(x0 + t * width + i, v);
        }
        return;
    }
    for (int i = threadIdx.x; i < width; i += kLnThreads) {
        const float v = p ? to_f(e[i]) * scale + to_f(p[i]) : to_f(e[i]) * scale;
        x[t * width + i] = v;
        if (x0) x0[t * width + i] = v;
    }
}

// out[r] = LN(x[row_idx ? row_idx[r] : r]) * w + b
template <typename T>
__global__ __launch_bounds__(kLnThreads) void layernorm_kernel(T *out, const float *x, const int32_t *row_idx,
                                                               const float *w, const float *b, float eps, int width) {
    extern __shared__ float lds[];
    float *row = lds, *red = lds + width;
    const int64_t r = blockIdx.x;
    const int64_t src = row_idx ? row_idx[r] : r;
    for (int i = threadIdx.x; i < width; i += kLnThreads) row[i] = x[src * width + i];
    __syncthreads();
    float mean, rstd;
    row_stats(row, width, eps, red, mean, rstd);
    for (int i = threadIdx.x; i < width; i += kLnThreads)
        out[r * width + i] = to_t<T>((row[i] - mean) * rstd * w[i] + b[i]);
}

// x <- x + mult * (LN(y) * w1 + b1)   [if y]
//        + x0                          [if x0]
//        + step                        [if step]
// out <- LN(x) * w2 + b2               [if out]
template <typename T>
__global__ __launch_bounds__(kLnThreads) void add_layernorm_kernel(float *x, const T *y, float mult, const float *w1,
                                                                   const float *b1, const float *x0, const float *step,
                                                                   T *out, const float *w2, const float *b2, float eps,
                                                                   int width) {
    extern __shared__ float lds[];
    float *row = lds, *red = lds + width;
    const int64_t t = blockIdx.x;
    float mean, rstd;
    if (y) {
        for (int i = threadIdx.x; i < width; i += kLnThreads) row[i] = to_f(y[t * width + i]);
        __syncthreads();
        row_stats(row, width, eps, red, mean, rstd);
    }
    for (int i = threadIdx.x; i < width; i += kLnThreads) {     // (each thread touches only its own columns of row[])
        float v = x[t * width + i];
        if (y) v += mult * ((row[i] - mean) * rstd * w1[i] + b1[i]);
        if (x0) v += x0[t * width + i];
        if (step) v += step[i];
        x[t * width + i] = v;
        row[i] = v;
    }
    if (!out) return;
    __syncthreads();
    row_stats(row, width, eps, red, mean, rstd);
    for (int i = threadIdx.x; i < width; i += kLnThreads)
        out[t * width + i] = to_t<T>((row[i] - mean) * rstd * w2[i] + b2[i]);
}

// The same with the row in registers (row_wide.h): rows of a multiple of four columns, up to 8192, on aligned addresses. Bound by memory: y and
// out in the compute dtype, x in and out in fp32 (and x0). bf16, 4500 x 2048: 47 -> 27 us (4.1 TB/s),
// 32 x 2048 7.7 -> 4.6 us.
template <int TPR, int NV>
__device__ __forceinline__ void wide_stats(const float (&v)[NV][4], int c0, int width, float eps, float *red, float &mean, float &rstd) {
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) s += v[j][e];       // (columns past the row are 0)
    mean = row_sum<TPR>(s, red) / static_cast<float>(width);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        if (c0 + 4 * TPR * j < width) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = v[j][e] - mean;
                q += d * d;
            }
        }
    }
    rstd = 1.0f / sqrtf(row_sum<TPR>(q, red + kRowThreads / 64) / static_cast<float>(width) + eps);
}

template <typename T, int TPR, int NV>
__global__ __launch_bounds__(kRowThreads) void add_layernorm_wide_kernel(float *x, const T *y, float mult, const float *w1, const float *b1,
                                                                         const float *x0, const float *step, T *out, const float *w2,
                                                                         const float *b2, float eps, int64_t rows, int width) {
    __shared__ float red[4][kRowThreads / 64];
    const int64_t id = static_cast<int64_t>(blockIdx.x) * (kRowThreads / TPR) + threadIdx.x / TPR, t = min(id, rows - 1);
    const bool live = id < rows;
    const int c0 = (threadIdx.x % TPR) * 4;
    float v[NV][4], s[NV][4], extra[NV][4], mean, rstd;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = s[j][e] = extra[j][e] = 0.f;
        if (c < width) {
            if (y) row_load<T>(s[j], y + t * width + c);
            row_load<float>(v[j], x + t * width + c);
            if (x0) row_load<float>(extra[j], x0 + t * width + c);
        }
    }
    if (y) wide_stats<TPR, NV>(s, c0, width, eps, red[0], mean, rstd);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
        if (c < width) {
            if (y) {
                float w[4], b[4];
                row_load<float>(w, w1 + c);
                row_load<float>(b, b1 + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[j][e] += mult * ((s[j][e] - mean) * rstd * w[e] + b[e]);
            }
            float add[4] = {0.f, 0.f, 0.f, 0.f};
            if (step) row_load<float>(add, step + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (x0) v[j][e] += extra[j][e];
                if (step) v[j][e] += add[e];
            }
            if (live) row_store<float>(x + t * width + c, v[j]);
        }
    }
    if (!out) return;
    wide_stats<TPR, NV>(v, c0, width, eps, red[2], mean, rstd);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
        if (live && c < width) {
            float w[4], b[4];
            row_load<float>(w, w2 + c);
            row_load<float>(b, b2 + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = (v[j][e] - mean) * rstd * w[e] + b[e];
            row_store<T>(out + t * width + c, w);
        }
    }
}

inline size_t ln_lds_bytes(int width) { return (static_cast<size_t>(width) + kLnThreads / 64) * sizeof(float); }

} // namespace swl

extern "C" int swl_embed_pos(float *x, float *x0, const void *embed, const void *pos, const int32_t *tokens,
                             const int32_t *positions, float scale, int64_t num_tokens, int32_t width, int32_t dtype,
                             swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!x || !embed || !tokens || (pos && !positions)) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::embed_pos_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kLnThreads), 0,
                           static_cast<hipStream_t>(stream), x, x0, static_cast<const T *>(embed),
                           static_cast<const T *>(pos), tokens, positions, scale, width);
    });
    return swl::check_launch();
}

extern "C" int swl_layernorm(void *out, const float *x, const int32_t *row_idx, const float *w, const float *b, float eps,
                             int64_t num_rows, int32_t width, int32_t dtype, swl_stream_t stream) {
    if (num_rows < 0 || width <= 0) return SWL_ERR_BAD_ARG;
    if (num_rows == 0) return SWL_OK;
    if (!out || !x || !w || !b) return SWL_ERR_BAD_ARG;
    if (num_rows > 0x7fffffffLL || swl::ln_lds_bytes(width) > 64 * 1024) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::layernorm_kernel<T>), dim3(static_cast<unsigned>(num_rows)), dim3(swl::kLnThreads),
                           swl::ln_lds_bytes(width), static_cast<hipStream_t>(stream), static_cast<T *>(out), x, row_idx,
                           w, b, eps, width);
    });
    return swl::check_launch();
}

extern "C" int swl_add_layernorm(float *x, const void *y, float mult, const float *w1, const float *b1, const float *x0,
                                 const float *step, void *out, const float *w2, const float *b2, float eps,
                                 int64_t num_tokens, int32_t width, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!x || (y && (!w1 || !b1)) || (out && (!w2 || !b2))) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL || swl::ln_lds_bytes(width) > 64 * 1024) return SWL_ERR_UNSUPPORTED;
#define SWL_GO(TPR, NV)                                                                                                                \
    hipLaunchKernelGGL((swl::add_layernorm_wide_kernel<T, TPR, NV>), dim3(static_cast<unsigned>((num_tokens * TPR + 255) / 256)),      \
                       dim3(swl::kRowThreads), 0, static_cast<hipStream_t>(stream), x, static_cast<const T *>(y), mult, w1, b1, x0,    \
                       step, static_cast<T *>(out), w2, b2, eps, num_tokens, width)
    SWL_DISPATCH_DTYPE3(dtype, T, {
        const bool wide = width % 4 == 0 && width <= swl::kRowMaxWidth && swl::row_aligned<float>(x) && swl::row_aligned<T>(y) &&
                          swl::row_aligned<T>(out) && swl::row_aligned<float>(w1) && swl::row_aligned<float>(b1) &&
                          swl::row_aligned<float>(w2) && swl::row_aligned<float>(b2) && swl::row_aligned<float>(x0) &&
                          swl::row_aligned<float>(step);
        if (wide) {
            SWL_ROW_SHAPE(num_tokens, width, SWL_GO);
            return swl::check_launch();
        }
        hipLaunchKernelGGL((swl::add_layernorm_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kLnThreads),
                           swl::ln_lds_bytes(width), static_cast<hipStream_t>(stream), x, static_cast<const T *>(y), mult,
                           w1, b1, x0, step, static_cast<T *>(out), w2, b2, eps, width);
    });
#undef SWL_GO
    return swl::check_launch();
}
