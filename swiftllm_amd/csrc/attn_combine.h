// attn_combine.h — the second launch of attention over key shares: what a share leaves (unnormalised fp32 result, running maximum in
// base-2 exponent units, sum) becomes one row per (token, head); plain sums of sigmoid attention are added up.
#pragma once

#include "swl_common.h"

namespace swl {

// Two fp32 weights as two 16-bit terms each, in the halves of a register. bf16: one conversion for two, and the first term as fp32 is a shift
// or a mask.
template <typename T>
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned &h, unsigned &l);
template <>
__device__ __forceinline__ void split_pair<bf16>(float x0, float x1, unsigned &h, unsigned &l) {
    typedef float float2_t __attribute__((ext_vector_type(2)));
    typedef bf16 bf2_t __attribute__((ext_vector_type(2)));
    h = __builtin_bit_cast(unsigned, __builtin_convertvector((float2_t{x0, x1}), bf2_t));
    const float2_t r = {x0 - __uint_as_float(h << 16), x1 - __uint_as_float(h & 0xffff0000u)};
    l = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf2_t));
}
template <>
__device__ __forceinline__ void split_pair<f16>(float x0, float x1, unsigned &h, unsigned &l) {
    const vec2_t<f16> a = {to_t<f16>(x0), to_t<f16>(x1)};
    const vec2_t<f16> b = {to_t<f16>(x0 - to_f(a[0])), to_t<f16>(x1 - to_f(a[1]))};
    h = __builtin_bit_cast(unsigned, a);
    l = __builtin_bit_cast(unsigned, b);
}
// ... eight
template <typename T>
__device__ __forceinline__ void split_weights(const float (&x)[8], vec8_t<T> &hi, vec8_t<T> &lo) {
    typedef unsigned uint4v __attribute__((ext_vector_type(4)));
    uint4v h, l;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        unsigned a, b;
        split_pair<T>(x[2 * j], x[2 * j + 1], a, b);
        h[j] = a;
        l[j] = b;
    }
    hi = __builtin_bit_cast(vec8_t<T>, h);
    lo = __builtin_bit_cast(vec8_t<T>, l);
}

// out[t][h][:] = sum_s e^{m_s - M} O_s / sum_s e^{m_s - M} l_s over the key shares s (a share without keys has l = 0).
// The first wave evaluates the shares' weights once (one share per lane, at most 64) and leaves them in LDS.
// NATURAL: the maxima are in natural units (the per-token kernel, whose arithmetic is full-precision throughout).
template <typename T, bool NATURAL = false>
__global__ __launch_bounds__(256) void window_attn_combine_kernel(T *out, const float *part_o, const float *part_ml,
                                                                  int64_t rows, int dv, int nsplit, const float *sink, int H,
                                                                  int out_f32, int out_dim, int64_t out_stride, const T *gate,
                                                                  int64_t gate_stride) {
    __shared__ float wgt[64];
    __shared__ float inv_den;
    const int64_t row = blockIdx.x;     // (token, head)
    if (threadIdx.x < 64) {
        const int sp = threadIdx.x;
        const bool live = sp < nsplit;
        const float m = live ? part_ml[(sp * rows + row) * 2] : kNegBig;     // (the maxima are in base-2 exponent units)
        const float l = live ? part_ml[(sp * rows + row) * 2 + 1] : 0.f;
        float mx = wave_allreduce_max(m);
        float extra = 0.f;
        if (sink) {
            const float sk = sink[row % H] * (NATURAL ? 1.0f : 1.4426950408889634f);
            mx = fmaxf(mx, sk);
            extra = NATURAL ? expf(sk - mx) : exp2f(sk - mx);
        }
        const float w = live ? (NATURAL ? expf(m - mx) : exp2f(m - mx)) : 0.f;
        const float den = wave_allreduce_sum(w * l) + extra;
        wgt[sp] = w;
        if (sp == 0) inv_den = 1.0f / den;
    }
    __syncthreads();
    const float inv = inv_den;
    const int64_t tok = row / H, hc0 = (row - tok * H) * out_dim;
    for (int c = threadIdx.x; c < out_dim; c += blockDim.x) {
        float a = 0.f;
        for (int s = 0; s < nsplit; ++s) a += wgt[s] * part_o[(s * rows + row) * dv + c];
        a *= inv;
        if (gate) a /= 1.0f + expf(-to_f(gate[tok * gate_stride + hc0 + c]));
        if (out_f32) reinterpret_cast<float *>(out)[tok * out_stride + hc0 + c] = a;
        else out[tok * out_stride + hc0 + c] = to_t<T>(a);
    }
}

// The same for rows of 64, 128 or 256 columns, four a lane: LP = dv / 4 lanes take a share and 64 / LP shares go side by side, up to eight a lane in
// flight; four rows a workgroup, a wave each.
// Above a column's shares are a chain of 4-byte loads. With the attention in front of it (window_attn.hip, fp32, 8 heads of 128, 16 shares) 3 tokens at 513
// keys 10.7 -> 8.4 us, 12 at 500 13.0 -> 11.3, 32 at 1000 20.0 -> 17.9, prompts of 100 (10 shares) 16.3 -> 14.3, of 500 (two) 39.2 -> 39.0.
template <typename T, bool NATURAL, int LP>
__global__ __launch_bounds__(256) void attn_combine_rows_kernel(T *out, const float *part_o, const float *part_ml, int64_t rows, int nsplit,
                                                                const float *sink, int H, int out_f32, int out_dim, int64_t out_stride,
                                                                const T *gate, int64_t gate_stride) {
    constexpr int dv = 4 * LP, SIDE = 64 / LP, DEEP = 8;
    // (a lane reads another's weight with all of them at work: inside a branch by its own share, the lane asked may have gone the other way)
    static_assert(64 % (DEEP * SIDE) == 0, "shares named below are lanes of the wave");
    const int lane = threadIdx.x & 63, sub = lane % LP, side = lane / LP;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // (token, head)
    if (row >= rows) return;
    const bool live = lane < nsplit;
    const float m = live ? part_ml[(lane * rows + row) * 2] : kNegBig, l = live ? part_ml[(lane * rows + row) * 2 + 1] : 0.f;
    const float sk = sink ? sink[row % H] * (NATURAL ? 1.0f : 1.4426950408889634f) : kNegBig;
    float4_t a = {0.f, 0.f, 0.f, 0.f};
    float w = 0.f, inv = 0.f;
    for (int s0 = 0; s0 < nsplit; s0 += DEEP * SIDE) {
        float4_t p[DEEP];
#pragma unroll
        for (int u = 0; u < DEEP; ++u)      // (the last share stands in for missing ones, whose weight is zero)
            p[u] = *reinterpret_cast<const float4_t *>(part_o + (min(s0 + u * SIDE + side, nsplit - 1) * rows + row) * dv + 4 * sub);
        if (s0 == 0) {
            const float mx = fmaxf(wave_allreduce_max(m), sk);
            w = live ? (NATURAL ? expf(m - mx) : exp2f(m - mx)) : 0.f;
            const float extra = sink ? (NATURAL ? expf(sk - mx) : exp2f(sk - mx)) : 0.f;
            inv = 1.0f / (wave_allreduce_sum(w * l) + extra);
        }
#pragma unroll
        for (int u = 0; u < DEEP; ++u) a += __shfl(w, s0 + u * SIDE + side, 64) * p[u];     // (lanes without a share have weight zero)
    }
#pragma unroll
    for (int d = LP; d < 64; d *= 2)
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] += __shfl_xor(a[c], d, 64);
    const int64_t tok = row / H, at = (row - tok * H) * out_dim + 4 * sub;
    if (side > 0 || 4 * sub >= out_dim) return;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        a[c] *= inv;
        if (gate && 4 * sub + c < out_dim) a[c] /= 1.0f + expf(-to_f(gate[tok * gate_stride + at + c]));
    }
    if (out_dim % 4 == 0 && out_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & (out_f32 ? 15 : 4 * sizeof(T) - 1)) == 0) {       // (uniform)
        if (out_f32) {
            *reinterpret_cast<float4_t *>(reinterpret_cast<float *>(out) + tok * out_stride + at) = a;
        } else {
            vec4_t<T> o;
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = to_t<T>(a[c]);
            *reinterpret_cast<vec4_t<T> *>(out + tok * out_stride + at) = o;
        }
        return;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (4 * sub + c >= out_dim) break;
        if (out_f32) reinterpret_cast<float *>(out)[tok * out_stride + at + c] = a[c];
        else out[tok * out_stride + at + c] = to_t<T>(a[c]);
    }
}

// The launch behind attention over key shares, one of the two above.
template <typename T, bool NATURAL = false>
inline void launch_attn_combine(T *out, const float *part_o, const float *part_ml, int64_t rows, int dv, int nsplit, const float *sink, int H,
                                int out_f32, int out_dim, int64_t out_stride, const T *gate, int64_t gate_stride, hipStream_t s) {
    const dim3 fours(static_cast<unsigned>((rows + 3) / 4));
#define SWL_COMBINE(LP)                                                                                                             \
    hipLaunchKernelGGL((attn_combine_rows_kernel<T, NATURAL, LP>), fours, dim3(256), 0, s, out, part_o, part_ml, rows, nsplit, sink, H, \
                       out_f32, out_dim, out_stride, gate, gate_stride)
    if (dv == 64) SWL_COMBINE(16);
    else if (dv == 128) SWL_COMBINE(32);
    else if (dv == 256) SWL_COMBINE(64);
    else
        hipLaunchKernelGGL((window_attn_combine_kernel<T, NATURAL>), dim3(static_cast<unsigned>(rows)), dim3(dv < 256 ? 64 : 256), 0, s, out,
                           part_o, part_ml, rows, dv, nsplit, sink, H, out_f32, out_dim, out_stride, gate, gate_stride);
#undef SWL_COMBINE
}

// out[i] = sum over the key shares s of part[s][i]
template <typename T>
__global__ __launch_bounds__(256) void sigmoid_attn_sum_kernel(T *out, const float *part, int64_t total, int nsplit) {
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    if (total & 3) {        // (uniform) odd rows: element by element
        for (int64_t k = i; k < min(i + 4, total); ++k) {
            float a = part[k];
            for (int s = 1; s < nsplit; ++s) a += part[s * total + k];
            out[k] = to_t<T>(a);
        }
        return;
    }
    float4_t a = *reinterpret_cast<const float4_t *>(part + i);
    for (int s = 1; s < nsplit; ++s) a += *reinterpret_cast<const float4_t *>(part + s * total + i);
    typedef T vec4 __attribute__((ext_vector_type(4)));
    vec4 w;
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = to_t<T>(a[r]);
    *reinterpret_cast<vec4 *>(out + i) = w;
}

} // namespace swl
