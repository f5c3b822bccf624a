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
