// rms_stream.hip — fp32 residual stream of models with RMS norms around every sublayer, a gate on every sublayer result and
// a short causal convolution in front of every sublayer.
//
//   swl_gated_add_rmsnorm: the step between two sublayers in one launch, one workgroup per token:
//       y   = m (+ sigmoid(s) * m2)            sublayer result (+ a second addend scaled by a per-token gate)
//       y  *= sigmoid(r + r_bias)              element-wise gate on the result
//       x  += y / rms(y) * w1                  into the fp32 stream
//       out = x / rms(x) * w2                  the next sublayer's input (or, with row_idx, the norm of selected rows only)
//     m may come as the fp32 slabs of a product whose K was split over workgroups (swl_gated_add_rmsnorm_parts): the launch that would
//     add them up is saved, and their rounding to the compute dtype with it.
//     Statistics, gates and the sum are fp32; m, m2, s, r and out are the compute dtype. Weights arrive as the factor itself
//     (a loader that stores "weight around zero" adds the one).
//     swl_gated_add_rmsnorm_conv, for steps of one token a sequence: the next sublayer's input convolution in the same launch. The row it
//     convolves is in registers, what came before it in the state slot, asked for with the stream's. A step's latency is a chain of
//     launches: 3 tokens x 1024 columns of 3 taps in fp32, 8 sublayers, 414 -> 396 us a step.
//   swl_post_norm_add: the same step for models whose sublayers read the stream itself (norm on the sublayer's RESULT only):
//       y   = c * (a' + b')      a' = a / rms(a) * wa when wa is given, else a; b' likewise (b optional)
//       x  += y / rms(y) * w1
//       out = x in the compute dtype, or x / rms(x) * w2 when w2 is given
//     Two results normed separately and averaged (mixers side by side: c = 0.5), or two addends summed as they are (routed
//     experts + a shared expert: c = 1), or one result alone.
//   Both are bound by memory: x in and out in fp32, the results, the gate and out once each. Rows of a multiple of four columns, up to 8192,
//   on aligned addresses are held in registers (row_wide.h); other rows go through LDS column by column. bf16, gated step:
//   8192 x 1024 48 -> 32 us, 4500 x 2048 56 -> 37 us, 32 x 2048 7.7 -> 4.9 us; two normed results 3663 x 2048 49 -> 26 us (4 TB/s).
//   swl_causal_conv_state: out[t] = (h[t] if add_input) + sum_j w[j][c] * h[t - taps + 1 + j] per channel (w tap-major) over the tokens of
//     one sequence, for any cut of the sequence into steps: inputs of earlier steps come from the sequence's state slot,
//     which keeps the last taps - 1 inputs. The tail is double-buffered: a step reads buffer `parity` and the workgroup of
//     a portion's last token writes the other one, so no launch reads what it writes.
//   swl_token_shift_mix: out[s][t] = h[t] + (h[t - 1] - h[t]) * mu[s] for several mixing vectors at once (h[-1] = 0); the last input
//     of every sequence is carried like a two-tap convolution's.
#include "swl_common.h"
#include "conv_tail.h"
#include "row_wide.h"

namespace swl {

constexpr int kRsThreads = 256;

__device__ __forceinline__ float rs_block_sum(float v, float *red) {
    v = wave_allreduce_sum(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kRsThreads / 64; ++w) t += red[w];
    return t;
}

__device__ __forceinline__ float sigmoidf_(float z) { return 1.0f / (1.0f + expf(-z)); }

template <typename T>
__global__ __launch_bounds__(kRsThreads) void gated_add_rmsnorm_kernel(
    float *x, const T *m, const T *m2, const T *m2_gate, int64_t m2_gate_stride, const T *r, int64_t r_stride,
    const float *r_bias, const float *w1, T *out, const float *w2, const int32_t *row_idx, float eps, int width) {
    extern __shared__ float lds[];
    float *row = lds, *red = lds + width;
    const int64_t o = blockIdx.x;
    const int64_t t = row_idx ? row_idx[o] : o;
    float *xr = x + t * width;
    if (m) {
        const float s2 = m2 ? sigmoidf_(to_f(m2_gate[t * m2_gate_stride])) : 0.f;
        float ss = 0.f;
        for (int i = threadIdx.x; i < width; i += kRsThreads) {
            float y = to_f(m[t * width + i]);
            if (m2) y += s2 * to_f(m2[t * width + i]);
            if (r) y *= sigmoidf_(to_f(r[t * r_stride + i]) + r_bias[i]);
            row[i] = y;
            ss += y * y;
        }
        const float rstd = 1.0f / sqrtf(rs_block_sum(ss, red) / static_cast<float>(width) + eps);
        for (int i = threadIdx.x; i < width; i += kRsThreads) {     // (each thread touches only its own columns of row[])
            const float v = xr[i] + row[i] * rstd * w1[i];
            xr[i] = v;
            row[i] = v;
        }
    } else {
        for (int i = threadIdx.x; i < width; i += kRsThreads) row[i] = xr[i];
    }
    if (!out) return;
    float ss = 0.f;
    for (int i = threadIdx.x; i < width; i += kRsThreads) ss += row[i] * row[i];
    const float rstd = 1.0f / sqrtf(rs_block_sum(ss, red) / static_cast<float>(width) + eps);
    for (int i = threadIdx.x; i < width; i += kRsThreads) out[o * width + i] = to_t<T>(row[i] * rstd * w2[i]);
}

// What a step of one token a sequence needs to convolve its rows where they are normed: tails and taps as swl_causal_conv_state's.
struct ConvStep {
    float *state;
    int64_t slot_stride, tail_off;
    const float *w;
    const int32_t *tok_pos, *tok_state;
    int taps;
};
constexpr int kConvStepTaps = 4;

// NC: 0, or kConvStepTaps: `sum` receives out + its causal convolution. The earlier inputs and the taps are asked for first, so that they
// come while the row is normed.
template <typename T, int TPR, int NV, int NC>
__global__ __launch_bounds__(kRowThreads) void gated_add_rmsnorm_wide_kernel(
    float *x, const T *m, const float *slabs, int parts, int64_t slab_stride, const T *m2, const T *m2_gate, int64_t m2_gate_stride, const T *r, int64_t r_stride,
    const float *r_bias, const float *w1, T *out, const float *w2, const int32_t *row_idx, float eps, int64_t rows, int width, T *sum, ConvStep conv) {
    __shared__ float red[2][kRowThreads / 64];
    const int64_t id = static_cast<int64_t>(blockIdx.x) * (kRowThreads / TPR) + threadIdx.x / TPR, o = min(id, rows - 1);
    const bool live = id < rows;
    const int64_t t = row_idx ? row_idx[o] : o;
    const int c0 = (threadIdx.x % TPR) * 4;
    float *xr = x + t * width;
    float v[NV][4];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = 0.f;
        if (c0 + 4 * TPR * j < width) row_load<float>(v[j], xr + c0 + 4 * TPR * j);
    }
    constexpr int MOST = NC > 0 ? NC - 1 : 1;
    float past[MOST][NV][4], taps[MOST + 1][NV][4];     // past[k - 1], taps[k]: the input k tokens back and its weights
    const int R = NC > 0 ? conv.taps - 1 : 0;
    float *new_tail = nullptr;
    int pos = 0;
    if constexpr (NC > 0) {
        pos = conv.tok_pos[o];
        const float *old_tail = nullptr;
        if (R > 0) {
            const int code = conv.tok_state[o];
            float *base = conv.state + static_cast<int64_t>(code >> 1) * conv.slot_stride + conv.tail_off;
            old_tail = base + static_cast<int64_t>(code & 1) * R * width;
            new_tail = base + static_cast<int64_t>(1 - (code & 1)) * R * width;
        }
#pragma unroll
        for (int k = 0; k <= MOST; ++k)
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int c = c0 + 4 * TPR * j;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    taps[k][j][e] = 0.f;
                    if (k > 0) past[k > 0 ? k - 1 : 0][j][e] = 0.f;
                }
                if (k <= R && c < width) {
                    row_load<float>(taps[k][j], conv.w + static_cast<int64_t>(R - k) * width + c);
                    if (k > 0 && pos >= k) row_load<float>(past[k > 0 ? k - 1 : 0][j], old_tail + static_cast<int64_t>(R - k) * width + c);
                }
            }
    }
    if (m || slabs) {
        float y[NV][4], a2[NV][4], rv[NV][4];
        const float s2 = m2 ? sigmoidf_(to_f(m2_gate[t * m2_gate_stride])) : 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = c0 + 4 * TPR * j;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[j][e] = a2[j][e] = rv[j][e] = 0.f;
            if (c < width) {
                if (m) row_load<T>(y[j], m + t * width + c);
                if (m2) row_load<T>(a2[j], m2 + t * width + c);
                if (r) row_load<T>(rv[j], r + t * r_stride + c);
            }
        }
        if (slabs) row_load_parts<TPR, NV>(y, slabs + t * width, c0, width, parts, slab_stride);
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = c0 + 4 * TPR * j;
            float bias[4] = {0.f, 0.f, 0.f, 0.f};
            if (r && c < width) row_load<float>(bias, r_bias + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (m2) y[j][e] += s2 * a2[j][e];
                if (r) y[j][e] *= sigmoidf_(rv[j][e] + bias[e]);
                ss += y[j][e] * y[j][e];
            }
        }
        const float rstd = 1.0f / sqrtf(row_sum<TPR>(ss, red[0]) / static_cast<float>(width) + eps);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = c0 + 4 * TPR * j;
            if (c < width) {
                float w[4];
                row_load<float>(w, w1 + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[j][e] = v[j][e] + y[j][e] * rstd * w[e];
                if (live) row_store<float>(xr + c, v[j]);
            }
        }
    }
    if (!out) return;
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += v[j][e] * v[j][e];
    const float rstd = 1.0f / sqrtf(row_sum<TPR>(ss, red[1]) / static_cast<float>(width) + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
        if (live && c < width) {
            float w[4];
            row_load<float>(w, w2 + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = v[j][e] * rstd * w[e];
            if constexpr (NC == 0) {
                row_store<T>(out + o * width + c, w);
            } else {
                // (one rounding for the row, the sum and the tail: left alone the compiler rounds the product to fp16 in one step for one
                // of them and in two for the others)
                typedef int Bits __attribute__((ext_vector_type(sizeof(T))));
                vec4_t<T> x;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = to_t<T>(w[e]);
                Bits bits = __builtin_bit_cast(Bits, x);
                asm volatile("" : "+v"(bits));
                x = __builtin_bit_cast(vec4_t<T>, bits);
                *reinterpret_cast<vec4_t<T> *>(out + o * width + c) = x;
                float cur[4], y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    cur[e] = to_f(x[e]);
                    y[e] = 0.f;
                }
#pragma unroll
                for (int k = MOST; k >= 1; --k) {
                    if (k <= R) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[e] += taps[k][j][e] * past[k - 1][j][e];
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    y[e] += taps[0][j][e] * cur[e];
                    y[e] += cur[e];
                }
                row_store<T>(sum + o * width + c, y);
#pragma unroll
                for (int k = 0; k < MOST; ++k)      // (the input k tokens back becomes entry R - 1 - k)
                    if (k < R && pos >= k) row_store<float>(new_tail + static_cast<int64_t>(R - 1 - k) * width + c, k == 0 ? cur : past[k > 0 ? k - 1 : 0][j]);
            }
        }
    }
}

template <typename T, int TPR, int NV>
__global__ __launch_bounds__(kRowThreads) void post_norm_add_wide_kernel(float *x, const T *a, const float *wa, const T *b, const float *wb,
                                                                         float coef, const float *w1, T *out, const float *w2, float eps,
                                                                         int64_t rows, int width) {
    __shared__ float red[4][kRowThreads / 64];
    const int64_t id = static_cast<int64_t>(blockIdx.x) * (kRowThreads / TPR) + threadIdx.x / TPR, t = min(id, rows - 1);
    const bool live = id < rows;
    const int c0 = (threadIdx.x % TPR) * 4;
    float *xr = x + t * width;
    float y[NV][4], z[NV][4], v[NV][4];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[j][e] = z[j][e] = v[j][e] = 0.f;
        if (c < width) {
            row_load<T>(y[j], a + t * width + c);
            if (b) row_load<T>(z[j], b + t * width + c);
            row_load<float>(v[j], xr + c);
        }
    }
    float na = 1.f, nb = 1.f;
    if (wa) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) s += y[j][e] * y[j][e];
        na = 1.0f / sqrtf(row_sum<TPR>(s, red[0]) / static_cast<float>(width) + eps);
    }
    if (b && wb) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) s += z[j][e] * z[j][e];
        nb = 1.0f / sqrtf(row_sum<TPR>(s, red[1]) / static_cast<float>(width) + eps);
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
        float w[4] = {1.f, 1.f, 1.f, 1.f}, u[4] = {1.f, 1.f, 1.f, 1.f};
        if (wa && c < width) row_load<float>(w, wa + c);
        if (b && wb && c < width) row_load<float>(u, wb + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float s = wa ? y[j][e] * na * w[e] : y[j][e];
            if (b) s += wb ? z[j][e] * nb * u[e] : z[j][e];
            s *= coef;
            y[j][e] = s;
            ss += s * s;
        }
    }
    const float rstd = 1.0f / sqrtf(row_sum<TPR>(ss, red[2]) / static_cast<float>(width) + eps);
    float sx = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
        if (c < width) {
            float w[4];
            row_load<float>(w, w1 + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[j][e] = v[j][e] + y[j][e] * rstd * w[e];
                sx += v[j][e] * v[j][e];
            }
            if (live) {
                row_store<float>(xr + c, v[j]);
                if (out && !w2) row_store<T>(out + t * width + c, v[j]);
            }
        }
    }
    if (!out || !w2) return;
    const float rx = 1.0f / sqrtf(row_sum<TPR>(sx, red[3]) / static_cast<float>(width) + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + 4 * TPR * j;
        if (live && c < width) {
            float w[4];
            row_load<float>(w, w2 + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = v[j][e] * rx * w[e];
            row_store<T>(out + t * width + c, w);
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kRsThreads) void post_norm_add_kernel(float *x, const T *a, const float *wa, const T *b,
                                                                   const float *wb, float coef, const float *w1, T *out,
                                                                   const float *w2, float eps, int width) {
    extern __shared__ float lds[];
    float *ra = lds, *rb = lds + width, *red = lds + 2 * width;
    const int64_t t = blockIdx.x;
    float *xr = x + t * width;
    float sa = 0.f, sb = 0.f;
    for (int i = threadIdx.x; i < width; i += kRsThreads) {
        const float va = to_f(a[t * width + i]);
        ra[i] = va;
        sa += va * va;
        if (b) {
            const float vb = to_f(b[t * width + i]);
            rb[i] = vb;
            sb += vb * vb;
        }
    }
    float na = 1.f, nb = 1.f;
    if (wa) na = 1.0f / sqrtf(rs_block_sum(sa, red) / static_cast<float>(width) + eps);
    if (b && wb) nb = 1.0f / sqrtf(rs_block_sum(sb, red) / static_cast<float>(width) + eps);
    float ss = 0.f;
    for (int i = threadIdx.x; i < width; i += kRsThreads) {     // (each thread touches only its own columns of the rows)
        float y = wa ? ra[i] * na * wa[i] : ra[i];
        if (b) y += wb ? rb[i] * nb * wb[i] : rb[i];
        y *= coef;
        ra[i] = y;
        ss += y * y;
    }
    const float rstd = 1.0f / sqrtf(rs_block_sum(ss, red) / static_cast<float>(width) + eps);
    float sx = 0.f;
    for (int i = threadIdx.x; i < width; i += kRsThreads) {
        const float v = xr[i] + ra[i] * rstd * w1[i];
        xr[i] = v;
        ra[i] = v;
        sx += v * v;
    }
    if (!out) return;
    if (!w2) {
        for (int i = threadIdx.x; i < width; i += kRsThreads) out[t * width + i] = to_t<T>(ra[i]);
        return;
    }
    const float rx = 1.0f / sqrtf(rs_block_sum(sx, red) / static_cast<float>(width) + eps);
    for (int i = threadIdx.x; i < width; i += kRsThreads) out[t * width + i] = to_t<T>(ra[i] * rx * w2[i]);
}

template <typename T>
__global__ __launch_bounds__(kRsThreads) void causal_conv_state_kernel(
    T *out, int64_t out_stride, const T *h, int64_t h_stride, const float *w, float *state, int64_t slot_stride,
    int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *tok_state, const int32_t *tok_seq,
    int64_t num_tokens, int C, int taps, int add_input) {
    const int64_t t = blockIdx.x;
    const ConvTail tail(state, slot_stride, tail_off, tok_pos, tok_start, tok_state, tok_seq, num_tokens, C, taps, t);
    if (ConvTail::wide_ok(h, h_stride, w, state, slot_stride, tail_off, C) && (out_stride & (16 / sizeof(T) - 1)) == 0 &&
        (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
        for (int c = threadIdx.x * 8; c < C; c += blockDim.x * 8) {
            float cur[8], a[8];
            ConvTail::row8(h + t * h_stride + c, cur);
            tail.conv_save8(h, h_stride, w, c, cur, a);
            if (add_input) {
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] += cur[j];
            }
            ConvTail::put8(out + t * out_stride + c, a);
        }
        return;
    }
    for (int c = threadIdx.x; c < C; c += blockDim.x) {
        const float cur = to_f(h[t * h_stride + c]);
        float a = tail.conv(h, h_stride, w, c, cur);
        if (add_input) a += cur;
        out[t * out_stride + c] = to_t<T>(a);
        tail.save(h, h_stride, c, cur);
    }
}

template <typename T, int TOK>
__global__ __launch_bounds__(kRsThreads) void causal_conv_run_kernel(
    T *out, int64_t out_stride, const T *h, int64_t h_stride, const float *w, float *state, int64_t slot_stride,
    int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *tok_state, const int32_t *tok_seq,
    int64_t num_tokens, int C, int taps, int add_input) {
    __shared__ int meta[TOK][4];
    const ConvRun<TOK> run(meta, state, slot_stride, tail_off, tok_pos, tok_start, tok_state, tok_seq, num_tokens, C, taps,
                           static_cast<int64_t>(blockIdx.x) * TOK);
    __syncthreads();
    for (int c = threadIdx.x * 8; c < C; c += blockDim.x * 8)
        run.walk(h, h_stride, w, c, [&](int i, const float (&cur)[8], float (&a)[8]) {
            if (add_input) {
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] += cur[j];
            }
            ConvTail::put8(out + (run.t0 + i) * out_stride + c, a);
        });
}

template <typename T>
__global__ __launch_bounds__(kRsThreads) void token_shift_mix_kernel(
    T *out, int64_t plane, const T *h, int64_t h_stride, const float *mu, int mixes, float *state, int64_t slot_stride,
    int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *tok_state, const int32_t *tok_seq,
    int64_t num_tokens, int C) {
    const int64_t t = blockIdx.x;
    const ConvTail tail(state, slot_stride, tail_off, tok_pos, tok_start, tok_state, tok_seq, num_tokens, C, 2, t);
    if constexpr (sizeof(T) == 2) {
        if (ConvTail::wide_ok(h, h_stride, mu, state, slot_stride, tail_off, C) && (plane & 7) == 0 &&
            (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
            for (int c = threadIdx.x * 8; c < C; c += kRsThreads * 8) {
                const vec8_t<T> x = load8(h + t * h_stride + c);
                float cur[8], prev[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) cur[j] = to_f(x[j]);
                tail.at8(h, h_stride, c, tail.pos - 1, prev);
                for (int s = 0; s < mixes; ++s) {
                    const float4_t m0 = *reinterpret_cast<const float4_t *>(mu + static_cast<int64_t>(s) * C + c);
                    const float4_t m1 = *reinterpret_cast<const float4_t *>(mu + static_cast<int64_t>(s) * C + c + 4);
                    vec8_t<T> o;
#pragma unroll
                    for (int j = 0; j < 8; ++j) o[j] = to_t<T>(cur[j] + (prev[j] - cur[j]) * (j < 4 ? m0[j & 3] : m1[j & 3]));
                    store8(out + s * plane + t * C + c, o);
                }
                tail.save8(h, h_stride, c, cur);
            }
            return;
        }
    }
    for (int c = threadIdx.x; c < C; c += kRsThreads) {
        const float cur = to_f(h[t * h_stride + c]), prev = tail.at(h, h_stride, c, tail.pos - 1);
        for (int s = 0; s < mixes; ++s)
            out[s * plane + t * C + c] = to_t<T>(cur + (prev - cur) * mu[static_cast<int64_t>(s) * C + c]);
        tail.save(h, h_stride, c, cur);
    }
}

inline size_t rs_lds_bytes(int width) { return (static_cast<size_t>(width) + kRsThreads / 64) * sizeof(float); }

} // namespace swl

static int gated_add_rmsnorm(float *x, const void *m, const float *slabs, int parts, const void *m2, const void *m2_gate, int64_t m2_gate_stride,
                                     const void *r, int64_t r_stride, const float *r_bias, const float *w1, void *out,
                                     const float *w2, const int32_t *row_idx, float eps, int64_t num_rows, int32_t width,
                                     int32_t dtype, swl_stream_t stream, void *sum = nullptr, const swl::ConvStep &conv = {}) {
    if (num_rows < 0 || width <= 0) return SWL_ERR_BAD_ARG;
    if (num_rows == 0) return SWL_OK;
    if (!x || ((m || slabs) && !w1) || (m2 && ((!m && !slabs) || !m2_gate)) || (r && ((!m && !slabs) || !r_bias)) || (out && !w2) ||
        (row_idx && (m || slabs)))
        return SWL_ERR_BAD_ARG;
    if (!m && !slabs && !out) return SWL_OK;
    if (num_rows > 0x7fffffffLL || swl::rs_lds_bytes(width) > 64 * 1024) return SWL_ERR_UNSUPPORTED;
#define SWL_GO_NC(TPR, NV, NC)                                                                                                         \
    hipLaunchKernelGGL((swl::gated_add_rmsnorm_wide_kernel<T, TPR, NV, NC>), dim3(static_cast<unsigned>((num_rows * TPR + 255) / 256)),    \
                       dim3(swl::kRowThreads), 0, static_cast<hipStream_t>(stream), x, static_cast<const T *>(m), slabs, parts,        \
                       num_rows * width, static_cast<const T *>(m2), static_cast<const T *>(m2_gate), m2_gate_stride, static_cast<const T *>(r),         \
                       r_stride, r_bias, w1, static_cast<T *>(out), w2, row_idx, eps, num_rows, width, static_cast<T *>(sum), conv)
#define SWL_GO(TPR, NV) SWL_GO_NC(TPR, NV, 0)
    SWL_DISPATCH_DTYPE3(dtype, T, {
        const bool wide = width % 4 == 0 && width <= swl::kRowMaxWidth && r_stride % 4 == 0 && swl::row_aligned<float>(x) &&
                          swl::row_aligned<T>(m) && swl::row_aligned<T>(m2) && swl::row_aligned<T>(r) && swl::row_aligned<T>(out) &&
                          swl::row_aligned<float>(r_bias) && swl::row_aligned<float>(w1) && swl::row_aligned<float>(w2) && swl::row_aligned<float>(slabs);
        if ((slabs || sum) && !wide) return SWL_ERR_UNSUPPORTED;
        if (sum) {
            if (!swl::row_aligned<T>(sum) || !swl::row_aligned<float>(conv.w) || !swl::row_aligned<float>(conv.state) || conv.slot_stride % 4 ||
                conv.tail_off % 4)
                return SWL_ERR_UNSUPPORTED;
            if (width <= 1024) SWL_GO_NC(256, 1, swl::kConvStepTaps);
            else if (width <= 2048) SWL_GO_NC(256, 2, swl::kConvStepTaps);
            else SWL_GO_NC(256, 4, swl::kConvStepTaps);
            return swl::check_launch();
        }
        if (wide) {
            SWL_ROW_SHAPE(num_rows, width, SWL_GO);
            return swl::check_launch();
        }
        hipLaunchKernelGGL((swl::gated_add_rmsnorm_kernel<T>), dim3(static_cast<unsigned>(num_rows)), dim3(swl::kRsThreads),
                           swl::rs_lds_bytes(width), static_cast<hipStream_t>(stream), x, static_cast<const T *>(m),
                           static_cast<const T *>(m2), static_cast<const T *>(m2_gate), m2_gate_stride,
                           static_cast<const T *>(r), r_stride, r_bias, w1, static_cast<T *>(out), w2, row_idx, eps, width);
    });
#undef SWL_GO
#undef SWL_GO_NC
    return swl::check_launch();
}

extern "C" int swl_gated_add_rmsnorm(float *x, const void *m, const void *m2, const void *m2_gate, int64_t m2_gate_stride,
                                     const void *r, int64_t r_stride, const float *r_bias, const float *w1, void *out,
                                     const float *w2, const int32_t *row_idx, float eps, int64_t num_rows, int32_t width,
                                     int32_t dtype, swl_stream_t stream) {
    return gated_add_rmsnorm(x, m, nullptr, 0, m2, m2_gate, m2_gate_stride, r, r_stride, r_bias, w1, out, w2, row_idx, eps, num_rows, width,
                             dtype, stream);
}

extern "C" int swl_gated_add_rmsnorm_parts(float *x, const float *slabs, int32_t parts, const void *m2, const void *m2_gate,
                                           int64_t m2_gate_stride, const void *r, int64_t r_stride, const float *r_bias,
                                           const float *w1, void *out, const float *w2, float eps, int64_t num_rows, int32_t width,
                                           int32_t dtype, swl_stream_t stream) {
    if (!slabs || parts < 1) return SWL_ERR_BAD_ARG;
    return gated_add_rmsnorm(x, nullptr, slabs, parts, m2, m2_gate, m2_gate_stride, r, r_stride, r_bias, w1, out, w2, nullptr, eps, num_rows,
                             width, dtype, stream);
}

extern "C" int swl_gated_add_rmsnorm_conv(float *x, const void *m, const float *slabs, int32_t parts, const void *m2, const void *m2_gate,
                                          int64_t m2_gate_stride, const void *r, int64_t r_stride, const float *r_bias, const float *w1,
                                          void *out, const float *w2, void *sum, const float *conv_w, int32_t taps, float *state,
                                          int64_t slot_stride, int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_state,
                                          float eps, int64_t num_rows, int32_t width, int32_t dtype, swl_stream_t stream) {
    if (taps < 1 || (m && slabs) || (slabs && parts < 1)) return SWL_ERR_BAD_ARG;
    if (num_rows > 0 && (!out || !sum || !conv_w || !tok_pos || (taps > 1 && (!state || !tok_state)))) return SWL_ERR_BAD_ARG;
    if (taps > swl::kConvStepTaps || width > 4096) return SWL_ERR_UNSUPPORTED;
    return gated_add_rmsnorm(x, m, slabs, parts, m2, m2_gate, m2_gate_stride, r, r_stride, r_bias, w1, out, w2, nullptr, eps, num_rows, width,
                             dtype, stream, sum, swl::ConvStep{state, slot_stride, tail_off, conv_w, tok_pos, tok_state, taps});
}

extern "C" int swl_causal_conv_state(void *out, int64_t out_stride, const void *h, int64_t h_stride, const float *w,
                                     float *state, int64_t slot_stride, int64_t tail_off, const int32_t *tok_pos,
                                     const int32_t *tok_start, const int32_t *tok_state, const int32_t *tok_seq,
                                     int64_t num_tokens, int32_t channels, int32_t taps, int32_t add_input, int32_t dtype,
                                     swl_stream_t stream) {
    if (num_tokens < 0 || channels <= 0 || taps < 1 || h_stride < channels || out_stride < channels) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!out || !h || !w || !tok_pos || !tok_start || !tok_seq) return SWL_ERR_BAD_ARG;
    if (taps > 1 && (!state || !tok_state)) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        // (a thread takes eight channels: no more waves than have some)
        const bool wide = swl::ConvTail::wide_ok(static_cast<const T *>(h), h_stride, w, state, slot_stride, tail_off, channels);
        const int threads = wide && channels < 8 * swl::kRsThreads ? (channels / 8 + 63) / 64 * 64 : swl::kRsThreads;
        if (wide && taps <= 4 && out_stride % (16 / sizeof(T)) == 0 && swl::aligned16(out) && swl::conv_run_pays(num_tokens, channels)) {
            hipLaunchKernelGGL((swl::causal_conv_run_kernel<T, 4>), dim3(static_cast<unsigned>((num_tokens + 3) / 4)), dim3(static_cast<unsigned>(threads)),
                               0, static_cast<hipStream_t>(stream), static_cast<T *>(out), out_stride, static_cast<const T *>(h), h_stride, w, state,
                               slot_stride, tail_off, tok_pos, tok_start, tok_state, tok_seq, num_tokens, channels, taps, add_input);
            return swl::check_launch();
        }
        hipLaunchKernelGGL((swl::causal_conv_state_kernel<T>), dim3(static_cast<unsigned>(num_tokens)),
                           dim3(static_cast<unsigned>(threads)), 0, static_cast<hipStream_t>(stream), static_cast<T *>(out), out_stride,
                           static_cast<const T *>(h), h_stride, w, state, slot_stride, tail_off, tok_pos, tok_start,
                           tok_state, tok_seq, num_tokens, channels, taps, add_input);
    });
    return swl::check_launch();
}

extern "C" int swl_token_shift_mix(void *out, const void *h, int64_t h_stride, const float *mu, int32_t mixes, float *state,
                                   int64_t slot_stride, int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start,
                                   const int32_t *tok_state, const int32_t *tok_seq, int64_t num_tokens, int32_t width,
                                   int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || mixes <= 0 || h_stride < width) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!out || !h || !mu || !state || !tok_pos || !tok_start || !tok_state || !tok_seq) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::token_shift_mix_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kRsThreads), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(out), num_tokens * width,
                           static_cast<const T *>(h), h_stride, mu, mixes, state, slot_stride, tail_off, tok_pos, tok_start,
                           tok_state, tok_seq, num_tokens, width);
    });
    return swl::check_launch();
}

extern "C" int swl_post_norm_add(float *x, const void *a, const float *wa, const void *b, const float *wb, float coef,
                                 const float *w1, void *out, const float *w2, float eps, int64_t num_rows, int32_t width,
                                 int32_t dtype, swl_stream_t stream) {
    if (num_rows < 0 || width <= 0) return SWL_ERR_BAD_ARG;
    if (num_rows == 0) return SWL_OK;
    if (!x || !a || !w1 || (wb && !b) || (w2 && !out)) return SWL_ERR_BAD_ARG;
    const size_t lds = (2 * static_cast<size_t>(width) + swl::kRsThreads / 64) * sizeof(float);
    if (num_rows > 0x7fffffffLL || lds > 64 * 1024) return SWL_ERR_UNSUPPORTED;
#define SWL_GO(TPR, NV)                                                                                                                \
    hipLaunchKernelGGL((swl::post_norm_add_wide_kernel<T, TPR, NV>), dim3(static_cast<unsigned>((num_rows * TPR + 255) / 256)),        \
                       dim3(swl::kRowThreads), 0, static_cast<hipStream_t>(stream), x, static_cast<const T *>(a), wa,                  \
                       static_cast<const T *>(b), wb, coef, w1, static_cast<T *>(out), w2, eps, num_rows, width)
    SWL_DISPATCH_DTYPE3(dtype, T, {
        const bool wide = width % 4 == 0 && width <= swl::kRowMaxWidth && swl::row_aligned<float>(x) && swl::row_aligned<T>(a) &&
                          swl::row_aligned<T>(b) && swl::row_aligned<T>(out) && swl::row_aligned<float>(wa) &&
                          swl::row_aligned<float>(wb) && swl::row_aligned<float>(w1) && swl::row_aligned<float>(w2);
        if (wide) {
            SWL_ROW_SHAPE(num_rows, width, SWL_GO);
            return swl::check_launch();
        }
        hipLaunchKernelGGL((swl::post_norm_add_kernel<T>), dim3(static_cast<unsigned>(num_rows)), dim3(swl::kRsThreads), lds,
                           static_cast<hipStream_t>(stream), x, static_cast<const T *>(a), wa, static_cast<const T *>(b), wb,
                           coef, w1, static_cast<T *>(out), w2, eps, width);
    });
#undef SWL_GO
    return swl::check_launch();
}
