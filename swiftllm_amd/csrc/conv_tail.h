// conv_tail.h — the carried inputs of a short causal convolution over time, shared by the kernels that convolve.
//
// A sequence's state slot keeps the last R = taps - 1 inputs of every channel, twice: buffer `parity` is what earlier steps
// left, the other buffer receives what this step leaves (written by the workgroup of the portion's last token). Entry r of a
// buffer holds the input at position (tokens consumed so far) - R + r; entries of positions before the sequence's start are
// never read (those inputs are zero by definition), so a slot needs no clearing when it changes hands.
#pragma once

#include "swl_common.h"

namespace swl {

struct ConvTail {
    const float *old_tail;
    float *new_tail;
    int64_t t;
    int R, C, taps, pos, start;
    bool last;

    __device__ ConvTail(float *state, int64_t slot_stride, int64_t tail_off, const int32_t *tok_pos,
                        const int32_t *tok_start, const int32_t *tok_state, const int32_t *tok_seq, int64_t num_tokens,
                        int channels, int taps_, int64_t token)
        : old_tail(nullptr), new_tail(nullptr), t(token), R(taps_ - 1), C(channels), taps(taps_) {
        pos = tok_pos[t];
        start = tok_start[t];
        last = (t + 1 == num_tokens) || tok_seq[t + 1] != tok_seq[t];
        if (R > 0) {
            const int code = tok_state[t];      // slot * 2 + parity
            float *base = state + static_cast<int64_t>(code >> 1) * slot_stride + tail_off;
            const int par = code & 1;
            old_tail = base + static_cast<int64_t>(par) * R * C;
            new_tail = base + static_cast<int64_t>(1 - par) * R * C;
        }
    }

    // input of channel c at position q < pos: zero before the sequence, a row of this step, or the carried tail
    template <typename T>
    __device__ __forceinline__ float at(const T *h, int64_t h_stride, int c, int q) const {
        if (q < 0) return 0.f;
        if (q >= start) return to_f(h[(t - (pos - q)) * h_stride + c]);
        return old_tail[static_cast<int64_t>(R - (start - q)) * C + c];
    }

    // sum_j w[j][c] * input(pos - taps + 1 + j); w is tap-major [taps, channels], the last tap multiplies the current input
    template <typename T>
    __device__ __forceinline__ float conv(const T *h, int64_t h_stride, const float *w, int c, float cur) const {
        float a = 0.f;
        for (int k = taps - 1; k >= 1; --k) a += w[static_cast<int64_t>(taps - 1 - k) * C + c] * at(h, h_stride, c, pos - k);
        return a + w[static_cast<int64_t>(taps - 1) * C + c] * cur;
    }

    // the portion's last token leaves the sequence's new tail (channel c)
    template <typename T>
    __device__ __forceinline__ void save(const T *h, int64_t h_stride, int c, float cur) const {
        if (!last || R == 0) return;
        for (int r = 0; r < R; ++r) {
            const int q = pos + 1 - R + r;
            if (q < 0) continue;
            new_tail[static_cast<int64_t>(r) * C + c] = q == pos ? cur : at(h, h_stride, c, q);
        }
    }

    // ---- the same for 8 consecutive channels (16-byte loads; c a multiple of 8, rows 16-byte aligned) ----
    template <typename T>
    static __device__ __forceinline__ void row8(const T *p, float (&v)[8]) {
        if constexpr (sizeof(T) == 2) {
            const vec8_t<T> x = load8(p);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = to_f(x[j]);
        } else {
            const float4_t a = *reinterpret_cast<const float4_t *>(p), b = *reinterpret_cast<const float4_t *>(p + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = a[j];
                v[4 + j] = b[j];
            }
        }
    }
    template <typename T>
    static __device__ __forceinline__ void put8(T *p, const float (&v)[8]) {
        if constexpr (sizeof(T) == 2) {
            vec8_t<T> x;
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = to_t<T>(v[j]);
            store8(p, x);
        } else {
            *reinterpret_cast<float4_t *>(p) = float4_t{v[0], v[1], v[2], v[3]};
            *reinterpret_cast<float4_t *>(p + 4) = float4_t{v[4], v[5], v[6], v[7]};
        }
    }
    template <typename T>
    __device__ __forceinline__ void at8(const T *h, int64_t h_stride, int c, int q, float (&v)[8]) const {
        if (q < 0) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = 0.f;
        } else if (q >= start) {
            row8(h + (t - (pos - q)) * h_stride + c, v);
        } else {
            row8(old_tail + static_cast<int64_t>(R - (start - q)) * C + c, v);
        }
    }

    // same sums in the same order as conv()
    template <typename T>
    __device__ __forceinline__ void conv8(const T *h, int64_t h_stride, const float *w, int c, const float (&cur)[8],
                                          float (&a)[8]) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = 0.f;
        for (int k = taps - 1; k >= 1; --k) {
            float v[8];
            at8(h, h_stride, c, pos - k, v);
            const float *wk = w + static_cast<int64_t>(taps - 1 - k) * C + c;
            const float4_t w0 = *reinterpret_cast<const float4_t *>(wk), w1 = *reinterpret_cast<const float4_t *>(wk + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                a[j] += w0[j] * v[j];
                a[4 + j] += w1[j] * v[4 + j];
            }
        }
        const float *wl = w + static_cast<int64_t>(taps - 1) * C + c;
        const float4_t w0 = *reinterpret_cast<const float4_t *>(wl), w1 = *reinterpret_cast<const float4_t *>(wl + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            a[j] += w0[j] * cur[j];
            a[4 + j] += w1[j] * cur[4 + j];
        }
    }

    template <typename T>
    __device__ __forceinline__ void save8(const T *h, int64_t h_stride, int c, const float (&cur)[8]) const {
        if (!last || R == 0) return;
        for (int r = 0; r < R; ++r) {
            const int q = pos + 1 - R + r;
            if (q < 0) continue;
            float v[8];
            if (q == pos) {
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = cur[j];
            } else {
                at8(h, h_stride, c, q, v);
            }
            float *p = new_tail + static_cast<int64_t>(r) * C + c;
            *reinterpret_cast<float4_t *>(p) = float4_t{v[0], v[1], v[2], v[3]};
            *reinterpret_cast<float4_t *>(p + 4) = float4_t{v[4], v[5], v[6], v[7]};
        }
    }

    // conv8 and save8 in one: up to three earlier inputs (four taps) and their weights are requested together and serve both; one behind
    // the other's sum they are a memory latency each, and the tail's as many again. 3 tokens in fp32: 1024
    // channels of 3 taps 8.5 -> 4.4 us (column by column before), the delta rule's 1536 of 4 taps with their norms 25 -> 8.2 us.
    template <typename T>
    __device__ __forceinline__ void conv_save8(const T *h, int64_t h_stride, const float *w, int c, const float (&cur)[8],
                                               float (&a)[8]) const {
        constexpr int MOST = 3;
        if (R > MOST) {
            conv8(h, h_stride, w, c, cur, a);
            save8(h, h_stride, c, cur);
            return;
        }
        float v[MOST][8], wk[MOST + 1][8];      // v[k - 1], wk[k]: the input k tokens back and its weights
#pragma unroll
        for (int k = 0; k <= MOST; ++k) {
            if (k <= R) {       // (uniform, as everything but c)
                row8(w + static_cast<int64_t>(R - k) * C + c, wk[k]);
                if (k > 0) at8(h, h_stride, c, pos - k, v[k > 0 ? k - 1 : 0]);
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = 0.f;
#pragma unroll
        for (int k = MOST; k >= 1; --k) {
            if (k <= R) {
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] += wk[k][j] * v[k - 1][j];
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] += wk[0][j] * cur[j];
        if (!last) return;
#pragma unroll
        for (int k = 0; k < MOST; ++k) {        // (the input k tokens back becomes entry R - 1 - k)
            if (k < R && pos - k >= 0) put8<float>(new_tail + static_cast<int64_t>(R - 1 - k) * C + c, k == 0 ? cur : v[k > 0 ? k - 1 : 0]);
        }
    }

    // whether the 8-channel forms may be used for rows of h (and a state region) laid out like this
    template <typename T>
    static __host__ __device__ __forceinline__ bool wide_ok(const T *h, int64_t h_stride, const float *w, const float *state,
                                                   int64_t slot_stride, int64_t tail_off, int channels) {
        return (channels & 7) == 0 && (h_stride & (16 / sizeof(T) - 1)) == 0 && (reinterpret_cast<uintptr_t>(h) & 15) == 0 &&
               (reinterpret_cast<uintptr_t>(w) & 15) == 0 && (reinterpret_cast<uintptr_t>(state) & 15) == 0 &&
               (slot_stride & 3) == 0 && (tail_off & 3) == 0;
    }
};

// The wide form for a workgroup that takes TOK tokens in a row (steps of many tokens): the taps, fp32 and four to eight times a 16-bit row, are
// read once for them, and a token's earlier inputs move on by one in registers. Up to four taps. meta: TOK x 4 ints of LDS, which a barrier has to
// stand behind before `walk`.
// When it pays: few tokens leave CUs idle, and a narrow row's workgroup is one wave, whose chain of four tokens takes its time. us of the causal convolution, a
// token a workgroup / four, bf16, 4 taps (2 taps and fp32 alike): 64 channels 4096 tokens 5.7 / 6.7, 6144 6.4 / 5.7; 256 2048 4.7 / 5.3, 4096 5.7 / 5.6, 8192
// 7.8 / 6.3; 512 2048 4.9 / 5.4, 3072 5.5 / 5.6, 4096 6.1 / 5.9, 8192 10.6 / 6.9; 1024 1024 4.7 / 5.4, 2048 6.2 / 6.1, 4096 10.5 / 7.0, 8192 18.1 / 11.4; 4096
// 2048 17.6 / 14.0, 8192 51.1 / 35.7. (The state space's 2304 channels, which end in fp32: 3663 tokens 26.4 / 24.6, too little to be seen in a pass.)
inline bool conv_run_pays(int64_t tokens, int64_t channels) { return tokens >= 6144 || (tokens >= 2048 && tokens * channels >= 1 << 21); }
template <int TOK>
struct ConvRun {
    static constexpr int MOST = 3;
    int64_t t0;
    int n, R, C, pos0, start0, code0;
    float *region;
    int64_t slot_stride;
    const int (*meta)[4];       // position, first position of the portion, state slot and parity, ends its portion

    __device__ ConvRun(int (*shared)[4], float *state, int64_t slot_stride_, int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start,
                       const int32_t *tok_state, const int32_t *tok_seq, int64_t num_tokens, int channels, int taps, int64_t first)
        : t0(first), R(taps - 1), C(channels), code0(0), region(state + tail_off), slot_stride(slot_stride_), meta(shared) {
        n = static_cast<int>(min<int64_t>(TOK, num_tokens - t0));
        pos0 = tok_pos[t0];
        start0 = tok_start[t0];
        if (R > 0) code0 = tok_state[t0];
        if (static_cast<int>(threadIdx.x) < n) {
            const int64_t t = t0 + threadIdx.x;
            int *m = shared[threadIdx.x];
            m[0] = tok_pos[t];
            m[1] = tok_start[t];
            m[2] = R > 0 ? tok_state[t] : 0;
            m[3] = t + 1 == num_tokens || tok_seq[t + 1] != tok_seq[t];
        }
    }

    __device__ __forceinline__ float *tail(int code, int parity) const {
        return region + static_cast<int64_t>(code >> 1) * slot_stride + static_cast<int64_t>(parity) * R * C;
    }

    // each(i, input[8], sum[8]) for tokens t0 + i, i < n, of channels c .. c + 7; the sums of ConvTail::conv8, in its order
    template <typename T, typename F>
    __device__ __forceinline__ void walk(const T *h, int64_t h_stride, const float *w, int c, F &&each) const {
        float past[MOST][8], wk[MOST + 1][8];
        typedef T Raw __attribute__((ext_vector_type(8)));
        Raw raw[TOK];
#pragma unroll
        for (int i = 0; i < TOK; ++i) raw[i] = *reinterpret_cast<const Raw *>(h + (t0 + min(i, n - 1)) * h_stride + c);
        auto earlier = [&](int64_t t, int code, int pos, int start) {
#pragma unroll
            for (int k = 1; k <= MOST; ++k)
                if (k <= R && pos >= k) {       // (uniform)
                    if (pos - k >= start) ConvTail::row8(h + (t - k) * h_stride + c, past[k - 1]);
                    else ConvTail::row8(tail(code, code & 1) + static_cast<int64_t>(R - (start - (pos - k))) * C + c, past[k - 1]);
                }
        };
        earlier(t0, code0, pos0, start0);
#pragma unroll
        for (int k = 0; k <= MOST; ++k)
            if (k <= R) ConvTail::row8(w + static_cast<int64_t>(R - k) * C + c, wk[k]);
#pragma unroll
        for (int i = 0; i < TOK; ++i) {
            if (i >= n) break;      // (uniform)
            auto of = [&](int what) { return __builtin_amdgcn_readfirstlane(meta[i][what]); };
            const int pos = of(0);
            if (i > 0 && R > 0 && of(1) == pos) earlier(t0 + i, of(2), pos, pos);      // (a portion begins)
            float cur[8], a[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                cur[j] = to_f(raw[i][j]);
                a[j] = 0.f;
            }
#pragma unroll
            for (int k = MOST; k >= 1; --k) {
                if (k <= R && pos >= k) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) a[j] += wk[k][j] * past[k - 1][j];
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] += wk[0][j] * cur[j];
            if (R > 0 && of(3)) {
                float *next = tail(of(2), 1 - (of(2) & 1));
#pragma unroll
                for (int k = 0; k < MOST; ++k)
                    if (k < R && pos >= k) ConvTail::put8<float>(next + static_cast<int64_t>(R - 1 - k) * C + c, k == 0 ? cur : past[k > 0 ? k - 1 : 0]);
            }
            each(i, cur, a);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
#pragma unroll
                for (int k = MOST - 1; k > 0; --k) past[k][j] = past[k - 1][j];
                past[0][j] = cur[j];
            }
        }
    }
};

} // namespace swl
