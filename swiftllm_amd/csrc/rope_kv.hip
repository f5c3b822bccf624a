// rope_kv.hip — rotary positions fused with the paged KV store, and what attention heads need after the softmax when they are
// gated or combined.
//
// Rotation: inside a head, for i < rot_dims / 2, dimension 2i is paired with dimension 2i + 1 (interleaved pairs) or dimension i
// with dimension i + rot_dims / 2 (halves: the kernels that take `half`); the pair (u, v) of a token at position p becomes
// (u cos a - v sin a, v cos a + u sin a), a = p * freq[i]. The frequencies come from the host as a float64 table (evaluated once
// per model, any interpolation included); the angle and its sine and cosine are evaluated in float64 per (token, i) into LDS —
// times a constant, where the kernel takes one — and used in fp32 by every head of the token: exact to fp32 rounding at any
// position. Dimensions from rot_dims on pass unchanged.
//
//   swl_rope_store_kv         rows [q: nq heads of d | k: nk heads of d | v: nv heads of dv]: q rotated in place, k rotated
//                             into the K pool, v copied into the V pool.
//   swl_qk_norm_rope_store_kv rows [q | k (| v)] of a projection whose biases are still to be added: per head bias, weighted RMS norm,
//                             rotation; q times a factor per head into a buffer of its own, k into the K pool, and into the V
//                             pool either the value columns or the KEYS AS PROJECTED (bias added, neither normed nor rotated).
//   swl_qkv_conv_rope_store_kv  rows [q | k | v] of a projection whose biases are still to be added, each step optional: bias, causal
//                             convolution over time per channel (inputs of earlier steps carried as projected, conv_tail.h),
//                             weighted RMS norm of the q / k heads, rotation; q into a buffer of its own, k into the K pool, v
//                             times a constant into the V pool. The row passes through LDS in fp32 and is rounded once.
//   swl_latent_rope_store_kv  latent attention. Rows hold H query heads [d unrotated | dr rotated] and (optionally) the
//                             compressed key/value row [r latent | dr shared rotated key part]. The rotated query parts go
//                             to qa[t][h][r : r + dr] (the caller fills qa[t][h][0 : r] with the queries folded through
//                             the key up-projection); the latent is RMS-normed (fp32 statistics, weight) and stored
//                             together with the rotated key part as ONE key head of r + dr, and once more, transposed, as
//                             the value head of r: attention over the pool then IS the latent attention with the
//                             up-projections applied outside (queries before, outputs after).
//   swl_diff_head_combine     out = unit_rms(a1 - lambda a2) * mult * sigmoid(gate) per head, a1 / a2 the fp32 results of two
//                             score maps over the same values, or (_shares) the key shares of them.
//   swl_head_gate             y[t][h][:] *= sigmoid(gate[t][h]).
//
// Pool layout as in qknorm_kv.hip: keys of a page [heads, 16, d], values transposed [heads, dv, 16]. The two kernels in the
// middle may lay heads out wider than they are (k_dim, v_dim: the row sizes that a compiled attention kernel serves); the
// columns beyond the head are written as zeros, which neither scores nor outputs see.
#include "swl_common.h"
#include "conv_tail.h"

namespace swl {

constexpr int kRkThreads = 256;
constexpr int kRkBlock = 16;        // tokens per KV block
constexpr int kRkMaxPairs = 256;    // rot_dims <= 512

__device__ __forceinline__ void rk_angles(float *cs, float *sn, const double *freq, int pos, int pairs, double mult = 1.0) {
    for (int i = threadIdx.x; i < pairs; i += kRkThreads) {
        const double a = static_cast<double>(pos) * freq[i];
        cs[i] = static_cast<float>(cos(a) * mult);
        sn[i] = static_cast<float>(sin(a) * mult);
    }
}

__device__ __forceinline__ float rk_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

template <typename T>
__global__ __launch_bounds__(kRkThreads) void rope_store_kv_kernel(
    T *qkv, const double *freq, T *k_cache, T *v_cache, const int32_t *block_table, const int32_t *tok_seq,
    const int32_t *tok_pos, int nq, int nk, int nv, int d, int dv, int rot_dims, int64_t tok_stride, int max_blocks_per_seq,
    int64_t block_stride) {
    __shared__ float cs[kRkMaxPairs], sn[kRkMaxPairs];
    const int64_t t = page_token();
    const int pos = tok_pos[t];
    const int pairs = rot_dims >> 1;
    rk_angles(cs, sn, freq, pos, pairs);
    __syncthreads();
    T *row = qkv + t * tok_stride;
    const bool store = k_cache != nullptr;
    int64_t blk = 0;
    if (store) blk = block_table[static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq + pos / kRkBlock];
    const int off = pos % kRkBlock;
    // queries: only the rotated pairs change
    for (int i = threadIdx.x; i < nq * pairs; i += kRkThreads) {
        const int h = i / pairs, j = i - h * pairs;
        T *p = row + static_cast<int64_t>(h) * d + 2 * j;
        const float u = to_f(p[0]), v = to_f(p[1]);
        p[0] = to_t<T>(u * cs[j] - v * sn[j]);
        p[1] = to_t<T>(v * cs[j] + u * sn[j]);
    }
    if (!store) return;
    // keys: every element goes to the pool, the first rot_dims of each head rotated
    const T *krow = row + static_cast<int64_t>(nq) * d;
    for (int i = threadIdx.x; i < nk * d; i += kRkThreads) {
        const int g = i / d, e = i - g * d;
        float x = to_f(krow[i]);
        if (e < rot_dims) {
            const int j = e >> 1;
            const float other = to_f(krow[i ^ 1]);      // (d is even: the partner is inside the head)
            x = (e & 1) ? x * cs[j] + other * sn[j] : x * cs[j] - other * sn[j];
        }
        k_cache[blk * block_stride + (static_cast<int64_t>(g) * kRkBlock + off) * d + e] = to_t<T>(x);
    }
    const T *vrow = krow + static_cast<int64_t>(nk) * d;
    for (int i = threadIdx.x; i < nv * dv; i += kRkThreads)
        v_cache[blk * block_stride + static_cast<int64_t>(i) * kRkBlock + off] = vrow[i];       // transposed page
}

template <typename T>
__global__ __launch_bounds__(kRkThreads) void qk_norm_rope_store_kv_kernel(
    const T *rows, T *q_out, const float *q_b, const float *k_b, const float *q_w, const float *k_w, const float *q_mult,
    const double *freq, T *k_cache, T *v_cache, const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos, int nq,
    int nk, int nv, int d, int dv, int rot_dims, int half, double rot_mult, int64_t tok_stride, int64_t q_out_stride, int k_dim,
    int v_dim, int keys_as_values, int max_blocks_per_seq, int64_t block_stride, float eps) {
    __shared__ float cs[kRkMaxPairs], sn[kRkMaxPairs];
    const int64_t t = page_token();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int pos = tok_pos[t];
    const int pairs = rot_dims >> 1;
    const T *row = rows + t * tok_stride;
    T *qrow = q_out + t * q_out_stride;
    const bool store = k_cache != nullptr;
    int64_t blk = 0;
    if (store) blk = block_table[static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq + pos / kRkBlock];
    const int off = pos % kRkBlock;
    T *kpage = k_cache + blk * block_stride, *vpage = v_cache + blk * block_stride;
    const int heads = store ? nq + nk : nq;
    bool wide = false;
    if constexpr (sizeof(T) == 2) {
        // 16-bit heads of a multiple of 8 elements up to 128 on 16-byte-aligned rows: a power-of-two group of lanes per head,
        // 8 elements per lane; a rotated lane's partner elements are 8 neighbours too (or, interleaved, its own)
        wide = d % 8 == 0 && d <= 128 && (tok_stride & 7) == 0 && (q_out_stride & 7) == 0 && (k_dim & 7) == 0 &&
               (half ? (pairs & 7) == 0 : (rot_dims & 7) == 0) && (block_stride & 7) == 0 &&
               ((reinterpret_cast<uintptr_t>(rows) | reinterpret_cast<uintptr_t>(q_out) | reinterpret_cast<uintptr_t>(k_cache) |
                 reinterpret_cast<uintptr_t>(q_b) | reinterpret_cast<uintptr_t>(k_b) | reinterpret_cast<uintptr_t>(q_w) |
                 reinterpret_cast<uintptr_t>(k_w)) & 15) == 0;
        if (wide) {
            const int lph = d <= 8 ? 1 : d <= 16 ? 2 : d <= 32 ? 4 : d <= 64 ? 8 : 16;      // lanes per head
            const int hpw = 64 / lph;
            const int slot = lane / lph, el = lane - slot * lph, e0 = el * 8;
            const bool turns = e0 < rot_dims, first = e0 < pairs;
            // (half) the partner elements of this lane's, and the pair index of its first element
            const int p0 = half && turns ? (first ? e0 + pairs : e0 - pairs) : e0;
            const int a0 = half ? (first ? e0 : p0) : e0 >> 1;
            // everything a head needs from memory is requested together, the first head's before the angles are evaluated
            vec8_t<T> own, other;
            float4_t bo[2], bp[2], wo[2], wp[2];
            float mult;
            auto fetch = [&](int hb) {
                const int h = hb + slot;
                const bool live = h < heads && e0 < d, is_q = h < nq;
                own = other = vec8_t<T>{};
                mult = 1.0f;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    bo[k] = bp[k] = float4_t{0.f, 0.f, 0.f, 0.f};
                    wo[k] = wp[k] = float4_t{1.f, 1.f, 1.f, 1.f};
                }
                if (!live) return;
                const T *src = row + static_cast<int64_t>(h) * d;
                const float *bias = is_q ? q_b : k_b, *wn = is_q ? q_w : k_w;
                own = load8(src + e0);
                other = load8(src + p0);
                if (bias) {
                    bias += static_cast<int64_t>(is_q ? h : h - nq) * d;
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        bo[k] = *reinterpret_cast<const float4_t *>(bias + e0 + 4 * k);
                        bp[k] = *reinterpret_cast<const float4_t *>(bias + p0 + 4 * k);
                    }
                }
                if (wn) {
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        wo[k] = *reinterpret_cast<const float4_t *>(wn + e0 + 4 * k);
                        wp[k] = *reinterpret_cast<const float4_t *>(wn + p0 + 4 * k);
                    }
                }
                if (is_q && q_mult) mult = q_mult[h];
            };
            fetch(wave * hpw);
            rk_angles(cs, sn, freq, pos, pairs, rot_mult);
            __syncthreads();
            for (int hb = wave * hpw; hb < heads; hb += (kRkThreads / 64) * hpw) {
                if (hb != wave * hpw) fetch(hb);
                const int h = hb + slot;
                const bool live = h < heads && e0 < d, is_q = h < nq;
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = to_f(own[j]) + bo[j >> 2][j & 3];
                float ss = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) ss += v[j] * v[j];
                ss = lph == 1 ? ss : lph == 2 ? group_allreduce_sum<2>(ss) : lph == 4 ? group_allreduce_sum<4>(ss)
                   : lph == 8 ? group_allreduce_sum<8>(ss) : group_allreduce_sum<16>(ss);
                if (!live) continue;
                const float r = (is_q ? q_w : k_w) ? 1.0f / sqrtf(ss / static_cast<float>(d) + eps) : 1.0f;
                if (!is_q && keys_as_values) {
                    T *dst = vpage + (static_cast<int64_t>(h - nq) * v_dim + e0) * kRkBlock + off;
#pragma unroll
                    for (int j = 0; j < 8; ++j) dst[j * kRkBlock] = to_t<T>(v[j]);
                }
                float n[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) n[j] = v[j] * r * wo[j >> 2][j & 3];
                if (turns && half) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float w = (to_f(other[j]) + bp[j >> 2][j & 3]) * r * wp[j >> 2][j & 3];
                        n[j] = first ? n[j] * cs[a0 + j] - w * sn[a0 + j] : n[j] * cs[a0 + j] + w * sn[a0 + j];
                    }
                } else if (turns) {
#pragma unroll
                    for (int j = 0; j < 8; j += 2) {
                        const float c = cs[a0 + (j >> 1)], sv = sn[a0 + (j >> 1)], u = n[j], w = n[j + 1];
                        n[j] = u * c - w * sv;
                        n[j + 1] = w * c + u * sv;
                    }
                }
                vec8_t<T> o;
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = to_t<T>(n[j] * mult);
                store8(is_q ? qrow + static_cast<int64_t>(h) * k_dim + e0
                            : kpage + (static_cast<int64_t>(h - nq) * kRkBlock + off) * k_dim + e0, o);
            }
        }
    }
    if (!wide) {
        rk_angles(cs, sn, freq, pos, pairs, rot_mult);
        __syncthreads();
    }
    for (int h = wave; h < heads && !wide; h += kRkThreads / 64) {
        const bool is_q = h < nq;
        const T *src = row + static_cast<int64_t>(h) * d;
        const float *bias = is_q ? q_b : k_b, *wn = is_q ? q_w : k_w;
        if (bias) bias += static_cast<int64_t>(is_q ? h : h - nq) * d;
        auto biased = [&](int e) { return to_f(src[e]) + (bias ? bias[e] : 0.f); };
        float ss = 0.f;
        for (int e = lane; e < d; e += 64) {
            const float v = biased(e);
            ss += v * v;
            if (!is_q && keys_as_values) vpage[(static_cast<int64_t>(h - nq) * v_dim + e) * kRkBlock + off] = to_t<T>(v);
        }
        ss = wave_allreduce_sum(ss);
        const float r = wn ? 1.0f / sqrtf(ss / static_cast<float>(d) + eps) : 1.0f;
        auto normed = [&](int e) { return wn ? biased(e) * r * wn[e] : biased(e); };
        const float mult = is_q && q_mult ? q_mult[h] : 1.0f;
        T *dst = is_q ? qrow + static_cast<int64_t>(h) * k_dim : kpage + (static_cast<int64_t>(h - nq) * kRkBlock + off) * k_dim;
        for (int e = lane; e < d; e += 64) {
            float n = normed(e);
            if (e < rot_dims) {
                const bool first = half ? e < pairs : (e & 1) == 0;
                const int p = half ? (first ? e + pairs : e - pairs) : e ^ 1, a = half ? (first ? e : p) : e >> 1;
                const float w = normed(p);
                n = first ? n * cs[a] - w * sn[a] : n * cs[a] + w * sn[a];
            }
            dst[e] = to_t<T>(n * mult);
        }
    }
    // zero the columns beyond the head
    const int kpad = k_dim - d;
    for (int i = threadIdx.x; i < heads * kpad; i += kRkThreads) {
        const int h = i / kpad, e = d + i - h * kpad;
        if (h < nq) qrow[static_cast<int64_t>(h) * k_dim + e] = to_t<T>(0.f);
        else kpage[(static_cast<int64_t>(h - nq) * kRkBlock + off) * k_dim + e] = to_t<T>(0.f);
    }
    if (!store) return;
    const int nval = keys_as_values ? nk : nv, dval = keys_as_values ? d : dv, vpad = v_dim - dval;
    if (!keys_as_values) {
        const T *vrow = row + static_cast<int64_t>(nq + nk) * d;
        for (int i = threadIdx.x; i < nv * dv; i += kRkThreads) {
            const int g = i / dv, c = i - g * dv;
            vpage[(static_cast<int64_t>(g) * v_dim + c) * kRkBlock + off] = vrow[i];
        }
    }
    for (int i = threadIdx.x; i < nval * vpad; i += kRkThreads) {
        const int g = i / vpad, c = dval + i - g * vpad;
        vpage[(static_cast<int64_t>(g) * v_dim + c) * kRkBlock + off] = to_t<T>(0.f);
    }
}

template <typename T>
__global__ __launch_bounds__(kRkThreads) void qkv_conv_rope_store_kv_kernel(
    const T *rows, int64_t tok_stride, T *q_out, int64_t q_out_stride, const float *bias, const float *conv_w, int taps,
    const float *q_w, const float *k_w, const double *freq, int rot_dims, int half, double rot_mult, float v_mult, T *k_cache,
    T *v_cache, const int32_t *block_table, int max_blocks_per_seq, int64_t block_stride, float *state, int64_t slot_stride,
    int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *tok_state, const int32_t *tok_seq,
    int64_t num_tokens, int nq, int nk, int d, int dv, int k_dim, int v_dim, float eps) {
    extern __shared__ float act[];      // [(nq + nk) d + nk dv] biased, convolved channels; then [nq + nk] the heads' 1 / rms
    __shared__ float cs[kRkMaxPairs], sn[kRkMaxPairs];
    const int64_t t = page_token();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int pos = tok_pos[t];
    const int pairs = rot_dims >> 1, heads = nq + nk, C = heads * d + nk * dv;
    float *rinv = act + C;
    const T *row = rows + t * tok_stride;
    if (conv_w) {
        const ConvTail tail(state, slot_stride, tail_off, tok_pos, tok_start, tok_state, tok_seq, num_tokens, C, taps, t);
        bool wide = false;
        if constexpr (sizeof(T) == 2) {
            wide = ConvTail::wide_ok(rows, tok_stride, conv_w, state, slot_stride, tail_off, C) &&
                   (reinterpret_cast<uintptr_t>(bias) & 15) == 0;
            if (wide) {
                for (int c = threadIdx.x * 8; c < C; c += kRkThreads * 8) {
                    const vec8_t<T> x = load8(row + c);
                    float cur[8], b[8], a[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        cur[j] = to_f(x[j]);
                        b[j] = bias ? bias[c + j] : 0.f;
                        a[j] = 0.f;
                    }
                    for (int k = taps - 1; k >= 1; --k) {       // inputs before the sequence are zero, biases included
                        if (pos - k < 0) continue;
                        float v[8];
                        tail.at8(rows, tok_stride, c, pos - k, v);
                        const float *wk = conv_w + static_cast<int64_t>(taps - 1 - k) * C + c;
#pragma unroll
                        for (int j = 0; j < 8; ++j) a[j] += wk[j] * (v[j] + b[j]);
                    }
                    const float *wl = conv_w + static_cast<int64_t>(taps - 1) * C + c;
#pragma unroll
                    for (int j = 0; j < 8; ++j) act[c + j] = a[j] + wl[j] * (cur[j] + b[j]);
                    tail.save8(rows, tok_stride, c, cur);
                }
            }
        }
        for (int c = threadIdx.x; c < C && !wide; c += kRkThreads) {
            const float cur = to_f(row[c]), b = bias ? bias[c] : 0.f;
            float a = 0.f;
            for (int k = taps - 1; k >= 1; --k)
                if (pos - k >= 0)
                    a += conv_w[static_cast<int64_t>(taps - 1 - k) * C + c] * (tail.at(rows, tok_stride, c, pos - k) + b);
            act[c] = a + conv_w[static_cast<int64_t>(taps - 1) * C + c] * (cur + b);
            tail.save(rows, tok_stride, c, cur);
        }
    } else {
        bool wide = false;
        if constexpr (sizeof(T) == 2) {
            wide = (C & 7) == 0 && (tok_stride & 7) == 0 && (reinterpret_cast<uintptr_t>(rows) & 15) == 0;
            if (wide) {
                for (int c = threadIdx.x * 8; c < C; c += kRkThreads * 8) {
                    const vec8_t<T> x = load8(row + c);
#pragma unroll
                    for (int j = 0; j < 8; ++j) act[c + j] = to_f(x[j]) + (bias ? bias[c + j] : 0.f);
                }
            }
        }
        for (int c = threadIdx.x; c < C && !wide; c += kRkThreads) act[c] = to_f(row[c]) + (bias ? bias[c] : 0.f);
    }
    rk_angles(cs, sn, freq, pos, pairs, rot_mult);
    __syncthreads();
    if (q_w) {
        for (int h = wave; h < heads; h += kRkThreads / 64) {
            float ss = 0.f;
            for (int e = lane; e < d; e += 64) ss += act[h * d + e] * act[h * d + e];
            ss = wave_allreduce_sum(ss);
            if (lane == 0) rinv[h] = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
        }
        __syncthreads();
    }
    auto element = [&](int h, int e) {      // element e of head h: normed and rotated
        const float *a = act + h * d, *w = h < nq ? q_w : k_w;
        const float r = q_w ? rinv[h] : 1.f;
        float n = q_w ? a[e] * r * w[e] : a[e];
        if (e < rot_dims) {
            const bool first = half ? e < pairs : (e & 1) == 0;
            const int p = half ? (first ? e + pairs : e - pairs) : e ^ 1, i = half ? (first ? e : p) : e >> 1;
            const float o = q_w ? a[p] * r * w[p] : a[p];
            n = first ? n * cs[i] - o * sn[i] : n * cs[i] + o * sn[i];
        }
        return n;
    };
    const bool store = k_cache != nullptr;
    int64_t blk = 0;
    if (store) blk = block_table[static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq + pos / kRkBlock];
    const int off = pos % kRkBlock;
    T *qrow = q_out + t * q_out_stride;
    T *kpage = k_cache + blk * block_stride, *vpage = v_cache + blk * block_stride;
    const int outs = store ? heads : nq;
    if (sizeof(T) == 2 && (k_dim & 7) == 0 && (q_out_stride & 7) == 0 && (block_stride & 7) == 0 &&
        ((reinterpret_cast<uintptr_t>(q_out) | reinterpret_cast<uintptr_t>(k_cache)) & 15) == 0) {
        const int per = k_dim >> 3;
        for (int i = threadIdx.x; i < outs * per; i += kRkThreads) {
            const int h = i / per, e0 = (i - h * per) * 8;
            vec8_t<T> o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = to_t<T>(e0 + j < d ? element(h, e0 + j) : 0.f);
            store8(h < nq ? qrow + static_cast<int64_t>(h) * k_dim + e0
                          : kpage + (static_cast<int64_t>(h - nq) * kRkBlock + off) * k_dim + e0, o);
        }
    } else {
        for (int i = threadIdx.x; i < outs * k_dim; i += kRkThreads) {
            const int h = i / k_dim, e = i - h * k_dim;
            T *dst = h < nq ? qrow + static_cast<int64_t>(h) * k_dim : kpage + (static_cast<int64_t>(h - nq) * kRkBlock + off) * k_dim;
            dst[e] = to_t<T>(e < d ? element(h, e) : 0.f);
        }
    }
    if (!store) return;
    for (int i = threadIdx.x; i < nk * v_dim; i += kRkThreads) {        // (the transposed page: 16 tokens of a column together)
        const int g = i / v_dim, c = i - g * v_dim;
        vpage[static_cast<int64_t>(i) * kRkBlock + off] = to_t<T>(c < dv ? act[heads * d + g * dv + c] * v_mult : 0.f);
    }
}

// The same for heads of 8 LPH columns (16, 32, 64 or 128), up to four taps and rows of whole aligned pieces of eight: a lane's eight channels
// stay in registers, a head's sum and its rotation are exchanges between neighbouring lanes. What bounds it is the chain of a token's
// workgroup, which above is a round trip for every earlier input and the norm's and the rotation's passes over LDS: here the row, up to
// three earlier ones, taps, bias and norm weights are asked for together. In steps of many tokens a workgroup takes four in a row, for which
// the taps (8 to 16 KiB a row of 2 KiB) are read once and whose earlier inputs move on by one in registers; its longer chain costs more where the
// workgroups of one token, few or of one wave each, are all on the chip at once (rk_four_pay).
// us, above -> one token / four, heads of 128, bf16: 8 over 2 with 4 taps and norm 32 tokens 10.5 -> 5.8, 500 11.7 -> 6.9, 1536 19.6 -> 12.5 / 11.7, 2030 25.6 -> 16.3 /
// 12.5, 5000 53.7 -> - / 24.8; without norm 3 7.6 -> 5.5, 500 9.1 -> 6.7, 1000 11.4 -> 7.8, 1500 14.3 -> 11.8, 2030 19.4 -> 15.7 / 11.7, 5000 36.8 -> - / 23.8; without
// norm and taps 500 7.5 -> 5.4, 2030 15.8 -> 11.7 / 9.4; 16 over 4 without norm 1000 18.1 -> 15.0, 2030 33.7 -> - / 18.9; fp32 without norm 3 11.4 -> 5.7, 1000
// 14.6 -> 9.1, 2030 25.0 -> 17.2 / 14.5. One / four by channels of q, k and v, 4 taps without norm: 96 3072 8.3 / 10.5, 4096 10.9 / 10.6, 8192 16.9 / 11.7; 384 1536 6.8 /
// 9.6, 3072 8.2 / 10.0, 4096 11.3 / 10.3; 768 1536 8.0 / 10.0, 2048 11.2 / 10.3, 3072 13.6 / 10.7; 1024 1536 8.2 / 10.9, 2048 12.0 / 11.2; 1536 1024 7.6 / 10.4, 1536 12.1 / 11.1.
inline bool rk_four_pay(int64_t tokens, int64_t channels) { return tokens >= 4096 || (tokens >= 1536 && tokens * channels >= 1 << 21); }
template <typename T, int LPH, int TOK>
__global__ __launch_bounds__(kRkThreads, 3) void qkv_conv_rope_rows_kernel(
    const T *rows, int64_t tok_stride, T *q_out, int64_t q_out_stride, const float *bias, const float *conv_w, int taps,
    const float *q_w, const float *k_w, const double *freq, int rot_dims, int half, double rot_mult, float v_mult, T *k_cache,
    T *v_cache, const int32_t *block_table, int max_blocks_per_seq, int64_t block_stride, float *state, int64_t slot_stride,
    int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *tok_state, const int32_t *tok_seq,
    int64_t num_tokens, int nq, int nk, int dv, int k_dim, int v_dim, float eps) {
    constexpr int d = 8 * LPH, MOST = 3;
    __shared__ float cs[TOK][d / 2], sn[TOK][d / 2];
    __shared__ int meta[TOK][5];        // position, first position of the portion, state slot and parity, ends its portion, block
    // workgroup -> its tokens; those of a page on one XCD (page_token)
    int64_t t0;
    if constexpr (TOK == 1) {
        t0 = page_token();
    } else {
        constexpr int RUN = 128 / TOK;
        const unsigned b = blockIdx.x, first = b & ~(RUN - 1u);
        t0 = (gridDim.x - first < RUN ? b : first + (b & 7) * (16 / TOK) + ((b >> 3) & (16 / TOK - 1))) * TOK;
    }
    const int n = static_cast<int>(min<int64_t>(TOK, num_tokens - t0));
    const int lane = threadIdx.x & 63, pairs = rot_dims >> 1, heads = nq + nk, C = heads * d + nk * dv;
    const int step = blockDim.x * 8, R = conv_w ? taps - 1 : 0;
    const bool store = k_cache != nullptr;
    float past[MOST][8], wk[MOST + 1][8], b[8], wn[8];      // past[k - 1], wk[k]: the input k tokens back and its weights
    T raw[TOK][8];
    auto earlier = [&](int64_t t, int code, int pos, int start, int c) {        // the inputs before token t, from rows of its portion or the tail
        const float *old_tail = state + static_cast<int64_t>(code >> 1) * slot_stride + tail_off + static_cast<int64_t>(code & 1) * R * C;
#pragma unroll
        for (int k = 1; k <= MOST; ++k)
            if (k <= R && pos >= k) {       // (uniform)
                if (pos - k >= start) ConvTail::row8(rows + (t - k) * tok_stride + c, past[k - 1]);
                else ConvTail::row8(old_tail + static_cast<int64_t>(R - (start - (pos - k))) * C + c, past[k - 1]);
            }
    };
    auto ask = [&](int c) {
#pragma unroll
        for (int i = 0; i < TOK; ++i) {
            const T *p = rows + (t0 + min(i, n - 1)) * tok_stride + c;
            if constexpr (sizeof(T) == 2) {
                const vec8_t<T> x = load8(p);
#pragma unroll
                for (int j = 0; j < 8; ++j) raw[i][j] = x[j];
            } else {
                ConvTail::row8(p, raw[i]);
            }
        }
        if (R > 0) earlier(t0, tok_state[t0], tok_pos[t0], tok_start[t0], c);
        if (conv_w) {
#pragma unroll
            for (int k = 0; k <= MOST; ++k)
                if (k <= R) ConvTail::row8(conv_w + static_cast<int64_t>(R - k) * C + c, wk[k]);
        }
        if (bias) ConvTail::row8(bias + c, b);
        if (q_w && c < heads * d) ConvTail::row8((c < nq * d ? q_w : k_w) + c % d, wn);
    };
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] = wn[j] = 0.f;
    if (threadIdx.x * 8 < C) ask(threadIdx.x * 8);
    if (static_cast<int>(threadIdx.x) < n) {
        const int64_t t = t0 + threadIdx.x;
        const int pos = tok_pos[t], seq = tok_seq[t];
        int *m = meta[threadIdx.x];
        m[0] = pos;
        m[1] = R > 0 ? tok_start[t] : 0;
        m[2] = R > 0 ? tok_state[t] : 0;
        m[3] = t + 1 == num_tokens || tok_seq[t + 1] != seq;
        m[4] = store ? block_table[static_cast<int64_t>(seq) * max_blocks_per_seq + pos / kRkBlock] : 0;
    }
    for (int i = threadIdx.x; i < n * pairs; i += blockDim.x) {
        const int u = i / pairs, p = i - u * pairs;
        const double a = static_cast<double>(tok_pos[t0 + u]) * freq[p];
        cs[u][p] = static_cast<float>(cos(a) * rot_mult);
        sn[u][p] = static_cast<float>(sin(a) * rot_mult);
    }
    __syncthreads();
    for (int c = threadIdx.x * 8; c < C; c += step) {
        if (c >= step) ask(c);
#pragma unroll
        for (int i = 0; i < TOK; ++i) {
            if (i >= n) break;      // (uniform)
            const int64_t t = t0 + i;
            auto of = [&](int what) { return __builtin_amdgcn_readfirstlane(meta[i][what]); };
            const int pos = of(0), off = pos % kRkBlock;
            const int64_t blk = of(4);
            T *qrow = q_out + t * q_out_stride, *kpage = k_cache + blk * block_stride, *vpage = v_cache + blk * block_stride;
            float a[8], cur[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) cur[j] = to_f(raw[i][j]);
            if (conv_w) {
                // (a token whose portion begins with it finds its earlier inputs in the tail; else they moved on by one)
                if (i > 0 && R > 0 && of(1) == pos) earlier(t, of(2), pos, pos, c);
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] = 0.f;
#pragma unroll
                for (int k = MOST; k >= 1; --k) {
                    if (k <= R && pos >= k) {       // inputs before the sequence are zero, biases included
#pragma unroll
                        for (int j = 0; j < 8; ++j) a[j] += wk[k][j] * (past[k - 1][j] + b[j]);
                    }
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] = a[j] + wk[0][j] * (cur[j] + b[j]);
                if (R > 0 && of(3)) {
                    const int code = of(2);     // (the layout of conv_tail.h; the input k tokens back becomes entry R - 1 - k)
                    float *new_tail = state + static_cast<int64_t>(code >> 1) * slot_stride + tail_off + static_cast<int64_t>(1 - (code & 1)) * R * C;
#pragma unroll
                    for (int k = 0; k < MOST; ++k)
                        if (k < R && pos >= k)
                            ConvTail::put8<float>(new_tail + static_cast<int64_t>(R - 1 - k) * C + c, k == 0 ? cur : past[k > 0 ? k - 1 : 0]);
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) {
#pragma unroll
                    for (int k = MOST - 1; k > 0; --k) past[k][j] = past[k - 1][j];
                    past[0][j] = cur[j];
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] = cur[j] + b[j];
            }
            if (c >= heads * d) {       // values: 16 tokens of a column together
                if (store) {
                    const int x = c - heads * d, g = x / dv;
                    T *dst = vpage + (static_cast<int64_t>(g) * v_dim + (x - g * dv)) * kRkBlock + off;
#pragma unroll
                    for (int j = 0; j < 8; ++j) dst[j * kRkBlock] = to_t<T>(a[j] * v_mult);
                }
                continue;
            }
            const int h = c / d, e0 = c - h * d;
            if (q_w) {
                float ss = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) ss += a[j] * a[j];
                ss = group_allreduce_sum<LPH>(ss);
                const float r = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] = a[j] * r * wn[j];
            }
            const bool turns = e0 < rot_dims, first = e0 < pairs;
            if (half) {     // (the partner's columns are another lane's of the head)
                const int from = !turns ? lane : first ? lane + pairs / 8 : lane - pairs / 8;
                float o[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = __shfl(a[j], from, 64);
                if (turns) {
                    const int a0 = first ? e0 : e0 - pairs;
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float co = cs[i][a0 + j], si = sn[i][a0 + j];
                        a[j] = first ? a[j] * co - o[j] * si : a[j] * co + o[j] * si;
                    }
                }
            } else if (turns) {
#pragma unroll
                for (int j = 0; j < 8; j += 2) {
                    const float co = cs[i][(e0 + j) >> 1], si = sn[i][(e0 + j) >> 1], u = a[j], v = a[j + 1];
                    a[j] = u * co - v * si;
                    a[j + 1] = v * co + u * si;
                }
            }
            if (h < nq) ConvTail::put8(qrow + static_cast<int64_t>(h) * k_dim + e0, a);
            else if (store) ConvTail::put8(kpage + (static_cast<int64_t>(h - nq) * kRkBlock + off) * k_dim + e0, a);
        }
    }
    const int kpad = k_dim - d, vpad = v_dim - dv;      // the columns beyond the heads are zero
    if (kpad == 0 && vpad == 0) return;
    for (int i = 0; i < n; ++i) {
        const int64_t t = t0 + i, blk = meta[i][4];
        const int off = meta[i][0] % kRkBlock;
        for (int x = threadIdx.x; x < (store ? heads : nq) * kpad; x += blockDim.x) {
            const int h = x / kpad, e = d + x - h * kpad;
            if (h < nq) q_out[t * q_out_stride + static_cast<int64_t>(h) * k_dim + e] = to_t<T>(0.f);
            else k_cache[blk * block_stride + (static_cast<int64_t>(h - nq) * kRkBlock + off) * k_dim + e] = to_t<T>(0.f);
        }
        for (int x = threadIdx.x; x < (store ? nk * vpad : 0); x += blockDim.x) {
            const int g = x / vpad, c = dv + x - g * vpad;
            v_cache[blk * block_stride + (static_cast<int64_t>(g) * v_dim + c) * kRkBlock + off] = to_t<T>(0.f);
        }
    }
}

template <typename T>
__device__ __forceinline__ void latent_rope_store_token(int64_t t,
    T *proj, T *qa, int64_t in_place, const double *freq, const float *c_w, T *k_cache, T *v_cache, const int32_t *block_table,
    const int32_t *tok_seq, const int32_t *tok_pos, int H, int d, int dr, int r, int64_t proj_stride, int64_t dkv_col,
    int64_t qa_stride, int max_blocks_per_seq, int64_t block_stride, float eps, int half, double rot_mult, int k_dim,
    int v_dim) {
    __shared__ float cs[kRkMaxPairs], sn[kRkMaxPairs];
    __shared__ float red[kRkThreads / 64];
    const int pos = tok_pos[t];
    const int pairs = dr >> 1;
    rk_angles(cs, sn, freq, pos, pairs, rot_mult);
    __syncthreads();
    T *row = proj + t * proj_stride;
    const bool here = t < in_place;     // (the query heads stay where they are)
    T *qrow = here ? row + d : qa + (t - in_place) * qa_stride + r;
    const int qhead = here ? d + dr : k_dim;
    // pair j of a rotated part: elements (2j, 2j + 1), or (j, j + pairs)
    const int step = half ? 1 : 2, gap = half ? pairs : 1;
    for (int i = threadIdx.x; i < H * pairs; i += kRkThreads) {
        const int h = i / pairs, j = i - h * pairs;
        const T *p = row + static_cast<int64_t>(h) * (d + dr) + d + step * j;
        T *o = qrow + static_cast<int64_t>(h) * qhead + step * j;
        const float u = to_f(p[0]), v = to_f(p[gap]);
        o[0] = to_t<T>(u * cs[j] - v * sn[j]);
        o[gap] = to_t<T>(v * cs[j] + u * sn[j]);
    }
    const int kpad = k_dim - r - dr, vpad = v_dim - r;
    for (int i = threadIdx.x; i < (here ? 0 : H * kpad); i += kRkThreads) {
        const int h = i / kpad;
        qrow[static_cast<int64_t>(h) * k_dim + dr + i - h * kpad] = to_t<T>(0.f);
    }
    if (dkv_col < 0 || k_cache == nullptr) return;
    const T *z = row + dkv_col;
    float ss = 0.f;
    for (int i = threadIdx.x; i < r; i += kRkThreads) {
        const float x = to_f(z[i]);
        ss += x * x;
    }
    ss = wave_allreduce_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < kRkThreads / 64; ++w) ss += red[w];
    const float rinv = 1.0f / sqrtf(ss / static_cast<float>(r) + eps);
    const int64_t blk = block_table[static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq + pos / kRkBlock];
    const int off = pos % kRkBlock;
    T *kdst = k_cache + blk * block_stride + static_cast<int64_t>(off) * k_dim;
    T *vdst = v_cache + blk * block_stride + off;
    for (int i = threadIdx.x; i < r; i += kRkThreads) {
        const T c = to_t<T>(to_f(z[i]) * rinv * c_w[i]);
        kdst[i] = c;
        vdst[static_cast<int64_t>(i) * kRkBlock] = c;
    }
    for (int j = threadIdx.x; j < pairs; j += kRkThreads) {
        const float u = to_f(z[r + step * j]), v = to_f(z[r + step * j + gap]);
        kdst[r + step * j] = to_t<T>(u * cs[j] - v * sn[j]);
        kdst[r + step * j + gap] = to_t<T>(v * cs[j] + u * sn[j]);
    }
    for (int i = threadIdx.x; i < kpad; i += kRkThreads) kdst[r + dr + i] = to_t<T>(0.f);
    for (int i = threadIdx.x; i < vpad; i += kRkThreads) vdst[static_cast<int64_t>(r + i) * kRkBlock] = to_t<T>(0.f);
}

template <typename T>
__global__ __launch_bounds__(kRkThreads) void latent_rope_store_kv_kernel(
    T *proj, T *qa, int64_t in_place, const double *freq, const float *c_w, T *k_cache, T *v_cache, const int32_t *block_table,
    const int32_t *tok_seq, const int32_t *tok_pos, int H, int d, int dr, int r, int64_t proj_stride, int64_t dkv_col,
    int64_t qa_stride, int max_blocks_per_seq, int64_t block_stride, float eps, int half, double rot_mult, int k_dim,
    int v_dim) {
    latent_rope_store_token<T>(page_token(), proj, qa, in_place, freq, c_w, k_cache, v_cache, block_table, tok_seq, tok_pos, H, d, dr, r, proj_stride,
                               dkv_col, qa_stride, max_blocks_per_seq, block_stride, eps, half, rot_mult, k_dim, v_dim);
}

// The same for a few tokens (the first workgroups, one a token) beside the queries folded through the key up-projection (the others): qa[t][h][:r]
// = W_uk,h^T q_th, W_uk transposed [H, r, d]. The two write different columns and read nothing of each other: one launch instead of two. A workgroup
// folds 64 columns of a head for all tokens, a wave 16 (16x16x32, columns as A, tokens as B): 2 MB of matrices over 128 workgroups at 16 heads of 128.
template <typename T>
__device__ __forceinline__ float4_t rk_mfma(vec8_t<T> a, vec8_t<T> b, float4_t c);
template <>
__device__ __forceinline__ float4_t rk_mfma<f16>(vec8_t<f16> a, vec8_t<f16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
template <>
__device__ __forceinline__ float4_t rk_mfma<bf16>(vec8_t<bf16> a, vec8_t<bf16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
constexpr int kFoldMaxDim = 256;

template <typename T>
__global__ __launch_bounds__(kRkThreads) void latent_fold_kernel(
    T *proj, T *qa, int n, const T *uk_t, const double *freq, const float *c_w, T *k_cache, T *v_cache, const int32_t *block_table,
    const int32_t *tok_seq, const int32_t *tok_pos, int H, int d, int dr, int r, int64_t proj_stride, int64_t dkv_col,
    int64_t qa_stride, int max_blocks_per_seq, int64_t block_stride, float eps, int half, double rot_mult, int k_dim,
    int v_dim) {
    if (blockIdx.x < static_cast<unsigned>(n)) {
        latent_rope_store_token<T>(blockIdx.x, proj, qa, 0, freq, c_w, k_cache, v_cache, block_table, tok_seq, tok_pos, H, d, dr, r, proj_stride,
                                   dkv_col, qa_stride, max_blocks_per_seq, block_stride, eps, half, rot_mult, k_dim, v_dim);
        return;
    }
    const int tiles = r / 64, at = static_cast<int>(blockIdx.x) - n, h = at / tiles, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lr = lane & 15, lk = lane >> 4, r0 = (at - h * tiles) * 64 + wave * 16, steps = d / 32;
    vec8_t<T> wf[kFoldMaxDim / 32];
    const T *wp = uk_t + (static_cast<int64_t>(h) * r + r0 + lr) * d + lk * 8;
#pragma unroll
    for (int e = 0; e < kFoldMaxDim / 32; ++e)
        if (e < steps) wf[e] = load8(wp + e * 32);
    for (int t0 = 0; t0 < n; t0 += 16) {
        const T *qp = proj + min(t0 + lr, n - 1) * proj_stride + static_cast<int64_t>(h) * (d + dr) + lk * 8;
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < kFoldMaxDim / 32; ++e)
            if (e < steps) acc = rk_mfma<T>(wf[e], load8(qp + e * 32), acc);
        mfma_results_ready<8>(acc);
        // acc[k]: column r0 + 4 lk + k of token t0 + lr
        vec4_t<T> v;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = to_t<T>(acc[k]);
        if (t0 + lr < n) *reinterpret_cast<vec4_t<T> *>(qa + (t0 + lr) * qa_stride + static_cast<int64_t>(h) * k_dim + r0 + 4 * lk) = v;
    }
}

constexpr int kDiffMaxDim = 256, kDiffMaxShares = 32;

// grid: (tokens, workgroups that share a token's heads), a wave takes every (4 grid.y)-th head.
template <typename T>
__global__ __launch_bounds__(256) void diff_head_combine_kernel(T *out, const float *a, const T *gate, int64_t gate_stride, float lambda, float mult,
                                                                float eps, int H, int dv) {
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63;
    for (int h = blockIdx.y * 4 + (threadIdx.x >> 6); h < H; h += 4 * gridDim.y) {
        const float *a1 = a + ((t * 2) * H + h) * dv, *a2 = a + ((t * 2 + 1) * H + h) * dv;
        float ss = 0.f;
        for (int e = lane; e < dv; e += 64) {
            const float o = a1[e] - lambda * a2[e];
            ss += o * o;
        }
        ss = wave_allreduce_sum(ss);
        const float g = gate ? rk_sigmoid(to_f(gate[t * gate_stride + h])) : 1.0f;
        const float f = mult * g / sqrtf(ss / static_cast<float>(dv) + eps);
        for (int e = lane; e < dv; e += 64) out[(t * H + h) * dv + e] = to_t<T>((a1[e] - lambda * a2[e]) * f);
    }
}
// Few tokens: a workgroup for every four heads, so that all are on the chip at once; many: one a token, whose rows lie together. us, one workgroup a token / one
// for four heads: 32 tokens x 16 heads of 128 5.6 / 3.5, 500 6.4 / 4.8, 1000 7.6 / 6.9, 2000 12.5 / 13.4, 4000 21.9 / 22.5, 8000 39.8 / 43.0; 8 of 128 8000
// 21.9 / 22.7.
constexpr int64_t kDiffManyTokens = 1536;
inline unsigned diff_groups(int H) { return static_cast<unsigned>(H < 4 * 65535 ? (H + 3) / 4 : 65535); }

// The same where a1 and a2 still are key shares (attn_combine.h; NATURAL: their maxima in natural units), which a wave, of one (token, head), weighs and
// adds up itself: lane s weighs share s of a1, lane 32 + s of a2, and each half of the wave reads its map's columns, eight shares in flight. Bound by
// latency: 32 tokens x 16 heads of 128, 8 shares: a launch that adds them up and the one above after it (four heads a wave) 4.8 + 6.6 us -> 4.7; with a
// lane on both maps' columns, a 4-byte load at a time, 8.8.
template <typename T, bool NATURAL>
__global__ __launch_bounds__(256) void diff_head_shares_kernel(T *out, const float *a, const float *part_ml, int shares, const T *gate, int64_t gate_stride,
                                                               float lambda, float mult, float eps, int64_t rows, int H, int dv) {
    const int lane = threadIdx.x & 63;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);     // t * H + h
    if (row >= rows) return;
    const int64_t t = row / H, r1 = row + t * H, r2 = r1 + H;      // (rows of the two maps: t * 2H + h, t * 2H + H + h)
    const float g = gate ? rk_sigmoid(to_f(gate[t * gate_stride + (row - t * H)])) : 1.0f;
    const float *a1 = a + r1 * dv, *a2 = a + r2 * dv;
    float ss = 0.f;
    constexpr int NE = kDiffMaxDim / 128;       // pieces of four columns of a lane, of its half's map
    const int sub = lane & 31;
    const bool live = sub < shares;
    const float *ml = part_ml + ((live ? sub : 0) * 2 * rows + (lane < 32 ? r1 : r2)) * 2;
    const float m = live ? ml[0] : kNegBig, l = live ? ml[1] : 0.f;
    const float *mine = lane < 32 ? a1 : a2;
    const int64_t plane = 2 * rows * dv;
    float4_t x[NE];
    float w = 0.f;
#pragma unroll
    for (int j = 0; j < NE; ++j) x[j] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < shares; s0 += 8) {
        float4_t p[8][NE];
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int j = 0; j < NE; ++j)        // (the last share and piece stand in for the missing ones)
                if (j == 0 || dv > 128 * j)
                    p[u][j] = *reinterpret_cast<const float4_t *>(mine + min(s0 + u, shares - 1) * plane + min(4 * sub + 128 * j, dv - 4));
        if (s0 == 0) {
            float mx = m;
#pragma unroll
            for (int d = 1; d < 32; d *= 2) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
            w = live ? (NATURAL ? expf(m - mx) : exp2f(m - mx)) : 0.f;
            float den = w * l;
#pragma unroll
            for (int d = 1; d < 32; d *= 2) den += __shfl_xor(den, d, 64);
            w *= 1.0f / den;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float ws = __shfl(w, (lane & 32) + min(s0 + u, 31), 64);       // (lanes without a share have weight zero)
#pragma unroll
            for (int j = 0; j < NE; ++j)
                if (j == 0 || dv > 128 * j) x[j] += ws * p[u][j];
        }
    }
#pragma unroll
    for (int j = 0; j < NE; ++j) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float other = __shfl_xor(x[j][c], 32, 64);
            x[j][c] = lane < 32 ? x[j][c] - lambda * other : 0.f;
            if (4 * sub + 128 * j < dv) ss += x[j][c] * x[j][c];
        }
    }
    ss = wave_allreduce_sum(ss);
    const float f = mult * g / sqrtf(ss / static_cast<float>(dv) + eps);
#pragma unroll
    for (int j = 0; j < NE; ++j) {
        if (lane < 32 && 4 * sub + 128 * j < dv) {
            vec4_t<T> o;
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = to_t<T>(x[j][c] * f);
            *reinterpret_cast<vec4_t<T> *>(out + row * dv + 4 * sub + 128 * j) = o;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void head_gate_kernel(T *y, const T *gate, int64_t gate_stride, int H, int dv) {
    const int64_t t = blockIdx.x;
    if constexpr (sizeof(T) == 2) {
        if ((dv & 7) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {      // 8 columns of one head per lane
            for (int i = threadIdx.x * 8; i < H * dv; i += 256 * 8) {
                const float g = rk_sigmoid(to_f(gate[t * gate_stride + i / dv]));
                vec8_t<T> v = load8(y + t * H * dv + i);
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = to_t<T>(to_f(v[j]) * g);
                store8(y + t * H * dv + i, v);
            }
            return;
        }
    }
    for (int i = threadIdx.x; i < H * dv; i += 256) {
        const float g = rk_sigmoid(to_f(gate[t * gate_stride + i / dv]));
        y[t * H * dv + i] = to_t<T>(to_f(y[t * H * dv + i]) * g);
    }
}

} // namespace swl

extern "C" int swl_rope_store_kv(void *qkv, const double *freq, void *k_cache, void *v_cache, const int32_t *block_table,
                                 const int32_t *tok_seq, const int32_t *tok_pos, int64_t num_tokens, int32_t num_q_heads,
                                 int32_t num_k_heads, int32_t num_v_heads, int32_t dim, int32_t vdim, int32_t rot_dims,
                                 int64_t tok_stride, int32_t max_blocks_per_seq, int64_t block_stride, int32_t dtype,
                                 swl_stream_t stream) {
    if (num_tokens < 0 || num_q_heads <= 0 || num_k_heads < 0 || num_v_heads < 0 || dim <= 0 || vdim <= 0) return SWL_ERR_BAD_ARG;
    if (rot_dims < 0 || (rot_dims & 1) || rot_dims > dim || (dim & 1)) return SWL_ERR_BAD_ARG;
    if (tok_stride < static_cast<int64_t>(num_q_heads + num_k_heads) * dim + static_cast<int64_t>(num_v_heads) * vdim)
        return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!qkv || !tok_pos || (rot_dims > 0 && !freq)) return SWL_ERR_BAD_ARG;
    if (k_cache && (!v_cache || !block_table || !tok_seq || max_blocks_per_seq <= 0)) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL || rot_dims > 2 * swl::kRkMaxPairs) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::rope_store_kv_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kRkThreads), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(qkv), freq, static_cast<T *>(k_cache),
                           static_cast<T *>(v_cache), block_table, tok_seq, tok_pos, num_q_heads, num_k_heads, num_v_heads,
                           dim, vdim, rot_dims, tok_stride, max_blocks_per_seq, block_stride);
    });
    return swl::check_launch();
}

extern "C" int swl_qk_norm_rope_store_kv(const void *rows, void *q_out, const float *q_b, const float *k_b, const float *q_w,
                                         const float *k_w, const float *q_mult, const double *freq, void *k_cache, void *v_cache,
                                         const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos,
                                         int64_t num_tokens, int32_t num_q_heads, int32_t num_k_heads, int32_t num_v_heads,
                                         int32_t dim, int32_t vdim, int32_t rot_dims, int32_t half, double rot_mult,
                                         int64_t tok_stride, int64_t q_out_stride, int32_t k_dim, int32_t v_dim,
                                         int32_t keys_as_values, int32_t max_blocks_per_seq, int64_t block_stride, float eps,
                                         int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_q_heads <= 0 || num_k_heads < 0 || num_v_heads < 0 || dim <= 0 || vdim <= 0) return SWL_ERR_BAD_ARG;
    if (rot_dims < 0 || (rot_dims & 1) || rot_dims > dim || (!half && (dim & 1))) return SWL_ERR_BAD_ARG;
    if (keys_as_values && (num_v_heads != 0 || vdim != dim)) return SWL_ERR_BAD_ARG;
    if (k_dim < dim || v_dim < vdim || q_out_stride < static_cast<int64_t>(num_q_heads) * k_dim) return SWL_ERR_BAD_ARG;
    if (tok_stride < static_cast<int64_t>(num_q_heads + num_k_heads) * dim + static_cast<int64_t>(num_v_heads) * vdim)
        return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!rows || !q_out || rows == q_out || !tok_pos || (rot_dims > 0 && !freq)) return SWL_ERR_BAD_ARG;
    if (k_cache && (!v_cache || !block_table || !tok_seq || max_blocks_per_seq <= 0)) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL || rot_dims > 2 * swl::kRkMaxPairs) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::qk_norm_rope_store_kv_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kRkThreads),
                           0, static_cast<hipStream_t>(stream), static_cast<const T *>(rows), static_cast<T *>(q_out), q_b, k_b,
                           q_w, k_w, q_mult, freq, static_cast<T *>(k_cache), static_cast<T *>(v_cache), block_table, tok_seq,
                           tok_pos, num_q_heads, num_k_heads, num_v_heads, dim, vdim, rot_dims, half, rot_mult, tok_stride,
                           q_out_stride, k_dim, v_dim, keys_as_values, max_blocks_per_seq, block_stride, eps);
    });
    return swl::check_launch();
}

extern "C" int swl_qkv_conv_rope_store_kv(
    const void *rows, int64_t tok_stride, void *q_out, int64_t q_out_stride, const float *bias, const float *conv_w, int32_t taps,
    const float *q_w, const float *k_w, const double *freq, int32_t rot_dims, int32_t half, double rot_mult, float v_mult,
    void *k_cache, void *v_cache, const int32_t *block_table, int32_t max_blocks_per_seq, int64_t block_stride, float *state,
    int64_t slot_stride, int64_t tail_off, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *tok_state,
    const int32_t *tok_seq, int64_t num_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t dim, int32_t vdim, int32_t k_dim,
    int32_t v_dim, float eps, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || dim <= 0 || vdim <= 0) return SWL_ERR_BAD_ARG;
    if (rot_dims < 0 || (rot_dims & 1) || rot_dims > dim || (!half && (dim & 1))) return SWL_ERR_BAD_ARG;
    if (k_dim < dim || v_dim < vdim || q_out_stride < static_cast<int64_t>(num_q_heads) * k_dim) return SWL_ERR_BAD_ARG;
    const int64_t C = static_cast<int64_t>(num_q_heads + num_kv_heads) * dim + static_cast<int64_t>(num_kv_heads) * vdim;
    if (tok_stride < C || (conv_w && taps < 1) || (!q_w) != (!k_w)) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!rows || !q_out || rows == q_out || !tok_pos || !tok_seq || (rot_dims > 0 && !freq)) return SWL_ERR_BAD_ARG;
    if (conv_w && (!tok_start || (taps > 1 && (!state || !tok_state)))) return SWL_ERR_BAD_ARG;
    if (k_cache && (!v_cache || !block_table || max_blocks_per_seq <= 0)) return SWL_ERR_BAD_ARG;
    const size_t lds = (static_cast<size_t>(C) + num_q_heads + num_kv_heads) * sizeof(float);
    if (num_tokens > 0x7fffffffLL || rot_dims > 2 * swl::kRkMaxPairs || lds > 60 * 1024) return SWL_ERR_UNSUPPORTED;
#define SWL_ROWS_TOK(LPH, TOK)                                                                                                            \
    hipLaunchKernelGGL((swl::qkv_conv_rope_rows_kernel<T, LPH, TOK>), dim3(static_cast<unsigned>((num_tokens + TOK - 1) / TOK)), dim3(threads), 0, \
                       static_cast<hipStream_t>(stream), static_cast<const T *>(rows), tok_stride, static_cast<T *>(q_out), q_out_stride, \
                       bias, conv_w, taps, q_w, k_w, freq, rot_dims, half, rot_mult, v_mult, static_cast<T *>(k_cache),                   \
                       static_cast<T *>(v_cache), block_table, max_blocks_per_seq, block_stride, state, slot_stride, tail_off, tok_pos,   \
                       tok_start, tok_state, tok_seq, num_tokens, num_q_heads, num_kv_heads, vdim, k_dim, v_dim, eps)
#define SWL_ROWS(LPH)                                                                                                                     \
    if (rows8 && dim == 8 * LPH) {                                                                                                        \
        if (swl::rk_four_pay(num_tokens, C)) SWL_ROWS_TOK(LPH, 4);                                                                         \
        else SWL_ROWS_TOK(LPH, 1);                                                                                                        \
        return swl::check_launch();                                                                                                       \
    }
    SWL_DISPATCH_DTYPE3(dtype, T, {
        constexpr int PIECE = 16 / static_cast<int>(sizeof(T));
        const bool rows8 = swl::aligned16(rows) && swl::aligned16(q_out) && tok_stride % PIECE == 0 && q_out_stride % PIECE == 0 && k_dim % 8 == 0 &&
                           vdim % 8 == 0 && (!bias || swl::aligned16(bias)) && (!q_w || (swl::aligned16(q_w) && swl::aligned16(k_w))) &&
                           (half ? rot_dims % 16 == 0 : rot_dims % 8 == 0) && (!k_cache || (swl::aligned16(k_cache) && block_stride % PIECE == 0)) &&
                           (!conv_w || (taps <= 4 && swl::aligned16(conv_w) &&
                                        (taps == 1 || (swl::aligned16(state) && slot_stride % 4 == 0 && tail_off % 4 == 0))));
        // (a thread takes eight channels: no more waves than have some)
        const int threads = static_cast<int>(C < 8 * swl::kRkThreads ? (C / 8 + 63) / 64 * 64 : swl::kRkThreads);
        SWL_ROWS(2)
        SWL_ROWS(4)
        SWL_ROWS(8)
        SWL_ROWS(16)
        hipLaunchKernelGGL((swl::qkv_conv_rope_store_kv_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kRkThreads),
                           lds, static_cast<hipStream_t>(stream), static_cast<const T *>(rows), tok_stride, static_cast<T *>(q_out),
                           q_out_stride, bias, conv_w, taps, q_w, k_w, freq, rot_dims, half, rot_mult, v_mult,
                           static_cast<T *>(k_cache), static_cast<T *>(v_cache), block_table, max_blocks_per_seq, block_stride,
                           state, slot_stride, tail_off, tok_pos, tok_start, tok_state, tok_seq, num_tokens, num_q_heads,
                           num_kv_heads, dim, vdim, k_dim, v_dim, eps);
    });
#undef SWL_ROWS
#undef SWL_ROWS_TOK
    return swl::check_launch();
}

extern "C" int swl_latent_rope_store_kv_rows(void *proj, void *qa, int64_t in_place, const double *freq, const float *c_norm,
                                        void *k_cache, void *v_cache, const int32_t *block_table, const int32_t *tok_seq,
                                        const int32_t *tok_pos, int64_t num_tokens, int32_t num_heads, int32_t dim,
                                        int32_t rot_dim, int32_t kv_rank, int64_t proj_stride, int64_t dkv_col,
                                        int64_t qa_stride, int32_t max_blocks_per_seq, int64_t block_stride, float eps,
                                        int32_t half, double rot_mult, int32_t k_dim, int32_t v_dim, int32_t dtype,
                                        swl_stream_t stream) {
    if (in_place < 0) return SWL_ERR_BAD_ARG;
    if (num_tokens < 0 || num_heads <= 0 || dim <= 0 || rot_dim <= 0 || (rot_dim & 1) || kv_rank <= 0) return SWL_ERR_BAD_ARG;
    if (k_dim < kv_rank + rot_dim || v_dim < kv_rank) return SWL_ERR_BAD_ARG;
    if (proj_stride < static_cast<int64_t>(num_heads) * (dim + rot_dim) || qa_stride < static_cast<int64_t>(num_heads) * k_dim)
        return SWL_ERR_BAD_ARG;
    if (dkv_col >= 0 && dkv_col + kv_rank + rot_dim > proj_stride) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!proj || (!qa && in_place < num_tokens) || !freq || !tok_pos) return SWL_ERR_BAD_ARG;
    if (dkv_col >= 0 && k_cache && (!v_cache || !c_norm || !block_table || !tok_seq || max_blocks_per_seq <= 0))
        return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL || rot_dim > 2 * swl::kRkMaxPairs) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::latent_rope_store_kv_kernel<T>), dim3(static_cast<unsigned>(num_tokens)),
                           dim3(swl::kRkThreads), 0, static_cast<hipStream_t>(stream), static_cast<T *>(proj),
                           static_cast<T *>(qa), in_place, freq, c_norm, static_cast<T *>(k_cache), static_cast<T *>(v_cache),
                           block_table, tok_seq, tok_pos, num_heads, dim, rot_dim, kv_rank, proj_stride, dkv_col, qa_stride,
                           max_blocks_per_seq, block_stride, eps, half, rot_mult, k_dim, v_dim);
    });
    return swl::check_launch();
}

extern "C" int swl_latent_rope_store_kv(const void *proj, void *qa, const double *freq, const float *c_norm, void *k_cache,
                                        void *v_cache, const int32_t *block_table, const int32_t *tok_seq,
                                        const int32_t *tok_pos, int64_t num_tokens, int32_t num_heads, int32_t dim,
                                        int32_t rot_dim, int32_t kv_rank, int64_t proj_stride, int64_t dkv_col,
                                        int64_t qa_stride, int32_t max_blocks_per_seq, int64_t block_stride, float eps,
                                        int32_t half, double rot_mult, int32_t k_dim, int32_t v_dim, int32_t dtype,
                                        swl_stream_t stream) {
    return swl_latent_rope_store_kv_rows(const_cast<void *>(proj), qa, 0, freq, c_norm, k_cache, v_cache, block_table, tok_seq, tok_pos,
                                         num_tokens, num_heads, dim, rot_dim, kv_rank, proj_stride, dkv_col, qa_stride,
                                         max_blocks_per_seq, block_stride, eps, half, rot_mult, k_dim, v_dim, dtype, stream);
}

/* 1 when swl_latent_fold serves these sizes. */
extern "C" int swl_latent_fold_supported(int32_t dim, int32_t rot_dim, int32_t kv_rank, int32_t k_dim, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    return dim > 0 && dim % 32 == 0 && dim <= swl::kFoldMaxDim && rot_dim > 0 && rot_dim % 8 == 0 && rot_dim <= 2 * swl::kRkMaxPairs && kv_rank > 0 &&
           kv_rank % 64 == 0 && k_dim >= kv_rank + rot_dim && k_dim % 4 == 0;
}

extern "C" int swl_latent_fold(const void *proj, void *qa, const void *uk_t, const double *freq, const float *c_norm, void *k_cache, void *v_cache,
                               const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos, int64_t num_tokens, int32_t num_heads,
                               int32_t dim, int32_t rot_dim, int32_t kv_rank, int64_t proj_stride, int64_t dkv_col, int64_t qa_stride,
                               int32_t max_blocks_per_seq, int64_t block_stride, float eps, int32_t half, double rot_mult, int32_t k_dim,
                               int32_t v_dim, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_heads <= 0 || v_dim < kv_rank) return SWL_ERR_BAD_ARG;
    if (!swl_latent_fold_supported(dim, rot_dim, kv_rank, k_dim, dtype)) return SWL_ERR_UNSUPPORTED;
    if (proj_stride < static_cast<int64_t>(num_heads) * (dim + rot_dim) || qa_stride < static_cast<int64_t>(num_heads) * k_dim)
        return SWL_ERR_BAD_ARG;
    if (dkv_col >= 0 && dkv_col + kv_rank + rot_dim > proj_stride) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!proj || !qa || !uk_t || !freq || !tok_pos) return SWL_ERR_BAD_ARG;
    if (dkv_col >= 0 && k_cache && (!v_cache || !c_norm || !block_table || !tok_seq || max_blocks_per_seq <= 0)) return SWL_ERR_BAD_ARG;
    // 16-byte loads of queries and matrices, 8-byte stores
    if (!swl::aligned16(proj) || (proj_stride & 7) || !swl::aligned16(uk_t) || (reinterpret_cast<uintptr_t>(qa) & 7) || (qa_stride & 3)) return SWL_ERR_BAD_ARG;
    const int64_t grid = num_tokens + static_cast<int64_t>(num_heads) * (kv_rank / 64);
    if (grid > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE(dtype, T, {
        hipLaunchKernelGGL((swl::latent_fold_kernel<T>), dim3(static_cast<unsigned>(grid)), dim3(swl::kRkThreads), 0, static_cast<hipStream_t>(stream),
                           static_cast<T *>(const_cast<void *>(proj)), static_cast<T *>(qa), static_cast<int>(num_tokens), static_cast<const T *>(uk_t), freq,
                           c_norm, static_cast<T *>(k_cache), static_cast<T *>(v_cache), block_table, tok_seq, tok_pos, num_heads, dim, rot_dim, kv_rank,
                           proj_stride, dkv_col, qa_stride, max_blocks_per_seq, block_stride, eps, half, rot_mult, k_dim, v_dim);
    });
    return swl::check_launch();
}

extern "C" int swl_diff_head_combine(void *out, const float *maps, const void *gate, int64_t gate_stride, float lambda,
                                     float mult, float eps, int64_t num_tokens, int32_t num_heads, int32_t vdim,
                                     int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_heads <= 0 || vdim <= 0 || (gate && gate_stride < num_heads)) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!out || !maps) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    const dim3 grid(static_cast<unsigned>(num_tokens), num_tokens >= swl::kDiffManyTokens ? 1 : swl::diff_groups(num_heads));
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::diff_head_combine_kernel<T>), grid, dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<T *>(out), maps,
                           static_cast<const T *>(gate), gate_stride, lambda, mult, eps, num_heads, vdim);
    });
    return swl::check_launch();
}

extern "C" int swl_diff_head_combine_shares(void *out, const float *shares, int32_t num_shares, int32_t natural, const void *gate,
                                            int64_t gate_stride, float lambda, float mult, float eps, int64_t num_tokens, int32_t num_heads,
                                            int32_t vdim, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_heads <= 0 || vdim <= 0 || num_shares < 1 || (gate && gate_stride < num_heads)) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!out || !shares) return SWL_ERR_BAD_ARG;
    const int64_t rows = num_tokens * num_heads;
    if (num_tokens > 0x7fffffffLL || rows / 4 >= 0x7fffffffLL || vdim > swl::kDiffMaxDim || vdim % 4 || num_shares > swl::kDiffMaxShares ||
        !swl::aligned16(out) || !swl::aligned16(shares)) return SWL_ERR_UNSUPPORTED;
    const float *part_ml = shares + num_shares * 2 * rows * vdim;
#define SWL_DIFF(NATURAL)                                                                                                                  \
    hipLaunchKernelGGL((swl::diff_head_shares_kernel<T, NATURAL>), dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0,              \
                       static_cast<hipStream_t>(stream), static_cast<T *>(out), shares, part_ml, num_shares, static_cast<const T *>(gate), \
                       gate_stride, lambda, mult, eps, rows, num_heads, vdim)
    SWL_DISPATCH_DTYPE3(dtype, T, {
        if (natural) SWL_DIFF(true);
        else SWL_DIFF(false);
    });
#undef SWL_DIFF
    return swl::check_launch();
}

extern "C" int swl_head_gate(void *y, const void *gate, int64_t gate_stride, int64_t num_tokens, int32_t num_heads,
                             int32_t vdim, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_heads <= 0 || vdim <= 0 || gate_stride < num_heads) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!y || !gate) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::head_gate_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(256), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(y), static_cast<const T *>(gate), gate_stride,
                           num_heads, vdim);
    });
    return swl::check_launch();
}
