// qknorm_kv.hip — per-head RMS norm of queries and keys fused with the paged KV store.
//
// One workgroup per token of the step (prompt portions and decoded tokens alike: every token carries its own sequence
// row and position). The query heads are normalised in place inside the fused qkv projection output; the key heads are
// normalised on their way into the K pool; the value heads are copied into the V pool. Norm statistics are fp32; the
// norm weight is shared by all heads (plain weight, not one-plus).
//
// Pool layout: block b of a layer run's keys starts at k_cache + b * block_stride and holds [kv_heads, 16, dim]; its values
// start at v_cache + b * block_stride and hold [kv_heads, vdim, 16] — TRANSPOSED, the 16 tokens of a column contiguous, which is
// how the matrix-core attention wants its value operand (block_stride in elements: a block of the pool may hold the
// keys and values of several layer runs side by side, so that swapping moves one contiguous piece per block).
#include "swl_common.h"
#include "conv_tail.h"

namespace swl {

constexpr int kQkThreads = 256;
constexpr int kQkBlock = 16;    // tokens per KV block

template <typename T>
__global__ __launch_bounds__(kQkThreads) void qknorm_store_kv_kernel(
    T *qkv, const float *q_w, const float *k_w, T *k_cache, T *v_cache, const int32_t *block_table,
    const int32_t *tok_seq, const int32_t *tok_pos, int H, int G, int d, int dv, int64_t tok_stride,
    int max_blocks_per_seq, int64_t block_stride, float eps, int store) {
    const int64_t t = page_token();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    T *row = qkv + t * tok_stride;
    const int pos = tok_pos[t];
    int64_t blk = 0;
    if (store) blk = block_table[static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq + pos / kQkBlock];
    const int off = pos % kQkBlock;
    // heads 0..H-1: queries (in place); H..H+G-1: keys (into the pool)
    bool wide = false;
    if constexpr (sizeof(T) == 2) {
        // 16-bit heads of 32 / 64 / 128 elements on 16-byte-aligned rows: d / 8 lanes per head move 16 bytes each and several
        // heads share a wave (the group reduction stays inside d / 8 aligned lanes)
        wide = (d == 32 || d == 64 || d == 128) && (tok_stride & 7) == 0 && (reinterpret_cast<uintptr_t>(qkv) & 15) == 0 &&
               (!store || ((reinterpret_cast<uintptr_t>(k_cache) & 15) == 0 && (block_stride & 7) == 0));
        if (wide) {
            const int lph = d >> 3;                 // lanes per head: 4, 8 or 16
            const int hpw = 64 / lph;               // heads per wave and pass
            const int slot = lane / lph, el = lane - slot * lph;
            for (int hb = wave * hpw; hb < H + G; hb += (kQkThreads / 64) * hpw) {
                const int h = hb + slot;
                const bool live = h < H + G;
                T *src = row + static_cast<int64_t>(live ? h : 0) * d + el * 8;
                vec8_t<T> v = vec8_t<T>{};
                if (live) v = load8(src);
                float ss = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) ss += to_f(v[j]) * to_f(v[j]);
                ss = lph == 4 ? group_allreduce_sum<4>(ss) : lph == 8 ? group_allreduce_sum<8>(ss) : group_allreduce_sum<16>(ss);
                const float r = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
                if (!live) continue;
                const bool is_q = h < H;
                if (!is_q && !store) continue;
                const float *wn = (is_q ? q_w : k_w) + el * 8;
                vec8_t<T> o;
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = to_t<T>(to_f(v[j]) * r * wn[j]);
                if (is_q) store8(src, o);
                else store8(k_cache + blk * block_stride + (static_cast<int64_t>(h - H) * kQkBlock + off) * d + el * 8, o);
            }
        }
    }
    for (int h = wave; h < H + G && !wide; h += kQkThreads / 64) {
        const bool is_q = h < H;
        const T *src = row + static_cast<int64_t>(h) * d;       // k heads follow the q heads: same formula
        float ss = 0.f;
        for (int e = lane; e < d; e += 64) {
            const float v = to_f(src[e]);
            ss += v * v;
        }
        ss = wave_allreduce_sum(ss);
        const float r = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
        if (is_q) {
            T *dst = row + static_cast<int64_t>(h) * d;
            for (int e = lane; e < d; e += 64) dst[e] = to_t<T>(to_f(src[e]) * r * q_w[e]);
        } else if (store) {
            const int g = h - H;
            T *dst = k_cache + blk * block_stride + (static_cast<int64_t>(g) * kQkBlock + off) * d;
            for (int e = lane; e < d; e += 64) dst[e] = to_t<T>(to_f(src[e]) * r * k_w[e]);
        }
    }
    if (store) {
        const T *vsrc = row + static_cast<int64_t>(H + G) * d;
        for (int i = threadIdx.x; i < G * dv; i += kQkThreads) {
            const int g = i / dv, c = i - g * dv;
            v_cache[blk * block_stride + (static_cast<int64_t>(g) * dv + c) * kQkBlock + off] = vsrc[i];    // transposed page
        }
    }
}


// The same store with ONE norm over the whole query projection and one over the whole key projection (all heads at once,
// a weight per element), and a query multiplier that grows with the logarithm of the position:
//   q <- q / rms(q) * q_w * (1 + temp_coef * ln(floor((pos + 1) / temp_every) + 1)).
// store = 0: the row holds queries only (a layer that attends over another layer's keys and values).
template <typename T>
__global__ __launch_bounds__(kQkThreads) void qknorm_full_store_kv_kernel(
    T *qkv, const float *q_w, const float *k_w, T *k_cache, T *v_cache, const int32_t *block_table,
    const int32_t *tok_seq, const int32_t *tok_pos, int H, int G, int d, int dv, int64_t tok_stride,
    int max_blocks_per_seq, int64_t block_stride, float eps, float temp_coef, int temp_every, int store) {
    __shared__ float red[2][kQkThreads / 64];
    const int64_t t = page_token();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    T *row = qkv + t * tok_stride;
    const int pos = tok_pos[t];
    const int nq = H * d, nk = G * d;
    float sq = 0.f, sk = 0.f;
    for (int i = threadIdx.x; i < nq; i += kQkThreads) {
        const float v = to_f(row[i]);
        sq += v * v;
    }
    if (store) {
        for (int i = threadIdx.x; i < nk; i += kQkThreads) {
            const float v = to_f(row[nq + i]);
            sk += v * v;
        }
    }
    sq = wave_allreduce_sum(sq);
    sk = wave_allreduce_sum(sk);
    if (lane == 0) {
        red[0][wave] = sq;
        red[1][wave] = sk;
    }
    __syncthreads();
    sq = sk = 0.f;
#pragma unroll
    for (int w = 0; w < kQkThreads / 64; ++w) {
        sq += red[0][w];
        sk += red[1][w];
    }
    float rq = 1.0f / sqrtf(sq / static_cast<float>(nq) + eps);
    if (temp_coef != 0.f) rq *= 1.0f + temp_coef * logf(static_cast<float>((pos + 1) / temp_every + 1));
    for (int i = threadIdx.x; i < nq; i += kQkThreads) row[i] = to_t<T>(to_f(row[i]) * q_w[i] * rq);
    if (!store) return;
    const float rk = 1.0f / sqrtf(sk / static_cast<float>(nk) + eps);
    const int64_t blk = block_table[static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq + pos / kQkBlock];
    const int off = pos % kQkBlock;
    for (int i = threadIdx.x; i < nk; i += kQkThreads) {
        const int g = i / d, e = i - g * d;
        k_cache[blk * block_stride + (static_cast<int64_t>(g) * kQkBlock + off) * d + e] = to_t<T>(to_f(row[nq + i]) * k_w[i] * rk);
    }
    const T *vsrc = row + nq + nk;
    for (int i = threadIdx.x; i < G * dv; i += kQkThreads) {
        const int g = i / dv, c = i - g * dv;
        v_cache[blk * block_stride + (static_cast<int64_t>(g) * dv + c) * kQkBlock + off] = vsrc[i];    // transposed page
    }
}


// The same store for projections WITH biases and values that may be blended with the values another layer made for the same
// token. Per token:
//   q_h <- (q_h + b_q) / rms(q_h + b_q) * w_q     in place, per head (w_q NULL: no weight)
//   k_g <- (k_g + b_k) / rms(k_g + b_k) * w_k     into the pool
//   v   <- v + b_v;  v <- (1 - mix) v + mix v_other[t]  (v_other given)   written back into the row AND into the pool
// so that the row's value columns can serve as v_other of a later layer. Biases and weights are fp32, all sums fp32.
template <typename T>
__global__ __launch_bounds__(kQkThreads) void qkv_bias_norm_store_kernel(
    T *qkv, const float *q_b, const float *k_b, const float *v_b, const float *q_w, const float *k_w, const T *v_other,
    int64_t v_other_stride, float mix, T *k_cache, T *v_cache, const int32_t *block_table, const int32_t *tok_seq,
    const int32_t *tok_pos, int H, int G, int d, int dv, int64_t tok_stride, int max_blocks_per_seq, int64_t block_stride,
    float eps, int store) {
    const int64_t t = page_token();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    T *row = qkv + t * tok_stride;
    const int pos = tok_pos[t];
    int64_t blk = 0;
    if (store) blk = block_table[static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq + pos / kQkBlock];
    const int off = pos % kQkBlock;
    for (int h = wave; h < H + G; h += kQkThreads / 64) {
        const bool is_q = h < H;
        if (!is_q && !store) continue;
        T *src = row + static_cast<int64_t>(h) * d;         // k heads follow the q heads
        const float *bias = is_q ? (q_b ? q_b + static_cast<int64_t>(h) * d : nullptr)
                                 : (k_b ? k_b + static_cast<int64_t>(h - H) * d : nullptr);
        const float *wn = is_q ? q_w : k_w;
        float ss = 0.f;
        for (int e = lane; e < d; e += 64) {
            const float v = to_f(src[e]) + (bias ? bias[e] : 0.f);
            ss += v * v;
        }
        ss = wave_allreduce_sum(ss);
        const float r = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
        T *dst = is_q ? src : k_cache + blk * block_stride + (static_cast<int64_t>(h - H) * kQkBlock + off) * d;
        for (int e = lane; e < d; e += 64) {
            const float v = (to_f(src[e]) + (bias ? bias[e] : 0.f)) * r;
            dst[e] = to_t<T>(wn ? v * wn[e] : v);
        }
    }
    T *vsrc = row + static_cast<int64_t>(H + G) * d;
    const T *vo = v_other ? v_other + t * v_other_stride : nullptr;
    for (int i = threadIdx.x; i < G * dv; i += kQkThreads) {
        float v = to_f(vsrc[i]) + (v_b ? v_b[i] : 0.f);
        if (vo) v = (1.0f - mix) * v + mix * to_f(vo[i]);
        const T vt = to_t<T>(v);
        vsrc[i] = vt;
        if (store) {
            const int g = i / dv, c = i - g * dv;
            v_cache[blk * block_stride + (static_cast<int64_t>(g) * dv + c) * kQkBlock + off] = vt;     // transposed page
        }
    }
}

// The last two, and the first in fp32, for rows of whole aligned pieces of eight, a piece a thread in registers: heads of 8 LPH columns (16, 32, 64 or
// 128) normed one by one, or (LPH 0) the whole query and the whole key projection. Bound by the chain of a token's workgroup and by the
// stores into the transposed page; everything a piece needs (row, bias, weights, the other layer's values) is asked for together, where a
// weight at a time after the norm's sum costs 15 us of 33. Before -> here, heads of 128: biased 3663 tokens 16 over 4 33.3 -> 16.4 us, 8 over 2
// 18.6 -> 9.9, 32 tokens 6.5 -> 4.0, 5000 of 32 over 32 169 -> 82; whole projections 8192 of 8 over 2 24.7 -> 15.5, 4500 of 16 over 4 25.8 -> 19.4, 32 6.1 ->
// 4.3, 3 in fp32 4.4 -> 3.8; per head in fp32 500 tokens 6.0 -> 4.8. Values that are no whole pieces (or blend in another layer's
// that are not) go one at a time behind heads normed one by one; in the kernel above / here, 3663 tokens: 8 over 2 heads of 64 with 33 columns of values
// 12.7 / 7.0, 16 over 4 of 128 blended with values three columns into a row 32.7 / 19.5, 16 over 4 of 64 with 36 (whole pieces over the heads) 20.4 / 8.9.
template <typename T>
struct QkvRows {
    T *qkv;
    const float *q_b, *k_b, *v_b, *q_w, *k_w;       // (each may be NULL: nothing to add, no weight)
    const T *v_other;
    T *k_cache, *v_cache;
    const int32_t *block_table, *tok_seq, *tok_pos;
    int64_t v_other_stride, tok_stride, block_stride;
    int H, G, d, dv, max_blocks, store, v_back, temp_every;     // v_back: values are written back into the row too
    float mix, eps, temp_coef;
};
constexpr int kQkRowsThreads = 512;

// V_PIECES: values in pieces of eight too (LPH 0: always)
template <typename T, int LPH, bool V_PIECES>
__global__ __launch_bounds__(kQkRowsThreads) void qkv_rows_kernel(QkvRows<T> a) {
    static_assert(LPH > 0 || V_PIECES, "");
    __shared__ float red[2][kQkRowsThreads / 64];
    extern __shared__ __attribute__((aligned(16))) char lds[];
    T *values = reinterpret_cast<T *>(lds);     // [G dv]
    const int64_t t = page_token();
    T *row = a.qkv + t * a.tok_stride;
    const int nq = a.H * a.d, nqk = nq + a.G * a.d, C = nqk + a.G * a.dv, step = blockDim.x * 8;
    const int pos = a.tok_pos[t], off = pos % kQkBlock;
    int64_t blk = 0;
    if (a.store) blk = a.block_table[static_cast<int64_t>(a.tok_seq[t]) * a.max_blocks + pos / kQkBlock];
    T *kpage = a.k_cache + blk * a.block_stride, *vpage = a.v_cache + blk * a.block_stride;
    const int end = !a.store && !a.v_back ? nq : V_PIECES ? C : nqk;
    float x[8], y[8], w[8], b[8];       // the row's piece, the other layer's values, weights, biases
    T raw[8];
    auto ask = [&](int c) {
        if constexpr (sizeof(T) == 2) {
            const vec8_t<T> v = load8(row + c);
#pragma unroll
            for (int j = 0; j < 8; ++j) raw[j] = v[j];
        } else {
            ConvTail::row8(row + c, raw);
        }
        const float *bias = c < nq ? a.q_b : c < nqk ? a.k_b : a.v_b, *wn = c < nq ? a.q_w : a.k_w;
        const int cc = c < nq ? c : c < nqk ? c - nq : c - nqk;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            b[j] = 0.f;
            w[j] = 1.f;
        }
        if (bias) ConvTail::row8(bias + cc, b);
        if (c < nqk && wn) ConvTail::row8(wn + (LPH ? cc % (LPH ? 8 * LPH : 1) : cc), w);
        if (c >= nqk && a.v_other) ConvTail::row8(a.v_other + t * a.v_other_stride + cc, y);
    };
    auto put = [&](int c) {     // one piece of x
        if (c < nq) ConvTail::put8(row + c, x);
        else if (c < nqk) {
            const int g = (c - nq) / a.d, e = c - nq - g * a.d;
            if (a.store) ConvTail::put8(kpage + (static_cast<int64_t>(g) * kQkBlock + off) * a.d + e, x);
        } else {
            if (a.v_b || a.v_other) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float v = x[j];
                    if (a.v_other) v = (1.0f - a.mix) * v + a.mix * y[j];
                    raw[j] = to_t<T>(v);
                }
                if (a.v_back) {
                    if constexpr (sizeof(T) == 2) {
                        vec8_t<T> v;
#pragma unroll
                        for (int j = 0; j < 8; ++j) v[j] = raw[j];
                        store8(row + c, v);
                    } else {
                        ConvTail::put8(row + c, raw);
                    }
                }
            }
            if (a.store) {
#pragma unroll
                for (int j = 0; j < 8; ++j) values[c - nqk + j] = raw[j];
            }
        }
    };
    if constexpr (LPH > 0) {
        for (int c = threadIdx.x * 8; c < end; c += step) {
            ask(c);
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = to_f(raw[j]) + b[j];
            if (c < nqk) {
                float ss = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
                ss = group_allreduce_sum<LPH>(ss);
                const float r = 1.0f / sqrtf(ss / static_cast<float>(8 * LPH) + a.eps);
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = x[j] * r * w[j];
            }
            put(c);
        }
    } else {        // (one piece a thread)
        const int c = threadIdx.x * 8, wave = threadIdx.x >> 6;
        float sq = 0.f, sk = 0.f;
        if (c < end) {
            ask(c);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                x[j] = to_f(raw[j]) + b[j];
                sq += c < nq ? x[j] * x[j] : 0.f;
                sk += c >= nq && c < nqk ? x[j] * x[j] : 0.f;
            }
        }
        sq = wave_allreduce_sum(sq);
        sk = wave_allreduce_sum(sk);
        if ((threadIdx.x & 63) == 0) {
            red[0][wave] = sq;
            red[1][wave] = sk;
        }
        __syncthreads();
        if (c < end) {
            float ss = 0.f;
            for (int i = 0; i < static_cast<int>(blockDim.x) / 64; ++i) ss += red[c < nq ? 0 : 1][i];
            float r = 1.0f / sqrtf(ss / static_cast<float>(c < nq ? nq : nqk - nq) + a.eps);
            if (c < nq && a.temp_coef != 0.f) r *= 1.0f + a.temp_coef * logf(static_cast<float>((pos + 1) / a.temp_every + 1));
            if (c < nqk) {
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = x[j] * w[j] * r;
            }
            put(c);
        }
    }
    if constexpr (!V_PIECES) {
        for (int i = threadIdx.x; i < (a.store || a.v_back ? a.G * a.dv : 0); i += blockDim.x) {
            float v = to_f(row[nqk + i]) + (a.v_b ? a.v_b[i] : 0.f);
            if (a.v_other) v = (1.0f - a.mix) * v + a.mix * to_f(a.v_other[t * a.v_other_stride + i]);
            const T vt = to_t<T>(v);
            if (a.v_back && (a.v_b || a.v_other)) row[nqk + i] = vt;
            if (a.store) vpage[static_cast<int64_t>(i) * kQkBlock + off] = vt;
        }
        return;
    }
    if (!a.store) return;
    __syncthreads();
    // the transposed page keeps the 16 tokens of a column together: neighbouring lanes take neighbouring columns, 32 bytes apart (a lane that
    // stores its own eight is 256 bytes from the next, and a store then touches four times the lines: 19.3 against 16.4 us at 3663 tokens)
    for (int i = threadIdx.x; i < a.G * a.dv; i += blockDim.x) vpage[static_cast<int64_t>(i) * kQkBlock + off] = values[i];
}

// Launches qkv_rows_kernel where it serves the rows; false: nothing was launched.
template <typename T>
static bool launch_rows(const QkvRows<T> &a, bool whole, int64_t num_tokens, hipStream_t s) {
    constexpr int PIECE = 16 / static_cast<int>(sizeof(T));
    const int64_t C = static_cast<int64_t>(a.H + a.G) * a.d + static_cast<int64_t>(a.G) * a.dv;
    auto ok = [](const void *p) { return aligned16(p); };       // (NULL is)
    if (a.d % 8 || a.tok_stride % PIECE || !ok(a.qkv) || !ok(a.q_b) || !ok(a.k_b) || !ok(a.q_w) || !ok(a.k_w) ||
        (a.store && (!ok(a.k_cache) || a.block_stride % PIECE)))
        return false;
    const size_t values = sizeof(T) * a.G * a.dv;
    const bool v_pieces = a.G * a.dv % 8 == 0 && ok(a.v_b) && (!a.v_other || (ok(a.v_other) && a.v_other_stride % PIECE == 0)) && values <= 32 * 1024;
    if (whole && (!v_pieces || C > 8 * kQkRowsThreads)) return false;
    const size_t lds = v_pieces ? values : 0;
    // (no more waves than have a piece)
    const dim3 grid(static_cast<unsigned>(num_tokens)), block(static_cast<unsigned>(C < 8 * kQkRowsThreads ? (C + 511) / 512 * 64 : kQkRowsThreads));
#define SWL_ROWS(LPH, PIECES) hipLaunchKernelGGL((qkv_rows_kernel<T, LPH, PIECES>), grid, block, lds, s, a)
#define SWL_ROWS_OF(LPH) do { if (v_pieces) SWL_ROWS(LPH, true); else SWL_ROWS(LPH, false); } while (0)
    if (whole) SWL_ROWS(0, true);
    else if (a.d == 16) SWL_ROWS_OF(2);
    else if (a.d == 32) SWL_ROWS_OF(4);
    else if (a.d == 64) SWL_ROWS_OF(8);
    else if (a.d == 128) SWL_ROWS_OF(16);
    else return false;
#undef SWL_ROWS_OF
#undef SWL_ROWS
    return true;
}

} // namespace swl

extern "C" int swl_qknorm_store_kv(void *qkv, const float *q_w, const float *k_w, void *k_cache, void *v_cache,
                                   const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos,
                                   int64_t num_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t dim,
                                   int32_t vdim, int64_t tok_stride, int32_t max_blocks_per_seq, int64_t block_stride,
                                   float eps, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || dim <= 0 || vdim <= 0) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!qkv || !q_w || !k_w || !tok_pos) return SWL_ERR_BAD_ARG;
    const int store = k_cache != nullptr;
    if (store && (!v_cache || !block_table || !tok_seq)) return SWL_ERR_BAD_ARG;
    if (tok_stride < static_cast<int64_t>(num_q_heads + num_kv_heads) * dim + static_cast<int64_t>(num_kv_heads) * vdim)
        return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        if constexpr (sizeof(T) == 4) {     // (16-bit rows: 15.2 us in the kernel below, 17.2 in this one, at 4500 tokens of 16 over 4 heads of 128)
            const swl::QkvRows<T> rows{static_cast<T *>(qkv), nullptr, nullptr, nullptr, q_w, k_w, nullptr, static_cast<T *>(k_cache),
                                       static_cast<T *>(v_cache), block_table, tok_seq, tok_pos, 0, tok_stride, block_stride, num_q_heads,
                                       num_kv_heads, dim, vdim, max_blocks_per_seq, store, 0, 1, 0.f, eps, 0.f};
            if (swl::launch_rows(rows, false, num_tokens, static_cast<hipStream_t>(stream))) return swl::check_launch();
        }
        hipLaunchKernelGGL((swl::qknorm_store_kv_kernel<T>), dim3(static_cast<unsigned>(num_tokens)),
                           dim3(swl::kQkThreads), 0, static_cast<hipStream_t>(stream), static_cast<T *>(qkv), q_w, k_w,
                           static_cast<T *>(k_cache), static_cast<T *>(v_cache), block_table, tok_seq, tok_pos,
                           num_q_heads, num_kv_heads, dim, vdim, tok_stride, max_blocks_per_seq, block_stride, eps, store);
    });
    return swl::check_launch();
}

extern "C" int swl_qknorm_full_store_kv(void *qkv, const float *q_w, const float *k_w, void *k_cache, void *v_cache,
                                        const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos,
                                        int64_t num_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t dim,
                                        int32_t vdim, int64_t tok_stride, int32_t max_blocks_per_seq,
                                        int64_t block_stride, float eps, float temp_coef, int32_t temp_every,
                                        int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || dim <= 0 || vdim <= 0 || temp_every < 1)
        return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!qkv || !q_w || !tok_pos) return SWL_ERR_BAD_ARG;
    const int store = k_cache != nullptr;
    if (store && (!k_w || !v_cache || !block_table || !tok_seq)) return SWL_ERR_BAD_ARG;
    const int64_t need = static_cast<int64_t>(num_q_heads) * dim +
                         (store ? static_cast<int64_t>(num_kv_heads) * (dim + vdim) : 0);
    if (tok_stride < need) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        const swl::QkvRows<T> rows{static_cast<T *>(qkv), nullptr, nullptr, nullptr, q_w, k_w, nullptr, static_cast<T *>(k_cache),
                                   static_cast<T *>(v_cache), block_table, tok_seq, tok_pos, 0, tok_stride, block_stride, num_q_heads,
                                   num_kv_heads, dim, vdim, max_blocks_per_seq, store, 0, temp_every, 0.f, eps, temp_coef};
        if (swl::launch_rows(rows, true, num_tokens, static_cast<hipStream_t>(stream))) return swl::check_launch();
        hipLaunchKernelGGL((swl::qknorm_full_store_kv_kernel<T>), dim3(static_cast<unsigned>(num_tokens)),
                           dim3(swl::kQkThreads), 0, static_cast<hipStream_t>(stream), static_cast<T *>(qkv), q_w, k_w,
                           static_cast<T *>(k_cache), static_cast<T *>(v_cache), block_table, tok_seq, tok_pos,
                           num_q_heads, num_kv_heads, dim, vdim, tok_stride, max_blocks_per_seq, block_stride, eps,
                           temp_coef, temp_every, store);
    });
    return swl::check_launch();
}

extern "C" int swl_qkv_bias_norm_store(void *qkv, const float *q_b, const float *k_b, const float *v_b, const float *q_w,
                                       const float *k_w, const void *v_other, int64_t v_other_stride, float mix,
                                       void *k_cache, void *v_cache, const int32_t *block_table, const int32_t *tok_seq,
                                       const int32_t *tok_pos, int64_t num_tokens, int32_t num_q_heads,
                                       int32_t num_kv_heads, int32_t dim, int32_t vdim, int64_t tok_stride,
                                       int32_t max_blocks_per_seq, int64_t block_stride, float eps, int32_t dtype,
                                       swl_stream_t stream) {
    if (num_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || dim <= 0 || vdim <= 0) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!qkv || !tok_pos) return SWL_ERR_BAD_ARG;
    const int store = k_cache != nullptr;
    if (store && (!v_cache || !block_table || !tok_seq)) return SWL_ERR_BAD_ARG;
    if (tok_stride < static_cast<int64_t>(num_q_heads + num_kv_heads) * dim + static_cast<int64_t>(num_kv_heads) * vdim)
        return SWL_ERR_BAD_ARG;
    if (v_other && v_other_stride < static_cast<int64_t>(num_kv_heads) * vdim) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        const swl::QkvRows<T> rows{static_cast<T *>(qkv), q_b, k_b, v_b, q_w, k_w, static_cast<const T *>(v_other), static_cast<T *>(k_cache),
                                   static_cast<T *>(v_cache), block_table, tok_seq, tok_pos, v_other_stride, tok_stride,
                                   block_stride, num_q_heads, num_kv_heads, dim, vdim, max_blocks_per_seq, store, 1, 1, mix, eps, 0.f};
        if (swl::launch_rows(rows, false, num_tokens, static_cast<hipStream_t>(stream))) return swl::check_launch();
        hipLaunchKernelGGL((swl::qkv_bias_norm_store_kernel<T>), dim3(static_cast<unsigned>(num_tokens)),
                           dim3(swl::kQkThreads), 0, static_cast<hipStream_t>(stream), static_cast<T *>(qkv), q_b, k_b, v_b,
                           q_w, k_w, static_cast<const T *>(v_other), v_other_stride, mix, static_cast<T *>(k_cache),
                           static_cast<T *>(v_cache), block_table, tok_seq, tok_pos, num_q_heads, num_kv_heads, dim, vdim,
                           tok_stride, max_blocks_per_seq, block_stride, eps, store);
    });
    return swl::check_launch();
}
