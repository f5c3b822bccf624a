// linear_scan.hip — recurrences that are linear in a matrix state, with a decay per key channel (or one per head), for any mixture
// of prompt portions and decoded tokens. Per head, with S [dim, vdim] fp32 in the sequence's state slot:
//     plain:   S <- diag(a) S + k v^T;   o = S^T q                       (gated linear attention; state-space duality: a scalar a)
//     bonus u: o = (S + diag(u) k v^T)^T q;   S <- diag(a) S + k v^T      (time mixing: the decay acts after the read-out)
//   optionally k times a factor per (token, head), and o + D v with D per head.
//
// Prompts run in tiles of 16 tokens (the plan's tiles: runs of up to 16 consecutive tokens of one portion). Inside a tile the
// recurrence unrolls into products whose decays are all products of factors in [0, 1], so nothing is divided and nothing overflows,
// however strong the decay:
//     o_t = (q_t * A_(0..t])^T S0 + sum_(s <= t) M[t][s] v_s,     M[t][s] = sum_i q_t[i] k_s[i] prod_(s < m <= t) a_m[i]
//     S   = diag(A_(0..n]) S0 + sum_s (k_s * A_(s..n]) v_s^T
//   (with the bonus the products end at t - 1 and M[t][t] = sum_i q_t[i] u[i] k_t[i]).
//   swl_linear_chunks: one workgroup per (tile, head), all tiles at once: decayed queries and keys, the tile's total decay and M.
//                      Running products over the tokens; nothing here depends on the state.
//   swl_linear_scan:   one workgroup (4 waves) per (portion, head, 16 state columns): walks the portion's tiles. The state lives in
//                      the accumulators of the fp32 matrix core (16x16x4: exact fp32 operands): the rows are shared out over the
//                      waves, and an accumulator tile is, register by register, the B operand of the read-out when the reduction
//                      index is taken in the order 4 (lane / 16) + r — so the state never moves. The waves' partial outputs meet
//                      in LDS, one barrier per tile; the next tiles' operands are requested ahead, as whole 1 KiB blocks. A head's
//                      column shares read the same operands: they run on one XCD (whose L2 holds them), neighbouring heads on the
//                      next, so that the long portions of a step that mixes prompts and decoded tokens spread over the chip: with
//                      the portion as the fastest grid index the two prompts beside 30 decoded tokens met on 16 CUs of two XCDs.
//                      2 x 1000 + 30 tokens, 8 heads of 128 x 128: 360 -> 85 us. 32 columns a workgroup (half the operand reads)
//                      took 136 us there and 106 instead of 99 us at 11 x 333 tokens, 16 heads.
//                      A step of few portions leaves the chip idle behind a chain of 1.3 us a tile. Its portions are cut into segments of
//                      several tiles: linear_segments_kernel walks every segment's state alone (from zero; the first from the portion's),
//                      without queries or outputs, and the scan's workgroup of a segment starts from those states, each taken on by
//                      the decays of the segments after it. 1 x 2000 tokens, 8 heads of 128 x
//                      128: 169 -> 45 us; 2 x 1000 + 30: 81 -> 52 us (both launches).
//   swl_linear_step:   steps whose portions are single tokens (decode): one workgroup per (sequence, head) streams the state once
//                      and finishes the head — read-out, RMS norm over the head, weight, gate — in the same launch.
// Everything after the loads of q, k, v is fp32.
#include "gemm_tile.h"

#include <algorithm>

namespace swl {

constexpr int kLsTile = 16;
constexpr int kLsThreads = 256;
constexpr int kLsWaves = kLsThreads / 64;
constexpr int kLsMaxDim = 320;          // padded key channels: 3 * 16 * 320 floats of LDS

__device__ __forceinline__ float ls_silu(float z) { return z / (1.0f + expf(-z)); }

// What bounds it: its rows and blocks are 30 MB for 2030 tokens and 8 heads of 128 channels (6 us); with one channel a load, each waited for behind
// a division and a predicate, eight turns of that latency took 22 us. WIDE: a thread takes eight channels of a token, loaded without a
// predicate and all at once, queries and keys are worked on by different waves, and the products read four channels at a time.
template <typename T, bool BONUS, bool WIDE>
__global__ __launch_bounds__(kLsThreads) void linear_chunks_kernel(
    float *qd, float *kd, float *total, float *intra, const T *q, int64_t q_stride, const T *k, int64_t k_stride, const float *decay,
    int64_t decay_stride, int per_channel, const float *k_scale, const float *bonus, float q_scale, const int32_t *tile_row0,
    const int32_t *tile_cnt, int H, int rep, int d, int dp) {
    extern __shared__ float lds[];
    float *qs = lds, *ks = qs + kLsTile * dp, *as = ks + kLsTile * dp;      // [16][dp] each
    const int tile = blockIdx.x, h = blockIdx.y;
    const int row0 = tile_row0[tile], cnt = tile_cnt[tile];
    const int64_t at = static_cast<int64_t>(tile) * H + h;
    const int qk0 = (h / rep) * d;
    // tokens beyond the tile's and channels beyond the head: q = k = 0, decay 1
    if constexpr (WIDE) {       // (whole blocks of 64 channels, rows on 16 bytes)
        const int per = d >> 3;
        for (int i = threadIdx.x; i < kLsTile * per; i += kLsThreads) {
            const int t = i / per, e = (i - t * per) * 8;
            const int64_t row = row0 + min(t, cnt - 1);
            const vec8_t<T> q8 = load8(q + row * q_stride + qk0 + e), k8 = load8(k + row * k_stride + qk0 + e);
            const float *ap = decay + row * decay_stride;
            float4_t a0, a1;
            if (per_channel) {      // (uniform)
                a0 = *reinterpret_cast<const float4_t *>(ap + h * d + e);
                a1 = *reinterpret_cast<const float4_t *>(ap + h * d + e + 4);
            } else {
                const float a = ap[h];
                a0 = a1 = float4_t{a, a, a, a};
            }
            const float scale = k_scale ? k_scale[row * H + h] : 1.f;
            const bool ok = t < cnt;
            float4_t o[6];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                o[c >> 2][c & 3] = ok ? to_f(q8[c]) * q_scale : 0.f;
                const float kv = to_f(k8[c]);
                o[2 + (c >> 2)][c & 3] = ok ? k_scale ? kv * scale : kv : 0.f;
                o[4 + (c >> 2)][c & 3] = ok ? c < 4 ? a0[c & 3] : a1[c & 3] : 1.f;
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                *reinterpret_cast<float4_t *>(qs + t * dp + e + 4 * c) = o[c];
                *reinterpret_cast<float4_t *>(ks + t * dp + e + 4 * c) = o[2 + c];
                *reinterpret_cast<float4_t *>(as + t * dp + e + 4 * c) = o[4 + c];
            }
        }
    }
    for (int i = threadIdx.x; !WIDE && i < kLsTile * dp; i += kLsThreads) {
        const int t = i / dp, e = i - t * dp;
        float qv = 0.f, kv = 0.f, av = 1.f;
        if (t < cnt && e < d) {
            const int64_t row = row0 + t;
            qv = to_f(q[row * q_stride + qk0 + e]) * q_scale;
            kv = to_f(k[row * k_stride + qk0 + e]);
            if (k_scale) kv *= k_scale[row * H + h];
            av = decay[row * decay_stride + (per_channel ? h * d + e : h)];
        }
        qs[i] = qv;
        ks[i] = kv;
        as[i] = av;
    }
    __syncthreads();
    // (WIDE: queries first, then keys: whole waves of either)
    for (int at_e = threadIdx.x; at_e < (WIDE ? 2 : 1) * dp; at_e += kLsThreads) {
        const bool of_q = !WIDE || at_e < dp, of_k = !WIDE || !of_q;
        const int e = of_q ? at_e : at_e - dp;
        const float *xs = of_q ? qs : ks;
        float x[kLsTile], a[kLsTile];
#pragma unroll
        for (int t = 0; t < kLsTile; ++t) {
            x[t] = xs[t * dp + e];
            a[t] = as[t * dp + e];
        }
        if (of_q) {
            float *qo = qd + at * kLsTile * dp + (e >> 4) * 256 + (e & 15);     // 16 x 16 blocks [channels / 16][token][channel]
            float p = 1.f;
#pragma unroll
            for (int t = 0; t < kLsTile; ++t) {
                if constexpr (BONUS) {
                    qo[t * 16] = x[t] * p;
                    p *= a[t];
                } else {
                    p *= a[t];
                    qo[t * 16] = x[t] * p;
                }
            }
            total[at * dp + e] = p;
        }
        if (!of_k) continue;
        if constexpr (!WIDE) {
#pragma unroll
            for (int t = 0; t < kLsTile; ++t) x[t] = ks[t * dp + e];
        }
        float p = 1.f;
#pragma unroll
        for (int t = kLsTile - 1; t >= 0; --t) {
            x[t] *= p;
            p *= a[t];
        }
        float *ko = kd + (at * dp + e) * kLsTile;
#pragma unroll
        for (int t = 0; t < kLsTile; t += 4) *reinterpret_cast<float4_t *>(ko + t) = float4_t{x[t], x[t + 1], x[t + 2], x[t + 3]};
    }
    // M: thread (s, g) takes key token s and the channels g, g + 16, ...; sixteen neighbouring lanes share an s
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s = threadIdx.x >> 4, g = threadIdx.x & 15;
    float acc[kLsTile];
#pragma unroll
    for (int t = 0; t < kLsTile; ++t) acc[t] = 0.f;
    auto products = [&](auto wc) {      // (a wave's key tokens are 4 wave .. 4 wave + 3)
        constexpr int FIRST = 4 * decltype(wc)::value;
        for (int e = 4 * g; e < d; e += 64) {
            float4_t p = *reinterpret_cast<const float4_t *>(ks + s * dp + e), diag = {};
            if constexpr (BONUS) {
#pragma unroll
                for (int c = 0; c < 4; ++c) diag[c] = p[c] * bonus[h * d + e + c];
            }
#pragma unroll
            for (int t = FIRST; t < kLsTile; ++t) {
                const float4_t a = *reinterpret_cast<const float4_t *>(as + t * dp + e), qv = *reinterpret_cast<const float4_t *>(qs + t * dp + e);
                const bool past = t >= FIRST + 4 || t > s, now = t >= FIRST + 4 || t >= s;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if constexpr (BONUS) {
                        acc[t] = fmaf(qv[c], past ? p[c] : now ? diag[c] : 0.f, acc[t]);
                        p[c] = past ? p[c] * a[c] : p[c];
                    } else {
                        p[c] = past ? p[c] * a[c] : p[c];
                        acc[t] = fmaf(qv[c], now ? p[c] : 0.f, acc[t]);
                    }
                }
            }
        }
    };
    if constexpr (WIDE) {
        switch (wave) {
        case 0: products(std::integral_constant<int, 0>{}); break;
        case 1: products(std::integral_constant<int, 1>{}); break;
        case 2: products(std::integral_constant<int, 2>{}); break;
        default: products(std::integral_constant<int, 3>{}); break;
        }
    }
    for (int e = g; !WIDE && e < d; e += 16) {
        float p = ks[s * dp + e];
        float diag = 0.f;
        if constexpr (BONUS) diag = p * bonus[h * d + e];
#pragma unroll
        for (int t = 0; t < kLsTile; ++t) {
            if (t >= 4 * wave) {        // (wave-uniform: the wave's key tokens are 4 wave .. 4 wave + 3)
                const float a = as[t * dp + e], qv = qs[t * dp + e];
                if constexpr (BONUS) {
                    acc[t] = fmaf(qv, t > s ? p : t == s ? diag : 0.f, acc[t]);
                    if (t > s) p *= a;
                } else {
                    if (t > s) p *= a;
                    acc[t] = fmaf(qv, t >= s ? p : 0.f, acc[t]);
                }
            }
        }
    }
    float mine = 0.f;
#pragma unroll
    for (int t = 0; t < kLsTile; ++t) {
        const float v = group_allreduce_sum<16>(acc[t]);
        if (g == t) mine = v;
    }
    intra[at * 256 + (s & 3) * 64 + (s >> 2) * 16 + g] = mine;      // (t = g) as the scan's waves read it: wave s % 4, lane 16 (s / 4) + t
}

__device__ __forceinline__ float4_t mfma_f32_16x16x4(float a, float b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// What a wave needs of one tile. Loaded without predicates (addresses are clamped, what does not count is masked at its use): a
// predicated load would be waited for on the spot, and the point is to have a tile's loads in flight while others are computed.
template <typename T, int TW>
struct LsOperands {
    float4_t q[TW], k[TW];
    float a[TW], m;
    T v[4];
};

// TW: 16-row state tiles per wave; AHEAD: tiles requested ahead of the one being computed
template <typename T, int TW, int AHEAD>
__global__ __launch_bounds__(kLsThreads) void linear_scan_kernel(
    float *o, int64_t o_stride, const float *qd, const float *kd, const float *total, const float *intra, const T *v,
    int64_t v_stride, const float *dskip, float *state, int64_t slot_stride, int64_t s_off, const int32_t *seq_row0,
    const int32_t *seq_cnt, const int32_t *seq_tile0, const int32_t *tok_pos, const int32_t *tok_state, int H, int d, int dp,
    int dv, int shares, int units, int segments, int seg_tiles, const float *seg_states, const float *seg_decays) {
    __shared__ float red[2][kLsWaves][256];
    const int id = blockIdx.x, unit = (id & 7) + 8 * ((id >> 3) / (shares * segments));     // (portion, head); id % 8 is the XCD
    if (unit >= units) return;
    const int seq = unit / H, h = unit - seq * H, col0 = ((id >> 3) % shares) * 16, seg = (id >> 3) / shares % segments;
    // this workgroup's segment of the portion (the whole portion without segments)
    const int first = seg * seg_tiles * kLsTile, all = seq_cnt[seq];
    if (first >= all) return;
    const bool last = all - first <= seg_tiles * kLsTile;
    const int start = seq_row0[seq], row0 = start + first, cnt = last ? all - first : seg_tiles * kLsTile;
    const int tile0 = seq_tile0[seq] + seg * seg_tiles;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int li = lane & 15, lq = lane >> 4;
    const int col = col0 + li;
    const bool okc = col < dv;
    const int ntiles = dp >> 4;
    float *S = state + static_cast<int64_t>(tok_state[start] >> 1) * slot_stride + s_off + static_cast<int64_t>(h) * d * dv;
    const bool fresh = tok_pos[start] == 0;     // a sequence starts from the zero state whatever the slot held
    // a portion of several segments: its own state is in the scratch too (the last segment may be done with the slot by now)
    const int64_t states = static_cast<int64_t>(d) * dv;
    const float *from_seg = seg_states + static_cast<int64_t>(unit) * (segments + 1) * states;
    const bool cut = !(last && seg == 0);
    const float *begin = !cut ? S : seg == 0 ? from_seg : from_seg + states;
    float4_t st[TW];        // st[j][r] = S[16 (wave TW + j) + 4 lq + r][col]
#pragma unroll
    for (int j = 0; j < TW; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (wave * TW + j) + 4 * lq + r;
            st[j][r] = ((cut || !fresh) && okc && row < d) ? begin[static_cast<int64_t>(row) * dv + col] : 0.f;
        }
    }
    for (int g = 1; g < seg; ++g) {
#pragma unroll
        for (int j = 0; j < TW; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * (wave * TW + j) + 4 * lq + r;
                if (okc && row < d)
                    st[j][r] = fmaf(st[j][r], seg_decays[(static_cast<int64_t>(unit) * segments + g) * dp + row],
                                    from_seg[(g + 1) * states + static_cast<int64_t>(row) * dv + col]);
            }
        }
    }
    const float dh = dskip ? dskip[h] : 0.f;
    const int nt = (cnt + kLsTile - 1) / kLsTile;
    const T *vcol = v + static_cast<int64_t>(row0) * v_stride + static_cast<int64_t>(h) * dv + (okc ? col : dv - 1);
    auto load = [&](int i, LsOperands<T, TW> &f) {
        i = min(i, nt - 1);
        const int64_t at = static_cast<int64_t>(tile0 + i) * H + h;
#pragma unroll
        for (int j = 0; j < TW; ++j) {
            const int tl = min(wave * TW + j, ntiles - 1);
            f.q[j] = *reinterpret_cast<const float4_t *>(qd + at * kLsTile * dp + tl * 256 + li * 16 + 4 * lq);
            f.k[j] = *reinterpret_cast<const float4_t *>(kd + (at * dp + 16 * tl + li) * kLsTile + 4 * lq);
            f.a[j] = total[at * dp + 16 * tl + 4 * lq + (li & 3)];
        }
        f.m = intra[at * 256 + wave * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) f.v[r] = vcol[static_cast<int64_t>(min(i * kLsTile + 4 * lq + r, cnt - 1)) * v_stride];
    };
    auto compute = [&](int i, const LsOperands<T, TW> &f) {
        float vv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) vv[r] = (i * kLsTile + 4 * lq + r < cnt && okc) ? to_f(f.v[r]) : 0.f;
        // this wave's share of the outputs: its state rows, and the in-tile keys 4 lq + wave
        float4_t part[TW + 1];
        part[TW] = mfma_f32_16x16x4(f.m, wave == 0 ? vv[0] : wave == 1 ? vv[1] : wave == 2 ? vv[2] : vv[3],
                                    float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int j = 0; j < TW; ++j) part[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int j = 0; j < TW; ++j) part[j] = mfma_f32_16x16x4(f.q[j][r], st[j][r], part[j]);
        }
#pragma unroll
        for (int j = 0; j < TW; ++j) {
            mfma_results_ready<8>(st[j]);
            st[j] *= quad_values(f.a[j]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int j = 0; j < TW; ++j) st[j] = mfma_f32_16x16x4(f.k[j][r], vv[r], st[j]);
        }
        float4_t out = part[TW];
        mfma_results_ready<8>(out);
#pragma unroll
        for (int j = 0; j < TW; ++j) {
            mfma_results_ready<8>(part[j]);
            if (wave * TW + j < ntiles) out += part[j];     // (wave-uniform; a row tile beyond the state repeats the last one)
        }
        if (dskip && wave == 0) {       // (v of this lane: token 4 lq + r, column li — the layout of the result)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = fmaf(dh, vv[r], out[r]);
        }
        float *rb = &red[i & 1][0][0];
        *reinterpret_cast<float4_t *>(rb + wave * 256 + lane * 4) = out;
        __syncthreads();        // (two buffers: the next tile's partials go to the other one)
        const int t = threadIdx.x >> 4, c = threadIdx.x & 15;
        const int from = ((t >> 2) * 16 + c) * 4 + (t & 3);
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < kLsWaves; ++w) sum += rb[w * 256 + from];
        const int tok = i * kLsTile + t;
        if (tok < cnt && col0 + c < dv) o[(row0 + tok) * o_stride + static_cast<int64_t>(h) * dv + col0 + c] = sum;
    };
    LsOperands<T, TW> f[AHEAD + 1];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) load(a, f[a]);
    int i = 0;
    for (; i + AHEAD < nt; i += AHEAD + 1) {
#pragma unroll
        for (int a = 0; a <= AHEAD; ++a) {
            load(i + a + AHEAD, f[(a + AHEAD) % (AHEAD + 1)]);
            compute(i + a, f[a]);
        }
    }
#pragma unroll
    for (int a = 0; a < AHEAD; ++a)
        if (i + a < nt) compute(i + a, f[a]);       // (uniform)
    if (!last) return;
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        float4_t s = st[j];
        mfma_results_ready<8>(s);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (wave * TW + j) + 4 * lq + r;
            if (okc && row < d) S[static_cast<int64_t>(row) * dv + col] = s[r];
        }
    }
}

// The states that the segments of cut portions leave when each starts from zero (segment 0: from the portion's state): of unit u
// seg_states[u][0] the portion's state, [1 + g] segment g's, seg_decays[u][g] the segment's total decay per row. Waves don't meet.
template <typename T, int TW>
__global__ __launch_bounds__(kLsThreads) void linear_segments_kernel(
    float *seg_states, float *seg_decays, const float *kd, const float *total, const T *v, int64_t v_stride, const float *state,
    int64_t slot_stride, int64_t s_off, const int32_t *seq_row0, const int32_t *seq_cnt, const int32_t *seq_tile0,
    const int32_t *tok_pos, const int32_t *tok_state, int H, int d, int dp, int dv, int shares, int units, int segments, int seg_tiles) {
    constexpr int AHEAD = 4;
    const int id = blockIdx.x, unit = (id & 7) + 8 * ((id >> 3) / (shares * segments));
    if (unit >= units) return;
    const int seq = unit / H, h = unit - seq * H, col0 = ((id >> 3) % shares) * 16, seg = (id >> 3) / shares % segments;
    const int first = seg * seg_tiles * kLsTile, all = seq_cnt[seq];
    if (all - first <= seg_tiles * kLsTile) return;     // a portion's last segment (an only one too) leaves its state to the scan
    const int start = seq_row0[seq], tile0 = seq_tile0[seq] + seg * seg_tiles;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int li = lane & 15, lq = lane >> 4, col = col0 + li, ntiles = dp >> 4;
    const bool okc = col < dv;
    const int64_t states = static_cast<int64_t>(d) * dv;
    const float *S = state + static_cast<int64_t>(tok_state[start] >> 1) * slot_stride + s_off + static_cast<int64_t>(h) * states;
    const bool fresh = tok_pos[start] == 0;
    float *out = seg_states + (static_cast<int64_t>(unit) * (segments + 1) + seg + 1) * states;
    float4_t st[TW], decay[TW];
#pragma unroll
    for (int j = 0; j < TW; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (wave * TW + j) + 4 * lq + r;
            const bool ok = okc && row < d;
            st[j][r] = seg == 0 && !fresh && ok ? S[static_cast<int64_t>(row) * dv + col] : 0.f;
            if (seg == 0 && ok) (out - states)[static_cast<int64_t>(row) * dv + col] = st[j][r];
            decay[j][r] = 1.f;
        }
    }
    struct Operands {
        float4_t k[TW];
        float a[TW];
        T v[4];
    };
    const T *vcol = v + static_cast<int64_t>(start + first) * v_stride + static_cast<int64_t>(h) * dv + (okc ? col : dv - 1);
    auto load = [&](int i, Operands &f) {
        i = min(i, seg_tiles - 1);
        const int64_t at = static_cast<int64_t>(tile0 + i) * H + h;
#pragma unroll
        for (int j = 0; j < TW; ++j) {
            const int tl = min(wave * TW + j, ntiles - 1);
            f.k[j] = *reinterpret_cast<const float4_t *>(kd + (at * dp + 16 * tl + li) * kLsTile + 4 * lq);
            f.a[j] = total[at * dp + 16 * tl + 4 * lq + (li & 3)];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) f.v[r] = vcol[static_cast<int64_t>(i * kLsTile + 4 * lq + r) * v_stride];
    };
    Operands f[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) load(a, f[a]);
    for (int i = 0; i < seg_tiles; i += AHEAD) {
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            if (i + a < seg_tiles) {
#pragma unroll
                for (int j = 0; j < TW; ++j) {
                    mfma_results_ready<8>(st[j]);
                    const float4_t by = quad_values(f[a].a[j]);
                    st[j] *= by;
                    decay[j] *= by;
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float vv = okc ? to_f(f[a].v[r]) : 0.f;       // (every tile of these segments is full)
#pragma unroll
                    for (int j = 0; j < TW; ++j) st[j] = mfma_f32_16x16x4(f[a].k[j][r], vv, st[j]);
                }
                load(i + a + AHEAD, f[a]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        float4_t s = st[j];
        mfma_results_ready<8>(s);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (wave * TW + j) + 4 * lq + r;
            if (row >= d) continue;
            if (okc) out[static_cast<int64_t>(row) * dv + col] = s[r];
            if (col == 0) seg_decays[(static_cast<int64_t>(unit) * segments + seg) * dp + row] = decay[j][r];
        }
    }
}

// ---- heads of 64 or 128 key channels: 64 columns a workgroup, 16 of all rows a wave ----------------------------------------------------
// In the walks above four waves have a quarter of the rows each and add their partial outputs up through LDS once a tile, and every 16 columns read all
// operands: 2.5 us a tile with two workgroups on a CU, a fifth of it matrix steps. Here a wave keeps all rows of its columns (NT accumulator
// tiles), and a tile's operands come to LDS once for four of them, two tiles ahead. (Straight to every wave's registers they took a CU's
// address units as long as the matrix steps: 1.6 us a tile.) The fp32 matrix core bounds it where every SIMD has a wave: 8 NT + 4 steps of 32 cycles.
struct LwParams {
    float *o;
    const float *qd, *kd, *total, *intra;
    const void *v;
    const float *dskip;
    float *state, *seg_states, *seg_decays;
    const int32_t *seq_row0, *seq_cnt, *seq_tile0, *tok_pos, *tok_state;
    int64_t o_stride, v_stride, slot_stride, s_off;
    int H, dv, shares, num_seqs, segments, seg_tiles;       // shares: of 64 columns
    Divisor span;           // tokens of a segment
};

// STATES false: the scan. true: the states that a cut portion's segments leave (linear_segments_kernel).
template <typename T, int NT, bool STATES>
__global__ __launch_bounds__(kLsThreads, 2) void linear_scan_wide_kernel(LwParams p) {
    constexpr int D = 16 * NT, SZ = sizeof(T), VB = SZ;     // (a tile's values: 16 rows of 64 columns, a KiB each fetch)
    constexpr int Q = 0, K = STATES ? 0 : NT, V = K + NT, A = V + VB, M = A + 1, FETCHES = M + (STATES ? 0 : 1), EACH = (FETCHES + 3) / 4;
    constexpr int SLOT = FETCHES * 1024, SLOTS = 3;
    __shared__ __attribute__((aligned(16))) char smem[SLOTS * SLOT];
    // This workgroup's segment: those that there are, counted from the portions' lengths (a grid of as many for each portion as the longest has kept a step
    // of 2 prompts beside 30 decoded tokens busy with workgroups that leave at once: 34 us instead of 27, 8 heads of 128 x 128), (segment, head) on the XCDs in turn,
    // all columns of one on one XCD
    const int id = static_cast<int>(blockIdx.x >> 3), rest = id / p.shares, at = rest * 8 + static_cast<int>(blockIdx.x & 7), piece = at / p.H, h = at - piece * p.H;
    const int lane = threadIdx.x & 63, dv = p.dv;
    int seq = piece, seg = 0, all, start, tile_0;       // (the three arrays asked for together: each wait is one for memory, the caches are cold)
    if (p.segments > 1) {
        int before = 0;
        for (int s0 = 0;; s0 += 64) {
            if (s0 >= p.num_seqs) return;
            const int s = min(s0 + lane, p.num_seqs - 1), cnt_s = p.seq_cnt[s], row_s = p.seq_row0[s], tile_s = p.seq_tile0[s];
            const int mine = s0 + lane < p.num_seqs ? min(p.segments, static_cast<int>(divide(static_cast<unsigned>(cnt_s) + p.span.by - 1, p.span))) : 0;
            int scan = mine;
            for (int o = 1; o < 64; o <<= 1) {
                const int x = __shfl_up(scan, o, 64);
                if (lane >= o) scan += x;
            }
            const unsigned long long past = __ballot(before + scan > piece);
            if (past) {
                const int l = __builtin_ctzll(past);
                seq = s0 + l;
                seg = piece - before - __builtin_amdgcn_readlane(scan - mine, l);
                all = __builtin_amdgcn_readlane(cnt_s, l), start = __builtin_amdgcn_readlane(row_s, l), tile_0 = __builtin_amdgcn_readlane(tile_s, l);
                break;
            }
            before += __builtin_amdgcn_readlane(scan, 63);
        }
    } else {
        if (piece >= p.num_seqs) return;
        const int cnt_s = p.seq_cnt[seq], row_s = p.seq_row0[seq], tile_s = p.seq_tile0[seq];
        all = __builtin_amdgcn_readfirstlane(cnt_s), start = __builtin_amdgcn_readfirstlane(row_s), tile_0 = __builtin_amdgcn_readfirstlane(tile_s);
    }
    const int unit = seq * p.H + h, first = seg * p.seg_tiles * kLsTile;
    if (first >= all) return;
    const bool last = all - first <= p.seg_tiles * kLsTile, cut = !(last && seg == 0);
    if (STATES && last) return;     // a portion's last segment (an only one too) leaves its state to the scan
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lq = lane >> 4;
    const int col0 = (id - rest * p.shares) * 64, cols = min(64, dv - col0), own = col0 + wave * 16 + li, col = min(own, dv - 1);
    const bool okc = own < dv;
    const int row0 = start + first, cnt = last ? all - first : p.seg_tiles * kLsTile, nt = (cnt + kLsTile - 1) / kLsTile;
    const int64_t tile0 = (tile_0 + static_cast<int64_t>(seg) * p.seg_tiles) * p.H + h;
    const int64_t states = static_cast<int64_t>(D) * dv;
    float *S = p.state + static_cast<int64_t>(p.tok_state[start] >> 1) * p.slot_stride + p.s_off + h * states;
    const bool fresh = p.tok_pos[start] == 0;       // a sequence starts from the zero state whatever the slot held
    float *const from_seg = p.seg_states + static_cast<int64_t>(unit) * (p.segments + 1) * states;

    // ---- fetches: KiB wave, wave + 4, ... of a tile's [queries | keys | values | decays | products] (as they are read: 16 bytes a lane); what is too
    // many repeats the decays, rows beyond the portion and tiles beyond the last are zeros without a memory access --------------------
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    const int64_t vb = p.v_stride * SZ;
    int4v rsrc[EACH];       // (of the next tile that is asked for)
    int64_t step[EACH];
    int to[EACH], v_row[EACH];
    unsigned off[EACH];
    auto v_bytes = [&](int rows) { return rows > 0 ? static_cast<int>(min(rows, kLsTile) * vb - vb) + cols * SZ : 0; };
#pragma unroll
    for (int n = 0; n < EACH; ++n) {
        const int f = wave + 4 * n < FETCHES ? wave + 4 * n : A;
        to[n] = f * 1024;
        v_row[n] = -1;
        off[n] = lane * 16;
        if (f < V) {
            rsrc[n] = tile_rsrc(reinterpret_cast<const char *>(f < K ? p.qd : p.kd) + (tile0 * NT + (f < K ? f : f - K)) * 1024, 1024);
            step[n] = static_cast<int64_t>(p.H) * NT * 1024;
            off[n] = li * 64 + lq * 16;
        } else if (f < A) {
            constexpr int PER = 4 * SZ;     // lanes of a row
            v_row[n] = (f - V) * (64 / PER);
            rsrc[n] = tile_rsrc(static_cast<const char *>(p.v) + (row0 + v_row[n]) * vb + (static_cast<int64_t>(h) * dv + col0) * SZ, v_bytes(cnt - v_row[n]));
            step[n] = kLsTile * vb;
            off[n] = static_cast<unsigned>(lane / PER * vb) + lane % PER * 16;
        } else if (f == A) {
            rsrc[n] = tile_rsrc(reinterpret_cast<const char *>(p.total + tile0 * D), D * 4);
            step[n] = static_cast<int64_t>(p.H) * D * 4;
        } else {
            rsrc[n] = tile_rsrc(reinterpret_cast<const char *>(p.intra + tile0 * 256), 1024);
            step[n] = static_cast<int64_t>(p.H) * 1024;
        }
    }
    int asked = 0;
    unsigned slot_to = lds0;
    auto ask = [&](int n) { tile_fetch(rsrc[n], off[n], 0, slot_to + to[n]); };
    auto asked_all = [&]() {        // on to the next tile
        ++asked;
        slot_to = slot_to == lds0 + (SLOTS - 1) * SLOT ? lds0 : slot_to + SLOT;
#pragma unroll
        for (int n = 0; n < EACH; ++n) {
            const uint64_t at = (static_cast<uint64_t>(static_cast<unsigned>(rsrc[n][1])) << 32 | static_cast<unsigned>(rsrc[n][0])) + step[n];
            rsrc[n][0] = static_cast<int>(at), rsrc[n][1] = static_cast<int>(at >> 32);
        }
        if (asked >= nt - 1) {
#pragma unroll
            for (int n = 0; n < EACH; ++n) rsrc[n][2] = asked >= nt ? 0 : v_row[n] < 0 ? rsrc[n][2] : v_bytes(cnt - asked * kLsTile - v_row[n]);
        }
    };
#pragma unroll
    for (int i = 0; i < SLOTS - 1; ++i) {
#pragma unroll
        for (int n = 0; n < EACH; ++n) ask(n);
        asked_all();
    }

    // ---- the state in front of the segment: st[j][r] = S[16 j + 4 lq + r][col] ---------------------------------------------------------
    float4_t st[NT], decay[STATES ? NT : 1];
    const int lane_at = 4 * lq * dv + col;
    auto load = [&](const float *s, float4_t (&x)[NT]) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[j][r] = s[lane_at + (16 * j + r) * dv];
    };
    const float *begin = STATES || !cut ? S : seg == 0 ? from_seg : from_seg + states;
    if (STATES ? seg > 0 || fresh : !cut && fresh) {
#pragma unroll
        for (int j = 0; j < NT; ++j) st[j] = float4_t{0.f, 0.f, 0.f, 0.f};
    } else {
        load(begin, st);
    }
    if constexpr (STATES) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            decay[j] = float4_t{1.f, 1.f, 1.f, 1.f};
            if (seg == 0 && okc) {      // (the last segment may be done with the slot before the first one's scan starts)
#pragma unroll
                for (int r = 0; r < 4; ++r) from_seg[lane_at + (16 * j + r) * dv] = st[j][r];
            }
        }
    } else {
        // each segment's own state behind what came before it, the next one asked for beside it
        const float *by = p.seg_decays + static_cast<int64_t>(unit) * p.segments * D + 4 * lq;
        float4_t more[2][NT], b[2][NT];
        auto load_segment = [&](int g, float4_t (&x)[NT], float4_t (&y)[NT]) {
            load(from_seg + (g + 1) * states, x);
#pragma unroll
            for (int j = 0; j < NT; ++j) y[j] = *reinterpret_cast<const float4_t *>(by + g * D + 16 * j);
        };
        auto behind = [&](const float4_t (&x)[NT], const float4_t (&y)[NT]) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) st[j][r] = fmaf(st[j][r], y[j][r], x[j][r]);
        };
        if (seg > 1) load_segment(1, more[0], b[0]);
        for (int g = 1; g < seg; g += 2) {
            load_segment(min(g + 1, seg - 1), more[1], b[1]);
            behind(more[0], b[0]);
            if (g + 1 >= seg) break;
            load_segment(min(g + 2, seg - 1), more[0], b[0]);
            behind(more[1], b[1]);
        }
    }
    float dh = !STATES && p.dskip ? p.dskip[h] : 0.f;
    // (arrived before the walk: a wait for them inside it is one for all fetches that are on their way)
#pragma unroll
    for (int j = 0; j < NT; ++j) mfma_results_tie(st[j]);
    mfma_results_tie(dh);

    constexpr int STORES = STATES ? 0 : 4;
    unsigned slot_at = 0;
    for (int i = 0; i < nt; ++i) {
        // this tile's fetches have landed (behind them: the next tile's and the last tile's stores), everyone is done with the slot before
        __builtin_amdgcn_sched_barrier(0);
        if (i == 0) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(EACH) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(EACH + STORES) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const char *slot = smem + slot_at;
        float vv[4], m[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) vv[r] = to_f(*reinterpret_cast<const T *>(slot + V * 1024 + ((4 * lq + r) * 64 + wave * 16 + li) * SZ));
        if constexpr (!STATES) {
#pragma unroll
            for (int r = 0; r < 4; ++r) m[r] = *reinterpret_cast<const float *>(slot + M * 1024 + (r * 64 + lane) * 4);
        }
        float4_t q[2], k[2], a[2];
        auto read = [&](int j) {
            if constexpr (!STATES) q[j & 1] = *reinterpret_cast<const float4_t *>(slot + (Q + j) * 1024 + lane * 16);
            k[j & 1] = *reinterpret_cast<const float4_t *>(slot + (K + j) * 1024 + lane * 16);
            a[j & 1] = *reinterpret_cast<const float4_t *>(slot + A * 1024 + (16 * j + 4 * lq) * 4);
        };
        read(0);
        // (sums of 16 rows each, added up in the order of linear_scan_kernel's: one long sum a register has 1.1 times the error)
        float4_t part[NT], in_tile[4];
        if constexpr (!STATES) {
#pragma unroll
            for (int r = 0; r < 4; ++r) in_tile[r] = mfma_f32_16x16x4(m[r], vv[r], float4_t{0.f, 0.f, 0.f, 0.f});
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {      // (operands are read while the rows before are multiplied)
            if (j + 1 < NT) read(j + 1);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (STATES) decay[j] *= a[j & 1];
            float4_t next = st[j] * a[j & 1];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (!STATES) part[j] = mfma_f32_16x16x4(q[j & 1][r], st[j][r], r ? part[j] : float4_t{0.f, 0.f, 0.f, 0.f});
                next = mfma_f32_16x16x4(k[j & 1][r], vv[r], next);
                if (EACH <= NT ? r == 1 && j < EACH : r == 0 || r == 2) {       // (requests between the matrix steps)
                    const int n = EACH <= NT ? j : 2 * j + (r >> 1);
                    if (n < EACH) ask(n);
                }
            }
            st[j] = next;
            __builtin_amdgcn_sched_barrier(0);
        }
        asked_all();
        slot_at = slot_at == (SLOTS - 1) * SLOT ? 0 : slot_at + SLOT;
        if constexpr (STATES) {
            mfma_results_ready<8>(st[NT - 1]);
            continue;
        }
#pragma unroll
        for (int j = 0; j < NT - 1; ++j) mfma_results_tie(part[j]);
        mfma_results_ready<8>(part[NT - 1]);
        float4_t out = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float4_t sum = in_tile[c];
#pragma unroll
            for (int j = c * NT / 4; j < (c + 1) * NT / 4; ++j) sum += part[j];
            out += sum;
        }
        if (p.dskip) {
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = fmaf(dh, vv[r], out[r]);
        }
        // (stores that are always made, so that they can be counted; tokens beyond the portion's and columns beyond the head's are dropped)
        const int rows = min(kLsTile, cnt - i * kLsTile);
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            p.o + (row0 + static_cast<int64_t>(i) * kLsTile) * p.o_stride + static_cast<int64_t>(h) * dv, 0, static_cast<int>((rows - 1) * p.o_stride + dv) * 4, 0x00020000);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(out[r]), rsrc, okc ? static_cast<int>((4 * lq + r) * p.o_stride + own) * 4 : 0x7fffffff, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");      // (fetches of no tile write zeros to LDS)
    if (!STATES && !last) return;
#pragma unroll
    for (int j = 0; j < NT - 1; ++j) mfma_results_tie(st[j]);
    mfma_results_ready<8>(st[NT - 1]);
    float *const into = STATES ? from_seg + (seg + 1) * states : S;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        if (okc) {
#pragma unroll
            for (int r = 0; r < 4; ++r) into[lane_at + (16 * j + r) * dv] = st[j][r];
        }
        if constexpr (STATES) {
            if (own == 0) *reinterpret_cast<float4_t *>(p.seg_decays + (static_cast<int64_t>(unit) * p.segments + seg) * D + 16 * j + 4 * lq) = decay[j];
        }
    }
}

// One token per sequence. Thread (rg, cg) owns columns V cg .. V cg + V - 1 and the state rows rg, rg + R, ...
constexpr int kLsBatch = 8;     // state rows in flight per thread

template <typename T, int V, bool BONUS>
__global__ __launch_bounds__(kLsThreads) void linear_step_kernel(
    T *out, int64_t out_stride, float *y, int64_t y_stride, const T *q, int64_t q_stride, const T *k, int64_t k_stride, const T *v,
    int64_t v_stride, const float *decay, int64_t decay_stride, int per_channel, const float *k_scale, const float *bonus,
    float q_scale, const float *dskip, float *state, int64_t slot_stride, int64_t s_off, const int32_t *seq_row0,
    const int32_t *tok_pos, const int32_t *tok_state, int H, int rep, int d, int dv, const float *norm_w, int norm_head_stride,
    const T *gate, int64_t gate_stride, float eps, float mult) {
    extern __shared__ float lds[];
    const int ncg = (dv + V - 1) / V, R = kLsThreads / ncg;
    float *qs = lds, *ks = qs + d, *as = ks + d, *us = as + d, *os = us + d;     // [d] x 4, then [R][ncg * V]
    __shared__ float red[kLsWaves];
    const int seq = blockIdx.x, h = blockIdx.y;
    const int64_t row = seq_row0[seq];
    const int cg = threadIdx.x % ncg, rg = threadIdx.x / ncg;
    const bool live = rg < R;
    float *S = state + static_cast<int64_t>(tok_state[row] >> 1) * slot_stride + s_off + static_cast<int64_t>(h) * d * dv;
    const bool fresh = tok_pos[row] == 0;
    // the first rows of the state are requested before anything else
    float sv[kLsBatch][V];
    auto fetch = [&](int b) {
#pragma unroll
        for (int j = 0; j < kLsBatch; ++j) {
            const int e = b + rg + j * R;
#pragma unroll
            for (int c = 0; c < V; ++c) sv[j][c] = 0.f;
            if (live && !fresh && e < d) {
                const float *p = S + static_cast<int64_t>(e) * dv + cg * V;
                if constexpr (V == 4) {
                    const float4_t x = *reinterpret_cast<const float4_t *>(p);
#pragma unroll
                    for (int c = 0; c < 4; ++c) sv[j][c] = x[c];
                } else {
                    sv[j][0] = p[0];
                }
            }
        }
    };
    fetch(0);
    for (int e = threadIdx.x; e < d; e += kLsThreads) {
        qs[e] = to_f(q[row * q_stride + static_cast<int64_t>(h / rep) * d + e]) * q_scale;
        const float kv = to_f(k[row * k_stride + static_cast<int64_t>(h / rep) * d + e]);
        ks[e] = k_scale ? kv * k_scale[row * H + h] : kv;
        as[e] = decay[row * decay_stride + (per_channel ? h * d + e : h)];
        if constexpr (BONUS) us[e] = bonus[h * d + e];
    }
    float vv[V], acc[V];
#pragma unroll
    for (int c = 0; c < V; ++c) {
        vv[c] = live ? to_f(v[row * v_stride + static_cast<int64_t>(h) * dv + cg * V + c]) : 0.f;
        acc[c] = 0.f;
    }
    __syncthreads();
    for (int b = 0; b < d; b += kLsBatch * R) {
        if (b) fetch(b);
#pragma unroll
        for (int j = 0; j < kLsBatch; ++j) {
            const int e = b + rg + j * R;
            if (live && e < d) {
                const float qe = qs[e], ke = ks[e], ae = as[e];
                float x[V];
#pragma unroll
                for (int c = 0; c < V; ++c) {
                    const float kv = ke * vv[c];
                    if constexpr (BONUS) {
                        acc[c] = fmaf(qe, fmaf(us[e], kv, sv[j][c]), acc[c]);
                        x[c] = fmaf(ae, sv[j][c], kv);
                    } else {
                        x[c] = fmaf(ae, sv[j][c], kv);
                        acc[c] = fmaf(qe, x[c], acc[c]);
                    }
                }
                float *p = S + static_cast<int64_t>(e) * dv + cg * V;
                if constexpr (V == 4) *reinterpret_cast<float4_t *>(p) = float4_t{x[0], x[1], x[2], x[3]};
                else p[0] = x[0];
            }
        }
    }
    const int cols = ncg * V;       // (V divides dv: cols == dv)
    if (live) {
#pragma unroll
        for (int c = 0; c < V; ++c) os[rg * cols + cg * V + c] = acc[c];
    }
    __syncthreads();
    float ss = 0.f;
    for (int c = threadIdx.x; c < dv; c += kLsThreads) {
        float a = 0.f;
        for (int r = 0; r < R; ++r) a += os[r * cols + c];
        if (dskip) a = fmaf(dskip[h], to_f(v[row * v_stride + static_cast<int64_t>(h) * dv + c]), a);
        if (y) y[row * y_stride + static_cast<int64_t>(h) * dv + c] = a;
        os[c] = a;          // (column c is read and written by this thread only)
        ss += a * a;
    }
    if (!out) return;
    ss = wave_allreduce_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < kLsWaves; ++w) ss += red[w];
    const float r = mult / sqrtf(ss / static_cast<float>(dv) + eps);
    for (int c = threadIdx.x; c < dv; c += kLsThreads) {
        const int64_t hc = static_cast<int64_t>(h) * dv + c;
        out[row * out_stride + hc] = to_t<T>(os[c] * r * norm_w[static_cast<int64_t>(h) * norm_head_stride + c] *
                                             ls_silu(to_f(gate[row * gate_stride + hc])));
    }
}

} // namespace swl

extern "C" int swl_linear_chunks(float *qd, float *kd, float *total, float *intra, const void *q, int64_t q_stride, const void *k,
                                 int64_t k_stride, const float *decay, int64_t decay_stride, int32_t per_channel,
                                 const float *k_scale, const float *bonus, float q_scale, const int32_t *tile_row0,
                                 const int32_t *tile_cnt, int32_t num_tiles, int32_t num_heads, int32_t num_qk_heads, int32_t dim,
                                 int32_t dtype, swl_stream_t stream) {
    if (num_tiles < 0 || num_heads <= 0 || num_qk_heads <= 0 || num_heads % num_qk_heads || dim <= 0) return SWL_ERR_BAD_ARG;
    const int64_t width = static_cast<int64_t>(num_qk_heads) * dim;
    if (q_stride < width || k_stride < width || decay_stride < (per_channel ? static_cast<int64_t>(num_heads) * dim : num_heads))
        return SWL_ERR_BAD_ARG;
    if (num_tiles == 0) return SWL_OK;
    if (!qd || !kd || !total || !intra || !q || !k || !decay || !tile_row0 || !tile_cnt || !swl::aligned16(kd))
        return SWL_ERR_BAD_ARG;
    const int dp = (dim + 15) / 16 * 16;
    if (dp > swl::kLsMaxDim || num_heads > 65535) return SWL_ERR_UNSUPPORTED;
    const size_t lds = 3ull * swl::kLsTile * dp * sizeof(float);
    const dim3 grid(static_cast<unsigned>(num_tiles), static_cast<unsigned>(num_heads));
    SWL_DISPATCH_DTYPE3(dtype, T, {
        // (eight channels of q and k a load, four of the decay)
        const bool wide = dim % 64 == 0 && swl::aligned16(q) && swl::aligned16(k) && q_stride * sizeof(T) % 16 == 0 && k_stride * sizeof(T) % 16 == 0 &&
                          (!per_channel || (swl::aligned16(decay) && decay_stride % 4 == 0));
        auto kernel = wide ? (bonus ? swl::linear_chunks_kernel<T, true, true> : swl::linear_chunks_kernel<T, false, true>)
                           : (bonus ? swl::linear_chunks_kernel<T, true, false> : swl::linear_chunks_kernel<T, false, false>);
        hipLaunchKernelGGL(kernel, grid, dim3(swl::kLsThreads), lds, static_cast<hipStream_t>(stream), qd, kd, total, intra,
                           static_cast<const T *>(q), q_stride, static_cast<const T *>(k), k_stride, decay, decay_stride,
                           per_channel, k_scale, bonus, q_scale, tile_row0, tile_cnt, num_heads, num_heads / num_qk_heads, dim, dp);
    });
    return swl::check_launch();
}

/* Bytes of scratch that swl_linear_scan_segments needs. */
extern "C" size_t swl_linear_scan_scratch_bytes(int64_t num_seqs, int32_t num_heads, int32_t dim, int32_t vdim, int32_t segments) {
    if (segments <= 1) return 0;
    const size_t states = static_cast<size_t>(segments + 1) * dim * vdim, decays = static_cast<size_t>(segments) * ((dim + 15) / 16 * 16);
    return sizeof(float) * static_cast<size_t>(num_seqs) * num_heads * (states + decays);
}

/* num_tiles: of the step (bounds the segments that there are; 0: as many for each portion) */
extern "C" int swl_linear_scan_cut(float *o, int64_t o_stride, const float *qd, const float *kd, const float *total, const float *intra,
                                   const void *v, int64_t v_stride, const float *dskip, float *state, int64_t slot_stride, int64_t s_off,
                                   const int32_t *seq_row0, const int32_t *seq_cnt, const int32_t *seq_tile0, const int32_t *tok_pos,
                                   const int32_t *tok_state, int32_t num_seqs, int32_t num_heads, int32_t dim, int32_t vdim, int32_t segments,
                                   int32_t seg_tiles, int32_t num_tiles, float *scratch, int32_t dtype, swl_stream_t stream) {
    if (num_tiles < 0) return SWL_ERR_BAD_ARG;
    if (num_seqs < 0 || num_heads <= 0 || dim <= 0 || vdim <= 0 || segments < 1 || segments > 64) return SWL_ERR_BAD_ARG;
    if (segments > 1 && (seg_tiles < 1 || !scratch)) return SWL_ERR_BAD_ARG;
    if (segments == 1) seg_tiles = 1 << 26;     // (one segment holds every portion)
    const int64_t width = static_cast<int64_t>(num_heads) * vdim;
    if (o_stride < width || v_stride < width) return SWL_ERR_BAD_ARG;
    if (num_seqs == 0) return SWL_OK;
    if (!o || !qd || !kd || !total || !intra || !v || !state || !seq_row0 || !seq_cnt || !seq_tile0 || !tok_pos || !tok_state)
        return SWL_ERR_BAD_ARG;
    if (!swl::aligned16(qd) || !swl::aligned16(kd) || !swl::aligned16(total)) return SWL_ERR_BAD_ARG;
    const int dp = (dim + 15) / 16 * 16, shares = (vdim + 15) / 16;
    const int64_t units = static_cast<int64_t>(num_seqs) * num_heads, blocks = 8 * ((units + 7) / 8) * shares * segments;
    if (dp > swl::kLsMaxDim || num_heads > 65535 || shares > 65535 || blocks > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    const hipStream_t on = static_cast<hipStream_t>(stream);
    const int tw = (dp / 16 + swl::kLsWaves - 1) / swl::kLsWaves;       // 1 .. 5
    const dim3 grid(static_cast<unsigned>(blocks));
    float *seg_states = scratch, *seg_decays = scratch ? scratch + units * (segments + 1) * dim * vdim : nullptr;
    // Rows of values in whole aligned pieces of 16 bytes; states by 32-bit offsets, a tile's rows within 2 GiB
    const int64_t size = dtype == SWL_F32 ? 4 : 2;
    if ((dim == 64 || dim == 128) && swl::aligned16(v) && v_stride * size % 16 == 0 && vdim * size % 16 == 0 && static_cast<int64_t>(dim) * vdim < (1LL << 29) &&
        16 * v_stride * size < (1LL << 31) && 16 * o_stride * 4 < (1LL << 31) && (segments == 1 || swl::aligned16(scratch))) {
        const int wide = (vdim + 63) / 64;
        swl::LwParams p = {o, qd, kd, total, intra, v, dskip, state, seg_states, seg_decays, seq_row0, seq_cnt, seq_tile0, tok_pos, tok_state,
                           o_stride, v_stride, slot_stride, s_off, num_heads, vdim, wide, num_seqs, segments, seg_tiles,
                           swl::Divisor::of(static_cast<unsigned>(seg_tiles) * swl::kLsTile)};
        int64_t pieces = static_cast<int64_t>(num_seqs) * segments;
        if (num_tiles > 0) pieces = std::min<int64_t>(pieces, num_seqs + static_cast<int64_t>(num_tiles) / seg_tiles);
        const dim3 by_64(static_cast<unsigned>(8 * ((pieces * num_heads + 7) / 8) * wide));
        SWL_DISPATCH_DTYPE3(dtype, T, {
            if (segments > 1)
                hipLaunchKernelGGL(dim == 64 ? (swl::linear_scan_wide_kernel<T, 4, true>) : (swl::linear_scan_wide_kernel<T, 8, true>), by_64, dim3(swl::kLsThreads), 0, on, p);
            hipLaunchKernelGGL(dim == 64 ? (swl::linear_scan_wide_kernel<T, 4, false>) : (swl::linear_scan_wide_kernel<T, 8, false>), by_64, dim3(swl::kLsThreads), 0, on, p);
        });
        return swl::check_launch();
    }
#define SWL_LS(N)                                                                                                             \
    case N:                                                                                                                   \
        if (segments > 1)                                                                                                     \
            hipLaunchKernelGGL((swl::linear_segments_kernel<T, N>), grid, dim3(swl::kLsThreads), 0,                           \
                               static_cast<hipStream_t>(stream), seg_states, seg_decays, kd, total,                           \
                               static_cast<const T *>(v), v_stride, state, slot_stride, s_off, seq_row0, seq_cnt, seq_tile0,  \
                               tok_pos, tok_state, num_heads, dim, dp, vdim, shares, static_cast<int>(units), segments,       \
                               seg_tiles);                                                                                    \
        hipLaunchKernelGGL((swl::linear_scan_kernel<T, N, (N <= 2 ? 2 : 1)>), grid, dim3(swl::kLsThreads), 0,                 \
                           static_cast<hipStream_t>(stream), o, o_stride, qd, kd, total, intra,                               \
                           static_cast<const T *>(v), v_stride, dskip, state, slot_stride, s_off,                             \
                           seq_row0, seq_cnt, seq_tile0, tok_pos, tok_state, num_heads, dim, dp, vdim, shares,                \
                           static_cast<int>(units), segments, seg_tiles, seg_states, seg_decays);                             \
        break
    SWL_DISPATCH_DTYPE3(dtype, T, {
        switch (tw) {
            SWL_LS(1);
            SWL_LS(2);
            SWL_LS(3);
            SWL_LS(4);
            SWL_LS(5);
        default: return SWL_ERR_UNSUPPORTED;
        }
    });
#undef SWL_LS
    return swl::check_launch();
}

extern "C" int swl_linear_scan_segments(float *o, int64_t o_stride, const float *qd, const float *kd, const float *total, const float *intra,
                               const void *v, int64_t v_stride, const float *dskip, float *state, int64_t slot_stride,
                               int64_t s_off, const int32_t *seq_row0, const int32_t *seq_cnt, const int32_t *seq_tile0,
                               const int32_t *tok_pos, const int32_t *tok_state, int32_t num_seqs, int32_t num_heads, int32_t dim,
                               int32_t vdim, int32_t segments, int32_t seg_tiles, float *scratch, int32_t dtype,
                                        swl_stream_t stream) {
    return swl_linear_scan_cut(o, o_stride, qd, kd, total, intra, v, v_stride, dskip, state, slot_stride, s_off, seq_row0, seq_cnt, seq_tile0,
                               tok_pos, tok_state, num_seqs, num_heads, dim, vdim, segments, seg_tiles, 0, scratch, dtype, stream);
}

extern "C" int swl_linear_scan(float *o, int64_t o_stride, const float *qd, const float *kd, const float *total, const float *intra,
                               const void *v, int64_t v_stride, const float *dskip, float *state, int64_t slot_stride,
                               int64_t s_off, const int32_t *seq_row0, const int32_t *seq_cnt, const int32_t *seq_tile0,
                               const int32_t *tok_pos, const int32_t *tok_state, int32_t num_seqs, int32_t num_heads, int32_t dim,
                               int32_t vdim, int32_t dtype, swl_stream_t stream) {
    return swl_linear_scan_segments(o, o_stride, qd, kd, total, intra, v, v_stride, dskip, state, slot_stride, s_off, seq_row0, seq_cnt,
                                    seq_tile0, tok_pos, tok_state, num_seqs, num_heads, dim, vdim, 1, 0, nullptr, dtype, stream);
}

extern "C" int swl_linear_step(void *out, int64_t out_stride, float *y, int64_t y_stride, const void *q, int64_t q_stride,
                               const void *k, int64_t k_stride, const void *v, int64_t v_stride, const float *decay,
                               int64_t decay_stride, int32_t per_channel, const float *k_scale, const float *bonus, float q_scale,
                               const float *dskip, float *state, int64_t slot_stride, int64_t s_off, const int32_t *seq_row0,
                               const int32_t *tok_pos, const int32_t *tok_state, int32_t num_seqs, int32_t num_heads,
                               int32_t num_qk_heads, int32_t dim, int32_t vdim, const float *norm_w, int32_t norm_head_stride,
                               const void *gate, int64_t gate_stride, float eps, float mult, int32_t dtype, swl_stream_t stream) {
    if (num_seqs < 0 || num_heads <= 0 || num_qk_heads <= 0 || num_heads % num_qk_heads || dim <= 0 || vdim <= 0)
        return SWL_ERR_BAD_ARG;
    const int64_t wq = static_cast<int64_t>(num_qk_heads) * dim, wv = static_cast<int64_t>(num_heads) * vdim;
    if (q_stride < wq || k_stride < wq || v_stride < wv) return SWL_ERR_BAD_ARG;
    if (decay_stride < (per_channel ? static_cast<int64_t>(num_heads) * dim : num_heads)) return SWL_ERR_BAD_ARG;
    if (num_seqs == 0) return SWL_OK;
    if ((!out && !y) || !q || !k || !v || !decay || !state || !seq_row0 || !tok_pos || !tok_state) return SWL_ERR_BAD_ARG;
    if (out && (!norm_w || !gate || out_stride < wv || gate_stride < wv)) return SWL_ERR_BAD_ARG;
    if (y && y_stride < wv) return SWL_ERR_BAD_ARG;
    const bool quads = vdim % 4 == 0 && swl::aligned16(state) && slot_stride % 4 == 0 && s_off % 4 == 0;
    const int ncg = quads ? vdim / 4 : vdim;
    if (ncg > swl::kLsThreads || num_heads > 65535) return SWL_ERR_UNSUPPORTED;
    const int R = swl::kLsThreads / ncg;
    const size_t lds = (4ull * dim + static_cast<size_t>(R) * vdim) * sizeof(float);
    if (lds > 60 * 1024) return SWL_ERR_UNSUPPORTED;
    const dim3 grid(static_cast<unsigned>(num_seqs), static_cast<unsigned>(num_heads));
    SWL_DISPATCH_DTYPE3(dtype, T, {
        auto kernel = quads ? (bonus ? swl::linear_step_kernel<T, 4, true> : swl::linear_step_kernel<T, 4, false>)
                            : (bonus ? swl::linear_step_kernel<T, 1, true> : swl::linear_step_kernel<T, 1, false>);
        hipLaunchKernelGGL(kernel, grid, dim3(swl::kLsThreads), lds, static_cast<hipStream_t>(stream), static_cast<T *>(out),
                           out_stride, y, y_stride, static_cast<const T *>(q), q_stride, static_cast<const T *>(k), k_stride,
                           static_cast<const T *>(v), v_stride, decay, decay_stride, per_channel, k_scale, bonus, q_scale, dskip,
                           state, slot_stride, s_off, seq_row0, tok_pos, tok_state, num_heads, num_heads / num_qk_heads, dim, vdim,
                           norm_w, norm_head_stride, static_cast<const T *>(gate), gate_stride, eps, mult);
    });
    return swl::check_launch();
}
