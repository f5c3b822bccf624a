// span_attn.hip — the matrix-core attention of prompt portions over the paged pool, for heads that are not mixed
// (swl_masked_attn_tiles' masks, bias, slopes, cap, sink, gate; same pool layout, same arithmetic up to the order of sums).
//
// What bounds it: the matrix cores, which a value product in two 16-bit terms (hi + lo, so that a weight keeps 16 bits of its
// fp32 value) loads with 2 (D + 2 DV) flops per (row, key). A workgroup is four waves = 128 ROWS over one key head's pages, a row
// being one (query, query head) pair: every head of a kv group reads the same keys, so one staged page serves all of them
// (QT = 128 / heads queries a workgroup, heads rounded up to a power of two). Each wave owns RW rows:
//   S^T = K Q^T   A = keys from LDS, B = its query fragments (registers for the whole walk)
//   online softmax: lane l owns row l % RW, the 64 / RW lanes of a row hold its keys between them
//   O^T += V^T P^T  A = value columns from LDS, B = the score registers. Which key an A row of S^T takes is chosen so that a lane's
//                   eight scores of a step are eight CONSECUTIVE keys, which is what the B operand wants and what a page's
//                   transposed values hold in 16 bytes — no data moves between lanes.
// RW = 32 (mfma 32x32x16, four waves) reads the least LDS per flop; wide rows (latent attention: 576 + 512 elements) take RW = 16
// (mfma 16x16x32, eight waves), whose query fragments and accumulators fit 256 registers, so that two waves share a SIMD.
// Pages are staged by LDS-DMA (1 KiB per wave instruction, full lines) into two buffers with one barrier a stage; the swizzles that
// keep the 16-byte fragment reads off each other's banks are applied to the source addresses.
// A value that is NaN or infinite reaches every row of a workgroup that stages its page (a weight of 0 times it), as it does in the tiles
// of window_attn_mfma.hip: rows of the same portion whose queries come before it, at most 127 of them; never another sequence's.
// Measured against the 16-row kernel of window_attn_mfma.hip (bf16, one layer): 4 prompts of about 2000 tokens, 8 heads of 128 over 2 key
// heads 489 -> 99 us, with a bias by distance 535 -> 104 us (330 TFLOP/s of useful 2 (D + DV), 490 with the second value term); 8 latent
// heads of 576 + 512 over one, window 1024: 1115 -> 253 us; 11 prompts of 333 tokens, 16 heads of 128 over 4: 120 -> 28 us.
#include "attn_combine.h"
#include "swl_common.h"

namespace swl {

__device__ __forceinline__ float4_t mfma_step(vec8_t<f16> a, vec8_t<f16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mfma_step(vec8_t<bf16> a, vec8_t<bf16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float16_t mfma_step(vec8_t<f16> a, vec8_t<f16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float16_t mfma_step(vec8_t<bf16> a, vec8_t<bf16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

struct SpanParams {
    void *out;
    const void *q, *k_cache, *v_cache;
    const int32_t *block_table, *tok_seq, *tok_pos, *tok_start, *span_row0, *span_cnt;
    const float *rel, *sink, *slopes;
    const void *gate;
    float *part_o, *part_ml;
    int rel_len, num_spans, H, G, GV, window, mask_kind, max_blocks, out_f32, out_dim, qt;
    float scale, softcap;
    int64_t q_stride, block_stride, out_stride, gate_stride, num_tokens;
};

constexpr int kSpan = 32;       // tokens of a span at most (the plan's chunks)

// LDS position of a K row's 16-byte unit: the low bits of the unit index are flipped by a function of the key that differs over the
// 16 rows that a group of lanes reads (rows are an even or an odd multiple of 128 bytes apart)
template <int KU, int RW>
__device__ __forceinline__ int span_k_flip(int key, int page) {
    if (RW == 16) return ((key >> 1) & 1) | ((key >> 2) & 2) | ((page & 1) << 2);      // keys 8 a + 4 t + b: a, b = 0 .. 3
    return KU % 16 == 0 ? key & 15 : (key >> 1) & 7;
}

template <int RW>
struct SpanTile;
template <>
struct SpanTile<32> {
    typedef float16_t acc_t;
    // key of A row m of score tile t
    static __device__ __forceinline__ int key(int m, int) { return (m & 19) | ((m & 4) << 1) | ((m & 8) >> 1); }
    static __device__ __forceinline__ float row_max(float v) {
        const auto o = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return fmaxf(__uint_as_float(o[0]), __uint_as_float(o[1]));
    }
    static __device__ __forceinline__ float row_sum(float v) { return v + __shfl_xor(v, 32, 64); }
};
template <>
struct SpanTile<16> {
    typedef float4_t acc_t;
    static __device__ __forceinline__ int key(int m, int t) { return 8 * (m >> 2) + 4 * (t & 1) + (m & 3); }
    static __device__ __forceinline__ float row_max(float v) {
        const auto o = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return SpanTile<32>::row_max(fmaxf(__uint_as_float(o[0]), __uint_as_float(o[1])));
    }
    static __device__ __forceinline__ float row_sum(float v) { return SpanTile<32>::row_sum(v + __shfl_xor(v, 16, 64)); }
};

template <typename T, int D, int DV, int KT, int RW, bool REL>
__global__ __launch_bounds__(8192 / RW, 2) void span_attn_kernel(SpanParams p) {
    static_assert(D % 64 == 0 && DV % 32 == 0 && KT % 32 == 0 && (RW == 32 || (D / 8) % 16 == 8) && !(REL && RW != 32), "");
    typedef SpanTile<RW> Tile;
    constexpr int NW = 128 / RW, ND = 8192 / RW;
    constexpr int KU = D / 8, KI = D / 32, VI = DV / 32, NP = KT / 16;      // units of a K row; DMA instructions of a page
    constexpr int ALL = NP * (KI + VI), PER = (ALL + NW - 1) / NW;          // ... of a stage, of a wave
    constexpr int KB = KT * D * 2, VB = KT * DV * 2, BUF = KB + VB;
    constexpr int KSTEP = 512 / RW;                 // depth of a matrix step: elements of a score product, keys of a value product
    constexpr int NT = KT / RW, NV = KT * RW / 64, PT = NV / NT;    // score tiles of a stage, scores of a lane: all, per tile
    constexpr int CT = DV / RW, KS = D / KSTEP, AC = RW * RW / 64;  // value tiles; score steps; values of an accumulator
    constexpr bool WIDE = RW == 16;
    constexpr float kLog2e = 1.4426950408889634f;
    constexpr float kLazy = 8.0f;       // (base-2 units: weights stay below 2^8)
    extern __shared__ __attribute__((aligned(16))) char smem[];     // two stages, then (REL) 4 x (KT + 32) floats

    const int tid = threadIdx.x, lane = tid & 63,
              wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane % RW, lk = lane / RW;       // row (or operand row); which of the row's lanes
    const int g = blockIdx.z, rep = p.H / p.G, qt = p.qt;
    // ---- which queries: qt of one portion, as several spans (qt > 32) or a part of one ------------------------------------------
    int span = blockIdx.x, sub = 0;
    if (qt < kSpan) {
        const int per = kSpan / qt;
        span = static_cast<int>(blockIdx.x) / per;
        sub = static_cast<int>(blockIdx.x) - span * per;
    }
    span = __builtin_amdgcn_readfirstlane(p.num_spans - 1 - span);      // (later spans of a portion see more keys: they go first)
    int row0 = __builtin_amdgcn_readfirstlane(p.span_row0[span]), cnt = __builtin_amdgcn_readfirstlane(p.span_cnt[span]);
    const int p_first = __builtin_amdgcn_readfirstlane(p.tok_pos[row0]);
    if (qt > kSpan) {
        const int per = qt / kSpan, nth = (p_first - __builtin_amdgcn_readfirstlane(p.tok_start[row0])) / kSpan;
        if (nth % per) return;      // (an earlier span's workgroup takes these queries)
        const int seq = __builtin_amdgcn_readfirstlane(p.tok_seq[row0]);
        for (int i = 1; i < per && span + i < p.num_spans; ++i) {
            const int r = __builtin_amdgcn_readfirstlane(p.span_row0[span + i]);
            if (p.tok_seq[r] != seq) break;
            cnt += __builtin_amdgcn_readfirstlane(p.span_cnt[span + i]);
        }
    } else {
        row0 += sub * qt;
        cnt = min(qt, cnt - sub * qt);
        if (cnt <= 0) return;
    }
    const int p0 = qt < kSpan ? p_first + sub * qt : p_first;
    const int32_t *bt = p.block_table + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(p.tok_seq[row0])) * p.max_blocks;

    // ---- this lane's row: head R / qt of the group, query R % qt --------------------------------------------------------------
    const int R = wave * RW + lr, hr = R / qt, qr = R - hr * qt;
    const bool live = hr < rep && qr < cnt;
    const int head = g * rep + min(hr, rep - 1), qi = min(qr, cnt - 1);
    const int qpos = p0 + qi;
    auto first_key = [&](int pos) {
        return p.window <= 0 ? 0 : p.mask_kind == 1 ? (pos / p.window) * p.window : max(pos - p.window + 1, 0);
    };
    const int qlo = first_key(qpos);
    // queries of this wave (uniform): positions [wp0, wp1]
    const int w_qr = qt >= RW ? (wave * RW) % qt : 0;
    const int wp0 = p0 + min(w_qr, cnt - 1), wp1 = p0 + min(qt >= RW ? w_qr + RW - 1 : qt - 1, cnt - 1);
    const bool idle = (wave * RW) / qt >= rep || (qt >= RW && w_qr >= cnt);     // no live row in this wave
    int kb0 = first_key(p0) / 16, kb1 = (p0 + cnt - 1) / 16;
    if (gridDim.y > 1) {        // key split: a contiguous share of the pages (possibly none), whole stages but for the last one's
        const int shares = static_cast<int>(gridDim.y), per = ((kb1 - kb0 + shares) / shares + NP - 1) / NP * NP;
        kb0 += per * static_cast<int>(blockIdx.y);
        kb1 = min(kb1, kb0 + per - 1);
    }
    const int nstages = kb1 >= kb0 ? (kb1 - kb0 + NP) / NP : 0;

    vec8_t<T> qf[KS];
    {
        const T *qp = static_cast<const T *>(p.q) + static_cast<int64_t>(row0 + qi) * p.q_stride + static_cast<int64_t>(head) * D + lk * 8;
#pragma unroll
        for (int e = 0; e < KS; ++e) qf[e] = load8(qp + e * KSTEP);
    }
    typename Tile::acc_t acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[ct] = typename Tile::acc_t{};
    float mrun = kNegBig, lrun = 0.f;

    // ---- staging --------------------------------------------------------------------------------------------------------------
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    const char *kc = static_cast<const char *>(p.k_cache) + static_cast<int64_t>(g) * 16 * D * 2;
    const char *vc = static_cast<const char *>(p.v_cache) + static_cast<int64_t>(g % p.GV) * 16 * DV * 2;
    const int64_t bstride = p.block_stride * 2;
    const unsigned v_off = static_cast<unsigned>((lane ^ ((lane >> 4) & 1)) * 16);
    int ids[NP];
    auto fetch_ids = [&](int stage) {       // block ids of a stage's pages (past the last visible page: that page again)
#pragma unroll
        for (int i = 0; i < NP; ++i) ids[i] = bt[min(kb0 + stage * NP + i, kb1)];
    };
    auto issue = [&](int stage) {
        const unsigned dst = lds0 + static_cast<unsigned>(stage & 1) * BUF;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int n = wave * PER + i;
            if (ALL % NW != 0 && n >= ALL) break;       // (uniform)
            const int page = n / (KI + VI), r = n - page * (KI + VI);
            int id = ids[0];
#pragma unroll
            for (int k = 1; k < NP; ++k) id = page == k ? ids[k] : id;
            const int64_t at = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(id)) * bstride;
            unsigned off, to;
            const char *base;
            if (r < KI) {
                const int unit = r * 64 + lane;
                off = static_cast<unsigned>((unit ^ span_k_flip<KU, RW>(unit / KU, page)) * 16);
                base = kc + at;
                to = dst + static_cast<unsigned>(page * 16 * D * 2 + r * 1024);
            } else {
                off = v_off;
                base = vc + at + (r - KI) * 1024;
                to = dst + static_cast<unsigned>(KB + page * 16 * DV * 2 + (r - KI) * 1024);
            }
            unsigned keep;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                         : "=&s"(keep) : "v"(off), "s"(base), "s"(to) : "memory");
        }
    };
    // fragment reads (bytes). K: row Tile::key(lr, t), unit e KSTEP / 8 + lk (the flip touches the unit's low bits only: a few
    // addresses, the rest are offsets of the instructions); V: column lr, keys 8 lk .. 8 lk + 7 of the step
    constexpr int TK = RW == 16 ? 2 : 1, KF = (KU % 16 == 0 ? 16 : 8) * 8 / KSTEP;
    int k_frag[TK][KF];
#pragma unroll
    for (int t = 0; t < TK; ++t)
#pragma unroll
        for (int e = 0; e < KF; ++e) {
            const int key = Tile::key(lr, t);
            k_frag[t][e] = key * D * 2 + (((e * KSTEP / 8 + lk) ^ span_k_flip<KU, RW>(key & 15, key >> 4)) * 16);
        }
    const unsigned v_frag = static_cast<unsigned>((lk >> 1) * 16 * DV * 2 + (((lr * 2 + (lk & 1)) ^ ((lr >> 3) & 1)) * 16));

    // bias by distance: the wave's window of the head's row, one stage ahead (REL: qt >= 32 = RW, so a wave has one head)
    float *rel_lds = reinterpret_cast<float *>(smem + 2 * BUF) + wave * (KT + 32);
    const float *rel_row = REL ? p.rel + static_cast<int64_t>(g * p.H / p.G + min((wave * 32) / qt, rep - 1)) * p.rel_len : nullptr;
    float rel_next[2] = {0.f, 0.f};
    auto fetch_rel = [&](int stage) {       // entry i: distance wp0 - (first key of the stage) - (KT - 1) + i
        const int d0 = wp0 - (kb0 + stage * NP) * 16 - (KT - 1);
        rel_next[0] = rel_row[min(max(d0 + lane, 0), p.rel_len - 1)];
        if (KT > 32) rel_next[1] = rel_row[min(max(d0 + 64 + lane, 0), p.rel_len - 1)];
    };

    // ---- score constants (base-2 exponent units) --------------------------------------------------------------------------------
    const bool capped = p.softcap > 0.f;
    const float c_mul = capped ? 2.0f * kLog2e * p.scale / p.softcap : p.scale * kLog2e;
    const float cap = p.softcap * kLog2e, cap2 = -2.0f * p.softcap * kLog2e;
    const float slope = p.slopes ? p.slopes[head] * kLog2e : 0.f;

    if (nstages > 0) {
        fetch_ids(0);
        issue(0);
        if constexpr (REL) fetch_rel(0);
        if (nstages > 1) fetch_ids(1);
    }
    for (int st = 0; st < nstages; ++st) {
        // this wave's pieces of the stage have landed, its reads of the other buffer have returned
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();       // ... and everyone's
        float rel_now[2];
        if constexpr (REL) { rel_now[0] = rel_next[0]; rel_now[1] = rel_next[1]; }
        if (st + 1 < nstages) {
            issue(st + 1);
            if constexpr (REL) fetch_rel(st + 1);
            if (st + 2 < nstages) fetch_ids(st + 2);
        }
        const int k0 = (kb0 + st * NP) * 16;
        if (idle || k0 > wp1 || k0 + KT - 1 < first_key(wp0)) continue;
        const char *kbuf = smem + (st & 1) * BUF, *vbuf = kbuf + KB;
        if constexpr (REL) {
            rel_lds[lane] = rel_now[0];
            if (KT > 32 && lane < KT - 32) rel_lds[64 + lane] = rel_now[1];
        }
        typename Tile::acc_t s[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            s[t] = typename Tile::acc_t{};
#pragma unroll
            for (int e = 0; e < KS; ++e) {
                const vec8_t<T> kf = *reinterpret_cast<const vec8_t<T> *>(kbuf + k_frag[t % TK][e % KF] + (t / TK) * 32 * D * 2 +
                                                                          (e / KF) * KF * KSTEP * 2);
                s[t] = mfma_step(kf, qf[e], s[t]);
            }
        }
#pragma unroll
        for (int t = 0; t + 1 < NT; ++t) mfma_results_tie(s[t]);
        mfma_results_ready<8>(s[NT - 1]);
        // score j of the lane, s[j / PT][j % PT]: key k0 + 8 lk + KSTEP (j / 8) + j % 8
        float x[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) x[j] = s[j / PT][j % PT];
        const int kd = qpos - k0 - 8 * lk;      // distance of this lane's first key
        if (capped) {       // cap tanh(x / cap) = cap - 2 cap / (2^(2 log2(e) x / cap) + 1); overflow gives cap, underflow -cap
#pragma unroll
            for (int j = 0; j < NV; ++j) x[j] = fmaf(cap2, __builtin_amdgcn_rcpf(fast_exp2(x[j] * c_mul) + 1.0f), cap);
        } else {
#pragma unroll
            for (int j = 0; j < NV; ++j) x[j] *= c_mul;
        }
        if constexpr (REL) {
            const float *rl = rel_lds + (qpos - wp0) + (KT - 1) - 8 * lk;
#pragma unroll
            for (int j = 0; j < NV; ++j) x[j] = fmaf(rl[-(KSTEP * (j / 8) + j % 8)], kLog2e, x[j]);
        }
        if (p.slopes) {
            const float d0 = static_cast<float>(kd);
#pragma unroll
            for (int j = 0; j < NV; ++j) x[j] = fmaf(-slope, d0 - static_cast<float>(KSTEP * (j / 8) + j % 8), x[j]);
        }
        if (k0 + KT - 1 > wp0 || (p.window > 0 && k0 < first_key(wp1))) {      // (uniform) the stage crosses a row's limits
            const int lo = qlo - k0 - 8 * lk;       // visible: lo <= key - (k0 + 8 lk) <= kd
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int at = KSTEP * (j / 8) + j % 8;
                if (at > kd || at < lo) x[j] = kNegBig;
            }
        }
        float mx = x[0];
#pragma unroll
        for (int j = 1; j < NV; ++j) mx = fmaxf(mx, x[j]);
        mx = Tile::row_max(mx);
        // lazy running maximum: a row moves its reference only when a stage raises it by more than kLazy
        const float mnew = mx - mrun > kLazy ? mx : mrun;
        const float alpha = fast_exp2(mrun - mnew);
        mrun = mnew;
        const float mref = mnew < 0.5f * kNegBig ? 0.f : mnew;      // (a row that has seen no key yet: all its weights are 2^-1e30 = 0)
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            x[j] = fast_exp2(x[j] - mref);
            psum += x[j];
        }
        lrun = fmaf(lrun, alpha, psum);
        if (!__all(alpha == 1.0f)) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int i = 0; i < AC; ++i) acc[ct][i] *= alpha;
        }
#pragma unroll
        for (int u = 0; u < NV / 8; ++u) {
            vec8_t<T> hi, lo;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                hi[j] = to_t<T>(x[8 * u + j]);
                lo[j] = to_t<T>(x[8 * u + j] - to_f(hi[j]));
            }
            const char *vp = vbuf + u * (KSTEP / 16) * 16 * DV * 2 + v_frag;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const vec8_t<T> vf = *reinterpret_cast<const vec8_t<T> *>(vp + ct * RW * 32);
                acc[ct] = mfma_step(vf, hi, acc[ct]);
                acc[ct] = mfma_step(vf, lo, acc[ct]);
            }
        }
    }
    // ---- epilogue: acc[ct][4 r + e] = O[row][ct RW + 8 r + 4 lk + e] ----------------------------------------------------------
#pragma unroll
    for (int ct = 0; ct + 1 < CT; ++ct) mfma_results_tie(acc[ct]);
    mfma_results_ready<8>(acc[CT - 1]);
    const float l = Tile::row_sum(lrun);
    if (!live) return;
    const int64_t orow = row0 + qr;
    if (gridDim.y > 1) {        // partial result of this key share: unnormalised O, running maximum, sum
        const int64_t slot = (static_cast<int64_t>(blockIdx.y) * p.num_tokens + orow) * p.H + head;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < AC / 4; ++r)
                *reinterpret_cast<float4_t *>(p.part_o + slot * DV + ct * RW + 8 * r + 4 * lk) =
                    float4_t{acc[ct][4 * r], acc[ct][4 * r + 1], acc[ct][4 * r + 2], acc[ct][4 * r + 3]};
        if (lk == 0) {
            p.part_ml[slot * 2] = mrun;
            p.part_ml[slot * 2 + 1] = l;
        }
        return;
    }
    float inv = 1.0f / l;
    if (p.sink) {       // the sink joins the denominator: rebase the row on max(m, sink)
        const float sk = p.sink[head] * kLog2e, big = fmaxf(mrun, sk);
        const float a = fast_exp2(mrun - big);
        inv = a / (l * a + fast_exp2(sk - big));
    }
    T *out = static_cast<T *>(p.out);
    const T *gate = static_cast<const T *>(p.gate);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int r = 0; r < AC / 4; ++r) {
            const int c = ct * RW + 8 * r + 4 * lk;
            if (c >= p.out_dim) continue;
            const int64_t hc = static_cast<int64_t>(head) * p.out_dim + c, at = orow * p.out_stride + hc;
            float4_t o = {acc[ct][4 * r], acc[ct][4 * r + 1], acc[ct][4 * r + 2], acc[ct][4 * r + 3]};
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] *= inv;
            if (p.out_dim & 3) {        // (uniform) element by element
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (c + e >= p.out_dim) continue;
                    if (gate) o[e] /= 1.0f + fast_exp2(-kLog2e * to_f(gate[orow * p.gate_stride + hc + e]));
                    if (p.out_f32) reinterpret_cast<float *>(p.out)[at + e] = o[e];
                    else out[at + e] = to_t<T>(o[e]);
                }
                continue;
            }
            if (gate) {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] /= 1.0f + fast_exp2(-kLog2e * to_f(gate[orow * p.gate_stride + hc + e]));
            }
            if (p.out_f32) {
                *reinterpret_cast<float4_t *>(reinterpret_cast<float *>(p.out) + at) = o;
            } else {
                vec4_t<T> w;
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = to_t<T>(o[e]);
                *reinterpret_cast<vec4_t<T> *>(out + at) = w;
            }
        }
}

template <typename T, int D, int DV, int KT, int RW>
int launch_span(const SpanParams &p, int key_splits, hipStream_t s) {
    const int per = p.qt < kSpan ? kSpan / p.qt : 1;
    const dim3 grid(static_cast<unsigned>(p.num_spans * per), static_cast<unsigned>(key_splits), static_cast<unsigned>(p.G));
    const size_t lds = 2 * static_cast<size_t>(KT) * (D + DV) * 2 + (p.rel ? 4 * (KT + 32) * sizeof(float) : 0);
    auto go = [&](auto kernel) {
        // (more LDS than a launch gets without asking)
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
            return false;
        hipLaunchKernelGGL(kernel, grid, dim3(8192 / RW), lds, s, p);
        return true;
    };
    bool ok;
    if constexpr (D <= 128 && DV <= 128) ok = p.rel ? go(&span_attn_kernel<T, D, DV, KT, RW, true>) : go(&span_attn_kernel<T, D, DV, KT, RW, false>);
    else ok = go(&span_attn_kernel<T, D, DV, KT, RW, false>);
    if (!ok) return SWL_ERR_LAUNCH;
    if (key_splits > 1) {
        const int64_t rows = p.num_tokens * p.H;
        hipLaunchKernelGGL((window_attn_combine_kernel<T>), dim3(static_cast<unsigned>(rows)), dim3(DV < 256 ? 64 : 256), 0, s,
                           static_cast<T *>(p.out), p.part_o, p.part_ml, rows, DV, key_splits, p.sink, p.H, p.out_f32, p.out_dim,
                           p.out_stride, static_cast<const T *>(p.gate), p.gate_stride);
    }
    return check_launch();
}

// queries of a workgroup for `rep` query heads a key head: 128 rows over rep rounded up to a power of two; 0: not served
static int span_queries(int rep) {
    int up = 1;
    while (up < rep) up *= 2;
    return up <= 64 ? 128 / up : 0;
}

} // namespace swl

#define SWL_SPAN_SHAPES(X) X(64, 64, 32, 32) X(64, 128, 32, 32) X(128, 64, 32, 32) X(128, 128, 32, 32) X(192, 128, 32, 32) X(320, 256, 32, 16) X(576, 512, 32, 16)

/* 1 when swl_span_attn serves this shape. */
extern "C" int swl_span_attn_supported(int32_t num_q_heads, int32_t num_kv_heads, int32_t num_v_heads, int32_t dim, int32_t vdim,
                                       int32_t has_rel, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    if (num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return 0;
    if (num_v_heads <= 0 || num_kv_heads % num_v_heads) return 0;
    const int qt = swl::span_queries(num_q_heads / num_kv_heads);
    if (qt == 0 || num_kv_heads > 65535) return 0;
    // (a wave's bias window is one head's: at least 32 queries of a head per wave)
    if (has_rel && (qt < 32 || dim > 128 || vdim > 128)) return 0;
#define SWL_SPAN_IS(DD, DDV, KT, RW) if (dim == DD && vdim == DDV) return 1;
    SWL_SPAN_SHAPES(SWL_SPAN_IS)
#undef SWL_SPAN_IS
    return 0;
}

extern "C" int swl_span_attn(void *out, const void *q, const void *k_cache, const void *v_cache, const int32_t *block_table,
                             const int32_t *tok_seq, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *span_row0,
                             const int32_t *span_cnt, const float *rel, int32_t rel_len, int32_t num_spans, int32_t num_q_heads,
                             int32_t num_kv_heads, int32_t num_v_heads, int32_t dim, int32_t vdim, int64_t q_tok_stride,
                             int32_t window, int32_t mask_kind, float scale, float softcap, int32_t max_blocks_per_seq,
                             int64_t block_stride, int32_t key_splits, float *scratch, int64_t num_tokens, const float *sink,
                             int32_t out_f32, const float *slopes, int32_t out_dim, int64_t out_stride, const void *gate,
                             int64_t gate_stride, int32_t dtype, swl_stream_t stream) {
    if (num_spans < 0 || window < 0 || mask_kind < 0 || mask_kind > 1 || key_splits < 1 || key_splits > 64) return SWL_ERR_BAD_ARG;
    if (key_splits > 1 && (!scratch || num_tokens <= 0 || !swl::aligned16(scratch))) return SWL_ERR_BAD_ARG;
    if (out_dim <= 0 || out_dim > vdim || out_stride < static_cast<int64_t>(num_q_heads) * out_dim) return SWL_ERR_BAD_ARG;
    if (gate && gate_stride < static_cast<int64_t>(num_q_heads) * out_dim) return SWL_ERR_BAD_ARG;
    if (out_dim % 4 == 0 && (out_stride & 3)) return SWL_ERR_BAD_ARG;      // (4-element stores)
    if (!swl_span_attn_supported(num_q_heads, num_kv_heads, num_v_heads, dim, vdim, rel != nullptr, dtype)) return SWL_ERR_UNSUPPORTED;
    if (num_spans == 0) return SWL_OK;
    if (!out || !q || !k_cache || !v_cache || !block_table || !tok_seq || !tok_pos || !tok_start || !span_row0 || !span_cnt ||
        (rel && rel_len <= 0))
        return SWL_ERR_BAD_ARG;
    // 16-byte operand loads
    if ((q_tok_stride & 7) || (block_stride & 7) || !swl::aligned16(q) || !swl::aligned16(k_cache) || !swl::aligned16(v_cache) ||
        (reinterpret_cast<uintptr_t>(out) & (out_f32 ? 15 : 7)))
        return SWL_ERR_BAD_ARG;
    swl::SpanParams p;
    p.out = out; p.q = q; p.k_cache = k_cache; p.v_cache = v_cache;
    p.block_table = block_table; p.tok_seq = tok_seq; p.tok_pos = tok_pos; p.tok_start = tok_start;
    p.span_row0 = span_row0; p.span_cnt = span_cnt;
    p.rel = rel; p.sink = sink; p.slopes = slopes; p.gate = gate;
    // scratch: [splits][tokens][H][vdim] fp32 partial outputs, then [splits][tokens][H][2] (maximum, sum)
    p.part_o = scratch;
    p.part_ml = scratch ? scratch + static_cast<int64_t>(key_splits) * num_tokens * num_q_heads * vdim : nullptr;
    p.rel_len = rel_len; p.num_spans = num_spans; p.H = num_q_heads; p.G = num_kv_heads; p.GV = num_v_heads;
    p.window = window; p.mask_kind = mask_kind; p.max_blocks = max_blocks_per_seq; p.out_f32 = out_f32; p.out_dim = out_dim;
    p.qt = swl::span_queries(num_q_heads / num_kv_heads);
    p.scale = scale; p.softcap = softcap;
    p.q_stride = q_tok_stride; p.block_stride = block_stride; p.out_stride = out_stride; p.gate_stride = gate_stride;
    p.num_tokens = num_tokens;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define SWL_SPAN_GO(DD, DDV, KT, RW) if (dim == DD && vdim == DDV) return swl::launch_span<T, DD, DDV, KT, RW>(p, key_splits, s);
    SWL_DISPATCH_DTYPE(dtype, T, { SWL_SPAN_SHAPES(SWL_SPAN_GO) });
#undef SWL_SPAN_GO
    return SWL_ERR_UNSUPPORTED;
}
