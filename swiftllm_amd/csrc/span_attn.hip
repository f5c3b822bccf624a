// span_attn.hip — the matrix-core attention of prompt portions over the paged pool, for heads that are not mixed
// (swl_masked_attn_tiles' masks, bias, slopes, cap, sink, gate; same pool layout, same arithmetic up to the order of sums).
//
// What bounds it: a value product in two 16-bit terms (hi + lo, so that a weight keeps 16 bits of its fp32 value) takes 2 (D + 2 DV) flops per
// (row, key) of the matrix cores, the softmax about as many cycles of the vector units (105 instructions a wave for 16 rows and 32 keys), the
// fragments read from LDS a little more: 64 rows of 128 + 128 columns and 64 keys take 1 us of a CU, 0.35 us of it matrix steps, and the two
// hardly overlap, as the waves of a stage start it together. A ROW is one (query, query head) pair: every head of a kv group reads the same keys, so
// one staged page serves all of them (QT = rows / heads queries a workgroup, heads rounded up to a power of two). Eight waves of 16 rows:
//   S^T = K Q^T   A = keys from LDS, B = its query fragments (registers for the whole walk)
//   online softmax: lane l owns row l % 16, the four lanes of a row hold its keys between them
//   O^T += V^T P^T  A = value columns from LDS, B = the score registers. Which key an A row of S^T takes is chosen so that a lane's
//                   eight scores of a step are eight CONSECUTIVE keys, which is what the B operand wants and what a page's
//                   transposed values hold in 16 bytes — no data moves between lanes.
// Rows of up to 320 elements (keys and values) in steps of a few workgroups a CU (launch_span_any): a stage is 64 keys, two waves share a
// row group and take 32 keys each, 64 rows a workgroup, two workgroups a CU: a workgroup's walk, the longest chain of a step, is half as many
// stages. Otherwise 32 keys, 128 rows. Four fragments are on their way from LDS ahead of their matrix step, and nothing the compiler loads is pending inside the walk: its
// waits for such loads would be waits for the stage that was just asked for.
// Pages are staged by LDS-DMA (1 KiB per wave instruction, full lines) into two buffers with one barrier a stage (three stages ahead instead of
// one changed nothing); the swizzle that keeps the 16-byte fragment reads of keys off each other's banks is applied to the source addresses.
// A value that is NaN or infinite reaches every row of a workgroup that stages its page (a weight of 0 times it), as it does in the tiles
// of window_attn_mfma.hip: rows of the same portion whose queries come before it, at most 127 of them; never another sequence's.
// us a launch, bf16, by the 16-row kernel of window_attn_mfma.hip / before these waves and this order of the spans / now: 4 prompts of 1000 to
// 2000 tokens, 8 heads of 128 over 2 key heads 489 / 100 / 77, with a bias by distance 535 / 108 / 75; 8 latent heads of 576 + 512 over one,
// window 1024: 1115 / 270 / 171; 11 prompts of 333 tokens, 16 heads of 128 over 4: 120 / 31 / 30.
#include "attn_combine.h"
#include "swl_common.h"

namespace swl {

__device__ __forceinline__ float4_t mfma_step(vec8_t<f16> a, vec8_t<f16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mfma_step(vec8_t<bf16> a, vec8_t<bf16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct SpanParams {
    void *out;
    const void *q, *k_cache, *v_cache;
    const int32_t *block_table, *tok_seq, *tok_pos, *tok_start, *span_row0, *span_cnt, *span_order;
    const float *rel, *sink, *slopes;
    const void *gate;
    float *part_o, *part_ml;
    int rel_len, num_spans, H, G, GV, window, mask_kind, max_blocks, out_f32, out_dim, qt;
    float scale, softcap;
    int64_t q_stride, block_stride, out_stride, gate_stride, num_tokens;
};

constexpr int kSpan = 32;       // tokens of a span at most (the plan's chunks)
constexpr int kSpanWaves = 8;
constexpr int kSpanKeys = 32;   // keys of a wave and stage

// Waves that share a row group's keys, at most: two where a stage of 64 keys leaves room for two workgroups a CU, one for wider rows
constexpr int span_halves(int D, int DV) { return 2 * 64 * (D + DV) * 2 <= 80 * 1024 ? 2 : 1; }

// LDS position of a K row's 16-byte unit: the low bits of the unit index are flipped by a function of the key that differs over the
// 16 rows that a group of lanes reads, keys 8 a + 4 t + b with a, b = 0 .. 3 (rows are an even or an odd multiple of 128 bytes apart)
template <int KU>
__device__ __forceinline__ int span_k_flip(int key, int page) {
    static_assert(KU % 8 == 0, "");
    if (KU % 16 == 0) return (key & 3) | ((key >> 1) & 4) | ((page & 1) << 3);
    return ((key >> 1) & 1) | ((key >> 2) & 2) | ((page & 1) << 2);
}
// key of A row m of score tile t
__device__ __forceinline__ int span_key(int m, int t) { return 8 * (m >> 2) + 4 * t + (m & 3); }

__device__ __forceinline__ float span_row_max(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float span_row_sum(float v) {
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// N matrix steps whose operand comes from LDS, AHEAD of them on their way. (Left alone, the compiler reads every fragment right in
// front of its step: a latency of LDS for each.)
template <int AHEAD, int N, int MFMAS, typename V, typename Load, typename Step>
__device__ __forceinline__ void span_steps(Load &&load, Step &&step) {
    constexpr int R = AHEAD < N ? AHEAD : N;
    V ring[R];
#pragma unroll
    for (int i = 0; i < R; ++i) ring[i] = load(i);
    __builtin_amdgcn_sched_group_barrier(0x100, R, 0);      // LDS reads
#pragma unroll
    for (int i = 0; i < N; ++i) {
        step(i, ring[i % R]);
        __builtin_amdgcn_sched_group_barrier(0x008, MFMAS, 0);      // matrix steps
        if (i + R < N) {
            ring[i % R] = load(i + R);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
    }
}

// The workgroup's place (at: along the spans, heaviest first; g: key head) from its number.
//   * Runs of `run` workgroups, the queries of four neighbouring spans, see the same keys but for 128. Workgroups go round the eight XCDs
//     by their number, so a run takes every eighth number: one XCD's L2 holds its keys once.
//   * The key heads alternate run by run: the heaviest spans of every head come first.
//   * PAIRS (two workgroups share a CU) and at most two a CU: all are there at once, and the second of a CU comes from the other end of
//     the list.
template <bool PAIRS>
__device__ __forceinline__ void span_place(int run, int &at, int &g) {
    const int gx = gridDim.x, G = gridDim.z, all = gx * G;
    constexpr int kCUs = 256;
    auto one_xcd = [&](int v, int n) {      // a permutation of 0 .. n - 1
        if (v >= n / (8 * run) * (8 * run)) return v;
        const int nth = v >> 3;
        return ((nth / run) * 8 + (v & 7)) * run + nth % run;
    };
    if (gridDim.y > 1) {
        at = one_xcd(at, gx);
        return;
    }
    int u = at + gx * g;
    if (PAIRS && all > kCUs && all <= 2 * kCUs) u = u < kCUs ? one_xcd(u, kCUs) : all - 1 - one_xcd(u - kCUs, all - kCUs);
    else u = one_xcd(u, all);
    const int whole = gx / run * run;
    if (u < whole * G) {
        const int q = u / run;
        g = q % G;
        at = (q / G) * run + u - q * run;
    } else {
        u -= whole * G;
        g = u / (gx - whole);
        at = whole + u - g * (gx - whole);
    }
}

template <typename T, int D, int DV, int KH, bool REL>
__global__ __launch_bounds__(kSpanWaves * 64, 2) void span_attn_kernel(SpanParams p) {
    static_assert(D % 64 == 0 && DV % 32 == 0, "");
    constexpr int NW = kSpanWaves, RG = NW / KH;                // (KH: waves of a row group) row groups
    constexpr int KW = kSpanKeys, KT = KW * KH, NP = KT / 16;   // keys of a stage: a wave's, all of them, their pages
    constexpr int KU = D / 8, KI = D / 32, VI = DV / 32;        // units of a K row; KiB of a page's keys, values
    constexpr int US = (KI + VI + NW - 1) / NW;                 // ... of a wave
    constexpr int kOddFlip = KU % 16 == 0 ? 8 : 4;              // (span_k_flip of an odd page)
    constexpr int KB = KT * D * 2, VB = KT * DV * 2, BUF = KB + VB;
    constexpr int NT = KW / 16, NV = 8;             // score tiles of a wave's keys, scores of a lane
    constexpr int CT = DV / 16, KS = D / 32;        // value tiles; steps of a score
    constexpr int AHEAD = 4;                        // fragments on their way from LDS
    constexpr float kLog2e = 1.4426950408889634f;
    constexpr float kLazy = 8.0f;       // (base-2 units: weights stay below 2^8)
    extern __shared__ __attribute__((aligned(16))) char smem[];     // two stages, then (REL) the waves' bias windows of both

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave % RG, kh = wave / RG;       // this wave's row group and which of its keys
    const int lr = lane & 15, lk = lane >> 4;       // row (or operand row); which of the row's lanes
    const int rep = p.H / p.G, qt = p.qt;
    // ---- which queries: qt of one portion, as several spans (qt > 32) or a part of one ------------------------------------------
    const int per_span = qt < kSpan ? kSpan / qt : 1;
    int at = blockIdx.x, g = blockIdx.z;
    span_place<(2 * BUF <= 80 * 1024)>(4 * per_span, at, g);
    int span = at / per_span;
    const int sub = at - span * per_span;
    // (later spans of a portion see more keys: they go first, over all portions where the caller says so)
    span = __builtin_amdgcn_readfirstlane(p.span_order ? min(max(p.span_order[span], 0), p.num_spans - 1) : p.num_spans - 1 - span);
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
    const int my_hr = (rg * 16 + lr) / qt, my_head = g * rep + min(my_hr, rep - 1), qi = min(rg * 16 + lr - my_hr * qt, cnt - 1);
    const int qpos = p0 + qi;
    auto first_key = [&](int pos) {
        return p.window <= 0 ? 0 : p.mask_kind == 1 ? (pos / p.window) * p.window : max(pos - p.window + 1, 0);
    };
    const int qlo = first_key(qpos);
    // queries of this wave (uniform): positions [wp0, wp1]
    const int w_qr = qt >= 16 ? (rg * 16) % qt : 0;
    const int wp0 = p0 + min(w_qr, cnt - 1), wp1 = p0 + min(qt >= 16 ? w_qr + 15 : qt - 1, cnt - 1);
    const bool idle = (rg * 16) / qt >= rep || (qt >= 16 && w_qr >= cnt);     // no live row in this wave
    int kb0 = first_key(p0) / 16, kb1 = (p0 + cnt - 1) / 16;
    if (gridDim.y > 1) {        // key split: a contiguous share of the pages (possibly none), whole stages but for the last one's
        const int shares = static_cast<int>(gridDim.y), per = ((kb1 - kb0 + shares) / shares + NP - 1) / NP * NP;
        kb0 += per * static_cast<int>(blockIdx.y);
        kb1 = min(kb1, kb0 + per - 1);
    }
    const int nstages = kb1 >= kb0 ? (kb1 - kb0 + NP) / NP : 0;

    vec8_t<T> qf[KS];
    {
        const T *qp = static_cast<const T *>(p.q) + static_cast<int64_t>(row0 + qi) * p.q_stride + static_cast<int64_t>(my_head) * D + lk * 8;
#pragma unroll
        for (int e = 0; e < KS; ++e) qf[e] = load8(qp + e * 32);
    }
    float4_t acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
    float mrun = kNegBig, lrun = 0.f;

    // ---- staging --------------------------------------------------------------------------------------------------------------
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    const char *kc = static_cast<const char *>(p.k_cache) + static_cast<int64_t>(g) * 16 * D * 2;
    const char *vc = static_cast<const char *>(p.v_cache) + static_cast<int64_t>(g % p.GV) * 16 * DV * 2;
    const int64_t bstride = p.block_stride * 2;
    // block ids: lane i holds that of page id_base + i of this share (past the last visible page: that page again), 64 pages a load
    int id_base = 0, id_lane = 0;
    auto fetch_ids = [&]() { id_lane = bt[min(kb0 + id_base + lane, kb1)]; };
    float *const rel_lds = reinterpret_cast<float *>(smem + 2 * BUF) + wave * 64;       // (REL) [2][NW][64]
    const float *rel_row = REL ? p.rel + static_cast<int64_t>(g * rep + min((rg * 16) / qt, rep - 1)) * p.rel_len : nullptr;
    // A page is KI + VI KiB, KiB u of every page of a stage is asked for by wave u % NW: its lanes' places in it are the same for every page
    // but for the flip of odd pages' keys.
    unsigned src[US];
#pragma unroll
    for (int j = 0; j < US; ++j) {
        const int u = wave + NW * j, unit = u * 64 + lane;
        src[j] = static_cast<unsigned>(u < KI ? (unit ^ span_k_flip<KU>(unit / KU, 0)) * 16 : lane * 16);
    }
    auto ask = [&](int stage) {
        const unsigned dst = lds0 + static_cast<unsigned>(stage & 1) * BUF;
        unsigned keep;
#pragma unroll
        for (int page = 0; page < NP; ++page) {
            const int64_t blk = static_cast<int64_t>(__builtin_amdgcn_readlane(id_lane, stage * NP - id_base + page)) * bstride;
#pragma unroll
            for (int j = 0; j < US; ++j) {
                const int u = wave + NW * j;        // (uniform)
                if (NW * (j + 1) > KI + VI && u >= KI + VI) break;
                const bool key = u < KI;
                const char *base = (key ? kc : vc + (u - KI) * 1024) + blk;
                const unsigned off = page & 1 ? src[j] ^ (key ? kOddFlip * 16 : 0) : src[j];
                const unsigned to = dst + static_cast<unsigned>(key ? page * 16 * D * 2 + u * 1024 : KB + page * 16 * DV * 2 + (u - KI) * 1024);
                asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                             : "=&s"(keep) : "v"(off), "s"(base), "s"(to) : "memory");
            }
        }
        if constexpr (REL) {    // the wave's window of its head's bias, entry i: distance wp0 - (its first key of the stage) - (KW - 1) + i
            const int d = wp0 - (kb0 + stage * NP) * 16 - kh * KW - (KW - 1) + lane;
            const unsigned off = static_cast<unsigned>(min(max(d, 0), p.rel_len - 1)) * 4,
                           to = lds0 + 2 * BUF + static_cast<unsigned>((stage & 1) * NW + wave) * 256;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
                         : "=&s"(keep) : "v"(off), "s"(rel_row), "s"(to) : "memory");
        }
    };
    // fragment reads (bytes). K: row span_key(lr, t), unit 4 e + lk (the flip touches the unit's low bits only: a few addresses, the rest
    // are offsets of the instructions); V: column lr, keys 8 lk .. 8 lk + 7
    constexpr int KF = KU % 16 == 0 ? 4 : 2;
    int k_frag[NT][KF];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < KF; ++e) {
            const int key = span_key(lr, t);
            k_frag[t][e] = kh * KW * D * 2 + key * D * 2 + (((e * 4 + lk) ^ span_k_flip<KU>(key & 15, key >> 4)) * 16);
        }
    const unsigned v_frag = static_cast<unsigned>(kh * KW * DV * 2 + (lk >> 1) * 16 * DV * 2 + (lr * 2 + (lk & 1)) * 16);

    // ---- scores as they are compared and their unit in powers of two: products of queries and keys where nothing is done to them but
    // the scale, the model's logits otherwise (capped ones in base-2 units already). A scale that leaves kNegBig no mask is applied first.
    const bool capped = p.softcap > 0.f, plain = !REL && !capped && !p.slopes && p.scale > 1e-20f;
    const float c_mul = capped ? 2.0f * kLog2e * p.scale / p.softcap : p.scale;
    const float unit = plain ? p.scale * kLog2e : capped ? 1.0f : kLog2e;
    const float cap = p.softcap * kLog2e, cap2 = -2.0f * p.softcap * kLog2e, rel_mul = capped ? kLog2e : 1.0f;
    const float slope = p.slopes ? p.slopes[my_head] * rel_mul : 0.f;

    if (nstages > 0) fetch_ids();
    // what the compiler itself loads has arrived before the walk: a load that might still be on its way at the loop's head is waited
    // for in every turn of it, and with it the stage that was asked for just before
#pragma unroll
    for (int e = 0; e < KS; ++e) asm volatile("" : "+v"(qf[e]));
    asm volatile("" : "+v"(id_lane));
    if (nstages > 0) ask(0);
    for (int st = 0; st < nstages; ++st) {
        const bool more = st + 1 < nstages;
        // this wave's pieces of the stage have landed, its reads of the other buffer have returned
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();       // ... and everyone's
        if (more && (st + 1) * NP - id_base >= 64) {
            id_base += 64;
            fetch_ids();
        }
        if (more) ask(st + 1);
        const int k0 = (kb0 + st * NP) * 16 + kh * KW;
        if (idle || k0 > wp1 || k0 + KW - 1 < first_key(wp0)) continue;
        const char *kbuf = smem + (st & 1) * BUF, *vbuf = kbuf + KB;
        float4_t s[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) s[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        // (step i: score tile i % NT, elements 32 (i / NT) ..)
        span_steps<AHEAD, NT * KS, 1, vec8_t<T>>(
            [&](int i) { return *reinterpret_cast<const vec8_t<T> *>(kbuf + k_frag[i % NT][(i / NT) % KF] + (i / NT) / KF * KF * 64); },
            [&](int i, vec8_t<T> kf) { s[i % NT] = mfma_step(kf, qf[i / NT], s[i % NT]); });
        mfma_results_tie(s[0]);
        mfma_results_ready<8>(s[1]);
        // score j of the lane: key k0 + 8 lk + j
        float x[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) x[j] = s[j / 4][j % 4];
        const int kd = qpos - k0 - 8 * lk;      // distance of this lane's first key
        if (capped) {       // cap tanh(x / cap) = cap - 2 cap / (2^(2 log2(e) x / cap) + 1); overflow gives cap, underflow -cap
#pragma unroll
            for (int j = 0; j < NV; ++j) x[j] = fmaf(cap2, __builtin_amdgcn_rcpf(fast_exp2(x[j] * c_mul) + 1.0f), cap);
        } else if (!REL && !plain) {
#pragma unroll
            for (int j = 0; j < NV; ++j) x[j] *= c_mul;
        }
        if constexpr (REL) {
            const float *rl = rel_lds + (st & 1) * NW * 64 + (qpos - wp0) + (KW - 1) - 8 * lk;
            if (capped) {
#pragma unroll
                for (int j = 0; j < NV; ++j) x[j] = fmaf(rl[-j], kLog2e, x[j]);
            } else {
#pragma unroll
                for (int j = 0; j < NV; ++j) x[j] = fmaf(x[j], c_mul, rl[-j]);
            }
        }
        if (p.slopes) {
            const float d0 = static_cast<float>(kd);
#pragma unroll
            for (int j = 0; j < NV; ++j) x[j] = fmaf(-slope, d0 - static_cast<float>(j), x[j]);
        }
        if (k0 + KW - 1 > wp0 || (p.window > 0 && k0 < first_key(wp1))) {      // (uniform) the keys cross a row's limits
            const int lo = qlo - k0 - 8 * lk;       // visible: lo <= key - (k0 + 8 lk) <= kd
#pragma unroll
            for (int j = 0; j < NV; ++j)
                if (j > kd || j < lo) x[j] = kNegBig;
        }
        float mx = x[0];
#pragma unroll
        for (int j = 1; j < NV; ++j) mx = fmaxf(mx, x[j]);
        mx = span_row_max(mx);
        // lazy running maximum: a row moves its reference only when a stage raises it by more than kLazy
        const float mnew = (mx - mrun) * unit > kLazy ? mx : mrun;
        const float alpha = fast_exp2((mrun - mnew) * unit);
        mrun = mnew;
        // (a row that has seen no key yet: all its weights are 2^-1e30 = 0)
        const float mref = mnew < 0.5f * kNegBig ? 0.f : -mnew * unit;
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            x[j] = fast_exp2(fmaf(x[j], unit, mref));
            psum += x[j];
        }
        lrun = fmaf(lrun, alpha, psum);
        if (!__all(alpha == 1.0f)) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[ct][i] *= alpha;
        }
        vec8_t<T> hi, lo;
        split_weights(x, hi, lo);
        const char *vp = vbuf + v_frag;
        span_steps<AHEAD, CT, 2, vec8_t<T>>([&](int ct) { return *reinterpret_cast<const vec8_t<T> *>(vp + ct * 512); },
                                            [&](int ct, vec8_t<T> vf) {
                                                acc[ct] = mfma_step(vf, hi, acc[ct]);
                                                acc[ct] = mfma_step(vf, lo, acc[ct]);
                                            });
    }
#pragma unroll
    for (int ct = 0; ct + 1 < CT; ++ct) mfma_results_tie(acc[ct]);
    mfma_results_ready<8>(acc[CT - 1]);
    if (!plain && !capped) mrun *= kLog2e;      // base-2 units from here on (kNegBig stays one)
    if (plain) mrun *= unit;
    // ---- the two waves of a row group: the second hands its sums to the first (the stages' place is free) -----------------------
    if constexpr (KH == 2) {
        static_assert(RG * (CT + 1) * 1024 <= 2 * BUF, "");
        __syncthreads();
        float4_t *mine = reinterpret_cast<float4_t *>(smem) + rg * (CT + 1) * 64 + lane;
        if (kh == 1) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) mine[ct * 64] = acc[ct];
            mine[CT * 64] = float4_t{mrun, lrun, 0.f, 0.f};
        }
        __syncthreads();
        if (kh == 1) return;
        const float4_t ml = mine[CT * 64];
        const float m = fmaxf(mrun, ml[0]), a0 = fast_exp2(mrun - m), a1 = fast_exp2(ml[0] - m);
        lrun = lrun * a0 + ml[1] * a1;
        mrun = m;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[ct] = acc[ct] * a0 + mine[ct * 64] * a1;
    }
    // ---- epilogue: acc[ct][e] = O[row][16 ct + 4 lk + e] ------------------------------------------------------------------------
    // (its parameters are loaded here: kept over the walk, they take the registers of other uniform values)
    const auto *again = (const __attribute__((address_space(4))) SpanParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(again));
    const auto &e = *again;
    const float l = span_row_sum(lrun);
    // (the lane's row once more: kept over the walk, it costs registers that the walk has no others for)
    int lane_again = lane;
    asm volatile("" : "+v"(lane_again));
    const int R = rg * 16 + (lane_again & 15), col = 4 * (lane_again >> 4), hr = R / qt, qr = R - hr * qt, head = g * rep + min(hr, rep - 1);
    if (hr >= rep || qr >= cnt) return;
    const int64_t orow = row0 + qr;
    if (gridDim.y > 1) {        // partial result of this key share: unnormalised O, running maximum, sum
        const int64_t slot = (static_cast<int64_t>(blockIdx.y) * e.num_tokens + orow) * e.H + head;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) *reinterpret_cast<float4_t *>(e.part_o + slot * DV + ct * 16 + col) = acc[ct];
        if (col == 0) {
            e.part_ml[slot * 2] = mrun;
            e.part_ml[slot * 2 + 1] = l;
        }
        return;
    }
    float inv = 1.0f / l;
    if (e.sink) {       // the sink joins the denominator: rebase the row on max(m, sink)
        const float sk = e.sink[head] * kLog2e, big = fmaxf(mrun, sk);
        const float a = fast_exp2(mrun - big);
        inv = a / (l * a + fast_exp2(sk - big));
    }
    T *out = static_cast<T *>(e.out);
    const T *gate = static_cast<const T *>(e.gate);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int c = ct * 16 + col;
        if (c >= e.out_dim) continue;
        const int64_t hc = static_cast<int64_t>(head) * e.out_dim + c, at = orow * e.out_stride + hc;
        float4_t o = acc[ct];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] *= inv;
        if (e.out_dim & 3) {        // (uniform) element by element
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (c + i >= e.out_dim) continue;
                if (gate) o[i] /= 1.0f + fast_exp2(-kLog2e * to_f(gate[orow * e.gate_stride + hc + i]));
                if (e.out_f32) reinterpret_cast<float *>(e.out)[at + i] = o[i];
                else out[at + i] = to_t<T>(o[i]);
            }
            continue;
        }
        if (gate) {
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] /= 1.0f + fast_exp2(-kLog2e * to_f(gate[orow * e.gate_stride + hc + i]));
        }
        if (e.out_f32) {
            *reinterpret_cast<float4_t *>(reinterpret_cast<float *>(e.out) + at) = o;
        } else {
            vec4_t<T> w;
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = to_t<T>(o[i]);
            *reinterpret_cast<vec4_t<T> *>(out + at) = w;
        }
    }
}

// queries of a workgroup for `rep` query heads a key head (64 at most): its rows over rep rounded up to a power of two
static int span_queries(int rep, int rows) {
    int up = 1;
    while (up < rep) up *= 2;
    return rows / up;
}

template <typename T, int D, int DV, int KH>
int launch_span(SpanParams &p, int key_splits, hipStream_t s) {
    p.qt = span_queries(p.H / p.G, 16 * kSpanWaves / KH);
    const int per = p.qt < kSpan ? kSpan / p.qt : 1;
    const dim3 grid(static_cast<unsigned>(p.num_spans * per), static_cast<unsigned>(key_splits), static_cast<unsigned>(p.G));
    const size_t lds = 2 * (static_cast<size_t>(kSpanKeys * KH) * (D + DV) * 2 + (p.rel ? kSpanWaves * 64 * sizeof(float) : 0));
    auto go = [&](auto kernel) {
        // (more LDS than a launch gets without asking)
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
            return false;
        hipLaunchKernelGGL(kernel, grid, dim3(kSpanWaves * 64), lds, s, p);
        return true;
    };
    bool ok;
    if constexpr (D <= 128 && DV <= 128) ok = p.rel ? go(&span_attn_kernel<T, D, DV, KH, true>) : go(&span_attn_kernel<T, D, DV, KH, false>);
    else ok = go(&span_attn_kernel<T, D, DV, KH, false>);
    if (!ok) return SWL_ERR_LAUNCH;
    if (key_splits > 1) {
        const int64_t rows = p.num_tokens * p.H;
        hipLaunchKernelGGL((window_attn_combine_kernel<T>), dim3(static_cast<unsigned>(rows)), dim3(DV < 256 ? 64 : 256), 0, s,
                           static_cast<T *>(p.out), p.part_o, p.part_ml, rows, DV, key_splits, p.sink, p.H, p.out_f32, p.out_dim,
                           p.out_stride, static_cast<const T *>(p.gate), p.gate_stride);
    }
    return check_launch();
}

// Two waves a row group halve a workgroup's walk, one halves the workgroups, the pages they stage and what each spends before its first
// stage. us by workgroups of 64 rows, 128 + 128 columns, two / one: 11 x 333 tokens, 458: 16.8 / 18.4; 3 x 1500, 562: 39 / 54; 32 x 100, 800: 21.5 /
// 15.3; 22 x 333, 916: 28.8 / 23.0; 8 x 920, 920: 44 / 41; 5 x 1472, 920: 54 / 53; 4 x 1841, 920: 73 / 73, with a bias 72 / 79; 3 x 2450, 924:
// 79 / 82; 7200, 900: 193 / 221; 4 x 1841, 1840: 120 / 115. The longest walk may be a decoded token's: 22 x 333 beside one at 2000 keys 43.6 / 66.9,
// beside one at 8000 141 / 240 (972). Rows of 192 + 128, a key head for each query head: two are never the slower ones (expansion and rotary of
// latent rows included, 16 heads: 4 x 2000 tokens 350 / 474, 40 x 100 98 / 110, 11 x 333 81 / 79).
template <typename T, int D, int DV>
int launch_span_any(SpanParams &p, int key_splits, int longest, hipStream_t s) {
    if constexpr (span_halves(D, DV) == 2) {
        const int64_t workgroups = static_cast<int64_t>(p.num_spans) * p.G * kSpan / span_queries(p.H / p.G, 64);
        if (D + DV > 256 || workgroups <= 640 || (workgroups <= 1024 && longest >= 1536)) return launch_span<T, D, DV, 2>(p, key_splits, s);
    }
    return launch_span<T, D, DV, 1>(p, key_splits, s);
}

} // namespace swl

#define SWL_SPAN_SHAPES(X) X(64, 64) X(64, 128) X(128, 64) X(128, 128) X(192, 128) X(320, 256) X(576, 512)

/* 1 when swl_span_attn serves this shape. */
extern "C" int swl_span_attn_supported(int32_t num_q_heads, int32_t num_kv_heads, int32_t num_v_heads, int32_t dim, int32_t vdim,
                                       int32_t has_rel, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    if (num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return 0;
    if (num_v_heads <= 0 || num_kv_heads % num_v_heads) return 0;
    const int rep = num_q_heads / num_kv_heads;
    if (rep > 64 || num_kv_heads > 65535) return 0;
    // (a wave's bias window is one head's: its 16 rows are queries of one)
    if (has_rel && (rep > 4 || dim > 128 || vdim > 128)) return 0;
#define SWL_SPAN_IS(DD, DDV) if (dim == DD && vdim == DDV) return 1;
    SWL_SPAN_SHAPES(SWL_SPAN_IS)
#undef SWL_SPAN_IS
    return 0;
}

/* span_order: the spans in the order in which workgroups take them up (a permutation, or NULL); longest: tokens of the longest sequence
 * (0: not known). */
extern "C" int swl_span_attn_ordered(const int32_t *span_order, int32_t longest, void *out, const void *q, const void *k_cache, const void *v_cache, const int32_t *block_table,
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
    p.span_row0 = span_row0; p.span_cnt = span_cnt; p.span_order = span_order;
    p.rel = rel; p.sink = sink; p.slopes = slopes; p.gate = gate;
    // scratch: [splits][tokens][H][vdim] fp32 partial outputs, then [splits][tokens][H][2] (maximum, sum)
    p.part_o = scratch;
    p.part_ml = scratch ? scratch + static_cast<int64_t>(key_splits) * num_tokens * num_q_heads * vdim : nullptr;
    p.rel_len = rel_len; p.num_spans = num_spans; p.H = num_q_heads; p.G = num_kv_heads; p.GV = num_v_heads;
    p.window = window; p.mask_kind = mask_kind; p.max_blocks = max_blocks_per_seq; p.out_f32 = out_f32; p.out_dim = out_dim;
    p.scale = scale; p.softcap = softcap;
    p.q_stride = q_tok_stride; p.block_stride = block_stride; p.out_stride = out_stride; p.gate_stride = gate_stride;
    p.num_tokens = num_tokens;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define SWL_SPAN_GO(DD, DDV) if (dim == DD && vdim == DDV) return swl::launch_span_any<T, DD, DDV>(p, key_splits, longest, s);
    SWL_DISPATCH_DTYPE(dtype, T, { SWL_SPAN_SHAPES(SWL_SPAN_GO) });
#undef SWL_SPAN_GO
    return SWL_ERR_UNSUPPORTED;
}

extern "C" int swl_span_attn(void *out, const void *q, const void *k_cache, const void *v_cache, const int32_t *block_table,
                             const int32_t *tok_seq, const int32_t *tok_pos, const int32_t *tok_start, const int32_t *span_row0,
                             const int32_t *span_cnt, const float *rel, int32_t rel_len, int32_t num_spans, int32_t num_q_heads,
                             int32_t num_kv_heads, int32_t num_v_heads, int32_t dim, int32_t vdim, int64_t q_tok_stride,
                             int32_t window, int32_t mask_kind, float scale, float softcap, int32_t max_blocks_per_seq,
                             int64_t block_stride, int32_t key_splits, float *scratch, int64_t num_tokens, const float *sink,
                             int32_t out_f32, const float *slopes, int32_t out_dim, int64_t out_stride, const void *gate,
                             int64_t gate_stride, int32_t dtype, swl_stream_t stream) {
    return swl_span_attn_ordered(nullptr, 0, out, q, k_cache, v_cache, block_table, tok_seq, tok_pos, tok_start, span_row0, span_cnt, rel,
                                 rel_len, num_spans, num_q_heads, num_kv_heads, num_v_heads, dim, vdim, q_tok_stride, window, mask_kind,
                                 scale, softcap, max_blocks_per_seq, block_stride, key_splits, scratch, num_tokens, sink, out_f32, slopes,
                                 out_dim, out_stride, gate, gate_stride, dtype, stream);
}
