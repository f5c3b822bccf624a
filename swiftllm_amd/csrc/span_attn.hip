// span_attn.hip — the matrix-core attention of prompt portions over the paged pool, for heads that are not mixed
// (swl_masked_attn_tiles' masks, bias, slopes, cap, sink, gate; same pool layout, same arithmetic up to the order of sums).
//
// A ROW is one (query, query head) pair: every head of a kv group reads the same keys, so one staged page serves all of them (QT = rows / heads
// queries a workgroup, heads rounded up to a power of two).
//   S^T = K Q^T   A = keys from LDS, B = a wave's query fragments (registers for the whole walk)
//   online softmax: lane l owns row l % 16 (32), the four (two) lanes of a row hold its keys between them
//   O^T += V^T P^T  A = value columns from LDS, B = the score registers. Which key an A row of S^T takes is chosen so that a lane's
//                   eight scores of a step are eight CONSECUTIVE keys, which is what the B operand wants and what a page's
//                   transposed values hold in 16 bytes - no data moves between lanes. (Values in two 16-bit terms, hi + lo, so that a weight
//                   keeps 16 bits of its fp32 value: the matrix steps are D + 2 DV columns a (row, key).)
// What bounds it: what a wave does between two barriers is a chain (addresses, scores, their maximum, weights, values), of which two to four
// waves a SIMD hide a part. 128 + 128 columns, a tile of 32 rows and 32 keys: matrix steps 770 cycles of a SIMD, vector work 760, fragments read
// 500 (32 rows a wave) or 1000 (16 rows) of the CU's LDS; 2700 are taken.
//   * span_attn_kernel, rows of 256 elements and more: eight waves of 16 rows, four a SIMD.
//   * span_attn_narrow_kernel: four waves of 32 rows (mfma 32x32x16: half the fragment reads), three a SIMD, the next stage's score products
//     between this stage's weights. At 128 + 128 columns its registers leave two waves a SIMD, and it takes as long as the other.
// Two waves share a row group and take 32 keys each of a stage of 64 (64 rows a workgroup) in steps of a few workgroups a CU: a workgroup's walk, the
// longest chain of a step, is half as many stages. Otherwise stages of 32 keys, 128 rows (launch_span_any). Four fragments are on their way from
// LDS ahead of their matrix step, and nothing the compiler loads is pending inside the walk: its waits for such loads would be waits for the
// stage that was just asked for.
// Pages are staged by LDS-DMA (1 KiB per wave instruction, full lines) into two buffers with one barrier a stage (three stages ahead instead of
// one changed nothing); the swizzle that keeps the 16-byte fragment reads of keys off each other's banks is applied to the source addresses.
// A value that is NaN or infinite reaches every row of a workgroup that stages its page (a weight of 0 times it), as it does in the tiles
// of window_attn_mfma.hip: rows of the same portion whose queries come before it, at most 127 of them; never another sequence's.
// us a launch, bf16, with sixteen rows a wave and an address for every KiB / now: 4 x 2000 tokens, 8 heads of 128 over 2 key heads 77 / 72, with a
// bias by distance 83 / 77; 11 x 333, 16 over 4: 26.3 / 26.0; 3 x 1500, 32 heads of 64 + 128 over 16 in windows of 1024: 160 / 87; 4 x 900, 8 of 128 +
// 64 over one 25.8 / 22.6; 3 x 1500, 4 of 64 30.1 / 26.8. (By the 16-row kernel of window_attn_mfma.hip the first took 489.)
#include "attn_combine.h"
#include "swl_common.h"

namespace swl {

__device__ __forceinline__ float4_t mfma_step(vec8_t<f16> a, vec8_t<f16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mfma_step(vec8_t<bf16> a, vec8_t<bf16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float16_t span_mfma(vec8_t<f16> a, vec8_t<f16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float16_t span_mfma(vec8_t<bf16> a, vec8_t<bf16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
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
constexpr int kSpanWaves = 8, kSpanNarrowWaves = 4;
constexpr int kSpanKeys = 32;   // keys of a wave and stage
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

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

// What a workgroup works on: qt queries of one portion, as several spans (qt > 32) or a part of one.
struct SpanWork {
    int row0, cnt, p0;      // first row, rows, position of the first (cnt <= 0: nothing)
    int g;                  // key head
    const int32_t *bt;      // the sequence's block table
    int kb0, kb1;           // first and last page of this workgroup's share of the visible keys

    __device__ __forceinline__ int nstages(int pages) const { return kb1 >= kb0 ? (kb1 - kb0 + pages) / pages : 0; }
};
__device__ __forceinline__ int span_first_key(const SpanParams &p, int pos) {
    return p.window <= 0 ? 0 : p.mask_kind == 1 ? (pos / p.window) * p.window : max(pos - p.window + 1, 0);
}
// stage_pages: pages of a stage (a key split's shares are whole stages but for the last one's)
template <bool PAIRS>
__device__ __forceinline__ SpanWork span_work(const SpanParams &p, int stage_pages) {
    SpanWork w;
    const int qt = p.qt, per_span = qt < kSpan ? kSpan / qt : 1;
    int at = blockIdx.x;
    w.g = blockIdx.z;
    w.cnt = 0;
    span_place<PAIRS>(4 * per_span, at, w.g);
    int span = at / per_span;
    const int sub = at - span * per_span;
    // (later spans of a portion see more keys: they go first, over all portions where the caller says so)
    span = __builtin_amdgcn_readfirstlane(p.span_order ? min(max(p.span_order[span], 0), p.num_spans - 1) : p.num_spans - 1 - span);
    w.row0 = __builtin_amdgcn_readfirstlane(p.span_row0[span]);
    int cnt = __builtin_amdgcn_readfirstlane(p.span_cnt[span]);
    const int p_first = __builtin_amdgcn_readfirstlane(p.tok_pos[w.row0]);
    if (qt > kSpan) {
        const int per = qt / kSpan, nth = (p_first - __builtin_amdgcn_readfirstlane(p.tok_start[w.row0])) / kSpan;
        if (nth % per) return w;      // (an earlier span's workgroup takes these queries)
        const int seq = __builtin_amdgcn_readfirstlane(p.tok_seq[w.row0]);
        for (int i = 1; i < per && span + i < p.num_spans; ++i) {
            const int r = __builtin_amdgcn_readfirstlane(p.span_row0[span + i]);
            if (p.tok_seq[r] != seq) break;
            cnt += __builtin_amdgcn_readfirstlane(p.span_cnt[span + i]);
        }
    } else {
        w.row0 += sub * qt;
        cnt = min(qt, cnt - sub * qt);
        if (cnt <= 0) return w;
    }
    w.cnt = cnt;
    w.p0 = qt < kSpan ? p_first + sub * qt : p_first;
    w.bt = p.block_table + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(p.tok_seq[w.row0])) * p.max_blocks;
    w.kb0 = span_first_key(p, w.p0) / 16;
    w.kb1 = (w.p0 + cnt - 1) / 16;
    if (gridDim.y > 1) {        // key split: a contiguous share of the pages (possibly none)
        const int shares = static_cast<int>(gridDim.y), per = ((w.kb1 - w.kb0 + shares) / shares + stage_pages - 1) / stage_pages * stage_pages;
        w.kb0 += per * static_cast<int>(blockIdx.y);
        w.kb1 = min(w.kb1, w.kb0 + per - 1);
    }
    return w;
}

// One lane's part of a row's result: groups of four columns, o(i) those from col(i) on, unnormalised; mrun in base-2 units, l the row's sum.
template <typename T, int DV, int GROUPS, typename Col, typename Get>
__device__ __forceinline__ void span_store(const __attribute__((address_space(4))) SpanParams &e, int64_t orow, int head, bool first, float mrun, float l,
                                           Col &&col, Get &&get) {
    constexpr float kLog2e = 1.4426950408889634f;
    if (gridDim.y > 1) {        // partial result of this key share: unnormalised O, running maximum, sum
        const int64_t slot = (static_cast<int64_t>(blockIdx.y) * e.num_tokens + orow) * e.H + head;
#pragma unroll
        for (int i = 0; i < GROUPS; ++i) *reinterpret_cast<float4_t *>(e.part_o + slot * DV + col(i)) = get(i);
        if (first) {
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
    for (int i = 0; i < GROUPS; ++i) {
        const int c = col(i);
        if (c >= e.out_dim) continue;
        const int64_t hc = static_cast<int64_t>(head) * e.out_dim + c, at = orow * e.out_stride + hc;
        float4_t o = get(i);
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] *= inv;
        if (e.out_dim & 3) {        // (uniform) element by element
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (c + k >= e.out_dim) continue;
                if (gate) o[k] /= 1.0f + fast_exp2(-kLog2e * to_f(gate[orow * e.gate_stride + hc + k]));
                if (e.out_f32) reinterpret_cast<float *>(e.out)[at + k] = o[k];
                else out[at + k] = to_t<T>(o[k]);
            }
            continue;
        }
        if (gate) {
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] /= 1.0f + fast_exp2(-kLog2e * to_f(gate[orow * e.gate_stride + hc + k]));
        }
        if (e.out_f32) {
            *reinterpret_cast<float4_t *>(reinterpret_cast<float *>(e.out) + at) = o;
        } else {
            vec4_t<T> w;
#pragma unroll
            for (int k = 0; k < 4; ++k) w[k] = to_t<T>(o[k]);
            *reinterpret_cast<vec4_t<T> *>(out + at) = w;
        }
    }
}

// 256 bytes (4 a lane) of `base` + the lane's `off` to the LDS address `to`
__device__ __forceinline__ void span_ask4(const void *base, unsigned off, unsigned to) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(off), "s"(base), "s"(to) : "memory");
}

// The scores as they are compared and their unit in powers of two: products of queries and keys where nothing is done to them but the scale,
// the model's logits otherwise (capped ones in base-2 units already). A scale that leaves kNegBig no mask is applied first.
struct SpanScores {
    bool capped, plain;
    float c_mul, unit, cap, cap2, rel_mul;
    template <bool REL>
    __device__ __forceinline__ static SpanScores of(const SpanParams &p) {
        constexpr float kLog2e = 1.4426950408889634f;
        SpanScores c;
        c.capped = p.softcap > 0.f;
        c.plain = !REL && !c.capped && !p.slopes && p.scale > 1e-20f;
        c.c_mul = c.capped ? 2.0f * kLog2e * p.scale / p.softcap : p.scale;
        c.unit = c.plain ? p.scale * kLog2e : c.capped ? 1.0f : kLog2e;
        c.cap = p.softcap * kLog2e;
        c.cap2 = -2.0f * p.softcap * kLog2e;
        c.rel_mul = c.capped ? kLog2e : 1.0f;
        return c;
    }
    // N scores; REL: entry rl[-off(j)] is score j's bias; slope: off the score a key of distance (d0 - off(j))
    template <bool REL, int N, typename Off>
    __device__ __forceinline__ void apply(float (&x)[N], bool sloped, float slope, float d0, const float *rl, Off &&off) const {
        constexpr float kLog2e = 1.4426950408889634f;
        if (capped) {       // cap tanh(x / cap) = cap - 2 cap / (2^(2 log2(e) x / cap) + 1); overflow gives cap, underflow -cap
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] = fmaf(cap2, __builtin_amdgcn_rcpf(fast_exp2(x[j] * c_mul) + 1.0f), cap);
        } else if (!REL && !plain) {
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] *= c_mul;
        }
        if constexpr (REL) {
            if (capped) {
#pragma unroll
                for (int j = 0; j < N; ++j) x[j] = fmaf(rl[-off(j)], kLog2e, x[j]);
            } else {
#pragma unroll
                for (int j = 0; j < N; ++j) x[j] = fmaf(x[j], c_mul, rl[-off(j)]);
            }
        }
        if (sloped) {
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] = fmaf(-slope, d0 - static_cast<float>(off(j)), x[j]);
        }
    }
};

// Rows of less than 256 elements (keys and values): four waves of 32 rows, KH of them share a row group's keys.
template <typename T, int D, int DV, int KH, bool REL>
__global__ __launch_bounds__(kSpanNarrowWaves * 64, 2) void span_attn_narrow_kernel(SpanParams p) {
    static_assert(D % 64 == 0 && DV % 32 == 0, "");
    constexpr int NW = kSpanNarrowWaves, RG = NW / KH;                // row groups
    constexpr int KW = kSpanKeys, KT = KW * KH, NP = KT / 16;   // keys of a stage: a wave's, all of them, their pages
    constexpr int KU = D / 8, KI = D / 32, VI = DV / 32;        // units of a K row; KiB of a page's keys, values
    constexpr int KA = KI * NP / NW, VA = VI * NP / NW;         // KiB of a stage's keys, values that a wave asks for
    static_assert(NW % NP == 0 && KI * NP % NW == 0 && VI * NP % NW == 0, "");
    constexpr int KB = KT * D * 2, VB = KT * DV * 2, BUF = KB + VB;
    constexpr int HW = KH == 2 ? 2 : 1;             // (REL) heads whose rows a wave may hold
    constexpr int NV = 16, CT = DV / 32, KS = D / 16;       // scores of a lane; value tiles; steps of a score
    constexpr int KF = KU % 16 == 0 ? 8 : 4;        // steps whose units the exchange tells apart
    constexpr int AHEAD = 4;                        // fragments on their way from LDS
    constexpr float kLog2e = 1.4426950408889634f;
    constexpr float kLazy = 8.0f;       // (base-2 units: weights stay below 2^8)
    extern __shared__ __attribute__((aligned(16))) char smem[];     // keys of two stages, values of two, then (REL) the waves' bias windows of both

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rg = wave % RG, kh = wave / RG;       // this wave's row group and which of its keys
    const int l32 = lane & 31, hf = lane >> 5;      // row (or operand row); which of the row's two lanes
    const int rep = p.H / p.G, qt = p.qt;
    const SpanWork w = span_work<(2 * BUF <= 80 * 1024)>(p, NP);
    if (w.cnt <= 0) return;
    const int row0 = w.row0, cnt = w.cnt, p0 = w.p0, g = w.g;

    // ---- this lane's row: head R / qt of the group, query R % qt --------------------------------------------------------------
    const int my_hr = (rg * 32 + l32) / qt, my_head = g * rep + min(my_hr, rep - 1), qi = min(rg * 32 + l32 - my_hr * qt, cnt - 1);
    const int qpos = p0 + qi;
    const int qlo = span_first_key(p, qpos);
    // queries of this wave (uniform): positions [wp0, wp1]
    const int w_qr = qt >= 32 ? (rg * 32) % qt : 0;
    const int wp0 = p0 + min(w_qr, cnt - 1), wp1 = p0 + min(qt >= 32 ? w_qr + 31 : qt - 1, cnt - 1);
    const bool idle = (rg * 32) / qt >= rep || (qt >= 32 && w_qr >= cnt);     // no live row in this wave
    const int nstages = w.nstages(NP);

    vec8_t<T> qf[KS];
    {
        const T *qp = static_cast<const T *>(p.q) + static_cast<int64_t>(row0 + qi) * p.q_stride + static_cast<int64_t>(my_head) * D + hf * 8;
#pragma unroll
        for (int e = 0; e < KS; ++e) qf[e] = load8(qp + e * 16);
    }
    float16_t acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[ct] = float16_t{};
    float mrun = kNegBig, lrun = 0.f;

    // ---- staging: a wave's KiB of a stage's keys, and of its values, are of one page (one address to work out; scalar work of the walk) ------
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    const char *kc = static_cast<const char *>(p.k_cache) + static_cast<int64_t>(g) * 16 * D * 2;
    const char *vc = static_cast<const char *>(p.v_cache) + static_cast<int64_t>(g % p.GV) * 16 * DV * 2;
    const int64_t bstride = p.block_stride * 2;
    // block ids: lane i holds that of page id_base + i of this share (past the last visible page: that page again), 64 pages a load; the
    // values are a stage behind the keys, and id_before the 64 pages before
    int id_base = 0, id_lane = 0, id_before = 0;
    auto fetch_ids = [&]() {
        id_before = id_lane;
        id_lane = w.bt[min(w.kb0 + id_base + lane, w.kb1)];
        asm volatile("" : "+v"(id_lane));       // (waited for here, not in front of every use, behind what is asked for in between)
    };
    constexpr int WP = NW / NP;         // waves of a page
    const int my_page = wave / WP, my_part = wave % WP;
    unsigned src[KA];
#pragma unroll
    for (int j = 0; j < KA; ++j) {
        const int unit = (my_part * KA + j) * 64 + lane;
        src[j] = static_cast<unsigned>((unit ^ span_k_flip<KU>(unit / KU, my_page)) * 16);
    }
    unsigned vsrc[VA];
#pragma unroll
    for (int j = 0; j < VA; ++j) vsrc[j] = static_cast<unsigned>((my_part * VA + j) * 1024 + lane * 16);
    auto block = [&](int stage) {
        const int i = stage * NP + my_page - id_base;
        const int now = __builtin_amdgcn_readlane(id_lane, i & 63), before = __builtin_amdgcn_readlane(id_before, i & 63);
        return static_cast<int64_t>(i >= 0 ? now : before) * bstride;
    };
    const unsigned to_keys = lds0 + static_cast<unsigned>(my_page * 16 * D * 2 + my_part * KA * 1024);
    const unsigned to_values = lds0 + 2 * KB + static_cast<unsigned>(my_page * 16 * DV * 2 + my_part * VA * 1024);
    auto ask_keys = [&](int stage) {
        lds_ask<KA>(kc + block(stage), src, to_keys + static_cast<unsigned>(stage & 1) * KB);
    };
    // (REL) the wave's windows of its heads' bias, entry i: distance wp0 - (its first key of the stage) - (KW - 1) + i
    float *const rel_lds = reinterpret_cast<float *>(smem + 2 * BUF) + wave * HW * 64;       // [2][NW][HW][64]
    auto ask_values = [&](int stage) {
        lds_ask<VA>(vc + block(stage), vsrc, to_values + static_cast<unsigned>(stage & 1) * VB);
        if constexpr (REL) {
            const int d = wp0 - (w.kb0 + stage * NP) * 16 - kh * KW - (KW - 1) + lane, head = (rg * 32) / qt;
            const unsigned off = static_cast<unsigned>(min(max(d, 0), p.rel_len - 1)) * 4,
                           to = lds0 + 2 * BUF + static_cast<unsigned>(((stage & 1) * NW + wave) * HW) * 256;
#pragma unroll
            for (int h = 0; h < HW; ++h)
                if (h == 0 || qt < 32) span_ask4(p.rel + static_cast<int64_t>(g * rep + min(head + h, rep - 1)) * p.rel_len, off, to + h * 256);
        }
    };
    // fragment reads (bytes). K: A row m is key 16 (m / 16) + 8 (m / 4 % 2) + 4 (m / 8 % 2) + m % 4, unit 2 e + hf (the exchange touches the
    // unit's low bits only); V: column l32, keys 8 hf .. 8 hf + 7 of a page
    int k_frag;
    {
        const int key = 16 * (l32 >> 4) + 8 * ((l32 >> 2) & 1) + 4 * ((l32 >> 3) & 1) + (l32 & 3);
        k_frag = (kh * KW + key) * D * 2 + ((hf ^ span_k_flip<KU>(key & 15, key >> 4)) * 16);
    }
    const unsigned v_frag = static_cast<unsigned>(kh * KW * DV * 2 + l32 * 32 + hf * 16);
    auto off = [](int j) { return 16 * (j >> 3) + (j & 7); };      // score j of the lane: key k0 + 8 hf + off(j)

    const SpanScores sc = SpanScores::of<REL>(p);
    const float slope = p.slopes ? p.slopes[my_head] * sc.rel_mul : 0.f;
    auto first_of = [&](int stage) { return (w.kb0 + stage * NP) * 16 + kh * KW; };
    // stages with a key that a query of this wave sees: first_live .. last_live (no test inside the walk: its other way would take the results'
    // registers once more)
    int first_live = nstages, last_live = -1;
    if (!idle) {
        constexpr int SK = NP * 16;
        const int before = span_first_key(p, wp0) - (first_of(0) + KW - 1), within = wp1 - first_of(0);
        first_live = before > 0 ? (before + SK - 1) / SK : 0;
        last_live = within >= 0 ? min(within / SK, nstages - 1) : -1;
        if (first_live > last_live) first_live = nstages;
    }
    float16_t s;        // scores of the stage to come
    auto key_at = [&](int stage, int e) {
        // (unit 2 e + hf, exchanged: rows start at multiples of KF units' bytes, so the step's bits are exchanged where they lie)
        return *reinterpret_cast<const vec8_t<T> *>(smem + (stage & 1) * KB + (k_frag ^ (e % KF * 32)) + e / KF * KF * 32);
    };

    if (nstages > 0) fetch_ids();
    // what the compiler itself loads has arrived before the walk: a load that might still be on its way at the loop's head is waited
    // for in every turn of it, and with it the stage that was asked for just before
#pragma unroll
    for (int e = 0; e < KS; ++e) asm volatile("" : "+v"(qf[e]));
    auto score = [&](int stage) {
        s = float16_t{};
        lds_steps<AHEAD, KS, 1, vec8_t<T>>([&](int e) { return key_at(stage, e); }, [&](int e, vec8_t<T> kf) { s = span_mfma(kf, qf[e], s); });
    };
    auto turn = [&](int st) {
        // this wave's pieces of the next keys and of these values have landed, its reads of what is overwritten now have returned
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();       // ... and everyone's
        if (st + 2 < nstages) {
            if ((st + 2) * NP - id_base >= 64) {
                id_base += 64;
                fetch_ids();
            }
            ask_keys(st + 2);
        }
        if (st + 1 < nstages) ask_values(st + 1);
    };
    if (nstages > 0) {
        ask_keys(0);
        ask_values(0);
        constexpr int VN = VA + (REL ? 1 : 0);      // (at least this many were asked for after the keys)
        if (nstages > 1) {
            ask_keys(1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(VN + KA) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(VN) : "memory");
        }
        __builtin_amdgcn_s_barrier();
    }
    for (int st = 0; st < first_live; ++st) turn(st);
    if (first_live < nstages) score(first_live);
    for (int st = first_live; st <= last_live; ++st) {
        turn(st);
        mfma_results_ready<8>(s);
        const int k0 = first_of(st);
        float x[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) x[j] = s[j];
        const int kd = qpos - k0 - 8 * hf;      // distance of this lane's first key
        const float *rl = REL ? rel_lds + ((st & 1) * NW * HW + (qt < 32 ? (rg * 32 + l32) / qt - (rg * 32) / qt : 0)) * 64 + (qpos - wp0) + (KW - 1) - 8 * hf : nullptr;
        sc.template apply<REL>(x, p.slopes != nullptr, slope, static_cast<float>(kd), rl, off);
        if (k0 + KW - 1 > wp0 || (p.window > 0 && k0 < span_first_key(p, wp1))) {      // (uniform) the keys cross a row's limits
            const int lo = qlo - k0 - 8 * hf;       // visible: lo <= key - (k0 + 8 hf) <= kd
#pragma unroll
            for (int j = 0; j < NV; ++j)
                if (off(j) > kd || off(j) < lo) x[j] = kNegBig;
        }
        // ---- the weights, and between them the score products of the next stage (of none after the last: never looked at) -------------
        // (the order is held step by step: left alone, the compiler takes the products one after another, each behind its own read)
        __builtin_amdgcn_sched_barrier(0);
        vec8_t<T> ring[AHEAD];
#pragma unroll
        for (int e = 0; e < AHEAD; ++e) ring[e] = key_at(st + 1, e);
        __builtin_amdgcn_sched_barrier(0);
        float mx = x[0];
#pragma unroll
        for (int j = 1; j < NV; ++j) mx = fmaxf(mx, x[j]);
        {
            const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
        }
        // lazy running maximum: a row moves its reference only when a stage raises it by more than kLazy
        const float mnew = (mx - mrun) * sc.unit > kLazy ? mx : mrun;
        const float alpha = fast_exp2((mrun - mnew) * sc.unit);
        mrun = mnew;
        // (a row that has seen no key yet: all its weights are 2^-1e30 = 0)
        const float mref = mnew < 0.5f * kNegBig ? 0.f : -mnew * sc.unit;
        float psum[2] = {0.f, 0.f};
        uint4v hi[2], lo[2];
        s = float16_t{};
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < KS; ++e) {
            s = span_mfma(ring[e % AHEAD], qf[e], s);
            if (e + AHEAD < KS) ring[e % AHEAD] = key_at(st + 1, e + AHEAD);
#pragma unroll
            for (int i = e * 8 / KS; i < (e + 1) * 8 / KS; ++i) {      // weights 2 i and 2 i + 1
                const float a = fast_exp2(fmaf(x[2 * i], sc.unit, mref)), b = fast_exp2(fmaf(x[2 * i + 1], sc.unit, mref));
                psum[0] += a;
                psum[1] += b;
                unsigned h, l;
                split_pair<T>(a, b, h, l);
                hi[i >> 2][i & 3] = h;
                lo[i >> 2][i & 3] = l;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        lrun = fmaf(lrun, alpha, psum[0] + psum[1]);
        asm volatile("" : "+v"(hi[0]), "+v"(hi[1]), "+v"(lo[0]), "+v"(lo[1]));       // (made here, not behind the branch)
        __builtin_amdgcn_sched_barrier(0);
        if (!__all(alpha == 1.0f)) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[ct][i] *= alpha;
        }
        // (step i: keys 16 (i % 2) .., value tile i / 2)
        const char *vp = smem + 2 * KB + (st & 1) * VB + v_frag;
        lds_steps<AHEAD, 2 * CT, 2, vec8_t<T>>(
            [&](int i) { return *reinterpret_cast<const vec8_t<T> *>(vp + (i & 1) * 16 * DV * 2 + (i >> 1) * 1024); },
            [&](int i, vec8_t<T> vf) {
                acc[i >> 1] = span_mfma(vf, __builtin_bit_cast(vec8_t<T>, hi[i & 1]), acc[i >> 1]);
                acc[i >> 1] = span_mfma(vf, __builtin_bit_cast(vec8_t<T>, lo[i & 1]), acc[i >> 1]);
            });
    }
    for (int st = max(last_live + 1, first_live); st < nstages; ++st) turn(st);
#pragma unroll
    for (int ct = 0; ct + 1 < CT; ++ct) mfma_results_tie(acc[ct]);
    mfma_results_ready<8>(acc[CT - 1]);
    if (!sc.plain && !sc.capped) mrun *= kLog2e;      // base-2 units from here on (kNegBig stays one)
    if (sc.plain) mrun *= sc.unit;
    // ---- the two waves of a row group: the second hands its sums to the first (the stages' place is free) -----------------------
    if constexpr (KH == 2) {
        static_assert(RG * (4 * CT + 1) * 1024 <= 2 * BUF, "");
        __syncthreads();
        float4_t *mine = reinterpret_cast<float4_t *>(smem) + rg * (4 * CT + 1) * 64 + lane;
        if (kh == 1) {
#pragma unroll
            for (int i = 0; i < 4 * CT; ++i) mine[i * 64] = float4_t{acc[i / 4][i % 4 * 4], acc[i / 4][i % 4 * 4 + 1], acc[i / 4][i % 4 * 4 + 2], acc[i / 4][i % 4 * 4 + 3]};
            mine[4 * CT * 64] = float4_t{mrun, lrun, 0.f, 0.f};
        }
        __syncthreads();
        if (kh == 1) return;
        const float4_t ml = mine[4 * CT * 64];
        const float m = fmaxf(mrun, ml[0]), a0 = fast_exp2(mrun - m), a1 = fast_exp2(ml[0] - m);
        lrun = lrun * a0 + ml[1] * a1;
        mrun = m;
#pragma unroll
        for (int i = 0; i < 4 * CT; ++i) {
            const float4_t o = mine[i * 64];
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[i / 4][i % 4 * 4 + k] = acc[i / 4][i % 4 * 4 + k] * a0 + o[k] * a1;
        }
    }
    // ---- epilogue: acc[ct][4 q + r] = O[row][32 ct + 8 q + 4 hf + r] ------------------------------------------------------------------
    // (its parameters are loaded here: kept over the walk, they take the registers of other uniform values)
    const auto *again = (const __attribute__((address_space(4))) SpanParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(again));
    const float l = lrun + __shfl_xor(lrun, 32, 64);
    const int R = rg * 32 + l32, hr = R / qt, qr = R - hr * qt;
    if (hr >= rep || qr >= cnt) return;
    span_store<T, DV, 4 * CT>(*again, row0 + qr, g * rep + hr, hf == 0, mrun, l, [&](int i) { return 8 * i + 4 * hf; },
                              [&](int i) { return float4_t{acc[i / 4][i % 4 * 4], acc[i / 4][i % 4 * 4 + 1], acc[i / 4][i % 4 * 4 + 2], acc[i / 4][i % 4 * 4 + 3]}; });
}

// Rows of 256 elements and more: eight waves of 16 rows, KH of them share a row group's keys.
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
    const SpanWork w = span_work<(2 * BUF <= 80 * 1024)>(p, NP);
    if (w.cnt <= 0) return;
    const int row0 = w.row0, cnt = w.cnt, p0 = w.p0, g = w.g;

    // ---- this lane's row: head R / qt of the group, query R % qt --------------------------------------------------------------
    const int my_hr = (rg * 16 + lr) / qt, my_head = g * rep + min(my_hr, rep - 1), qi = min(rg * 16 + lr - my_hr * qt, cnt - 1);
    const int qpos = p0 + qi;
    const int qlo = span_first_key(p, qpos);
    // queries of this wave (uniform): positions [wp0, wp1]
    const int w_qr = qt >= 16 ? (rg * 16) % qt : 0;
    const int wp0 = p0 + min(w_qr, cnt - 1), wp1 = p0 + min(qt >= 16 ? w_qr + 15 : qt - 1, cnt - 1);
    const bool idle = (rg * 16) / qt >= rep || (qt >= 16 && w_qr >= cnt);     // no live row in this wave
    const int nstages = w.nstages(NP);

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
    auto fetch_ids = [&]() { id_lane = w.bt[min(w.kb0 + id_base + lane, w.kb1)]; };
    float *const rel_lds = reinterpret_cast<float *>(smem + 2 * BUF) + wave * 64;       // (REL) [2][NW][64]
    const float *rel_row = REL ? p.rel + static_cast<int64_t>(g * rep + min((rg * 16) / qt, rep - 1)) * p.rel_len : nullptr;
    // Rows that are not too wide: a wave asks for a part of one page's keys or of its values, one address a stage to work out (the scalar work of
    // eight waves' addresses was a tenth of a walk: 4 x 2000 tokens, 8 heads of 128 over 2, 77.1 -> 71.8 us). Else a page is KI + VI KiB, KiB u of
    // every page of a stage is asked for by wave u % NW: its lanes' places in it are the same for every page but for the flip of odd pages' keys.
    constexpr int WP = NW / (2 * NP);       // waves of a page's keys, and of its values
    constexpr bool PARTS = KI % WP == 0 && VI % WP == 0 && KI / WP <= 6 && VI / WP <= 6;
    constexpr int PK = PARTS ? KI / WP : 1, PV = PARTS ? VI / WP : 1, PM = PARTS ? (PK > PV ? PK : PV) : US;       // KiB of a wave
    const int my_page = wave / (2 * WP), my_part = wave % WP;
    const bool my_keys = wave / WP % 2 == 0;
    unsigned src[PM];
#pragma unroll
    for (int j = 0; j < PM; ++j) {
        if constexpr (PARTS) {
            const int unit = (my_part * (my_keys ? PK : PV) + j) * 64 + lane;
            src[j] = static_cast<unsigned>((my_keys ? unit ^ span_k_flip<KU>(unit / KU, my_page) : unit) * 16);
        } else {
            const int u = wave + NW * j, unit = u * 64 + lane;
            src[j] = static_cast<unsigned>(u < KI ? (unit ^ span_k_flip<KU>(unit / KU, 0)) * 16 : lane * 16);
        }
    }
    const char *my_base = my_keys ? kc : vc;
    const unsigned my_dst = lds0 + static_cast<unsigned>(my_keys ? my_page * 16 * D * 2 + my_part * PK * 1024 : KB + my_page * 16 * DV * 2 + my_part * PV * 1024);
    auto ask = [&](int stage) {
        if constexpr (PARTS) {
            const int64_t blk = static_cast<int64_t>(__builtin_amdgcn_readlane(id_lane, stage * NP - id_base + my_page)) * bstride;
            const unsigned dst = my_dst + static_cast<unsigned>(stage & 1) * BUF;
            if (PK == PV || my_keys) lds_ask<PK>(my_base + blk, src, dst);
            else lds_ask<PV>(my_base + blk, src, dst);
        } else {
            const unsigned dst = lds0 + static_cast<unsigned>(stage & 1) * BUF;
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
                    lds_ask<1>(base, {off}, to);
                }
            }
        }
        if constexpr (REL) {    // the wave's window of its head's bias, entry i: distance wp0 - (its first key of the stage) - (KW - 1) + i
            const int d = wp0 - (w.kb0 + stage * NP) * 16 - kh * KW - (KW - 1) + lane;
            const unsigned off = static_cast<unsigned>(min(max(d, 0), p.rel_len - 1)) * 4,
                           to = lds0 + 2 * BUF + static_cast<unsigned>((stage & 1) * NW + wave) * 256;
            span_ask4(rel_row, off, to);
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

    const SpanScores sc = SpanScores::of<REL>(p);
    const float slope = p.slopes ? p.slopes[my_head] * sc.rel_mul : 0.f;

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
        const int k0 = (w.kb0 + st * NP) * 16 + kh * KW;
        if (idle || k0 > wp1 || k0 + KW - 1 < span_first_key(p, wp0)) continue;
        const char *kbuf = smem + (st & 1) * BUF, *vbuf = kbuf + KB;
        float4_t s[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) s[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        // (step i: score tile i % NT, elements 32 (i / NT) ..)
        lds_steps<AHEAD, NT * KS, 1, vec8_t<T>>(
            [&](int i) { return *reinterpret_cast<const vec8_t<T> *>(kbuf + k_frag[i % NT][(i / NT) % KF] + (i / NT) / KF * KF * 64); },
            [&](int i, vec8_t<T> kf) { s[i % NT] = mfma_step(kf, qf[i / NT], s[i % NT]); });
        mfma_results_tie(s[0]);
        mfma_results_ready<8>(s[1]);
        // score j of the lane: key k0 + 8 lk + j
        float x[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) x[j] = s[j / 4][j % 4];
        const int kd = qpos - k0 - 8 * lk;      // distance of this lane's first key
        const float *rl = REL ? rel_lds + (st & 1) * NW * 64 + (qpos - wp0) + (KW - 1) - 8 * lk : nullptr;
        sc.template apply<REL>(x, p.slopes != nullptr, slope, static_cast<float>(kd), rl, [](int j) { return j; });
        if (k0 + KW - 1 > wp0 || (p.window > 0 && k0 < span_first_key(p, wp1))) {      // (uniform) the keys cross a row's limits
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
        const float mnew = (mx - mrun) * sc.unit > kLazy ? mx : mrun;
        const float alpha = fast_exp2((mrun - mnew) * sc.unit);
        mrun = mnew;
        // (a row that has seen no key yet: all its weights are 2^-1e30 = 0)
        const float mref = mnew < 0.5f * kNegBig ? 0.f : -mnew * sc.unit;
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            x[j] = fast_exp2(fmaf(x[j], sc.unit, mref));
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
        split_weights<T>(x, hi, lo);
        const char *vp = vbuf + v_frag;
        lds_steps<AHEAD, CT, 2, vec8_t<T>>([&](int ct) { return *reinterpret_cast<const vec8_t<T> *>(vp + ct * 512); },
                                            [&](int ct, vec8_t<T> vf) {
                                                acc[ct] = mfma_step(vf, hi, acc[ct]);
                                                acc[ct] = mfma_step(vf, lo, acc[ct]);
                                            });
    }
#pragma unroll
    for (int ct = 0; ct + 1 < CT; ++ct) mfma_results_tie(acc[ct]);
    mfma_results_ready<8>(acc[CT - 1]);
    if (!sc.plain && !sc.capped) mrun *= kLog2e;      // base-2 units from here on (kNegBig stays one)
    if (sc.plain) mrun *= sc.unit;
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
    const float l = span_row_sum(lrun);
    // (the lane's row once more: kept over the walk, it costs registers that the walk has no others for)
    int lane_again = lane;
    asm volatile("" : "+v"(lane_again));
    const int R = rg * 16 + (lane_again & 15), col = 4 * (lane_again >> 4), hr = R / qt, qr = R - hr * qt, head = g * rep + min(hr, rep - 1);
    if (hr >= rep || qr >= cnt) return;
    span_store<T, DV, CT>(*again, row0 + qr, head, col == 0, mrun, l, [&](int i) { return i * 16 + col; }, [&](int i) { return acc[i]; });
}

// queries of a workgroup for `rep` query heads a key head (64 at most): its rows over rep rounded up to a power of two
static int span_queries(int rep, int rows) {
    int up = 1;
    while (up < rep) up *= 2;
    return rows / up;
}

// KH: waves that share a row group's keys; 128 / KH (query, head) pairs a workgroup
template <typename T, int D, int DV, int KH>
int launch_span(SpanParams &p, int key_splits, hipStream_t s) {
    constexpr bool narrow = D + DV < 256;
    constexpr int waves = narrow ? kSpanNarrowWaves : kSpanWaves, windows = narrow ? kSpanNarrowWaves * KH : kSpanWaves;
    p.qt = span_queries(p.H / p.G, 128 / KH);
    if (p.rel && p.qt < (narrow && KH == 1 ? 32 : 16)) return SWL_ERR_UNSUPPORTED;      // (a wave's rows are of more heads than it has bias windows)
    const int per = p.qt < kSpan ? kSpan / p.qt : 1;
    const dim3 grid(static_cast<unsigned>(p.num_spans * per), static_cast<unsigned>(key_splits), static_cast<unsigned>(p.G));
    const size_t lds = 2 * (static_cast<size_t>(kSpanKeys * KH) * (D + DV) * 2 + (p.rel ? windows * 64 * sizeof(float) : 0));
    auto go = [&](auto kernel) {
        // (more LDS than a launch gets without asking)
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
            return false;
        hipLaunchKernelGGL(kernel, grid, dim3(waves * 64), lds, s, p);
        return true;
    };
    bool ok;
    if constexpr (narrow) ok = p.rel ? go(&span_attn_narrow_kernel<T, D, DV, KH, true>) : go(&span_attn_narrow_kernel<T, D, DV, KH, false>);
    else if constexpr (D <= 128 && DV <= 128) ok = p.rel ? go(&span_attn_kernel<T, D, DV, KH, true>) : go(&span_attn_kernel<T, D, DV, KH, false>);
    else ok = go(&span_attn_kernel<T, D, DV, KH, false>);
    if (!ok) return SWL_ERR_LAUNCH;
    if (key_splits > 1) {
        const int64_t rows = p.num_tokens * p.H;
        launch_attn_combine<T>(static_cast<T *>(p.out), p.part_o, p.part_ml, rows, DV, key_splits, p.sink, p.H, p.out_f32, p.out_dim,
                               p.out_stride, static_cast<const T *>(p.gate), p.gate_stride, s);
    }
    return check_launch();
}

// Two waves a row group halve a workgroup's walk, one halves the workgroups, the pages they stage and what each spends before its first
// stage. us by workgroups of 64 rows, 128 + 128 columns, two / one: 11 x 333 tokens, 458: 16.8 / 18.4; 3 x 1500, 562: 39 / 54; 32 x 100, 800: 21.5 /
// 15.3; 22 x 333, 916: 28.8 / 23.0; 8 x 920, 920: 44 / 41; 5 x 1472, 920: 54 / 53; 4 x 1841, 920: 73 / 73, with a bias 72 / 79; 3 x 2450, 924:
// 79 / 82; 7200, 900: 193 / 221; 4 x 1841, 1840: 120 / 115. The longest walk may be a decoded token's: 22 x 333 beside one at 2000 keys 43.6 / 66.9,
// beside one at 8000 141 / 240 (972). Of 128 rows and one or two heads a key
// head, the queries are several spans, whose other workgroups are launched to leave at once: two / one waves a row group, 16 heads over 16 of 64 + 128,
// 40 x 100 tokens 37.5 / 47.3; 32 over 16, 3 x 1500, 86 / 119; 16 over 16 of 192 + 128, 3 x 1500, 114 / 167 (of 128 + 128 both ways: the old line).
template <typename T, int D, int DV>
int launch_span_any(SpanParams &p, int key_splits, int longest, hipStream_t s) {
    if constexpr (span_halves(D, DV) == 2) {
        const int rep = p.H / p.G;
        const int64_t workgroups = static_cast<int64_t>(p.num_spans) * p.G * kSpan / span_queries(rep, 64);
        if ((D + DV != 256 && rep <= 2) || workgroups <= 640 || (workgroups <= 1024 && longest >= 1536))
            return launch_span<T, D, DV, 2>(p, key_splits, s);
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
    // (a wave holds the bias windows of one head, in the narrow kernel with two waves a row group of two: up to four heads a key head leave 16 or
    // 32 queries of a head to a workgroup of 64 or 128 rows; launch_span checks it)
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
