// window_attn.hip — attention over the paged KV pool with a sliding window, tanh soft-capping and pre-softmax head
// mixing ("talking heads": the capped scores of all query heads at one (query, key) pair are mixed by an [H, H] matrix
// before the softmax; without a matrix every head keeps its own) and an optional learned bias per (distance, head) added to
// the mixed scores, for any mixture of prompt portions and single decoded tokens.
//
// Every query token carries its sequence row and position; its own key/value are already in the pool (qknorm_kv.hip ran
// first), so a prompt portion that continues a cached prefix, a whole prompt and a decoded token are the same case:
// keys [max(0, p - window + 1), p] of the token's sequence, read through the block table.
//
// Because the mix couples the heads, one workgroup owns ALL heads of its query token. Keys are taken in chunks of four 16-key pages:
//   1. capped scores s[g][j] for every head g (fp32 dot products, fp32 tanh),
//   2. mixed scores  m[h][j] = sum_g talk[h][g] s[g][j], online softmax per mixed head h (fp32, full-precision exp),
//   3. acc[h][:] = acc[h][:] * alpha[h] + sum_j p[h][j] v[kv(h)][j][:]   (fp32 weights, fp32 accumulation).
// This is the reference-grade kernel: everything after the loads is fp32 whatever the storage dtype.
// What bounds it is latency: a step of a few tokens is a few workgroups, each a chain of chunks. Key rows are read by neighbouring lanes
// (one 512-byte row of 128 fp32 by half a wave) and serve four heads, a page's values are read once for the heads that share them
// (token_attn.h), and key_splits > 1 shares a token's pages out over workgroups whose partial results a second launch combines.
// 3 tokens at 513 keys, 8 heads of 128 over 2, fp32: 685 us with a key per thread and no shares, 18 us (16 shares and their sum; 8.4 in the
// form below).
//
// The general entry point (swl_masked_attn) adds what other designs need of the same loop:
//   * mask_kind 1: chunked visibility — keys [floor(p / window) * window, p], chunks counted from position 0;
//   * sink[H]: a learned logit per head that joins the softmax denominator only (no key, no value, not scaled);
//   * num_v_heads < num_kv_heads: several key heads share one value head (value head = key head % num_v_heads) — two
//     score maps over the same values, laid out map-major, are 2 G key heads over G value heads;
//   * out_f32: the result leaves in fp32 (for a combination of maps that cancels);
//   * slopes[H]: slope times the distance (query position - key position) is taken off the (capped) score;
//   * out_dim / out_stride: pages may hold values wider than the heads are (vdim columns, of which the first out_dim count) and the
//     result may be a column slice of wider rows; gate: the result is multiplied by sigmoid(gate[t][h * out_dim + c]);
//   * without a mixing matrix the heads are independent: more than 32 of them (or more than the accumulators and the LDS of
//     one workgroup hold) are shared out over blockIdx.y, every workgroup taking a group of consecutive heads.
#include "attn_combine.h"
#include "swl_common.h"
#include "token_attn.h"

namespace swl {

// fp32 words ahead of the page table (offsets of four blocks)
__host__ __device__ inline size_t wa_float_count(int H, int d) {
    const size_t n = static_cast<size_t>(H) * d + static_cast<size_t>(H) * H + 2 * static_cast<size_t>(H) * kTaChunk + 2 * static_cast<size_t>(H);
    return (n + 3) / 4 * 4 + 8;     // (the rows of weights start on 16-byte boundaries)
}

template <typename T, int R>
__global__ __launch_bounds__(kTaThreads, 2) void window_attn_kernel(
    T *out, const T *q, const T *k_cache, const T *v_cache, const int32_t *block_table, const int32_t *tok_seq,
    const int32_t *tok_pos, const float *talk, const float *rel, int rel_len, int H, int G, int d, int dv,
    int64_t q_tok_stride, int window, float scale, float softcap, int max_blocks_per_seq, int64_t block_stride,
    int mask_kind, const float *sink, int GV, int out_f32, int Hall, const float *slopes, int out_dim, int64_t out_stride,
    const T *gate, int64_t gate_stride, float *part_o, float *part_ml, int k_wide, int v_wide) {
    // H: heads of this workgroup, starting at head hb of the token's Hall heads (G: key heads per Hall query heads)
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float *s = lds;                         // [H][64] capped scores
    float *p = s + H * kTaChunk;            // [H][64] softmax numerators
    float *qf = p + H * kTaChunk;           // [H * d]
    float *tk = qf + (H * d + 3) / 4 * 4;   // [H * H]
    float *alpha = tk + H * H;              // [H]
    int64_t *pages = reinterpret_cast<int64_t *>(lds + wa_float_count(H, d));   // [4] element offset of each page's block

    const int64_t t = blockIdx.x;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int pos = tok_pos[t];
    const int32_t *bt = block_table + static_cast<int64_t>(tok_seq[t]) * max_blocks_per_seq;
    const int lo = window <= 0 ? 0 : mask_kind == 1 ? (pos / window) * window : (pos - window + 1 > 0 ? pos - window + 1 : 0);
    int kb0 = lo / kTaPage, kb1 = pos / kTaPage;
    if (gridDim.z > 1) {        // key split: a contiguous share of the pages (possibly none)
        const int per = (kb1 - kb0 + static_cast<int>(gridDim.z)) / static_cast<int>(gridDim.z);
        kb0 += per * static_cast<int>(blockIdx.z);
        kb1 = min(kb1, kb0 + per - 1);
    }
    const int rep = Hall / G;
    const int hb = static_cast<int>(blockIdx.y) * H;
    if (hb + H > Hall) H = Hall - hb;
    if (sink) sink += hb;
    if (rel) rel += static_cast<int64_t>(hb) * rel_len;
    if (slopes) slopes += hb;

    const T *qrow = q + t * q_tok_stride + static_cast<int64_t>(hb) * d;
    for (int i = tid; i < H * d; i += kTaThreads) qf[i] = to_f(qrow[i]);
    if (talk)
        for (int i = tid; i < H * H; i += kTaThreads) tk[i] = talk[i];

    float acc[kTaMaxAcc / R][R];
#pragma unroll
    for (int i = 0; i < kTaMaxAcc / R; ++i)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[i][r] = 0.f;
    // running maximum and sum of mixed head h live in the lanes of the wave that owns h (wave = h % 4): replicated
    float mrun[8], lrun[8];     // heads per wave <= 8: H <= 32
#pragma unroll
    for (int i = 0; i < 8; ++i) { mrun[i] = kNegBig; lrun[i] = 0.f; }
    const int hpw = (H + 3) / 4;     // heads per wave (host guarantees <= 8)

    for (int kb = kb0; kb <= kb1; kb += 4) {
        const int first = max(lo - kb * kTaPage, 0), last = min(min(pos, kb1 * kTaPage + kTaPage - 1) - kb * kTaPage, kTaChunk - 1);
        __syncthreads();    // previous chunk's p / alpha / pages fully consumed (and qf / tk written, first time)
        if (tid < 4) pages[tid] = bt[min(kb + tid, kb1)] * block_stride;
        __syncthreads();
        // 1. scores, capped in passing by the next step
        ta_scores(s, qf, k_cache, pages, first, last, H, hb, rep, d, k_wide != 0);
        __syncthreads();
        if (talk) {     // (every head's capped scores are mixed by every wave)
            for (int idx = tid; idx < H * kTaChunk; idx += kTaThreads) {
                const float a = s[idx] * scale;
                s[idx] = softcap > 0.f ? softcap * tanhf(a / softcap) : a;
            }
            __syncthreads();
        }
        // 2. mix the heads, online softmax per mixed head (wave `wave` owns heads wave, wave + 4, ...)
        const bool ok = lane >= first && lane <= last;
        const int dist = pos - (kb * kTaPage + lane);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int h = wave + 4 * i;
            if (i >= hpw || h >= H) break;
            float mixed = kNegBig;
            if (ok) {
                float a = 0.f;
                if (talk) {
                    for (int g = 0; g < H; ++g) a += tk[h * H + g] * s[g * kTaChunk + lane];
                } else {
                    a = s[h * kTaChunk + lane] * scale;
                    if (softcap > 0.f) a = softcap * tanhf(a / softcap);
                }
                // learned bias by distance (query position - key position), one row of the table per head
                if (rel) a += rel[static_cast<int64_t>(h) * rel_len + min(dist, rel_len - 1)];
                if (slopes) a -= slopes[h] * static_cast<float>(dist);
                mixed = a;
            }
            const float cmax = wave_allreduce_max(mixed);
            const float mnew = fmaxf(mrun[i], cmax);
            const float pj = ok ? expf(mixed - mnew) : 0.f;
            const float csum = wave_allreduce_sum(pj);
            const float al = expf(mrun[i] - mnew);      // first chunk: exp(-1e30 - m) = 0
            lrun[i] = lrun[i] * al + csum;
            mrun[i] = mnew;
            p[h * kTaChunk + lane] = pj;
            if (lane == 0) alpha[h] = al;
        }
        __syncthreads();
        // 3. weighted values
#pragma unroll
        for (int i = 0; i < kTaMaxAcc / R; ++i) {
            const int idx = tid + i * kTaThreads;
            if (i * kTaThreads >= H / R * dv) break;
            if (idx >= H / R * dv) continue;
#pragma unroll
            for (int r = 0; r < R; ++r) acc[i][r] *= alpha[idx / dv * R + r];
        }
        ta_values<T, R>(acc, p, v_cache, pages, first, last, H, hb, rep, GV, dv, v_wide != 0);
    }
    if (gridDim.z > 1) {        // partial result of this key share: unnormalised sums, running maximum, sum of weights
        const int64_t slot = (static_cast<int64_t>(blockIdx.z) * gridDim.x + t) * Hall + hb;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int h = wave + 4 * i;
            if (i >= hpw || h >= H) break;
            if (lane == 0) {
                part_ml[(slot + h) * 2] = mrun[i];
                part_ml[(slot + h) * 2 + 1] = lrun[i];
            }
        }
#pragma unroll
        for (int i = 0; i < kTaMaxAcc / R; ++i) {
            const int idx = tid + i * kTaThreads;
            if (i * kTaThreads >= H / R * dv) break;
            if (idx >= H / R * dv) continue;
#pragma unroll
            for (int r = 0; r < R; ++r) part_o[(slot + idx / dv * R + r) * dv + idx % dv] = acc[i][r];
        }
        return;
    }
    __syncthreads();
    // final scale of every head: 1 / sum, or with a sink e^(m - M) / (sum e^(m - M) + e^(sink - M)), M = max(m, sink)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int h = wave + 4 * i;
        if (i >= hpw || h >= H) break;
        float al = 1.f, l = lrun[i];
        if (sink) {
            const float sk = sink[h], big = fmaxf(mrun[i], sk);
            al = expf(mrun[i] - big);
            l = l * al + expf(sk - big);
        }
        if (lane == 0) alpha[h] = al / l;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTaMaxAcc / R; ++i) {
        const int idx = tid + i * kTaThreads;
        if (i * kTaThreads >= H / R * dv) break;
        const int c = idx % dv;
        if (idx >= H / R * dv || c >= out_dim) continue;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int h = idx / dv * R + r;
            float o = acc[i][r] * alpha[h];
            const int64_t hc = static_cast<int64_t>(hb + h) * out_dim + c;
            if (gate) o /= 1.0f + expf(-to_f(gate[t * gate_stride + hc]));
            if (out_f32) reinterpret_cast<float *>(out)[t * out_stride + hc] = o;
            else out[t * out_stride + hc] = to_t<T>(o);
        }
    }
}

inline size_t wa_lds_bytes(int H, int d) {
    return wa_float_count(H, d) * 4 + 4 * sizeof(int64_t);
}

// The same loop in fp32 for the H heads of one key head, D columns a key and DV a value, nothing mixed. What bounds a share of 64 keys is the
// chain of its memory round trips: above they are the blocks' ids, the queries, two rounds of keys, the distance bias and the values, one
// behind the other. Here the ids are scalar loads and a chunk's keys, bias and values are all asked for before the first score (the next
// chunk's as soon as the registers are free); a lane has its queries in registers, and where a value row has 64 or 128 columns two or four
// groups of threads share the pages. 90 to 145 registers: a sum left alone sinks below the next chunk's loads and takes 256.
// us with the launch that adds up the shares, both as they were -> both as they are (heads of 128, 8 over 2, fp32; other sizes named): 3 tokens at 513 keys
// 18.0 -> 8.4, one at 100 14.1 -> 8.1, 3 at 4000 50 -> 17.5, 12 at 500 18.2 -> 11.3, 32 at 1000 32 -> 18; prompts of 100 23 -> 14, 500 120 -> 39, 4 x 125
// 48 -> 21, 500 with 8 key heads 365 -> 73, 500 of 64 / 128 columns 73 -> 30. Nothing measured was slower, so whatever it takes goes to it. Error
// against 64 bits 2.0 to 3.7e-7 (2-norm) where it is 2.1 to 3.8e-7 above.
struct HeadsParams {
    void *out;
    const float *q, *k, *v;
    const int32_t *block_table, *tok_seq, *tok_pos;
    const float *rel, *sink, *slopes, *gate;
    float *part_o, *part_ml;
    int64_t q_stride, block_stride, out_stride, gate_stride;
    int rel_len, window, mask_kind, max_blocks, G, GV, out_dim;
    float scale, softcap;
};

template <int D, int DV, int H>
__global__ __launch_bounds__(kTaThreads, 2) void window_attn_heads_kernel(HeadsParams a) {
    constexpr int LPR = D / 4, ROWS = 64 / LPR, KU = kTaChunk / (4 * ROWS);     // lanes of a key row, keys a wave loads at once, loads a chunk
    constexpr int VP = kTaThreads / DV, PV = kTaChunk / kTaPage / VP;           // groups of threads that share the pages, pages of each
    constexpr int HW = (H + 3) / 4;                                             // heads a wave
    __shared__ __attribute__((aligned(16))) float s[H][kTaChunk], p[H][kTaChunk], red[VP > 1 ? VP - 1 : 1][H][DV], alpha[H];
    const int64_t t = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kv = blockIdx.y, hb = kv * H, gv = kv % a.GV, Hall = a.G * H;
    const int pos = a.tok_pos[t];
    const int32_t *bt = a.block_table + static_cast<int64_t>(a.tok_seq[t]) * a.max_blocks;
    const int lo = a.window <= 0 ? 0 : a.mask_kind == 1 ? (pos / a.window) * a.window : max(pos - a.window + 1, 0);
    int kb0 = lo / kTaPage, kb1 = pos / kTaPage;
    if (gridDim.z > 1) {        // a contiguous share of the pages (possibly none)
        const int per = (kb1 - kb0 + static_cast<int>(gridDim.z)) / static_cast<int>(gridDim.z);
        kb0 += per * static_cast<int>(blockIdx.z);
        kb1 = min(kb1, kb0 + per - 1);
    }
    const int sub = lane % LPR, row = lane / LPR;
    const int col = tid % DV, grp = __builtin_amdgcn_readfirstlane(tid / DV);
    float4_t qv[H], x[KU];
    float v[PV][kTaPage], relv[HW], acc[H], mrun[HW], lrun[HW];
#pragma unroll
    for (int h = 0; h < H; ++h) acc[h] = 0.f;
#pragma unroll
    for (int i = 0; i < HW; ++i) {
        mrun[i] = kNegBig;
        lrun[i] = relv[i] = 0.f;
    }
    auto ask_keys = [&](int kb) {
#pragma unroll
        for (int i = 0; i < HW; ++i) {
            const int h = wave + 4 * i, dist = pos - (kb * kTaPage + lane);
            if (a.rel && h < H) relv[i] = a.rel[static_cast<int64_t>(hb + h) * a.rel_len + max(min(dist, a.rel_len - 1), 0)];
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int pg = u * 4 * ROWS / kTaPage, in = u * 4 * ROWS % kTaPage;
            const float *page = a.k + bt[min(kb + pg, kb1)] * a.block_stride + (static_cast<int64_t>(kv) * kTaPage + in) * D;
            x[u] = *reinterpret_cast<const float4_t *>(page + (wave * ROWS + row) * D + 4 * sub);
        }
    };
    auto ask_values = [&](int kb) {
#pragma unroll
        for (int i = 0; i < PV; ++i) {
            const float *page = a.v + bt[min(kb + grp + VP * i, kb1)] * a.block_stride + static_cast<int64_t>(gv) * DV * kTaPage;
#pragma unroll
            for (int k = 0; k < kTaPage; k += 4) {
                const float4_t w = *reinterpret_cast<const float4_t *>(page + col * kTaPage + k);
#pragma unroll
                for (int c = 0; c < 4; ++c) v[i][k + c] = w[c];
            }
        }
    };
    if (kb0 <= kb1) {
#pragma unroll
        for (int h = 0; h < H; ++h) qv[h] = *reinterpret_cast<const float4_t *>(a.q + t * a.q_stride + (hb + h) * D + 4 * sub);
        ask_keys(kb0);
        ask_values(kb0);
    }
    for (int kb = kb0; kb <= kb1; kb += 4) {
        const int first = max(lo - kb * kTaPage, 0), last = min(min(pos, kb1 * kTaPage + kTaPage - 1) - kb * kTaPage, kTaChunk - 1);
        // 1. scores (what a key outside first .. last gives is not looked at)
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            float mine = 0.f;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                float d = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) d = fmaf(qv[h][c], x[u][c], d);
                d = ta_lane_sum(d, LPR);
                mine = sub == h ? d : mine;
            }
            if (sub < H) s[sub][(u * 4 + wave) * ROWS + row] = mine;
            if ((u + 1) * H % 16 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        float bias[HW];
#pragma unroll
        for (int i = 0; i < HW; ++i) bias[i] = relv[i];
        if (kb + 4 <= kb1) ask_keys(kb + 4);
        __syncthreads();
        // 2. online softmax: wave w owns heads w and w + 4, a lane a key
        const bool ok = lane >= first && lane <= last;
#pragma unroll
        for (int i = 0; i < HW; ++i) {
            const int h = wave + 4 * i;
            if (h < H) {
                float m = kNegBig;
                if (ok) {
                    m = s[h][lane] * a.scale;
                    if (a.softcap > 0.f) m = a.softcap * tanhf(m / a.softcap);
                    if (a.rel) m += bias[i];
                    if (a.slopes) m -= a.slopes[hb + h] * static_cast<float>(pos - (kb * kTaPage + lane));
                }
                const float mnew = fmaxf(mrun[i], wave_allreduce_max(m));
                const float pj = ok ? expf(m - mnew) : 0.f;
                const float csum = wave_allreduce_sum(pj);
                const float al = expf(mrun[i] - mnew);      // first chunk: exp(-1e30 - m) = 0
                lrun[i] = lrun[i] * al + csum;
                mrun[i] = mnew;
                p[h][lane] = pj;
                if (lane == 0) alpha[h] = al;
            }
        }
        __syncthreads();
        // 3. weighted values (those outside first .. last do not count, whatever they hold)
#pragma unroll
        for (int h = 0; h < H; ++h) acc[h] *= alpha[h];
#pragma unroll
        for (int i = 0; i < PV; ++i) {
            const int j0 = (grp + VP * i) * kTaPage;
            if (j0 < first || j0 + kTaPage - 1 > last) {
#pragma unroll
                for (int k = 0; k < kTaPage; ++k)
                    if (j0 + k < first || j0 + k > last) v[i][k] = 0.f;
            }
#pragma unroll
            for (int k = 0; k < kTaPage; k += 4) {
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const float4_t w = *reinterpret_cast<const float4_t *>(&p[h][j0 + k]);
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[h] = fmaf(w[c], v[i][k + c], acc[h]);
                }
                if ((k / 4 + 1) * H % (H > 1 ? 8 : 4) == 0) {     // (else the sums sink below the next loads, and all the weights stay in registers)
#pragma unroll
                    for (int h = 0; h < H; ++h) asm volatile("" : "+v"(acc[h]));
                }
            }
        }
        if (kb + 4 <= kb1) ask_values(kb + 4);
    }
    if constexpr (VP > 1) {
        if (grp > 0) {
#pragma unroll
            for (int h = 0; h < H; ++h) red[grp - 1][h][col] = acc[h];
        }
        __syncthreads();
        if (grp == 0) {
#pragma unroll
            for (int g = 0; g < VP - 1; ++g)
#pragma unroll
                for (int h = 0; h < H; ++h) acc[h] += red[g][h][col];
        }
    }
    if (gridDim.z > 1) {
        const int64_t slot = (static_cast<int64_t>(blockIdx.z) * gridDim.x + t) * Hall + hb;
#pragma unroll
        for (int i = 0; i < HW; ++i) {
            const int h = wave + 4 * i;
            if (h < H && lane == 0) {
                a.part_ml[(slot + h) * 2] = mrun[i];
                a.part_ml[(slot + h) * 2 + 1] = lrun[i];
            }
        }
        if (grp == 0) {
#pragma unroll
            for (int h = 0; h < H; ++h) a.part_o[(slot + h) * DV + col] = acc[h];
        }
        return;
    }
    __syncthreads();
    // final scale of every head, as in window_attn_kernel
#pragma unroll
    for (int i = 0; i < HW; ++i) {
        const int h = wave + 4 * i;
        if (h < H) {
            float al = 1.f, l = lrun[i];
            if (a.sink) {
                const float sk = a.sink[hb + h], big = fmaxf(mrun[i], sk);
                al = expf(mrun[i] - big);
                l = l * al + expf(sk - big);
            }
            if (lane == 0) alpha[h] = al / l;
        }
    }
    __syncthreads();
    if (grp > 0 || col >= a.out_dim) return;
#pragma unroll
    for (int h = 0; h < H; ++h) {
        float o = acc[h] * alpha[h];
        const int64_t hc = static_cast<int64_t>(hb + h) * a.out_dim + col;
        if (a.gate) o /= 1.0f + expf(-a.gate[t * a.gate_stride + hc]);
        static_cast<float *>(a.out)[t * a.out_stride + hc] = o;
    }
}

// Launches window_attn_heads_kernel where it serves the heads; false: nothing was launched.
static bool launch_heads(const HeadsParams &a, int rep, int d, int dv, const dim3 &grid, hipStream_t st) {
#define SWL_HEADS(D, DV, H)                                                                                         \
    if (d == D && dv == DV && rep == H) {                                                                           \
        hipLaunchKernelGGL((window_attn_heads_kernel<D, DV, H>), grid, dim3(kTaThreads), 0, st, a);                 \
        return true;                                                                                                \
    }
#define SWL_HEADS_OF(D, DV) SWL_HEADS(D, DV, 1) SWL_HEADS(D, DV, 2) SWL_HEADS(D, DV, 4) SWL_HEADS(D, DV, 8)
    SWL_HEADS_OF(128, 128)
    SWL_HEADS_OF(64, 64)
    SWL_HEADS_OF(64, 128)
#undef SWL_HEADS_OF
#undef SWL_HEADS
    return false;
}

} // namespace swl

extern "C" int swl_masked_attn_shares(void *out, const void *q, const void *k_cache, const void *v_cache,
                               const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos,
                               const float *talk, const float *rel, int32_t rel_len, int64_t num_tokens,
                               int32_t num_q_heads, int32_t num_kv_heads,
                               int32_t dim, int32_t vdim, int64_t q_tok_stride, int32_t window, float scale,
                               float softcap, int32_t max_blocks_per_seq, int64_t block_stride, int32_t mask_kind,
                               const float *sink, int32_t num_v_heads, int32_t out_f32, const float *slopes,
                               int32_t out_dim, int64_t out_stride, const void *gate, int64_t gate_stride, int32_t key_splits,
                               float *scratch, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || dim <= 0 || vdim <= 0 || window < 0)
        return SWL_ERR_BAD_ARG;
    if (num_q_heads % num_kv_heads) return SWL_ERR_BAD_ARG;
    if (mask_kind < 0 || mask_kind > 1 || num_v_heads <= 0 || num_kv_heads % num_v_heads) return SWL_ERR_BAD_ARG;
    if (out_dim <= 0 || out_dim > vdim || out_stride < static_cast<int64_t>(num_q_heads) * out_dim) return SWL_ERR_BAD_ARG;
    if (gate && gate_stride < static_cast<int64_t>(num_q_heads) * out_dim) return SWL_ERR_BAD_ARG;
    if (key_splits < 1 || key_splits > 64 || (key_splits > 1 && (!scratch || !swl::aligned16(scratch)))) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (out_f32 == SWL_OUT_SHARES && (key_splits < 2 || sink || gate)) return SWL_ERR_BAD_ARG;
    if ((!out && out_f32 != SWL_OUT_SHARES) || !q || !k_cache || !v_cache || !block_table || !tok_seq || !tok_pos || (rel && rel_len <= 0))
        return SWL_ERR_BAD_ARG;
    // heads per workgroup: all of them when they are mixed, else as many as its accumulators and LDS hold
    int hpg = num_q_heads;
    if (!talk) {
        if (hpg > 32) hpg = 32;
        while (hpg > 1 && (static_cast<int64_t>(hpg) * vdim > swl::kTaMaxAcc * swl::kTaThreads ||
                           swl::wa_lds_bytes(hpg, dim) > 64 * 1024))
            --hpg;
        // a few workgroups: one for the heads of every key head (whose keys and values no other heads read). A chunk's scores are a chain
        // over the key heads of a workgroup. 3 tokens at 513 keys, 8 heads of 128 over 2, fp32, 16 shares: 21.4 -> 14.8 us
        const int rep = num_q_heads / num_kv_heads;
        if (hpg > rep && num_tokens * key_splits <= 256) hpg = rep;
    }
    const size_t lds = swl::wa_lds_bytes(hpg, dim);
    if (num_tokens > 0x7fffffffLL || hpg > 32 ||
        static_cast<int64_t>(hpg) * vdim > swl::kTaMaxAcc * swl::kTaThreads || lds > 64 * 1024)
        return SWL_ERR_UNSUPPORTED;
    const unsigned groups = static_cast<unsigned>((num_q_heads + hpg - 1) / hpg);
    const size_t esize = dtype == SWL_F32 ? 4 : 2;
    auto whole = [&](const void *c, size_t piece, int elems) {     // rows of whole pieces on their boundaries
        return elems * esize % piece == 0 && block_stride * static_cast<int64_t>(esize) % static_cast<int64_t>(piece) == 0 &&
               reinterpret_cast<uintptr_t>(c) % piece == 0;
    };
    const int k_wide = whole(k_cache, 4 * esize, dim), v_wide = whole(v_cache, 16, 16);
    // scratch: [splits][tokens][H][vdim] fp32 partial sums, then [splits][tokens][H][2] (maximum, sum)
    float *part_o = scratch;
    float *part_ml = key_splits > 1 ? scratch + static_cast<int64_t>(key_splits) * num_tokens * num_q_heads * vdim : nullptr;
    const dim3 grid(static_cast<unsigned>(num_tokens), groups, static_cast<unsigned>(key_splits));
    hipStream_t st = static_cast<hipStream_t>(stream);
    bool served = false;
    if (!talk && dtype == SWL_F32 && k_wide && v_wide && q_tok_stride % 4 == 0 && swl::aligned16(q) && num_kv_heads <= 65535) {
        const swl::HeadsParams a{out, static_cast<const float *>(q), static_cast<const float *>(k_cache), static_cast<const float *>(v_cache),
                                 block_table, tok_seq, tok_pos, rel, sink, slopes, static_cast<const float *>(gate), part_o, part_ml, q_tok_stride,
                                 block_stride, out_stride, gate_stride, rel_len, window, mask_kind, max_blocks_per_seq, num_kv_heads, num_v_heads,
                                 out_dim, scale, softcap};
        served = swl::launch_heads(a, num_q_heads / num_kv_heads, dim, vdim,
                                   dim3(static_cast<unsigned>(num_tokens), static_cast<unsigned>(num_kv_heads), static_cast<unsigned>(key_splits)), st);
    }
    SWL_DISPATCH_DTYPE3(dtype, T, {
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(swl::kTaThreads), lds, st, static_cast<T *>(out), static_cast<const T *>(q),
                               static_cast<const T *>(k_cache), static_cast<const T *>(v_cache), block_table, tok_seq, tok_pos, talk,
                               rel, rel_len, hpg, num_kv_heads, dim, vdim, q_tok_stride, window, scale, softcap, max_blocks_per_seq,
                               block_stride, mask_kind, sink, num_v_heads, out_f32, num_q_heads, slopes, out_dim, out_stride,
                               static_cast<const T *>(gate), gate_stride, part_o, part_ml, k_wide, v_wide);
        };
        if (!served) switch (swl::ta_share(num_q_heads / num_kv_heads, hpg)) {
        case 8: go(&swl::window_attn_kernel<T, 8>); break;
        case 4: go(&swl::window_attn_kernel<T, 4>); break;
        case 2: go(&swl::window_attn_kernel<T, 2>); break;
        default: go(&swl::window_attn_kernel<T, 1>); break;
        }
        if (key_splits > 1 && out_f32 != SWL_OUT_SHARES) {
            const int64_t rows = num_tokens * num_q_heads;
            if (rows > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
            swl::launch_attn_combine<T, true>(static_cast<T *>(out), part_o, part_ml, rows, vdim, key_splits, sink, num_q_heads, out_f32, out_dim,
                                              out_stride, static_cast<const T *>(gate), gate_stride, st);
        }
    });
    return swl::check_launch();
}

extern "C" int swl_masked_attn(void *out, const void *q, const void *k_cache, const void *v_cache,
                               const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos,
                               const float *talk, const float *rel, int32_t rel_len, int64_t num_tokens,
                               int32_t num_q_heads, int32_t num_kv_heads,
                               int32_t dim, int32_t vdim, int64_t q_tok_stride, int32_t window, float scale,
                               float softcap, int32_t max_blocks_per_seq, int64_t block_stride, int32_t mask_kind,
                               const float *sink, int32_t num_v_heads, int32_t out_f32, const float *slopes,
                               int32_t out_dim, int64_t out_stride, const void *gate, int64_t gate_stride, int32_t dtype,
                               swl_stream_t stream) {
    return swl_masked_attn_shares(out, q, k_cache, v_cache, block_table, tok_seq, tok_pos, talk, rel, rel_len, num_tokens, num_q_heads,
                                  num_kv_heads, dim, vdim, q_tok_stride, window, scale, softcap, max_blocks_per_seq, block_stride,
                                  mask_kind, sink, num_v_heads, out_f32, slopes, out_dim, out_stride, gate, gate_stride, 1, nullptr,
                                  dtype, stream);
}

extern "C" int swl_window_attn(void *out, const void *q, const void *k_cache, const void *v_cache,
                               const int32_t *block_table, const int32_t *tok_seq, const int32_t *tok_pos,
                               const float *talk, const float *rel, int32_t rel_len, int64_t num_tokens,
                               int32_t num_q_heads, int32_t num_kv_heads,
                               int32_t dim, int32_t vdim, int64_t q_tok_stride, int32_t window, float scale,
                               float softcap, int32_t max_blocks_per_seq, int64_t block_stride, int32_t dtype,
                               swl_stream_t stream) {
    return swl_masked_attn(out, q, k_cache, v_cache, block_table, tok_seq, tok_pos, talk, rel, rel_len, num_tokens,
                           num_q_heads, num_kv_heads, dim, vdim, q_tok_stride, window, scale, softcap, max_blocks_per_seq,
                           block_stride, 0, nullptr, num_kv_heads > 0 ? num_kv_heads : 1, 0, nullptr, vdim,
                           static_cast<int64_t>(num_q_heads) * vdim, nullptr, 0, dtype, stream);
}
