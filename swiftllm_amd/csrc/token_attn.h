// token_attn.h — the two passes over a chunk of four 16-key pages that the per-token attention kernels share (window_attn.hip,
// sigmoid_attn.hip): 256 threads, fp32 arithmetic whatever the storage type.
#pragma once

#include "swl_common.h"

namespace swl {

constexpr int kTaThreads = 256, kTaChunk = 64, kTaPage = 16;
constexpr int kTaMaxAcc = 32;       // (head, value column) accumulators per thread: heads * vdim <= 8192

// Sum over aligned groups of lpr lanes (8, 16, 32 or 64; uniform): every lane ends with the total.
__device__ __forceinline__ float ta_lane_sum(float v, int lpr) {
    v = group_allreduce_sum<8>(v);
    if (lpr >= 16) v += dpp_mov<kDppRowMirror>(v);
    if (lpr >= 32) v += __shfl_xor(v, 16, 64);
    if (lpr >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

template <typename T>
__device__ __forceinline__ float4_t ta_load4(const T *p) {
    if constexpr (sizeof(T) == 4) {
        return *reinterpret_cast<const float4_t *>(p);
    } else {
        vec4_t<T> v;
        load4(v, p);
        return float4_t{to_f(v[0]), to_f(v[1]), to_f(v[2]), to_f(v[3])};
    }
}

// s[h][j] = q_h . k_j for keys first .. last of the chunk and heads hb .. hb + H - 1 of the token (qf: their rows, fp32, in LDS).
// A key row is read by 8 .. 64 neighbouring lanes, four elements each, once for four heads; four keys are in flight per lane.
// `wide`: rows are whole 4-element pieces on their boundaries. pages[4]: element offsets of the chunk's blocks.
template <typename T>
__device__ __forceinline__ void ta_scores(float *s, const float *qf, const T *k_cache, const int64_t *pages, int first, int last, int H,
                                          int hb, int rep, int d, bool wide) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lpr = d <= 32 ? 8 : d <= 64 ? 16 : d <= 128 ? 32 : 64, rows = 64 / lpr, sub = lane % lpr, row = lane / lpr;
    for (int kv = hb / rep; kv <= (hb + H - 1) / rep; ++kv) {
        const int h_hi = min((kv + 1) * rep, hb + H) - hb;
        for (int h0 = max(kv * rep, hb) - hb; h0 < h_hi; h0 += 4) {
            for (int j0 = wave * rows; j0 < kTaChunk; j0 += 16 * rows) {
                if (j0 > last) break;       // (uniform; a wave's keys are j0 + 4 rows u + row)
                const T *kr[4];
                float a[4][4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int j = min(max(j0 + 4 * rows * u + row, first), last);
                    kr[u] = k_cache + pages[j >> 4] + (static_cast<int64_t>(kv) * kTaPage + (j & 15)) * d;
#pragma unroll
                    for (int h = 0; h < 4; ++h) a[u][h] = 0.f;
                }
                if (wide) {
                    for (int e = 4 * sub; e < d; e += 4 * lpr) {
                        float4_t x[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) x[u] = ta_load4(kr[u] + e);
#pragma unroll
                        for (int h = 0; h < 4; ++h) {
                            const float4_t qv = *reinterpret_cast<const float4_t *>(qf + min(h0 + h, H - 1) * d + e);
#pragma unroll
                            for (int u = 0; u < 4; ++u)
#pragma unroll
                                for (int c = 0; c < 4; ++c) a[u][h] = fmaf(qv[c], x[u][c], a[u][h]);
                        }
                    }
                } else {
                    for (int e = sub; e < d; e += lpr) {
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float x = to_f(kr[u][e]);
#pragma unroll
                            for (int h = 0; h < 4; ++h) a[u][h] = fmaf(qf[min(h0 + h, H - 1) * d + e], x, a[u][h]);
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int j = j0 + 4 * rows * u + row;
#pragma unroll
                    for (int h = 0; h < 4; ++h) {
                        const float v = ta_lane_sum(a[u][h], lpr);
                        if (sub == 0 && h0 + h < h_hi && j >= first && j <= last) s[(h0 + h) * kTaChunk + j] = v;
                    }
                }
            }
        }
    }
}

// acc[i][r] += sum_j p[h0 + r][j] v_j[col] over the chunk's pages first / 16 .. last / 16 (p is zero outside first .. last). A thread owns
// column idx % dv of the R heads h0 = R (idx / dv), idx = thread + 256 i: a page keeps a column's sixteen values together, which are
// read once for the R heads. `wide`: columns on 16-byte boundaries. Values outside first .. last do not count, whatever they hold.
template <typename T, int R>
__device__ __forceinline__ void ta_values(float (&acc)[kTaMaxAcc / R][R], const float *p, const T *v_cache, const int64_t *pages,
                                          int first, int last, int H, int hb, int rep, int GV, int dv, bool wide) {
#pragma unroll
    for (int i = 0; i < kTaMaxAcc / R; ++i) {
        const int idx = threadIdx.x + i * kTaThreads;
        if (i * kTaThreads >= H / R * dv) break;        // (uniform)
        if (idx >= H / R * dv) continue;
        const int h0 = idx / dv * R, col = idx % dv, gv = ((hb + h0) / rep) % GV;
        for (int pg = first >> 4; pg <= last >> 4; ++pg) {
            const T *vr = v_cache + pages[pg] + (static_cast<int64_t>(gv) * dv + col) * kTaPage;
            float v[kTaPage];
            if (wide) {
                if constexpr (sizeof(T) == 4) {
#pragma unroll
                    for (int k = 0; k < kTaPage; k += 4) {
                        const float4_t x = *reinterpret_cast<const float4_t *>(vr + k);
#pragma unroll
                        for (int c = 0; c < 4; ++c) v[k + c] = x[c];
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < kTaPage; k += 8) {
                        const vec8_t<T> x = load8(vr + k);
#pragma unroll
                        for (int c = 0; c < 8; ++c) v[k + c] = to_f(x[c]);
                    }
                }
            } else {
#pragma unroll
                for (int k = 0; k < kTaPage; ++k) v[k] = to_f(vr[k]);
            }
            if (pg * kTaPage < first || pg * kTaPage + kTaPage - 1 > last) {        // (uniform)
#pragma unroll
                for (int k = 0; k < kTaPage; ++k)
                    if (pg * kTaPage + k < first || pg * kTaPage + k > last) v[k] = 0.f;
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float *pr = p + (h0 + r) * kTaChunk + pg * kTaPage;
#pragma unroll
                for (int k = 0; k < kTaPage; k += 4) {
                    const float4_t w = *reinterpret_cast<const float4_t *>(pr + k);
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[i][r] = fmaf(w[c], v[k + c], acc[i][r]);
                }
            }
        }
    }
}

// heads a thread's value loads serve: the largest of 8, 4, 2, 1 that divides the query heads of a key head and of a workgroup
inline int ta_share(int rep, int heads) {
    for (int r = 8; r > 1; r /= 2)
        if (rep % r == 0 && heads % r == 0) return r;
    return 1;
}

} // namespace swl
