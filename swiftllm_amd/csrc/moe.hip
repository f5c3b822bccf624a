// moe.hip — mixture-of-experts feed-forward: fp32 router with top-k selection, and the expert products for the
// token counts where an expert's weights are streamed once per assignment (decode and short portions).
//
//   swl_moe_route:        logits = router h + bias in fp32; the `top` largest (ties: lowest expert id); weights =
//                         softmax over the chosen logits only.
//   swl_moe_gate_up:      for every (token, chosen expert): g = min(W_gate h, limit), u = clamp(W_up h, +-limit),
//                         y = g * sigmoid(1.702 g) * (u + 1); fp32 accumulation, y rounded to the compute dtype.
//   swl_moe_down_combine: out[t] = sum_j weight[t][j] * (W_down[e_j] y[t][j]) with fp32 accumulation through the weighted
//                         sum (fixed order j = 0, 1, ...: the result does not depend on what else is in the batch).
//
//   swl_moe_route_grouped: scores s = sigmoid(router h); experts are CHOSEN by s + correction, inside the `keep` best of
//                         `count` equal groups of neighbouring experts (a group's score: the sum of its two largest choice
//                         scores); the weights are the chosen experts' s, divided by their sum when `normalize` is set.
//   in_w (swl_moe_gate_up, swl_glu_clamp, swl_moe_expert_stationary): a weight per assignment on the expert's INPUT. The first
//                         products are linear, so it multiplies their fp32 sums: act(w g, w u). The combination then takes no
//                         weights (NULL: all one).
//   act (swl_moe_gate_up, swl_glu_clamp; glu = 3 of swl_moe_expert_stationary): 0 the clamped unit above, 1 the plain gated
//                         unit y = silu(g) * u, 2 (swl_glu_clamp only) the same on rows [up | gate].
//
// Expert weights are stacked: gate_up [experts, 2 ff, width] (gate rows, then up rows), down [experts, width, ff].
#include "swl_common.h"

namespace swl {

__device__ __forceinline__ bool aligned16_dev(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int kMoeThreads = 256;
constexpr int kMoeWaves = kMoeThreads / 64;

// Per-lane shares of sum_i x[i] * w[r][i] over N rows of n elements (x: fp32 in LDS or a row in global memory; the caller reduces over
// the wave): 16 bytes per lane and row where the rows allow it, all rows' loads of a turn in flight together.
template <int N, typename X, typename T>
__device__ __forceinline__ void lane_dots(float (&a)[N], const X *x, const T *const (&w)[N], int n, int lane) {
    constexpr int V = 16 / sizeof(T);
    bool wide = n % V == 0 && (sizeof(X) != 2 || aligned16_dev(x));
#pragma unroll
    for (int r = 0; r < N; ++r) {
        a[r] = 0.f;
        wide = wide && aligned16_dev(w[r]);
    }
    if (wide) {
#pragma unroll 2
        for (int i = lane * V; i < n; i += 64 * V) {
            typedef T vec __attribute__((ext_vector_type(V)));
            vec v[N];
            float xv[V];
#pragma unroll
            for (int r = 0; r < N; ++r) v[r] = *reinterpret_cast<const vec *>(w[r] + i);
#pragma unroll
            for (int k = 0; k < V; ++k) xv[k] = to_f(x[i + k]);
#pragma unroll
            for (int r = 0; r < N; ++r)
#pragma unroll
                for (int k = 0; k < V; ++k) a[r] += xv[k] * to_f(v[r][k]);
        }
        return;
    }
    for (int i = lane; i < n; i += 64) {
        const float xv = to_f(x[i]);
#pragma unroll
        for (int r = 0; r < N; ++r) a[r] += xv * to_f(w[r][i]);
    }
}

// The token's row as fp32 in LDS, for the whole workgroup (the caller synchronises).
template <typename T>
__device__ __forceinline__ void stage_row(float *dst, const T *src, int n) {
    if constexpr (sizeof(T) == 2) {
        if ((n & 7) == 0 && aligned16_dev(src)) {
            for (int i = threadIdx.x * 8; i < n; i += kMoeThreads * 8) {
                const vec8_t<T> v = load8(src + i);
                *reinterpret_cast<float4_t *>(dst + i) = float4_t{to_f(v[0]), to_f(v[1]), to_f(v[2]), to_f(v[3])};
                *reinterpret_cast<float4_t *>(dst + i + 4) = float4_t{to_f(v[4]), to_f(v[5]), to_f(v[6]), to_f(v[7])};
            }
            return;
        }
    }
    for (int i = threadIdx.x; i < n; i += kMoeThreads) dst[i] = to_f(src[i]);
}
// Router logit: x . w over n fp32 elements (x in LDS), reduced over the wave; 16 bytes per lane when the rows allow it.
__device__ __forceinline__ float router_dot(const float *x, const float *w, int n, int lane) {
    float a = 0.f;
    if ((n & 3) == 0 && aligned16_dev(w)) {
#pragma unroll 4
        for (int i = lane * 4; i < n; i += 64 * 4) {
            const float4_t u = *reinterpret_cast<const float4_t *>(x + i), v = *reinterpret_cast<const float4_t *>(w + i);
            a += (u[0] * v[0] + u[1] * v[1]) + (u[2] * v[2] + u[3] * v[3]);
        }
    } else {
        for (int i = lane; i < n; i += 64) a += x[i] * w[i];
    }
    return wave_allreduce_sum(a);
}

// Arg-max over an LDS array of n floats for the whole wave (ties: the lowest index; NaN, -inf and taken entries never win: 0x7fffffff).
// A lane scans entries lane, lane + 64, ...; the exchange is a chain of LDS latencies, so up to eight entries take three steps, not six.
__device__ __forceinline__ void wave_argmax(const float *v, int n, int lane, float &best, int &besti) {
    best = -INFINITY;
    besti = 0x7fffffff;
    for (int e = lane; e < n; e += 64) {
        if (v[e] > best) {      // strict: keeps the lowest id among a lane's equals
            best = v[e];
            besti = e;
        }
    }
    auto exchange = [&](int m) {
        const float ob = __shfl_xor(best, m, 64);
        const int oi = __shfl_xor(besti, m, 64);
        if (ob > best || (ob == best && oi < besti)) {
            best = ob;
            besti = oi;
        }
    };
    if (n > 8) {
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) exchange(m);
        return;
    }
#pragma unroll
    for (int m = 4; m >= 1; m >>= 1) exchange(m);
    best = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(best)));
    besti = __builtin_amdgcn_readfirstlane(besti);
}

template <typename T>
__global__ __launch_bounds__(kMoeThreads) void moe_route_kernel(int32_t *idx_out, float *w_out, const T *h,
                                                                const float *router, const float *bias, int width,
                                                                int experts, int top, int all_scores, float scale) {
    extern __shared__ __align__(16) float lds[];
    float *hf = lds;                // [width]
    float *logit = lds + width;     // [experts]
    const int64_t t = blockIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    stage_row(hf, h + t * width, width);
    __syncthreads();
    for (int e = wave; e < experts; e += kMoeWaves) {
        const float a = router_dot(hf, router + static_cast<int64_t>(e) * width, width, lane);
        if (lane == 0) logit[e] = a + (bias ? bias[e] : 0.f);
    }
    __syncthreads();
    if (wave != 0) return;
    // all_scores: the weights are scale * softmax over ALL experts (not renormalised over the chosen ones)
    float all_max = -INFINITY, all_den = 0.f;
    if (all_scores) {
        for (int e = lane; e < experts; e += 64) all_max = fmaxf(all_max, logit[e]);
        all_max = wave_allreduce_max(all_max);
        for (int e = lane; e < experts; e += 64) all_den += expf(logit[e] - all_max);
        all_den = wave_allreduce_sum(all_den);
    }
    // top-k by repeated arg-max over the wave (each lane scans experts lane, lane + 64, ...)
    // Latency bounds the choice. Lane j keeps the j-th one until the sum is known: a store to global memory in the loop is waited for at
    // every fence. With the shorter exchange, 3663 tokens of 2048, two of eight experts, bf16: 12.8 to 11.3 us, in groups 15.4 to 13.3;
    // six or eight of 64 or 128 experts: 1 to 4 % less.
    float chosen_max = 0.f, denom = 0.f, mine = 0.f;
    int mine_idx = 0;
    for (int j = 0; j < top; ++j) {
        float best;
        int besti;
        wave_argmax(logit, experts, lane, best, besti);
        if (besti >= experts) besti = 0;        // (only NaN, -inf or taken scores are left: an expert that exists, its weight 0 or NaN)
        if (j == 0) chosen_max = all_scores ? all_max : best;
        const float pj = expf(best - chosen_max);
        denom += pj;
        if (lane == j) {
            mine = pj;
            mine_idx = besti;
        }
        if (lane == 0) {
            if (top > 64) {     // (more choices than lanes)
                idx_out[t * top + j] = besti;
                w_out[t * top + j] = pj;
            }
            logit[besti] = -INFINITY;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    const float mult = all_scores ? scale / all_den : 1.0f / denom;
    if (top <= 64) {
        if (lane < top) {
            idx_out[t * top + lane] = mine_idx;
            w_out[t * top + lane] = mine * mult;
        }
    } else if (lane == 0) {
        for (int j = 0; j < top; ++j) w_out[t * top + j] *= mult;
    }
}

// Sigmoid scores with group-limited choice. One workgroup per token; the first wave chooses.
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void moe_route_grouped_kernel(int32_t *idx_out, float *w_out, const T *h,
                                                                        const float *router, const float *correction,
                                                                        int width, int experts, int top, int count,
                                                                        int keep, int normalize) {
    extern __shared__ __align__(16) float lds[];
    float *hf = lds;                    // [width]
    float *score = hf + width;          // [experts] s = sigmoid(logit)
    float *choice = score + experts;    // [experts] s + correction; -inf once taken or outside the kept groups
    float *gscore = choice + experts;   // [count]
    float *gkeep = gscore + count;      // [count] 1 for the groups whose experts may be chosen
    const int64_t t = blockIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    stage_row(hf, h + t * width, width);
    __syncthreads();
    for (int e = wave; e < experts; e += kMoeWaves) {
        const float a = router_dot(hf, router + static_cast<int64_t>(e) * width, width, lane);
        if (lane == 0) {
            const float sc = 1.0f / (1.0f + expf(-a));
            score[e] = sc;
            choice[e] = sc + (correction ? correction[e] : 0.f);
        }
    }
    __syncthreads();
    if (wave != 0) return;
    if (count > 1 && keep < count) {
        const int per = experts / count;
        for (int g = lane; g < count; g += 64) {    // a group's score: its two largest choice scores (one, in groups of one)
            float a = -INFINITY, b = -INFINITY;
            for (int e = g * per; e < (g + 1) * per; ++e) {
                const float v = choice[e];
                if (v > a) {
                    b = a;
                    a = v;
                } else if (v > b) {
                    b = v;
                }
            }
            gscore[g] = per > 1 ? a + b : a;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int g = lane; g < count; g += 64) gkeep[g] = 0.f;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int j = 0; j < keep; ++j) {
            float best;
            int besti;
            wave_argmax(gscore, count, lane, best, besti);
            if (lane == 0 && besti < count) {
                gscore[besti] = -INFINITY;      // (taken)
                gkeep[besti] = 1.f;
            }
            __builtin_amdgcn_wave_barrier();
            __threadfence_block();
        }
        for (int e = lane; e < experts; e += 64)
            if (gkeep[e / per] == 0.f) choice[e] = -INFINITY;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    float denom = 0.f, mine = 0.f;      // (lane j keeps the j-th choice, as above)
    int mine_idx = 0;
    for (int j = 0; j < top; ++j) {
        float best;
        int besti;
        wave_argmax(choice, experts, lane, best, besti);
        if (besti >= experts) besti = 0;        // (as above)
        const float sc = score[besti];
        denom += sc;
        if (lane == j) {
            mine = sc;
            mine_idx = besti;
        }
        if (lane == 0) {
            if (top > 64) {
                idx_out[t * top + j] = besti;
                w_out[t * top + j] = sc;
            }
            choice[besti] = -INFINITY;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    const float mult = normalize ? 1.0f / (denom + 1e-20f) : 1.0f;
    if (top <= 64) {
        if (lane < top) {
            idx_out[t * top + lane] = mine_idx;
            w_out[t * top + lane] = mine * mult;
        }
    } else if (lane == 0) {
        for (int j = 0; j < top; ++j) w_out[t * top + j] *= mult;
    }
}

// Routers of five to eight experts for steps of many tokens: a wave takes two or four tokens, whose rows meet each load of the router's, and the choice is
// made by a lane a token from registers. What bounds it is vector work (eight multiplies and adds a quad and expert, which stay apart) and the
// chain of a choice; a workgroup a token, as above, also waits for its row, its two meetings and the router's rows (32 KiB of 1024 columns a token from
// L2). The same sums in the same order, the same bits.
// us, bf16, two of eight, before -> now: 7452 tokens of 1024 plain 13.6 -> 9.7, all scores 13.5 -> 11.3, in groups 17.5 -> 12.3; 3657 of 2048 12.0 -> 9.8, 11.9 ->
// 11.3, 13.6 -> 11.9; 16000 of 2048 40 -> 22, 39 -> 23, 44 -> 25; fp32, 7452 of 2048 29 -> 13.
constexpr int kRouteFew = 8;

struct RouteParams {
    int32_t *idx;
    float *w;
    const void *h;
    const float *router, *bias;     // (or the correction)
    int64_t num_tokens;
    int width, experts, top, all_scores, count, keep, normalize;
    float scale;
};

template <typename T, bool GROUPED, int N>
__global__ __launch_bounds__(kMoeThreads) void moe_route_few_kernel(RouteParams p) {
    constexpr int E = kRouteFew;
    const int lane = threadIdx.x & 63, experts = p.experts;
    const int64_t t0 = (static_cast<int64_t>(blockIdx.x) * kMoeWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * N;
    if (t0 >= p.num_tokens) return;
    const T *x[N];
#pragma unroll
    for (int n = 0; n < N; ++n) x[n] = static_cast<const T *>(p.h) + min(t0 + n, p.num_tokens - 1) * p.width;
    float a[N][E];
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int e = 0; e < E; ++e) a[n][e] = 0.f;
    vec4_t<T> u[2][N];
    float4_t r[2][E];
    auto load = [&](int i, vec4_t<T> (&u)[N], float4_t (&r)[E]) {
#pragma unroll
        for (int n = 0; n < N; ++n) u[n] = *reinterpret_cast<const vec4_t<T> *>(x[n] + i);
#pragma unroll
        for (int e = 0; e < E; ++e) r[e] = *reinterpret_cast<const float4_t *>(p.router + static_cast<int64_t>(min(e, experts - 1)) * p.width + i);
    };
    auto add = [&](const vec4_t<T> (&u)[N], const float4_t (&r)[E]) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const float u0 = to_f(u[n][0]), u1 = to_f(u[n][1]), u2 = to_f(u[n][2]), u3 = to_f(u[n][3]);
#pragma unroll
            for (int e = 0; e < E; ++e) a[n][e] += (u0 * r[e][0] + u1 * r[e][1]) + (u2 * r[e][2] + u3 * r[e][3]);
        }
    };
    const int last = p.width - 4;       // (columns past the row: the last ones again, which nobody adds)
    load(min(lane * 4, last), u[0], r[0]);
    for (int i = lane * 4; i - lane * 4 < p.width; i += 512) {
        load(min(i + 256, last), u[1], r[1]);
        if (i < p.width) add(u[0], r[0]);
        load(min(i + 512, last), u[0], r[0]);
        if (i + 256 < p.width) add(u[1], r[1]);
    }
    // lane n: token n's logits
    float v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        v[e] = 0.f;
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const float sum = wave_allreduce_sum(a[n][e]);
            v[e] = lane == n ? sum : v[e];
        }
    }
    const int64_t t = t0 + lane;
    if (lane >= N || t >= p.num_tokens) return;
    // the largest of eight, ties to the lowest (NaN and -inf never win: 0x7fffffff)
    auto argmax = [](const float (&s)[E], float &best, int &besti) {
        best = -INFINITY;
        besti = 0x7fffffff;
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (s[e] > best) {
                best = s[e];
                besti = e;
            }
    };
    auto take = [](float (&s)[E], int i) {
#pragma unroll
        for (int e = 0; e < E; ++e) s[e] = e == i ? -INFINITY : s[e];
    };
    float c[E], mine[E], denom = 0.f;       // c: choice
    int mine_idx[E];
    float all_max = -INFINITY, all_den = 0.f, chosen_max = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if constexpr (GROUPED) {
            v[e] = 1.0f / (1.0f + expf(-v[e]));
            c[e] = e < experts ? v[e] + (p.bias ? p.bias[e] : 0.f) : -INFINITY;
        } else {
            c[e] = e < experts ? v[e] + (p.bias ? p.bias[e] : 0.f) : -INFINITY;
        }
    }
    if constexpr (GROUPED) {
        if (p.count > 1 && p.keep < p.count) {
            const int per = experts / p.count;
            float g[E];
            unsigned kept = 0;
            auto scores = [&](int size) {       // a group's score: its two largest choice scores (one, in groups of one)
#pragma unroll
                for (int i = 0; i < E; ++i) {
                    float a0 = -INFINITY, b0 = -INFINITY;
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        if (e >= i * size && e < (i + 1) * size) {
                            if (c[e] > a0) {
                                b0 = a0;
                                a0 = c[e];
                            } else if (c[e] > b0) {
                                b0 = c[e];
                            }
                        }
                    }
                    g[i] = i < p.count ? size > 1 ? a0 + b0 : a0 : -INFINITY;
                }
            };
            auto leave = [&](int size) {
#pragma unroll
                for (int e = 0; e < E; ++e)
                    if (!(kept >> e / size & 1)) c[e] = -INFINITY;
            };
            if (per == 2) scores(2);        // (sizes that are known leave few of the comparisons)
            else if (per == 4) scores(4);
            else scores(per);
            for (int j = 0; j < p.keep; ++j) {
                float best;
                int besti;
                argmax(g, best, besti);
                take(g, besti);
                if (besti < E) kept |= 1u << besti;
            }
            if (per == 2) leave(2);
            else if (per == 4) leave(4);
            else leave(per);
        }
    } else if (p.all_scores) {      // (sums in the order of a wave's exchange)
        float q[E];
#pragma unroll
        for (int e = 0; e < E; ++e) all_max = e < experts ? fmaxf(all_max, c[e]) : all_max;
#pragma unroll
        for (int e = 0; e < E; ++e) q[e] = e < experts ? expf(c[e] - all_max) : 0.f;
        all_den = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
    }
#pragma unroll
    for (int j = 0; j < E; ++j) {
        if (j >= p.top) break;
        float best;
        int besti;
        argmax(c, best, besti);
        if (besti >= experts) besti = 0;        // (as above)
        if constexpr (GROUPED) {
            mine[j] = v[0];
#pragma unroll
            for (int e = 1; e < E; ++e) mine[j] = e == besti ? v[e] : mine[j];
        } else {
            if (j == 0) chosen_max = p.all_scores ? all_max : best;
            mine[j] = expf(best - chosen_max);
        }
        denom += mine[j];
        mine_idx[j] = besti;
        take(c, besti);
    }
    const float mult = GROUPED ? p.normalize ? 1.0f / (denom + 1e-20f) : 1.0f : p.all_scores ? p.scale / all_den : 1.0f / denom;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        if (j >= p.top) break;
        p.idx[t * p.top + j] = mine_idx[j];
        p.w[t * p.top + j] = mine[j] * mult;
    }
}

// Where that pays, us by a workgroup a token -> so, bf16 (two tokens a wave). Seven and eight experts: from 3072 tokens on (2048 columns, 3000 tokens 10.8 -> 9.8
// plain, 12.8 -> 11.7 in four groups; 1024 columns in groups 2000 tokens 1.13 times as long). All scores and one group, whose choice a workgroup makes
// quickly, from 5632 on (1024 columns, 4500 tokens 10.0 -> 10.5, 6000 11.9 -> 10.5). Five and six, for which some of the eight sums are for nothing, from 6600 on (2048
// columns, all scores 4500 tokens 11.9 -> 13.7, 7000 15.9 -> 13.7 by four). Fewer never (two, 2048 columns: 4700 tokens 8.8 -> 12.4 to 14.6, 9000 14.9 -> 17.0 to
// 19.0). Four tokens a wave, not of fp32, from 6600 on: 2048 columns plain, two and four, 4500 tokens 12.4, 12.0, 7000 14.7, 12.5; 1024 6000 9.1, 9.5, 7000 10.3, 9.5.
constexpr int64_t kRouteFewTokens = 3072, kRouteQuickTokens = 5632, kRouteFourTokens = 6600;
constexpr int kRouteLeast = 5, kRouteMost = 7;
template <typename T, bool GROUPED>
bool route_few(const RouteParams &p, hipStream_t s) {
    const bool quick = GROUPED ? p.count <= 1 || p.keep >= p.count : p.all_scores != 0;
    const int64_t least = p.experts < kRouteMost ? kRouteFourTokens : quick ? kRouteQuickTokens : kRouteFewTokens;
    if (p.num_tokens < least || p.experts > kRouteFew || p.experts < kRouteLeast || p.width % 4 || !aligned16(p.router) || (reinterpret_cast<uintptr_t>(p.h) & (4 * sizeof(T) - 1))) return false;
    const int each = sizeof(T) == 4 || p.num_tokens < kRouteFourTokens ? 2 : 4;
    const dim3 grid(static_cast<unsigned>((p.num_tokens + each * kMoeWaves - 1) / (each * kMoeWaves)));
    if (each == 2) hipLaunchKernelGGL((moe_route_few_kernel<T, GROUPED, 2>), grid, dim3(kMoeThreads), 0, s, p);
    else hipLaunchKernelGGL((moe_route_few_kernel<T, GROUPED, 4>), grid, dim3(kMoeThreads), 0, s, p);
    return true;
}

// The per-assignment kernels: every (token, chosen expert) streams its expert's rows. Bound by latency at decode sizes (3 tokens, two
// experts of 1024 x 1024, fp32: 25 MB), so a workgroup owns sixteen outputs and a wave four rows at a time, whose loads are in flight
// together. That shape: up 115 and down 228 us with 64 outputs a workgroup and one row
// of 4-byte loads at a time, 7.5 and 8 us.
constexpr int kMoeRows = 16;        // outputs of a workgroup
inline int moe_rows(int n) { return (n + kMoeRows - 1) / kMoeRows <= 65535 ? kMoeRows : 64; }

// grid (assignments, ceil(ff / rows))
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void moe_gate_up_kernel(T *y, const T *h, const T *gate_up,
                                                                  const int32_t *expert_idx, const float *in_w, int width,
                                                                  int ff, int top, float limit, int act, int rows) {
    extern __shared__ __align__(16) float lds[];
    float *hf = lds;    // [width]
    const int64_t a = blockIdx.x;           // assignment = token * top + j
    const int64_t t = a / top;
    const int e = expert_idx[a];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int i = threadIdx.x; i < width; i += kMoeThreads) hf[i] = to_f(h[t * width + i]);
    __syncthreads();
    const T *wg = gate_up + static_cast<int64_t>(e) * 2 * ff * width;
    const T *wu = wg + static_cast<int64_t>(ff) * width;
    const int f0 = blockIdx.y * rows, f1 = min(ff, f0 + rows);
    for (int f = f0 + 2 * wave; f < f1; f += 2 * kMoeWaves) {
        const int64_t at0 = static_cast<int64_t>(f) * width, at1 = static_cast<int64_t>(min(f + 1, f1 - 1)) * width;
        const T *const w[4] = {wg + at0, wu + at0, wg + at1, wu + at1};
        float v[4];
        lane_dots(v, hf, w, width, lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] = wave_allreduce_sum(v[r]);
            if (in_w) v[r] *= in_w[a];
        }
        if (lane == 0) y[a * ff + f] = to_t<T>(gated_unit(v[0], v[1], limit, act));
        if (lane == 0 && f + 1 < f1) y[a * ff + f + 1] = to_t<T>(gated_unit(v[2], v[3], limit, act));
    }
}

// Experts without a gate: y = relu(W_up h)^2 for every (token, chosen expert); up [experts, ff, width]. Same grid.
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void moe_up_relu2_kernel(T *y, const T *h, const T *up, const int32_t *expert_idx,
                                                                   int width, int ff, int top, int rows) {
    extern __shared__ __align__(16) float lds[];
    float *hf = lds;    // [width]
    const int64_t a = blockIdx.x;
    const int64_t t = a / top;
    const int e = expert_idx[a];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int i = threadIdx.x; i < width; i += kMoeThreads) hf[i] = to_f(h[t * width + i]);
    __syncthreads();
    const T *wu = up + static_cast<int64_t>(e) * ff * width;
    const int f0 = blockIdx.y * rows, f1 = min(ff, f0 + rows);
    for (int f = f0 + 4 * wave; f < f1; f += 4 * kMoeWaves) {
        const T *w[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = wu + static_cast<int64_t>(min(f + r, f1 - 1)) * width;
        float v[4];
        lane_dots(v, hf, w, width, lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float u = fmaxf(wave_allreduce_sum(v[r]), 0.f);
            if (lane == 0 && f + r < f1) y[a * ff + f + r] = to_t<T>(u * u);
        }
    }
}

// y[r][f] = relu(z[r][f])^2 over rows of z that may be wider than ff (in_stride)
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void relu_sq_kernel(T *y, const T *z, int64_t total, int ff, int64_t in_stride) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kMoeThreads + threadIdx.x;
    if (i >= total) return;
    const int64_t r = i / ff;
    const float v = fmaxf(to_f(z[r * in_stride + (i - r * ff)]), 0.f);
    y[i] = to_t<T>(v * v);
}

// the same for 16-bit rows of a multiple of 8 elements on 16-byte boundaries: 8 elements (16 bytes) per lane
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void relu_sq_wide_kernel(T *y, const T *z, int64_t total8, int ff8,
                                                                   int64_t in_stride) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kMoeThreads + threadIdx.x;
    if (i >= total8) return;
    const int64_t r = i / ff8;
    const int c = static_cast<int>(i - r * ff8) * 8;
    const vec8_t<T> x = load8(z + r * in_stride + c);
    vec8_t<T> o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float v = fmaxf(to_f(x[j]), 0.f);
        o[j] = to_t<T>(v * v);
    }
    store8(y + r * static_cast<int64_t>(ff8) * 8 + c, o);
}

// grid (tokens, ceil(width / rows)): out[t][c] = sum_j w[t][j] y[t * top + j] . down[e_j][c]
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void moe_down_combine_kernel(T *out, const T *y, const T *down,
                                                                       const int32_t *expert_idx, const float *expert_w,
                                                                       int width, int ff, int top, int rows) {
    const int64_t t = blockIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c0 = blockIdx.y * rows, c1 = min(width, c0 + rows);
    for (int c = c0 + 4 * wave; c < c1; c += 4 * kMoeWaves) {
        float total[4] = {0.f, 0.f, 0.f, 0.f};
        for (int j = 0; j < top; ++j) {
            const T *wd = down + static_cast<int64_t>(expert_idx[t * top + j]) * width * ff;
            const T *w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = wd + static_cast<int64_t>(min(c + r, c1 - 1)) * ff;
            float v[4];
            lane_dots(v, y + (t * top + j) * ff, w, ff, lane);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float a = wave_allreduce_sum(v[r]);
                total[r] += expert_w ? expert_w[t * top + j] * a : a;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (lane == 0 && c + r < c1) out[t * width + c + r] = to_t<T>(total[r]);
    }
}


// ---- expert-stationary products for decode-sized steps -----------------------------------------------------------------------
// out[a][n] = sum_k W[e][n][k] X[xrow(a)][k] for the assignments a of expert e, on the matrix core. A workgroup owns (expert,
// 64 outputs n), a wave 16 of them: per 16-wide k step it loads its weight fragment ONCE (A operand: row n, 8 bytes per lane)
// and multiplies it with the input fragments of up to four tiles of 16 assignments (B operand: the assignment's input row,
// read through the caches — the rows of a decode step are few and stay resident). An expert's weights are thus streamed once
// per step however many tokens chose it (the per-assignment kernels above stream them once per token). GLU: n indexes ff,
// the gate row n and the up row ff + n share the input fragments and meet in the clamped gated unit; X rows are tokens
// (a / top). Otherwise (down projection) X rows are assignments and the output is the plain product, rounded to T.
constexpr int kEsRows = 64;         // outputs per workgroup at most (16 per wave; fewer waves when the grid would be small)
constexpr int kEsTiles = 4;         // tiles of 16 assignments per pass over the weights
constexpr int kEsMaxAssign = 1024;  // assignments per step (the sorted library path serves larger steps)

template <typename T, int MODE>
__global__ __launch_bounds__(kMoeThreads, 2) void moe_expert_stationary_kernel(T *out, const T *x, const T *w,
                                                                            const int32_t *expert_idx, const float *in_w,
                                                                            int assignments, int K, int N, int top, float limit, int ksplit) {
    // ksplit = 1: every wave of the workgroup owns 16 outputs and the whole reduction. ksplit = waves of the workgroup: all
    // waves own the SAME 16 outputs and a quarter (half) of the reduction each; their accumulators meet in LDS and wave 0
    // finishes (short reductions and few outputs would otherwise leave most of the chip idle in a decode step).
    // MODE 0: plain product, X rows are assignments; 1: clamped gated unit, X rows are tokens; 2: squared ReLU of the plain
    // product (experts without a gate), X rows are tokens
    constexpr bool GLU = MODE == 1 || MODE == 3;      // (3: the plain gated unit silu(g) u)
    __shared__ int mine[kEsMaxAssign];
    __shared__ int count;
    __shared__ float red[3][2 * kEsTiles][256];
    const int e = blockIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nwaves = blockDim.x >> 6;
    const int li = lane & 15, lq = lane >> 4;
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    for (int a = threadIdx.x; a < assignments; a += blockDim.x)
        if (expert_idx[a] == e) mine[atomicAdd(&count, 1)] = a;
    __syncthreads();
    const int m = count;
    const int n0 = ksplit > 1 ? blockIdx.y * 16 : (blockIdx.y * nwaves + wave) * 16;
    if (m == 0 || (ksplit == 1 && n0 >= N)) return;
    const int kper = K / ksplit;                       // (ksplit > 1: a multiple of 32, checked on the host)
    const int kbeg = ksplit > 1 ? wave * kper : 0, kend = kbeg + kper;
    const int nrow = min(n0 + li, N - 1);       // (rows past N compute a duplicate that is never stored)
    // this lane's share of a 32-wide reduction step: elements 8 lq .. 8 lq + 7 (one 16-byte load), fed to the matrix core as
    // two 4-element halves — the same split on both operands, so the order inside a step does not matter
    const T *wg = w + (static_cast<int64_t>(e) * (GLU ? 2 : 1) * N + nrow) * K + 8 * lq;
    const T *wu = wg + static_cast<int64_t>(N) * K;
    const bool wide = (kper & 31) == 0 && ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(x)) & 15) == 0 && (K & 7) == 0;
    for (int pass = 0; pass < m; pass += 16 * kEsTiles) {
        const int ntile = min(kEsTiles, (m - pass + 15) / 16);
        int arow[kEsTiles];
        const T *xp[kEsTiles];
#pragma unroll
        for (int t = 0; t < kEsTiles; ++t) {
            const int i = pass + t * 16 + li;
            const int a = i < m ? mine[i] : -1;
            arow[t] = a;
            xp[t] = x + static_cast<int64_t>(a < 0 ? 0 : (MODE != 0 ? a / top : a)) * K + 8 * lq;
        }
        float4_t accg[kEsTiles], accu[kEsTiles];
#pragma unroll
        for (int t = 0; t < kEsTiles; ++t) accg[t] = accu[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        if (wide) {
#pragma unroll 2
            for (int k0 = kbeg; k0 < kend; k0 += 32) {
                const vec8_t<T> ag = load8(wg + k0);
                vec8_t<T> au = vec8_t<T>{};
                if constexpr (GLU) au = load8(wu + k0);
#pragma unroll
                for (int t = 0; t < kEsTiles; ++t) {
                    if (t < ntile) {
                        vec8_t<T> b = vec8_t<T>{};
                        if (arow[t] >= 0) b = load8(xp[t] + k0);
                        const vec4_t<T> b0 = {b[0], b[1], b[2], b[3]}, b1 = {b[4], b[5], b[6], b[7]};
                        accg[t] = mfma16(vec4_t<T>{ag[0], ag[1], ag[2], ag[3]}, b0, accg[t]);
                        accg[t] = mfma16(vec4_t<T>{ag[4], ag[5], ag[6], ag[7]}, b1, accg[t]);
                        if constexpr (GLU) {
                            accu[t] = mfma16(vec4_t<T>{au[0], au[1], au[2], au[3]}, b0, accu[t]);
                            accu[t] = mfma16(vec4_t<T>{au[4], au[5], au[6], au[7]}, b1, accu[t]);
                        }
                    }
                }
            }
        } else {
            // 16-wide steps, 8-byte fragments (this lane: elements 4 lq .. 4 lq + 3 of the step)
            const T *wg4 = wg - 4 * lq, *wu4 = wu - 4 * lq;
#pragma unroll 4
            for (int k0 = kbeg; k0 < kend; k0 += 16) {
                vec4_t<T> ag, au;
                load4(ag, wg4 + k0);
                if constexpr (GLU) load4(au, wu4 + k0);
#pragma unroll
                for (int t = 0; t < kEsTiles; ++t) {
                    if (t < ntile) {
                        vec4_t<T> b = vec4_t<T>{};
                        if (arow[t] >= 0) load4(b, xp[t] - 4 * lq + k0);
                        accg[t] = mfma16(ag, b, accg[t]);
                        if constexpr (GLU) accu[t] = mfma16(au, b, accu[t]);
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < kEsTiles; ++t) {
            mfma_results_tie(accg[t]);
            mfma_results_ready<4>(accu[t]);
        }
        if (ksplit > 1) {       // (workgroup-uniform) sum the waves' partial accumulators in wave 0
            __syncthreads();    // (the previous pass's partials have been read)
            if (wave > 0) {
#pragma unroll
                for (int t = 0; t < kEsTiles; ++t) {
                    if (t < ntile) {
                        *reinterpret_cast<float4_t *>(&red[wave - 1][2 * t][lane * 4]) = accg[t];
                        if constexpr (GLU) *reinterpret_cast<float4_t *>(&red[wave - 1][2 * t + 1][lane * 4]) = accu[t];
                    }
                }
            }
            __syncthreads();
            if (wave > 0) continue;
            for (int o = 0; o + 1 < nwaves; ++o) {
#pragma unroll
                for (int t = 0; t < kEsTiles; ++t) {
                    if (t < ntile) {
                        accg[t] += *reinterpret_cast<const float4_t *>(&red[o][2 * t][lane * 4]);
                        if constexpr (GLU) accu[t] += *reinterpret_cast<const float4_t *>(&red[o][2 * t + 1][lane * 4]);
                    }
                }
            }
        }
        // accumulator r of lane (li, lq): output row n0 + 4 lq + r of the assignment in column li
#pragma unroll
        for (int t = 0; t < kEsTiles; ++t) {
            if (t < ntile && arow[t] >= 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = n0 + 4 * lq + r;
                    if (n < N) {
                        float v = accg[t][r];
                        if constexpr (GLU) {
                            const float iw = in_w ? in_w[arow[t]] : 1.f;
                            v = gated_unit(v * iw, accu[t][r] * iw, limit, MODE == 3 ? 1 : 0);
                        }
                        if constexpr (MODE == 2) {
                            v = fmaxf(v, 0.f);
                            v *= v;
                        }
                        out[static_cast<int64_t>(arow[t]) * N + n] = to_t<T>(v);
                    }
                }
            }
        }
    }
}

// y[r][f] = act(w[r] gu[r][f], w[r] gu[r][ff + f]) for rows of [gate | up] products that came from a library GEMM (in_w NULL: 1)
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void glu_clamp_kernel(T *y, const T *gu, const float *in_w, int64_t total, int ff,
                                                                float limit, int act, int64_t y_stride, int64_t gu_stride,
                                                                int64_t up_off) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kMoeThreads + threadIdx.x;
    if (i >= total) return;
    const int64_t r = i / ff;
    const int f = static_cast<int>(i - r * ff);
    const float w = in_w ? in_w[r] : 1.f;
    const T *g = gu + r * gu_stride + f;
    y[r * y_stride + f] = to_t<T>(gated_unit(w * to_f(g[0]), w * to_f(g[up_off]), limit, act));
}

// the same for 16-bit rows of a multiple of 8 elements on 16-byte boundaries: 8 elements (16 bytes) per lane
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void glu_clamp_wide_kernel(T *y, const T *gu, const float *in_w, int64_t total8,
                                                                     int ff8, float limit, int act, int64_t y_stride,
                                                                     int64_t gu_stride, int64_t up_off) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kMoeThreads + threadIdx.x;
    if (i >= total8) return;
    const int64_t r = i / ff8;
    const int f = static_cast<int>(i - r * ff8) * 8;
    const float w = in_w ? in_w[r] : 1.f;
    const vec8_t<T> g = load8(gu + r * gu_stride + f), u = load8(gu + r * gu_stride + up_off + f);
    vec8_t<T> o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = to_t<T>(gated_unit(w * to_f(g[j]), w * to_f(u[j]), limit, act));
    store8(y + r * y_stride + f, o);
}

// out[t] = sum_j w[t][j] * rows[where[t * top + j]]  (fp32 sum in the order j = 0, 1, ...)
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void moe_combine_kernel(T *out, const T *rows, const int64_t *where,
                                                                  const float *w, int width, int top) {
    const int64_t t = blockIdx.x;
    for (int c = threadIdx.x; c < width; c += kMoeThreads) {
        float a = 0.f;
        for (int j = 0; j < top; ++j) a += (w ? w[t * top + j] : 1.f) * to_f(rows[where[t * top + j] * width + c]);
        out[t * width + c] = to_t<T>(a);
    }
}

// The same for 16-bit rows of whole 16-byte pieces: 8 columns a lane, flat over (token, piece). Bound by HBM: `top` + 1 rows a token;
// 8000 tokens of 1024, two rows each: 20 us with one 2-byte access a lane and row, 10 us.
template <typename T>
__global__ __launch_bounds__(kMoeThreads) void moe_combine_wide_kernel(T *out, const T *rows, const int64_t *where, const float *w,
                                                                       int64_t pieces, int width8, int top) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kMoeThreads + threadIdx.x;
    if (i >= pieces) return;
    const int64_t t = i / width8, c = (i - t * width8) * 8, width = static_cast<int64_t>(width8) * 8;
    float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < top; ++j) {
        const float wj = w ? w[t * top + j] : 1.f;
        const vec8_t<T> r = load8(rows + where[t * top + j] * width + c);
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] += wj * to_f(r[k]);
    }
    vec8_t<T> o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = to_t<T>(a[k]);
    store8(out + t * width + c, o);
}

} // namespace swl

/* 1 when swl_moe_expert_stationary serves the shape: 16-bit, both reduction lengths multiples of 16, at most 1024
 * assignments. */
extern "C" int swl_moe_expert_stationary_supported(int64_t num_tokens, int32_t width, int32_t ff, int32_t top, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    if (width <= 0 || ff <= 0 || (width & 15) || (ff & 15)) return 0;
    return num_tokens * top <= swl::kEsMaxAssign;
}

extern "C" int swl_moe_expert_stationary(void *out, const void *x, const void *w, const int32_t *expert_idx, const float *in_w,
                                         int64_t num_tokens, int32_t experts, int32_t width, int32_t ff, int32_t top,
                                         int32_t glu, float limit, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || experts <= 0 || top <= 0) return SWL_ERR_BAD_ARG;
    if (!swl_moe_expert_stationary_supported(num_tokens, width, ff, top, dtype)) return SWL_ERR_UNSUPPORTED;
    if (num_tokens == 0) return SWL_OK;
    if (!out || !x || !w || !expert_idx || !swl::aligned16(x) || !swl::aligned16(w)) return SWL_ERR_BAD_ARG;
    const int K = glu ? width : ff, N = glu ? ff : width;
    const int assignments = static_cast<int>(num_tokens * top);
    const size_t lds = 0;
    // Four waves per workgroup. With plenty of outputs each wave owns 16 of them; when that would launch under ~2048 waves
    // (a decode step must fill 256 CUs x 4 SIMDs, with latency to hide) the four waves share 16 outputs and split the reduction.
    const int nw = 4;
    const int64_t tiles16 = (N + 15) / 16;
    const int ksplit = (experts * tiles16 < 2048 && K % (32 * nw) == 0) ? nw : 1;
    const dim3 grid(static_cast<unsigned>(experts),
                    static_cast<unsigned>(ksplit > 1 ? tiles16 : (N + 16 * nw - 1) / (16 * nw)));
    if (grid.y > 65535) return SWL_ERR_UNSUPPORTED;
    hipStream_t s = static_cast<hipStream_t>(stream);
    SWL_DISPATCH_DTYPE(dtype, T, {
        if (glu == 1)
            hipLaunchKernelGGL((swl::moe_expert_stationary_kernel<T, 1>), grid, dim3(64 * nw), lds, s,
                               static_cast<T *>(out), static_cast<const T *>(x), static_cast<const T *>(w), expert_idx,
                               in_w, assignments, K, N, top, limit, ksplit);
        else if (glu == 2)
            hipLaunchKernelGGL((swl::moe_expert_stationary_kernel<T, 2>), grid, dim3(64 * nw), lds, s,
                               static_cast<T *>(out), static_cast<const T *>(x), static_cast<const T *>(w), expert_idx,
                               in_w, assignments, K, N, top, limit, ksplit);
        else if (glu == 3)
            hipLaunchKernelGGL((swl::moe_expert_stationary_kernel<T, 3>), grid, dim3(64 * nw), lds, s,
                               static_cast<T *>(out), static_cast<const T *>(x), static_cast<const T *>(w), expert_idx,
                               in_w, assignments, K, N, top, limit, ksplit);
        else
            hipLaunchKernelGGL((swl::moe_expert_stationary_kernel<T, 0>), grid, dim3(64 * nw), lds, s,
                               static_cast<T *>(out), static_cast<const T *>(x), static_cast<const T *>(w), expert_idx,
                               in_w, assignments, K, N, top, limit, ksplit);
    });
    return swl::check_launch();
}

extern "C" int swl_glu_rows(void *y, int64_t y_stride, const void *gate_up, int64_t gu_stride, int64_t up_off, const float *in_w,
                            int64_t num_rows, int32_t ff, float limit, int32_t act, int32_t dtype, swl_stream_t stream) {
    if (num_rows < 0 || ff <= 0 || act < 0 || act > 2 || y_stride < ff || up_off < ff || gu_stride < up_off + ff)
        return SWL_ERR_BAD_ARG;
    if (num_rows == 0) return SWL_OK;
    if (!y || !gate_up) return SWL_ERR_BAD_ARG;
    const bool wide = dtype != SWL_F32 && ((ff | y_stride | gu_stride | up_off) & 7) == 0 && swl::aligned16(y) &&
                      swl::aligned16(gate_up);
    const int64_t total = num_rows * ff / (wide ? 8 : 1);
    const int64_t blocks = (total + swl::kMoeThreads - 1) / swl::kMoeThreads;
    if (blocks > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    if (wide) {
        SWL_DISPATCH_DTYPE(dtype, T, {
            hipLaunchKernelGGL((swl::glu_clamp_wide_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(swl::kMoeThreads), 0,
                               static_cast<hipStream_t>(stream), static_cast<T *>(y), static_cast<const T *>(gate_up), in_w,
                               total, ff / 8, limit, act, y_stride, gu_stride, up_off);
        });
        return swl::check_launch();
    }
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::glu_clamp_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(swl::kMoeThreads), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(y), static_cast<const T *>(gate_up), in_w, total,
                           ff, limit, act, y_stride, gu_stride, up_off);
    });
    return swl::check_launch();
}

extern "C" int swl_glu_clamp(void *y, const void *gate_up, const float *in_w, int64_t num_rows, int32_t ff, float limit,
                             int32_t act, int32_t dtype, swl_stream_t stream) {
    return swl_glu_rows(y, ff, gate_up, 2 * static_cast<int64_t>(ff), ff, in_w, num_rows, ff, limit, act, dtype, stream);
}

extern "C" int swl_moe_combine(void *out, const void *rows, const int64_t *where, const float *expert_w,
                               int64_t num_tokens, int32_t width, int32_t top, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || top <= 0) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!out || !rows || !where) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    const int64_t pieces = num_tokens * (width / 8), blocks = (pieces + swl::kMoeThreads - 1) / swl::kMoeThreads;
    if (width % 8 == 0 && swl::aligned16(out) && swl::aligned16(rows) && blocks <= 0x7fffffffLL && dtype != SWL_F32) {
        SWL_DISPATCH_DTYPE(dtype, T, {
            hipLaunchKernelGGL((swl::moe_combine_wide_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(swl::kMoeThreads), 0,
                               static_cast<hipStream_t>(stream), static_cast<T *>(out), static_cast<const T *>(rows), where, expert_w,
                               pieces, width / 8, top);
        });
        return swl::check_launch();
    }
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::moe_combine_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kMoeThreads), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(out), static_cast<const T *>(rows), where,
                           expert_w, width, top);
    });
    return swl::check_launch();
}

extern "C" int swl_moe_route(int32_t *idx_out, float *w_out, const void *h, const float *router, const float *bias,
                             int64_t num_tokens, int32_t width, int32_t experts, int32_t top, int32_t dtype,
                             swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || experts <= 0 || top <= 0 || top > experts) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!idx_out || !w_out || !h || !router || !bias) return SWL_ERR_BAD_ARG;
    const size_t lds = (static_cast<size_t>(width) + experts) * 4;
    if (num_tokens > 0x7fffffffLL || lds > 64 * 1024) return SWL_ERR_UNSUPPORTED;
    const swl::RouteParams few = {idx_out, w_out, h, router, bias, num_tokens, width, experts, top, 0, 1, 1, 0, 1.0f};
    SWL_DISPATCH_DTYPE3(dtype, T, {
        if (swl::route_few<T, false>(few, static_cast<hipStream_t>(stream))) return swl::check_launch();
        hipLaunchKernelGGL((swl::moe_route_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kMoeThreads),
                           lds, static_cast<hipStream_t>(stream), idx_out, w_out, static_cast<const T *>(h), router, bias,
                           width, experts, top, 0, 1.0f);
    });
    return swl::check_launch();
}

extern "C" int swl_moe_route_scores(int32_t *idx_out, float *w_out, const void *h, const float *router, const float *bias,
                                    int64_t num_tokens, int32_t width, int32_t experts, int32_t top, float scale,
                                    int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || experts <= 0 || top <= 0 || top > experts) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!idx_out || !w_out || !h || !router) return SWL_ERR_BAD_ARG;
    const size_t lds = (static_cast<size_t>(width) + experts) * 4;
    if (num_tokens > 0x7fffffffLL || lds > 64 * 1024) return SWL_ERR_UNSUPPORTED;
    const swl::RouteParams few = {idx_out, w_out, h, router, bias, num_tokens, width, experts, top, 1, 1, 1, 0, scale};
    SWL_DISPATCH_DTYPE3(dtype, T, {
        if (swl::route_few<T, false>(few, static_cast<hipStream_t>(stream))) return swl::check_launch();
        hipLaunchKernelGGL((swl::moe_route_kernel<T>), dim3(static_cast<unsigned>(num_tokens)), dim3(swl::kMoeThreads),
                           lds, static_cast<hipStream_t>(stream), idx_out, w_out, static_cast<const T *>(h), router, bias,
                           width, experts, top, 1, scale);
    });
    return swl::check_launch();
}

extern "C" int swl_moe_gate_up(void *y, const void *h, const void *gate_up, const int32_t *expert_idx, const float *in_w,
                               int64_t num_tokens, int32_t width, int32_t ff, int32_t top, float limit, int32_t act,
                               int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || ff <= 0 || top <= 0 || act < 0 || act > 1) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!y || !h || !gate_up || !expert_idx) return SWL_ERR_BAD_ARG;
    const size_t lds = static_cast<size_t>(width) * 4;
    const int64_t assignments = num_tokens * top;
    if (assignments > 0x7fffffffLL || lds > 64 * 1024 || (ff + 63) / 64 > 65535) return SWL_ERR_UNSUPPORTED;
    const int rows = swl::moe_rows(ff);
    const dim3 grid(static_cast<unsigned>(assignments), static_cast<unsigned>((ff + rows - 1) / rows));
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::moe_gate_up_kernel<T>), grid, dim3(swl::kMoeThreads), lds,
                           static_cast<hipStream_t>(stream), static_cast<T *>(y), static_cast<const T *>(h),
                           static_cast<const T *>(gate_up), expert_idx, in_w, width, ff, top, limit, act, rows);
    });
    return swl::check_launch();
}

extern "C" int swl_moe_down_combine(void *out, const void *y, const void *down, const int32_t *expert_idx,
                                    const float *expert_w, int64_t num_tokens, int32_t width, int32_t ff, int32_t top,
                                    int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || ff <= 0 || top <= 0) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!out || !y || !down || !expert_idx) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL || (width + 63) / 64 > 65535) return SWL_ERR_UNSUPPORTED;
    const int rows = swl::moe_rows(width);
    const dim3 grid(static_cast<unsigned>(num_tokens), static_cast<unsigned>((width + rows - 1) / rows));
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::moe_down_combine_kernel<T>), grid, dim3(swl::kMoeThreads), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(out), static_cast<const T *>(y),
                           static_cast<const T *>(down), expert_idx, expert_w, width, ff, top, rows);
    });
    return swl::check_launch();
}

extern "C" int swl_moe_up_relu2(void *y, const void *h, const void *up, const int32_t *expert_idx, int64_t num_tokens,
                                int32_t width, int32_t ff, int32_t top, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || ff <= 0 || top <= 0) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!y || !h || !up || !expert_idx) return SWL_ERR_BAD_ARG;
    const size_t lds = static_cast<size_t>(width) * 4;
    const int64_t assignments = num_tokens * top;
    if (assignments > 0x7fffffffLL || lds > 64 * 1024 || (ff + 63) / 64 > 65535) return SWL_ERR_UNSUPPORTED;
    const int rows = swl::moe_rows(ff);
    const dim3 grid(static_cast<unsigned>(assignments), static_cast<unsigned>((ff + rows - 1) / rows));
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::moe_up_relu2_kernel<T>), grid, dim3(swl::kMoeThreads), lds,
                           static_cast<hipStream_t>(stream), static_cast<T *>(y), static_cast<const T *>(h),
                           static_cast<const T *>(up), expert_idx, width, ff, top, rows);
    });
    return swl::check_launch();
}

extern "C" int swl_relu_sq(void *y, const void *z, int64_t num_rows, int32_t ff, int64_t in_stride, int32_t dtype,
                           swl_stream_t stream) {
    if (num_rows < 0 || ff <= 0 || in_stride < ff) return SWL_ERR_BAD_ARG;
    if (num_rows == 0) return SWL_OK;
    if (!y || !z) return SWL_ERR_BAD_ARG;
    const int64_t total = num_rows * ff;
    if (dtype != SWL_F32 && ff % 8 == 0 && in_stride % 8 == 0 && swl::aligned16(y) && swl::aligned16(z)) {
        const int64_t total8 = total / 8, blocks8 = (total8 + swl::kMoeThreads - 1) / swl::kMoeThreads;
        SWL_DISPATCH_DTYPE(dtype, T, {
            hipLaunchKernelGGL((swl::relu_sq_wide_kernel<T>), dim3(static_cast<unsigned>(blocks8)), dim3(swl::kMoeThreads),
                               0, static_cast<hipStream_t>(stream), static_cast<T *>(y), static_cast<const T *>(z), total8,
                               ff / 8, in_stride);
        });
        return swl::check_launch();
    }
    const int64_t blocks = (total + swl::kMoeThreads - 1) / swl::kMoeThreads;
    if (blocks > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    SWL_DISPATCH_DTYPE3(dtype, T, {
        hipLaunchKernelGGL((swl::relu_sq_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(swl::kMoeThreads), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(y), static_cast<const T *>(z), total, ff,
                           in_stride);
    });
    return swl::check_launch();
}

extern "C" int swl_moe_route_grouped(int32_t *idx_out, float *w_out, const void *h, const float *router,
                                     const float *correction, int64_t num_tokens, int32_t width, int32_t experts, int32_t top,
                                     int32_t group_count, int32_t group_keep, int32_t normalize, int32_t dtype,
                                     swl_stream_t stream) {
    if (num_tokens < 0 || width <= 0 || experts <= 0 || top <= 0 || top > experts) return SWL_ERR_BAD_ARG;
    if (group_count < 1 || group_keep < 1 || group_keep > group_count || experts % group_count) return SWL_ERR_BAD_ARG;
    if (static_cast<int64_t>(group_keep) * (experts / group_count) < top) return SWL_ERR_BAD_ARG;
    if (num_tokens == 0) return SWL_OK;
    if (!idx_out || !w_out || !h || !router) return SWL_ERR_BAD_ARG;
    const size_t lds = (static_cast<size_t>(width) + 2 * experts + 2 * group_count) * 4;
    if (num_tokens > 0x7fffffffLL || lds > 64 * 1024) return SWL_ERR_UNSUPPORTED;
    const swl::RouteParams few = {idx_out, w_out, h, router, correction, num_tokens, width, experts, top, 0, group_count, group_keep, normalize, 1.0f};
    SWL_DISPATCH_DTYPE3(dtype, T, {
        if (swl::route_few<T, true>(few, static_cast<hipStream_t>(stream))) return swl::check_launch();
        hipLaunchKernelGGL((swl::moe_route_grouped_kernel<T>), dim3(static_cast<unsigned>(num_tokens)),
                           dim3(swl::kMoeThreads), lds, static_cast<hipStream_t>(stream), idx_out, w_out,
                           static_cast<const T *>(h), router, correction, width, experts, top, group_count, group_keep,
                           normalize);
    });
    return swl::check_launch();
}
