// mix_attn.hip — prompt attention whose heads are mixed by an [H, H] matrix at every (query, key) pair, on the matrix cores:
//   softmax form (swl_mix_attn):          p = softmax_j(sum_g talk[h][g] cap(scale q_g . k_j)), windows
//   sigmoid form (swl_mix_sigmoid_attn):  p = sum_g talk[h][g] sigmoid(scale q_g . k_j - r1_g ln(1 + r2_g dist) + pb_g)
// the arithmetic of window_attn_mfma.hip and sigmoid_attn.hip (fp32 scores and weights, weights into the value product as two 16-bit
// terms), another split of the work.
//
// What bounds it: H^2 multiply-adds per pair for the mix beside 2 H (D + 2 DV) for the products, and the exchange of the scores between
// the waves that own the heads. One workgroup of eight waves takes 16 consecutive queries and walks 32 keys a stage; wave w owns HPW
// heads (of one key head) for the score and the value products. In between, the scores of all heads lie in LDS as a matrix [g][pair] and
// the mix is a matrix product on the fp32 matrix core (16x16x4: talk as A, 16 pairs as B, exact fp32 operands), 4 of the stage's 32
// blocks of pairs a wave; its result goes back the same way. The VALU mix it replaces read every head's scores from LDS in every wave
// and spent H FMAs per score. A pair's place in a row is (lane of its owner) x 8 + key % 8: owners write and read 32 bytes a lane, and
// the row pitches (528 and 516 floats) keep the transposed accesses on different banks. The key that A row m of a score product takes
// is chosen as in span_attn.hip, so that a lane's eight scores are eight consecutive keys, the B operand of the value product. The score products of a stage are
// made where the weights of the one before are: one uses the matrix core, the other the vector units. Tiles are taken from the back: the long ones start first.
// Measured, 16 heads of 128 over 4, bf16, against the 16-query tiles with the mix on the VALU: softmax, 3 prompts of 1500 tokens, window 1024
// 697 -> 143 us; sigmoid, 11 prompts of 333 tokens 231 -> 61 us. With the score products of a stage beside the weights of the one before, the
// reads of the mix together and no load that only some paths make (each is waited for on all of them, with what was asked for before it):
// softmax 139 -> 130 us, sigmoid 71 us both (the same prompts, in a step). Vector instructions, 3500 cycles a stage, and matrix steps, 2600,
// still run mostly one after the other.
#include "attn_combine.h"
#include "swl_common.h"

namespace swl {

__device__ __forceinline__ float4_t mx_mfma(vec8_t<f16> a, vec8_t<f16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mx_mfma(vec8_t<bf16> a, vec8_t<bf16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float mx_rows_max(float v) {     // over the four lanes of a query
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

constexpr int kMxThreads = 512, kMxWaves = 8, kMxTile = 16, kMxKeys = 32;
constexpr int kMxIn = 528, kMxOut = 516;        // row pitches of the scores before and after the mix (512 pairs)

struct MixParams {
    void *out;
    const void *q, *k_cache, *v_cache;
    const int32_t *block_table, *tok_seq, *tok_pos, *tile_row0, *tile_cnt;
    const float *talk, *r1, *r2, *pb;
    float *part_o, *part_ml;
    int num_tiles, H, G, window, max_blocks;
    float scale, softcap;
    int64_t q_stride, block_stride, num_tokens;
};

template <typename T, int D, int DV, int HPW, bool SIG>
__global__ __launch_bounds__(kMxThreads, 2) void mix_attn_kernel(MixParams p) {
    constexpr int HM = 16;                      // heads of the mix product's tile
    constexpr int KS = D / 32, CT = DV / 16;
    constexpr float kLog2e = 1.4426950408889634f, kLazy = 8.0f;
    __shared__ __attribute__((aligned(16))) float s_in[HM * kMxIn];
    __shared__ __attribute__((aligned(16))) float s_out[HM * kMxOut];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lq = lane >> 4;
    const int tile = p.num_tiles - 1 - static_cast<int>(blockIdx.x), H = p.H;
    const int row0 = __builtin_amdgcn_readfirstlane(p.tile_row0[tile]), cnt = __builtin_amdgcn_readfirstlane(p.tile_cnt[tile]);
    const int p0 = __builtin_amdgcn_readfirstlane(p.tok_pos[row0]);
    const int32_t *bt = p.block_table + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(p.tok_seq[row0])) * p.max_blocks;
    const bool qok = li < cnt;
    const int qi = min(li, cnt - 1), qpos = p0 + qi;
    const int qlo = p.window > 0 ? max(qpos - p.window + 1, 0) : 0;
    int kb0 = (p.window > 0 ? max(p0 - p.window + 1, 0) : 0) / 16, kb1 = (p0 + cnt - 1) / 16;
    if (gridDim.y > 1) {        // key split: a contiguous share of the pages (possibly none), whole stages but for the last one's
        const int shares = static_cast<int>(gridDim.y), per = ((kb1 - kb0 + shares) / shares + 1) / 2 * 2;
        kb0 += per * static_cast<int>(blockIdx.y);
        kb1 = min(kb1, kb0 + per - 1);
    }
    // heads of this wave (a wave without heads still takes its blocks of the mix)
    const int h0 = wave * HPW, nh = max(0, min(HPW, H - h0)), kv = min(h0, H - 1) / (H / p.G);
    // rows of the mix that belong to no head: zero once, so that their products with a zero of talk are zero
    for (int i = H * kMxIn + tid; i < HM * kMxIn; i += kMxThreads) s_in[i] = 0.f;
    // A operand of the mix: talk[h = li][g = 4 s + lq]; softmax scores come out in base-2 exponent units
    constexpr int STEPS = 2 * HPW;              // (eight heads or fewer: one a wave, two steps; rows of no head are zero on both sides)
    float mixw[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const int g = 4 * s + lq;
        mixw[s] = li < H && g < H ? p.talk[li * H + g] * (SIG ? 1.0f : kLog2e) : 0.f;
    }
    vec8_t<T> qf[HPW][KS], kf[2][KS], vf[CT];
    const T *v_now = nullptr, *v_next = nullptr;        // values of the stage at hand and of the one whose keys were asked for last
    float4_t acc[HPW][CT];
    float mrun[HPW], lrun[HPW], hr1[HPW], hr2[HPW], hpb[HPW];
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        const int h = min(h0 + hh, H - 1);
        const T *qp = static_cast<const T *>(p.q) + static_cast<int64_t>(row0 + qi) * p.q_stride + static_cast<int64_t>(h) * D + 8 * lq;
#pragma unroll
        for (int e = 0; e < KS; ++e) qf[hh][e] = load8(qp + 32 * e);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[hh][ct] = float4_t{0.f, 0.f, 0.f, 0.f};
        mrun[hh] = kNegBig;
        lrun[hh] = 0.f;
        hr1[hh] = SIG && p.r1 ? p.r1[h] : 0.f;
        hr2[hh] = SIG && p.r2 ? p.r2[h] : 0.f;
        hpb[hh] = (SIG && p.pb ? p.pb[h] : 0.f) * kLog2e;
    }
    const bool capped = !SIG && p.softcap > 0.f;
    const float c_mul = capped ? 2.0f * kLog2e * p.scale / p.softcap : SIG ? p.scale * kLog2e : p.scale, cap2 = -2.0f * p.softcap;

    // operand addresses inside a block (elements). K: row li of score tile t is key 8 (li / 4) + 4 t + li % 4 of the stage's 32, dims
    // 8 lq ..; V: column li of a tile, keys 8 lq .. 8 lq + 7 of the stage's
    const T *kc = static_cast<const T *>(p.k_cache) + (static_cast<int64_t>(kv) * 16 + (8 * (li >> 2) & 15) + (li & 3)) * D + 8 * lq;
    const T *vc = static_cast<const T *>(p.v_cache) + (static_cast<int64_t>(kv) * DV + li) * 16 + 8 * (lq & 1);
    const int nstages = kb1 >= kb0 ? (kb1 - kb0) / 2 + 1 : 0;
    // (scalar loads: a vector load of the ids inside the walk would be waited for with all keys and values that are on their way)
    const auto *ids = (const __attribute__((address_space(4))) int32_t *)bt;
    int b0 = 0, b1 = 0;
    auto fetch_ids = [&](int st) {      // past the last page: that page again
        b0 = ids[min(kb0 + 2 * st, kb1)];
        b1 = ids[min(kb0 + 2 * st + 1, kb1)];
    };
    auto fetch_k = [&]() {
        const T *kp = kc + static_cast<int64_t>(li >> 3 ? b1 : b0) * p.block_stride;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < KS; ++e) kf[t][e] = load8(kp + 4 * t * D + 32 * e);
        v_next = vc + static_cast<int64_t>(lq >> 1 ? b1 : b0) * p.block_stride;
    };
    auto fetch_v = [&]() {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) vf[ct] = load8(v_now + ct * 256);
    };
    // scores of a stage: the products of this wave's heads, and what is done to them on their way to LDS
    float4_t sc[HPW][2];
    auto products = [&]() {     // (a wave without heads goes along: what it makes is not stored)
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
            sc[hh][0] = sc[hh][1] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < KS; ++e)
#pragma unroll
                for (int t = 0; t < 2; ++t) sc[hh][t] = mx_mfma(kf[t][e], qf[hh][e], sc[hh][t]);
        }
    };
    auto hand_in = [&](int st) {
        const int k0 = (kb0 + 2 * st) * 16, kd = qpos - k0 - 8 * lq, lo = qlo - k0 - 8 * lq;     // visible: lo <= key - (k0 + 8 lq) <= kd
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
            mfma_results_tie(sc[hh][0]);
            mfma_results_ready<8>(sc[hh][1]);
            if (hh < nh) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    float4_t s = sc[hh][t];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {       // key 8 lq + 4 t + r of the stage
                        float x = s[r];
                        if constexpr (SIG) {
                            const int at = 4 * t + r;
                            float z = fmaf(x, c_mul, hpb[hh]);
                            if (p.r1) z -= hr1[hh] * fast_log2(fmaf(hr2[hh], static_cast<float>(max(kd - at, 0)), 1.0f));
                            x = at <= kd && at >= lo && qok ? __builtin_amdgcn_rcpf(1.0f + fast_exp2(-z)) : 0.f;
                        } else if (capped) {
                            x = fmaf(cap2, __builtin_amdgcn_rcpf(fast_exp2(x * c_mul) + 1.0f), p.softcap);
                        } else {
                            x *= c_mul;
                        }
                        s[r] = x;
                    }
                    *reinterpret_cast<float4_t *>(s_in + (h0 + hh) * kMxIn + lane * 8 + 4 * t) = s;
                }
            }
        }
    };
    if (nstages > 0) {
        fetch_ids(0);
        fetch_k();
        v_now = v_next;
        products();
        fetch_ids(1);
        fetch_k();
        __builtin_amdgcn_sched_barrier(0);      // (the order of the walk: keys, then values)
        fetch_v();
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();        // (the zero rows)
    if (nstages > 0) hand_in(0);
    for (int st = 0; st < nstages; ++st) {
        const int k0 = (kb0 + 2 * st) * 16, kd = qpos - k0 - 8 * lq, lo = qlo - k0 - 8 * lq;     // visible: lo <= key - (k0 + 8 lq) <= kd
        __syncthreads();
        fetch_ids(st + 2);      // (past the last stage: its keys again. A load that only some paths make is waited for on all of them)
        // ---- 1. the mix: blocks 4 wave .. 4 wave + 3 of 16 pairs -------------------------------------------------------------------
        {
            float4_t m[4];
            float b[4][STEPS];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                m[u] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < STEPS; ++s) b[u][s] = s_in[(4 * s + lq) * kMxIn + (4 * wave + u) * 16 + li];
            }
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int u = 0; u < 4; ++u) m[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(mixw[s], b[u][s], m[u], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 3; ++u) mfma_results_tie(m[u]);
            mfma_results_ready<8>(m[3]);
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * STEPS, 0);     // (the LDS reads together, before the first matrix step)
            __builtin_amdgcn_sched_group_barrier(0x008, 4 * STEPS, 0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) s_out[(4 * lq + r) * kMxOut + (4 * wave + u) * 16 + li] = m[u][r];
        }
        __syncthreads();
        // ---- 2. score products of the next stage, which the matrix core works off beside the weights of this one -------------------
        const T *v_after = v_next;
        products();
        fetch_k();
        // ---- 3. weights and value products of this wave's heads ---------------------------------------------------------------------
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
            float x[8];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float4_t v = *reinterpret_cast<const float4_t *>(s_out + (h0 + hh) * kMxOut + lane * 8 + 4 * t);
#pragma unroll
                for (int r = 0; r < 4; ++r) x[4 * t + r] = v[r];
            }
            if constexpr (!SIG) {
                if (k0 + kMxKeys - 1 > p0 || (p.window > 0 && k0 < p0 + cnt - p.window)) {        // (uniform) the keys cross a query's limits
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (j > kd || j < lo) x[j] = kNegBig;
                }
                float mx = x[0];
#pragma unroll
                for (int j = 1; j < 8; ++j) mx = fmaxf(mx, x[j]);
                mx = mx_rows_max(mx);
                // lazy running maximum: a row moves its reference only when a stage raises it by more than kLazy
                const float mnew = mx - mrun[hh] > kLazy ? mx : mrun[hh];
                const float alpha = fast_exp2(mrun[hh] - mnew);
                mrun[hh] = mnew;
                const float mref = mnew < 0.5f * kNegBig ? 0.f : mnew;
                float psum = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    x[j] = fast_exp2(x[j] - mref);
                    psum += x[j];
                }
                lrun[hh] = fmaf(lrun[hh], alpha, psum);
                if (!__all(alpha == 1.0f)) {
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[hh][ct][r] *= alpha;
                }
            }
            vec8_t<T> phi, plo;
            split_weights<T>(x, phi, plo);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                acc[hh][ct] = mx_mfma(vf[ct], phi, acc[hh][ct]);
                acc[hh][ct] = mx_mfma(vf[ct], plo, acc[hh][ct]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        v_now = v_after;
        fetch_v();
        __builtin_amdgcn_sched_barrier(0);
        if (st + 1 < nstages) hand_in(st + 1);
    }
    // ---- epilogue: acc[hh][ct][r] = O[query li][head][ct * 16 + 4 lq + r] --------------------------------------------------------
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) mfma_results_tie(acc[hh][ct]);
    mfma_results_ready<8>(acc[HPW - 1][CT - 1]);
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        const int h = h0 + hh;
        if (hh < nh) {
            const int64_t orow = row0 + li;
            float l = lrun[hh];
            l += __shfl_xor(l, 16, 64);
            l += __shfl_xor(l, 32, 64);
            const int64_t slot = (static_cast<int64_t>(blockIdx.y) * p.num_tokens + orow) * H + h;
            const float inv = SIG ? 1.0f : 1.0f / l;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                if (!qok) continue;
                if (gridDim.y > 1) {
                    *reinterpret_cast<float4_t *>(p.part_o + slot * DV + ct * 16 + 4 * lq) = acc[hh][ct];
                    continue;
                }
                vec4_t<T> w;
#pragma unroll
                for (int r = 0; r < 4; ++r) w[r] = to_t<T>(acc[hh][ct][r] * inv);
                *reinterpret_cast<vec4_t<T> *>(static_cast<T *>(p.out) + (orow * H + h) * DV + ct * 16 + 4 * lq) = w;
            }
            if (!SIG && gridDim.y > 1 && qok && lq == 0) {
                p.part_ml[slot * 2] = mrun[hh];
                p.part_ml[slot * 2 + 1] = l;
            }
        }
    }
}

template <typename T, int D, int DV, bool SIG>
int launch_mix(const MixParams &p, int key_splits, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(p.num_tiles), static_cast<unsigned>(key_splits));
    if (p.H <= kMxWaves) hipLaunchKernelGGL((mix_attn_kernel<T, D, DV, 1, SIG>), grid, dim3(kMxThreads), 0, s, p);
    else hipLaunchKernelGGL((mix_attn_kernel<T, D, DV, 2, SIG>), grid, dim3(kMxThreads), 0, s, p);
    if (key_splits > 1) {
        const int64_t rows = p.num_tokens * p.H;
        if constexpr (SIG)
            hipLaunchKernelGGL((sigmoid_attn_sum_kernel<T>), dim3(static_cast<unsigned>((rows * DV / 4 + 255) / 256)), dim3(256), 0, s,
                               static_cast<T *>(p.out), p.part_o, rows * DV, key_splits);
        else
            launch_attn_combine<T>(static_cast<T *>(p.out), p.part_o, p.part_ml, rows, DV, key_splits, nullptr, p.H, 0, DV,
                                   static_cast<int64_t>(p.H) * DV, nullptr, 0, s);
    }
    return check_launch();
}

} // namespace swl

#define SWL_MIX_SHAPES(X) X(64, 64) X(64, 128) X(128, 64) X(128, 128)

/* 1 when swl_mix_attn / swl_mix_sigmoid_attn serve this shape: at most 16 heads, the heads of a wave (two from nine heads on) on one key head. */
extern "C" int swl_mix_attn_supported(int32_t num_q_heads, int32_t num_kv_heads, int32_t dim, int32_t vdim, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    if (num_q_heads <= 0 || num_q_heads > 16 || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return 0;
    if (num_q_heads > swl::kMxWaves && (num_q_heads / num_kv_heads) % 2) return 0;
#define SWL_MIX_IS(DD, DDV) if (dim == DD && vdim == DDV) return 1;
    SWL_MIX_SHAPES(SWL_MIX_IS)
#undef SWL_MIX_IS
    return 0;
}

static int mix_attn(bool sigmoid, void *out, const void *q, const void *k_cache, const void *v_cache, const int32_t *block_table,
                    const int32_t *tok_seq, const int32_t *tok_pos, const int32_t *tile_row0, const int32_t *tile_cnt,
                    const float *talk, const float *r1, const float *r2, const float *pb, int32_t num_tiles, int32_t num_q_heads,
                    int32_t num_kv_heads, int32_t dim, int32_t vdim, int64_t q_tok_stride, int32_t window, float scale, float softcap,
                    int32_t max_blocks_per_seq, int64_t block_stride, int32_t key_splits, float *scratch, int64_t num_tokens,
                    int32_t dtype, swl_stream_t stream) {
    if (num_tiles < 0 || window < 0 || key_splits < 1 || key_splits > 64 || (r1 == nullptr) != (r2 == nullptr)) return SWL_ERR_BAD_ARG;
    if (key_splits > 1 && (!scratch || num_tokens <= 0 || !swl::aligned16(scratch))) return SWL_ERR_BAD_ARG;
    if (!swl_mix_attn_supported(num_q_heads, num_kv_heads, dim, vdim, dtype)) return SWL_ERR_UNSUPPORTED;
    if (num_tiles == 0) return SWL_OK;
    if (!out || !q || !k_cache || !v_cache || !block_table || !tok_seq || !tok_pos || !tile_row0 || !tile_cnt || !talk) return SWL_ERR_BAD_ARG;
    // 16-byte operand loads
    if ((q_tok_stride & 7) || (block_stride & 7) || !swl::aligned16(q) || !swl::aligned16(k_cache) || !swl::aligned16(v_cache) ||
        (reinterpret_cast<uintptr_t>(out) & 7))
        return SWL_ERR_BAD_ARG;
    swl::MixParams p;
    p.out = out; p.q = q; p.k_cache = k_cache; p.v_cache = v_cache;
    p.block_table = block_table; p.tok_seq = tok_seq; p.tok_pos = tok_pos; p.tile_row0 = tile_row0; p.tile_cnt = tile_cnt;
    p.talk = talk; p.r1 = r1; p.r2 = r2; p.pb = pb;
    // scratch: [splits][tokens][H][vdim] fp32 partial outputs, then (softmax) [splits][tokens][H][2] (maximum, sum)
    p.part_o = scratch;
    p.part_ml = scratch ? scratch + static_cast<int64_t>(key_splits) * num_tokens * num_q_heads * vdim : nullptr;
    p.num_tiles = num_tiles; p.H = num_q_heads; p.G = num_kv_heads; p.window = window; p.max_blocks = max_blocks_per_seq;
    p.scale = scale; p.softcap = softcap;
    p.q_stride = q_tok_stride; p.block_stride = block_stride; p.num_tokens = num_tokens;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define SWL_MIX_GO(DD, DDV)                                                         \
    if (dim == DD && vdim == DDV)                                                   \
        return sigmoid ? swl::launch_mix<T, DD, DDV, true>(p, key_splits, s) : swl::launch_mix<T, DD, DDV, false>(p, key_splits, s);
    SWL_DISPATCH_DTYPE(dtype, T, { SWL_MIX_SHAPES(SWL_MIX_GO) });
#undef SWL_MIX_GO
    return SWL_ERR_UNSUPPORTED;
}

extern "C" int swl_mix_attn(void *out, const void *q, const void *k_cache, const void *v_cache, const int32_t *block_table,
                            const int32_t *tok_seq, const int32_t *tok_pos, const int32_t *tile_row0, const int32_t *tile_cnt,
                            const float *talk, int32_t num_tiles, int32_t num_q_heads, int32_t num_kv_heads, int32_t dim, int32_t vdim,
                            int64_t q_tok_stride, int32_t window, float scale, float softcap, int32_t max_blocks_per_seq,
                            int64_t block_stride, int32_t key_splits, float *scratch, int64_t num_tokens, int32_t dtype,
                            swl_stream_t stream) {
    return mix_attn(false, out, q, k_cache, v_cache, block_table, tok_seq, tok_pos, tile_row0, tile_cnt, talk, nullptr, nullptr, nullptr,
                    num_tiles, num_q_heads, num_kv_heads, dim, vdim, q_tok_stride, window, scale, softcap, max_blocks_per_seq, block_stride,
                    key_splits, scratch, num_tokens, dtype, stream);
}

extern "C" int swl_mix_sigmoid_attn(void *out, const void *q, const void *k_cache, const void *v_cache, const int32_t *block_table,
                                    const int32_t *tok_seq, const int32_t *tok_pos, const int32_t *tile_row0, const int32_t *tile_cnt,
                                    const float *talk, const float *r1, const float *r2, const float *pb, int32_t num_tiles,
                                    int32_t num_q_heads, int32_t num_kv_heads, int32_t dim, int32_t vdim, int64_t q_tok_stride,
                                    int32_t window, float scale, int32_t max_blocks_per_seq, int64_t block_stride, int32_t key_splits,
                                    float *scratch, int64_t num_tokens, int32_t dtype, swl_stream_t stream) {
    return mix_attn(true, out, q, k_cache, v_cache, block_table, tok_seq, tok_pos, tile_row0, tile_cnt, talk, r1, r2, pb, num_tiles,
                    num_q_heads, num_kv_heads, dim, vdim, q_tok_stride, window, scale, 0.f, max_blocks_per_seq, block_stride, key_splits,
                    scratch, num_tokens, dtype, stream);
}
