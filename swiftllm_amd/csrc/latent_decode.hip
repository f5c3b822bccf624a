// latent_decode.hip — latent attention of single tokens (a decode step): all query heads of a token attend to the ONE cached row of each earlier
// token, key (latent of rank R | rotated part) and value (latent), queries folded through the key up-projection before and results unfolded
// through the value up-projection after. Three launches:
//   swl_latent_fold     qa[t][h] = (W_uk,h^T q_th | rotated part), and the token's own cached row (the work of swl_latent_rope_store_kv)
//   swl_latent_decode   attention over shares of the keys, partial results
//   swl_latent_unfold   y[t][h] = sigmoid(gate) W_uv,h (sum of the shares)
// Made for one row, R = 512 and 64 rotated columns, whose fragments, LDS places and loads of a page are constants below: at any other a step takes the
// folded chain (two batched library products around the attention of window_attn_mfma.hip).
//
// What bounds it: 32 tokens at 1000 keys are 38 MB of cached rows, 6 to 8 us; every launch of a step costs about 4 us whatever it does.
// window_attn_mfma.hip reads the values' transposed copy beside the rows (71 MB) with one-wave workgroups, two a CU, and leaves 16 shares of 32 x 16
// x 512 fp32 results to a combining launch; two batched library products and a gate were launches of their own.
//
// The attention: a workgroup of four waves takes a token's share of pages, a wave every fourth, each on its own (no barrier in the walk): a page of
// 16 rows (18 KiB) is staged by LDS-DMA, two pages a wave in flight, 147 KB a CU. The rows serve as keys (S^T = C Q^T, 16x16x32) and, read back
// transposed (ds_read_b64_tr_b16), as values (O^T += C^T P^T, 16x16x16: the score registers are the B operand as they are, weights in two
// 16-bit terms). The waves' results meet in LDS at the end.
// Measured (bf16, 32 tokens at 1024 keys, 16 heads of 128, in a replayed step): attention 26 + 6.3 (shares combined) -> 15.8 us, value product and gate
// 9.2 + 4.7 -> 7.8, with rotary, store and folded queries 56 -> 30. What is left of the attention is a chain of loads (position, block ids, page),
// two pages of 1.2 us and the meeting of the waves.
#include "attn_combine.h"
#include "swl_common.h"

namespace swl {

constexpr int kLdRank = 512, kLdRot = 64, kLdRow = kLdRank + kLdRot;        // elements of a cached row
constexpr int kLdPage = 16 * kLdRow * 2, kLdUnits = kLdRow / 8;             // bytes of a page's rows; 16-byte units of a row
constexpr int kLdWaves = 4, kLdHeads = 16;

__device__ __forceinline__ float4_t ld_mfma(vec8_t<f16> a, vec8_t<f16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t ld_mfma(vec8_t<bf16> a, vec8_t<bf16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct LatentDecodeParams {
    const void *q, *k_cache;
    const int32_t *block_table, *tok_seq, *tok_pos;
    float *part_o, *part_ml;
    int n, H, window, max_blocks;
    float scale;
    int64_t q_stride, block_stride;
};

// LDS place of a row's unit: its low bits are exchanged by a function of the row that tells the 16 rows of a fragment read apart (rows are an odd
// multiple of 128 bytes apart)
__device__ __forceinline__ int ld_flip(int row) { return (row >> 1) & 7; }

// four rows' elements of column lane % 16 (gfx950 transpose read: 16 lanes hand in four rows of 16 columns, 8 bytes each)
template <typename T>
__device__ __forceinline__ vec4_t<T> ld_transposed(const char *p) {
    return __builtin_bit_cast(vec4_t<T>, __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3))) *)(p)));
}

__device__ __forceinline__ float ld_keys_max(float v) {     // over the four lanes of a head
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// grid: (tokens, shares, groups of 16 heads)
template <typename T>
__global__ __launch_bounds__(kLdWaves * 64, 1) void latent_decode_kernel(LatentDecodeParams p) {
    constexpr int KS = kLdRow / 32, CT = kLdRank / 16;      // steps of a score, value tiles
    constexpr float kLog2e = 1.4426950408889634f, kLazy = 8.0f;
    extern __shared__ __attribute__((aligned(16))) char smem[];     // [wave][2] pages; then the waves' results
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lk = lane >> 4, i16 = lane & 15;
    const int t = blockIdx.x, pos = __builtin_amdgcn_readfirstlane(p.tok_pos[t]);
    const int32_t *bt = p.block_table + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(p.tok_seq[t])) * p.max_blocks;
    const int first = p.window > 0 ? max(pos - p.window + 1, 0) : 0;
    const int shares = static_cast<int>(gridDim.y), all = pos / 16 - first / 16 + 1, per = (all + shares - 1) / shares;
    const int kb0 = first / 16 + per * static_cast<int>(blockIdx.y), kb1 = min(pos / 16, kb0 + per - 1);
    const int pages = kb1 >= kb0 + wave ? (kb1 - kb0 - wave) / kLdWaves + 1 : 0;       // of this wave: kb0 + wave + 4 i
    const int head = static_cast<int>(blockIdx.z) * kLdHeads + lr;

    vec8_t<T> qf[KS];
    {
        const T *qp = static_cast<const T *>(p.q) + t * p.q_stride + static_cast<int64_t>(min(head, p.H - 1)) * kLdRow + lk * 8;
#pragma unroll
        for (int e = 0; e < KS; ++e) qf[e] = load8(qp + e * 32);
    }
    // block ids: lane i holds that of this wave's page id_base + i, 64 a load
    int id_base = 0, id_lane = 0;
    auto fetch_ids = [&]() {
        id_lane = bt[min(kb0 + wave + kLdWaves * (id_base + lane), max(kb1, 0))];
        asm volatile("" : "+v"(id_lane));       // (waited for here)
    };
    if (pages > 0) fetch_ids();
#pragma unroll
    for (int e = 0; e < KS; ++e) asm volatile("" : "+v"(qf[e]));
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    unsigned src[18];
#pragma unroll
    for (int j = 0; j < 18; ++j) {
        const int unit = j * 64 + lane, row = unit / kLdUnits, c = unit - row * kLdUnits;
        src[j] = static_cast<unsigned>((row * kLdUnits + (c ^ ld_flip(row))) * 16);
    }
    auto ask = [&](int i) {     // page i of this wave
        const char *base = static_cast<const char *>(p.k_cache) + static_cast<int64_t>(__builtin_amdgcn_readlane(id_lane, i - id_base)) * p.block_stride * 2;
        const unsigned to = lds0 + static_cast<unsigned>((wave * 2 + (i & 1)) * kLdPage);
        const unsigned a[6] = {src[0], src[1], src[2], src[3], src[4], src[5]}, b[6] = {src[6], src[7], src[8], src[9], src[10], src[11]},
                       c[6] = {src[12], src[13], src[14], src[15], src[16], src[17]};
        lds_ask<6>(base, a, to);
        lds_ask<6>(base, b, to + 6 * 1024);
        lds_ask<6>(base, c, to + 12 * 1024);
    };
    // scores: row lr, unit 4 e + lk; values: rows 4 lk .. + 3, columns 16 ct + 4 (i16 % 4) of row 4 lk + i16 / 4
    unsigned k_frag[2], v_frag[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) k_frag[e] = static_cast<unsigned>((lr * kLdUnits + ((4 * e + lk) ^ ld_flip(lr))) * 16);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int row = 4 * lk + (i16 >> 2);
        v_frag[c] = static_cast<unsigned>((row * kLdUnits + ((2 * c + ((i16 & 3) >> 1)) ^ ld_flip(row))) * 16 + (i16 & 1) * 8);
    }
    float4_t acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
    float mrun = kNegBig, lrun = 0.f;
    // (a scale that leaves kNegBig no mask is applied first, as in span_attn.hip)
    const bool plain = p.scale > 1e-20f;
    const float unit = plain ? p.scale * kLog2e : kLog2e;

    if (pages > 0) ask(0);
    if (pages > 1) ask(1);
    for (int i = 0; i < pages; ++i) {
        // the page has landed; the one after it may be on its way
        if (i + 1 < pages) asm volatile("s_waitcnt vmcnt(18)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const char *page = smem + (wave * 2 + (i & 1)) * kLdPage;
        float4_t s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        lds_steps<8, KS, 1, vec8_t<T>>([&](int e) { return *reinterpret_cast<const vec8_t<T> *>(page + k_frag[e & 1] + (e >> 1) * 128); },
                                       [&](int e, vec8_t<T> kf) { s[e & 1] = ld_mfma(kf, qf[e], s[e & 1]); });
        mfma_results_tie(s[0]);
        mfma_results_ready<8>(s[1]);
        // score j of the lane: key 16 page + 4 lk + j, head lr
        const int key = (kb0 + wave + kLdWaves * i) * 16 + 4 * lk;
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[j] = s[0][j] + s[1][j];
            if (!plain) x[j] *= p.scale;
            if (key + j > pos || key + j < first) x[j] = kNegBig;
        }
        const float mx = ld_keys_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
        const float mnew = (mx - mrun) * unit > kLazy ? mx : mrun;
        const float alpha = fast_exp2((mrun - mnew) * unit);
        mrun = mnew;
        const float mref = mnew < 0.5f * kNegBig ? 0.f : -mnew * unit;
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[j] = fast_exp2(fmaf(x[j], unit, mref));
            psum += x[j];
        }
        lrun = fmaf(lrun, alpha, psum);
        if (i > 0 && !__all(alpha == 1.0f)) {       // (nothing to rescale at the first page)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[ct] *= alpha;
        }
        typedef unsigned uint2v __attribute__((ext_vector_type(2)));
        uint2v h, l;
        {
            unsigned a, b;
            split_pair<T>(x[0], x[1], a, b);
            h[0] = a, l[0] = b;
            split_pair<T>(x[2], x[3], a, b);
            h[1] = a, l[1] = b;
        }
        const vec4_t<T> hi = __builtin_bit_cast(vec4_t<T>, h), lo = __builtin_bit_cast(vec4_t<T>, l);
        lds_steps<16, CT, 2, vec4_t<T>>([&](int ct) { return ld_transposed<T>(page + v_frag[ct & 3] + (ct >> 2) * 128); },
                                        [&](int ct, vec4_t<T> vf) {
                                            acc[ct] = mfma16(vf, hi, acc[ct]);
                                            acc[ct] = mfma16(vf, lo, acc[ct]);
                                        });
        if (i + 2 < pages) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (its reads have returned before the page is overwritten)
            if (i + 2 - id_base >= 64) {
                id_base += 64;
                fetch_ids();
            }
            ask(i + 2);
        }
    }
#pragma unroll
    for (int ct = 0; ct + 1 < CT; ++ct) mfma_results_tie(acc[ct]);
    mfma_results_ready<8>(acc[CT - 1]);
    mrun *= unit;       // base-2 units from here on
    float l = lrun + __shfl_xor(lrun, 16, 64);
    l += __shfl_xor(l, 32, 64);
    // ---- the waves' results meet ------------------------------------------------------------------------------------------------------
    float *ml = reinterpret_cast<float *>(smem + kLdWaves * CT * 1024);     // [wave][16 heads][maximum, sum], behind the results
    __syncthreads();        // every wave is done with its pages
    if (lk == 0) {
        ml[(wave * 16 + lr) * 2] = mrun;
        ml[(wave * 16 + lr) * 2 + 1] = l;
    }
    __syncthreads();
    float big = kNegBig, sum = 0.f;
#pragma unroll
    for (int w = 0; w < kLdWaves; ++w) big = fmaxf(big, ml[(w * 16 + lr) * 2]);
#pragma unroll
    for (int w = 0; w < kLdWaves; ++w) sum += fast_exp2(ml[(w * 16 + lr) * 2] - big) * ml[(w * 16 + lr) * 2 + 1];
    const float a = fast_exp2(mrun - big);
    float4_t *mine = reinterpret_cast<float4_t *>(smem) + wave * CT * 64 + lane;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) mine[ct * 64] = acc[ct] * a;
    __syncthreads();
    if (head >= p.H) return;
    const int64_t slot = (static_cast<int64_t>(blockIdx.y) * p.n + t) * p.H + head;
    const float4_t *from = reinterpret_cast<const float4_t *>(smem) + lane;
#pragma unroll
    for (int c = 0; c < CT / kLdWaves; ++c) {
        const int ct = wave * (CT / kLdWaves) + c;
        float4_t o = from[ct * 64];
#pragma unroll
        for (int w = 1; w < kLdWaves; ++w) o += from[(w * CT + ct) * 64];
        *reinterpret_cast<float4_t *>(p.part_o + slot * kLdRank + ct * 16 + 4 * lk) = o;
    }
    if (wave == 0 && lk == 0) {
        p.part_ml[slot * 2] = big;
        p.part_ml[slot * 2 + 1] = sum;
    }
}

// ---- y[t][h][:] = sigmoid(gate[t][h]) W_uv,h (sum of the shares, rounded once) ------------------------------------------------------------
// A workgroup takes four tokens of a head: two waves add up one token's shares (the weights asked for before that are on their way meanwhile),
// then each of eight waves multiplies 16 rows of the matrix.
constexpr int kLuTokens = 4, kLuPitch = kLdRank + 8;

template <typename T>
__global__ __launch_bounds__(512, 2) void latent_unfold_kernel(T *y, const float *part_o, const float *part_ml, const T *uv, const float *sink, const T *gate,
                                                               int64_t gate_stride, int n, int H, int e_rows, int nsplit) {
    constexpr int KS = kLdRank / 32;
    constexpr float kLog2e = 1.4426950408889634f;
    __shared__ __attribute__((aligned(16))) T att[kLuTokens * kLuPitch];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lk = lane >> 4;
    const int h = blockIdx.x, t0 = blockIdx.y * kLuTokens;
    vec8_t<T> wf[KS];
    const T *wp = uv + (static_cast<int64_t>(h) * e_rows + min(wave * 16 + lr, e_rows - 1)) * kLdRank + lk * 8;
#pragma unroll
    for (int e = 0; e < KS; ++e) wf[e] = load8(wp + e * 32);
    {
        const int t = min(t0 + (wave >> 1), n - 1), c0 = (wave & 1) * (kLdRank / 2) + lane * 4;
        const int64_t rows = static_cast<int64_t>(n) * H, row = static_cast<int64_t>(t) * H + h;
        const bool live = lane < nsplit;
        const float m = live ? part_ml[(lane * rows + row) * 2] : kNegBig, l = live ? part_ml[(lane * rows + row) * 2 + 1] : 0.f;
        float big = wave_allreduce_max(m), extra = 0.f;
        if (sink) {
            const float sk = sink[h] * kLog2e;
            big = fmaxf(big, sk);
            extra = fast_exp2(sk - big);
        }
        const float w = live ? fast_exp2(m - big) : 0.f;
        const float inv = 1.0f / (wave_allreduce_sum(w * l) + extra);
        float4_t a = {0.f, 0.f, 0.f, 0.f};
        const float *po = part_o + row * kLdRank + c0;
        for (int s0 = 0; s0 < nsplit; s0 += 8) {        // (shares past the last: that one again, with no weight)
            float4_t v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = *reinterpret_cast<const float4_t *>(po + min(s0 + k, nsplit - 1) * rows * kLdRank);
#pragma unroll
            for (int k = 0; k < 8; ++k) a += v[k] * (s0 + k < nsplit ? __shfl(w, min(s0 + k, 63), 64) : 0.f);
        }
        vec4_t<T> o;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = to_t<T>(a[k] * inv);
        *reinterpret_cast<vec4_t<T> *>(att + (wave >> 1) * kLuPitch + c0) = o;
    }
    __syncthreads();
    const int t = t0 + lr % kLuTokens;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int row0 = 0;;) {
        if (row0 + wave * 16 < e_rows) {
#pragma unroll
            for (int e = 0; e < KS; ++e) acc = ld_mfma(wf[e], *reinterpret_cast<const vec8_t<T> *>(att + lr % kLuTokens * kLuPitch + e * 32 + lk * 8), acc);
            mfma_results_ready<8>(acc);
            const int c = row0 + wave * 16 + 4 * lk;
            if (lr < kLuTokens && t < n && c < e_rows) {
                float g = 1.0f;
                if (gate) g = 1.0f / (1.0f + expf(-to_f(gate[t * gate_stride + h])));
                vec4_t<T> v;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = to_t<T>(acc[k] * g);
                *reinterpret_cast<vec4_t<T> *>(y + (static_cast<int64_t>(t) * H + h) * e_rows + c) = v;
            }
        }
        row0 += 128;
        if (row0 >= e_rows) break;
        wp = uv + (static_cast<int64_t>(h) * e_rows + min(row0 + wave * 16 + lr, e_rows - 1)) * kLdRank + lk * 8;
#pragma unroll
        for (int e = 0; e < KS; ++e) wf[e] = load8(wp + e * 32);
        acc = float4_t{0.f, 0.f, 0.f, 0.f};
    }
}

} // namespace swl

/* 1 when swl_latent_decode and swl_latent_unfold serve these sizes (k_dim: elements of a cached row). */
extern "C" int swl_latent_decode_supported(int32_t kv_rank, int32_t rot_dim, int32_t k_dim, int32_t vdim, int32_t dtype) {
    if (dtype != SWL_F16 && dtype != SWL_BF16) return 0;
    return kv_rank == swl::kLdRank && rot_dim == swl::kLdRot && k_dim == swl::kLdRow && vdim > 0 && vdim % 16 == 0 && vdim <= 4096;
}

extern "C" int swl_latent_decode(float *scratch, const void *q, const void *k_cache, const int32_t *block_table, const int32_t *tok_seq,
                                 const int32_t *tok_pos, int64_t num_tokens, int32_t num_heads, int64_t q_stride, int32_t window, float scale,
                                 int32_t max_blocks_per_seq, int64_t block_stride, int32_t shares, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_heads <= 0 || window < 0 || shares < 1 || shares > 64 || max_blocks_per_seq <= 0) return SWL_ERR_BAD_ARG;
    if (dtype != SWL_F16 && dtype != SWL_BF16) return SWL_ERR_UNSUPPORTED;
    if (num_tokens == 0) return SWL_OK;
    if (!scratch || !q || !k_cache || !block_table || !tok_seq || !tok_pos) return SWL_ERR_BAD_ARG;
    if (!swl::aligned16(scratch) || !swl::aligned16(q) || !swl::aligned16(k_cache) || (q_stride & 7) || (block_stride & 7)) return SWL_ERR_BAD_ARG;
    if (q_stride < static_cast<int64_t>(num_heads) * swl::kLdRow) return SWL_ERR_BAD_ARG;
    if (num_tokens > 0x7fffffffLL || num_heads > 16 * 65535) return SWL_ERR_UNSUPPORTED;
    swl::LatentDecodeParams p;
    p.q = q; p.k_cache = k_cache; p.block_table = block_table; p.tok_seq = tok_seq; p.tok_pos = tok_pos;
    // scratch: [shares][tokens][heads][rank] fp32 partial results, then [shares][tokens][heads][2] (maximum, sum)
    p.part_o = scratch;
    p.part_ml = scratch + static_cast<int64_t>(shares) * num_tokens * num_heads * swl::kLdRank;
    p.n = static_cast<int>(num_tokens); p.H = num_heads; p.window = window; p.max_blocks = max_blocks_per_seq;
    p.scale = scale; p.q_stride = q_stride; p.block_stride = block_stride;
    const dim3 grid(static_cast<unsigned>(num_tokens), static_cast<unsigned>(shares), static_cast<unsigned>((num_heads + swl::kLdHeads - 1) / swl::kLdHeads));
    constexpr int lds = swl::kLdWaves * 2 * swl::kLdPage;
    static_assert(lds >= swl::kLdWaves * (swl::kLdRank / 16) * 1024 + swl::kLdWaves * 16 * 8, "");
    SWL_DISPATCH_DTYPE(dtype, T, {
        if (hipFuncSetAttribute(reinterpret_cast<const void *>(&swl::latent_decode_kernel<T>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
            return SWL_ERR_LAUNCH;
        hipLaunchKernelGGL((swl::latent_decode_kernel<T>), grid, dim3(swl::kLdWaves * 64), lds, static_cast<hipStream_t>(stream), p);
    });
    return swl::check_launch();
}

extern "C" int swl_latent_unfold(void *y, const float *scratch, const void *uv, const float *sink, const void *gate, int64_t gate_stride, int64_t num_tokens,
                                 int32_t num_heads, int32_t vdim, int32_t shares, int32_t dtype, swl_stream_t stream) {
    if (num_tokens < 0 || num_heads <= 0 || vdim <= 0 || vdim % 16 || vdim > 4096 || shares < 1 || shares > 64) return SWL_ERR_BAD_ARG;
    if (dtype != SWL_F16 && dtype != SWL_BF16) return SWL_ERR_UNSUPPORTED;
    if (num_tokens == 0) return SWL_OK;
    if (!y || !scratch || !uv || (gate && gate_stride < num_heads)) return SWL_ERR_BAD_ARG;
    if (!swl::aligned16(scratch) || !swl::aligned16(uv) || (reinterpret_cast<uintptr_t>(y) & 7)) return SWL_ERR_BAD_ARG;
    const int64_t groups = (num_tokens + swl::kLuTokens - 1) / swl::kLuTokens;
    if (groups > 65535) return SWL_ERR_UNSUPPORTED;
    const float *ml = scratch + static_cast<int64_t>(shares) * num_tokens * num_heads * swl::kLdRank;
    SWL_DISPATCH_DTYPE(dtype, T, {
        hipLaunchKernelGGL((swl::latent_unfold_kernel<T>), dim3(static_cast<unsigned>(num_heads), static_cast<unsigned>(groups)), dim3(512), 0,
                           static_cast<hipStream_t>(stream), static_cast<T *>(y), scratch, ml, static_cast<const T *>(uv), sink, static_cast<const T *>(gate),
                           gate_stride, static_cast<int>(num_tokens), num_heads, vdim, shares);
    });
    return swl::check_launch();
}
