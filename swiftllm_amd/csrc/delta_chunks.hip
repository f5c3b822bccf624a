// delta_chunks.hip — the gated delta rule (delta_rule.hip) over a step's prompt portions, sixteen tokens at a time, on the fp32 matrix core.
//
// Inside a run of 16 tokens (a tile of the step) that starts from the state S, with b_i = g_0 .. g_i and r_ij = g_(j+1) .. g_i,
//     u_i = beta_i (v_i - b_i S^T k_i - sum_(j<i) r_ij (k_i . k_j) u_j),   o_i = b_i S^T q_i + sum_(j<=i) r_ij (q_i . k_j) u_j,
//     S  <- b_15 S + sum_j r_(15)j k_j u_j^T
// so with L_ij = beta_i r_ij (k_i . k_j) (j < i), T = (I + L)^-1:  U = T diag(beta) V - T diag(beta b) K S.
// Everything but the products with S is known before the walk:
//   delta_chunk_kernel: one wave per (tile, head): K K^T and Q K^T, T by forward substitution (a column a lane), then
//                       W = -T diag(beta b) K, U0 = T diag(beta) V, A_ij = r_ij (q_i . k_j), b and r_(15)j. The r are products of the
//                       decays (never quotients: a decay may be 0). Tokens past the tile's end have beta = 0 and g = 1.
//   delta_walk_kernel:  one workgroup per (portion, head, 16 columns of S), eight waves. Four keep dim / 4 rows of S each and carry the
//                       chain: per tile U = U0 + W S (summed over the waves through LDS, one barrier a tile), S = b_15 S + (K^T diag(r)) U;
//                       they leave S and U in LDS, from where the other four form O = diag(b) Q S + A U while the chain goes on.
//                       The operands of the next three tiles are in registers, read as whole 1 KiB blocks. A lane's four accumulator
//                       rows 4 g .. 4 g + 3 are the k indices that it feeds to the next product (step s takes row 4 g + s), so nothing
//                       is transposed between products.
// What bounds the walk: the chain of tiles (two products of 16 x 16 x dim on four SIMDs and an exchange through LDS a tile: about 1400
// cycles, 512 of them matrix core). Splitting off the outputs and reading blocks took a tile from 3100 to 2100 cycles.
// The column shares of a (portion, head) pair read the same operands: consecutive numbers on one XCD.
// Measured against the walk token by token (8 heads of 128 x 128): 4 prompts of 2048 tokens 756 -> 159 us (both launches, back to back), 2 of 1000
// beside 30 decoded tokens 921 -> 94 us. Error of o against 64 bits: 1 to 2e-7 of the largest value (0.6 to 1.3e-7 token by token); of
// a model's logits in fp32: 0.98e-6 against 1.0e-6.
// A NaN or an infinity of a token reaches the outputs of its whole tile, the tokens before it included (a zero of a triangular factor times
// it), as it does in linear_scan.hip; token by token it reaches the later ones only. Other sequences never see it.
#include "swl_common.h"

namespace swl {

constexpr int kDcPitch = 20;        // floats a row of the 16 x 16 transposes

__device__ __forceinline__ float4_t dc_mfma(float a, float b, float4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// scratch of one (tile, head), in whole blocks of the order in which the walk's lanes read them:
//   W [D / 16][16 tokens][16 dims] | K^T diag(r) [D / 16][16 dims][16 tokens] | U0 [dv / 16][token % 4][token / 4][16 columns] |
//   A [key % 4][key / 4][query] | b [16] | b_15 [16] (once a lane: a scalar load would be waited for together with the exchange through LDS)
__host__ __device__ inline int64_t dc_floats(int D, int dv) { return 16LL * (2 * D + dv) + 256 + 32; }

template <int D>
__global__ __launch_bounds__(64, 3) void delta_chunk_kernel(float *scratch, const float *qn, const float *kn, const float *vv,
                                                            const float *beta, const float *decay, const int32_t *tile_row0,
                                                            const int32_t *tile_cnt, int H, int G, int dv) {
    constexpr int ND = D / 16;
    __shared__ __attribute__((aligned(16))) float lds[16 * kDcPitch];
    const int tile = blockIdx.x, h = blockIdx.y, kvh = h / (H / G);
    const int lane = threadIdx.x, li = lane & 15, g = lane >> 4;
    const int row0 = __builtin_amdgcn_readfirstlane(tile_row0[tile]), cnt = __builtin_amdgcn_readfirstlane(tile_cnt[tile]);
    const int64_t qk = static_cast<int64_t>(G) * D, hv = static_cast<int64_t>(H) * dv;
    const float *kt = kn + row0 * qk + static_cast<int64_t>(kvh) * D, *qt = qn + row0 * qk + static_cast<int64_t>(kvh) * D;
    const float *vt = vv + row0 * hv + static_cast<int64_t>(h) * dv;
    const int mine = min(li, cnt - 1);
    // K K^T and Q K^T: lane (li, g) feeds dims 16 S + 4 g + s of row li at step (S, s)
    // (four partial sums each: short sums round less)
    float4_t m, p;
    {
        float4_t ms[4], ps[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) ms[s] = ps[s] = float4_t{0.f, 0.f, 0.f, 0.f};
        float4_t kf[ND], qf[ND];
#pragma unroll
        for (int e = 0; e < ND; ++e) {
            kf[e] = *reinterpret_cast<const float4_t *>(kt + mine * qk + 16 * e + 4 * g);
            qf[e] = *reinterpret_cast<const float4_t *>(qt + mine * qk + 16 * e + 4 * g);
        }
#pragma unroll
        for (int e = 0; e < ND; ++e)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                ms[s] = dc_mfma(kf[e][s], kf[e][s], ms[s]);
                ps[s] = dc_mfma(qf[e][s], kf[e][s], ps[s]);
            }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            mfma_results_tie(ms[s]);
            mfma_results_tie(ps[s]);
        }
        mfma_results_ready<8>(ps[3]);
        m = (ms[0] + ms[1]) + (ms[2] + ms[3]);
        p = (ps[0] + ps[1]) + (ps[2] + ps[3]);
    }
    const int64_t at = static_cast<int64_t>(row0 + mine) * H + h;
    const float gl = li < cnt ? decay[at] : 1.0f, bl = li < cnt ? beta[at] : 0.0f;
    // lane's column j = li: r_ij down the rows, b_j
    float r = 1.0f, b = 1.0f, rr[4];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float gi = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(gl), i));
        if (i > li) r *= gi;
        else b *= gi;
        if ((i >> 2) == g) rr[i & 3] = r;
    }
    float sw[4], su[4], sr[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        su[s] = __shfl(bl, 4 * g + s, 64);
        sw[s] = -su[s] * __shfl(b, 4 * g + s, 64);
        sr[s] = __shfl(r, 4 * g + s, 64);
    }
    float *out = scratch + (static_cast<int64_t>(tile) * H + h) * dc_floats(D, dv);
    float *w_out = out, *k_out = w_out + 16 * D, *u_out = k_out + 16 * D, *a_out = u_out + 16 * dv, *b_out = a_out + 256;
    float4_t lcol, acol;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = 4 * g + e;
        lcol[e] = li < i ? su[e] * rr[e] * m[e] : 0.f;
        acol[e] = li <= i ? rr[e] * p[e] : 0.f;
    }
    *reinterpret_cast<float4_t *>(a_out + (li & 3) * 64 + (li >> 2) * 16 + 4 * g) = acol;
    if (g == 0) {
        b_out[li] = b;
        b_out[16 + li] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(b), 15));
    }
    *reinterpret_cast<float4_t *>(lds + li * kDcPitch + 4 * g) = lcol;      // column li of L
    __syncthreads();
    // column li of T: x[i] is final once columns 0 .. i - 1 have been taken off
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = i == li ? 1.0f : 0.0f;
#pragma unroll
    for (int i = 0; i < 15; ++i) {
#pragma unroll
        for (int k4 = i / 4; k4 < 4; ++k4) {
            const float4_t c = *reinterpret_cast<const float4_t *>(lds + i * kDcPitch + 4 * k4);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * k4 + e > i) x[4 * k4 + e] = fmaf(-c[e], x[i], x[4 * k4 + e]);
        }
    }
    __syncthreads();
    if (g == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) lds[i * kDcPitch + li] = x[i];
    }
    __syncthreads();
    const float4_t tf = *reinterpret_cast<const float4_t *>(lds + li * kDcPitch + 4 * g);      // T[li][4 g + s]
    int rows[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) rows[s] = min(4 * g + s, cnt - 1);
    // T times the scaled rows, four column blocks at a time: their loads are in flight together
    auto product = [&](const float *src, int stride, const float *scale, int cols, auto &&write) {
        for (int c0 = 0; c0 < cols; c0 += 64) {
            float in[4][4];
            float4_t d[4];
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int s = 0; s < 4; ++s) in[n][s] = src[rows[s] * stride + min(c0 + 16 * n, cols - 16) + li];
#pragma unroll
            for (int n = 0; n < 4; ++n) d[n] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int n = 0; n < 4; ++n) d[n] = dc_mfma(tf[s], in[n][s] * scale[s], d[n]);
#pragma unroll
            for (int n = 0; n < 3; ++n) mfma_results_tie(d[n]);
            mfma_results_ready<8>(d[3]);
#pragma unroll
            for (int n = 0; n < 4; ++n)
                if (c0 + 16 * n < cols) write((c0 + 16 * n) * 16, in[n], d[n]);       // (uniform)
        }
    };
    product(kt, static_cast<int>(qk), sw, D, [&](int block, const float *in, const float4_t &d) {
        *reinterpret_cast<float4_t *>(k_out + block + li * 16 + 4 * g) = float4_t{in[0] * sr[0], in[1] * sr[1], in[2] * sr[2], in[3] * sr[3]};
#pragma unroll
        for (int e = 0; e < 4; ++e) w_out[block + (4 * g + e) * 16 + li] = d[e];
    });
    product(vt, static_cast<int>(hv), su, dv, [&](int block, const float *, const float4_t &d) {
#pragma unroll
        for (int e = 0; e < 4; ++e) u_out[block + e * 64 + lane] = d[e];
    });
}

// A load from a wave-uniform base and a lane's byte offset.
__device__ __forceinline__ float dc_load(const float *base, uint32_t off) {
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + off);
}
__device__ __forceinline__ float4_t dc_load4(const float *base, uint32_t off) {
    return *reinterpret_cast<const float4_t *>(reinterpret_cast<const char *>(base) + off);
}

template <int D>
__global__ __launch_bounds__(512, 4) void delta_walk_kernel(float *o, const float *scratch, const float *qn, float *state,
                                                            int64_t slot_stride, int64_t s_off, const int32_t *seq_row0,
                                                            const int32_t *seq_cnt, const int32_t *seq_tile0, const int32_t *tok_pos,
                                                            const int32_t *tok_state, int pairs, int H, int G, int dv) {
    constexpr int NT = D / 64, DEPTH = 3;
    __shared__ __attribute__((aligned(16))) float4_t s_u[2][4][64], s_o[2][4][64], s_st[2][4][NT][64];
    const int groups = dv / 16, xcd = blockIdx.x & 7, nth = blockIdx.x >> 3;
    const int pair = nth / groups * 8 + xcd, col0 = nth % groups * 16;
    if (pair >= pairs) return;      // (the whole workgroup)
    const int seq = pair / H, h = pair % H, kvh = h / (H / G);
    const int lane = threadIdx.x & 63, role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), li = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const int row0 = __builtin_amdgcn_readfirstlane(seq_row0[seq]), cnt = __builtin_amdgcn_readfirstlane(seq_cnt[seq]);
    const int tile0 = __builtin_amdgcn_readfirstlane(seq_tile0[seq]), ntiles = (cnt + 15) / 16, base = wave * 16 * NT;
    const uint32_t qk = static_cast<uint32_t>(G * D);
    const int64_t hv = static_cast<int64_t>(H) * dv, per = dc_floats(D, dv), pre_step = per * H;
    const float *pre = scratch + (static_cast<int64_t>(tile0) * H + h) * per;       // the tile that the next fetch reads
    const float *rows = qn + static_cast<int64_t>(row0) * qk + static_cast<int64_t>(kvh) * D;
    int next = 0;
    auto advance = [&]() {      // (past the last tile: read again, never used)
        const bool more = ++next < ntiles;
        pre += more ? pre_step : 0;
        rows += more ? 16 * qk : 0;
    };
    if (role == 0) {
        // ---- the chain: U and the state, four waves of D / 4 rows -----------------------------------------------------------------
        float *S = state + static_cast<int64_t>(tok_state[row0] >> 1) * slot_stride + s_off + static_cast<int64_t>(h) * D * dv + col0 + li;
        const bool fresh = tok_pos[row0] == 0;      // a sequence starts from the zero state whatever the slot held
        float4_t st[NT];        // S[base + 16 t + 4 g + e][col0 + li]
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) st[t][e] = fresh ? 0.f : S[static_cast<int64_t>(base + 16 * t + 4 * g + e) * dv];
        struct Ops {
            float4_t w[NT], k[NT];
            float u0, total;
        };
        const uint32_t w_off = 4 * (wave * NT * 256 + li * 16 + 4 * g), k_off = w_off + 64 * D;
        const uint32_t u_off = 4 * (32 * D + col0 * 16 + wave * 64 + lane), t_off = 4 * (32 * D + 16 * dv + 256 + 16 + li);
        auto fetch = [&](Ops &f) {
#pragma unroll
            for (int t = 0; t < NT; ++t) f.w[t] = dc_load4(pre, w_off + 1024 * t);
            f.u0 = dc_load(pre, u_off);
#pragma unroll
            for (int t = 0; t < NT; ++t) f.k[t] = dc_load4(pre, k_off + 1024 * t);
            f.total = dc_load(pre, t_off);
            advance();
        };
        // sums stay short (a partial sum per 16 rows of S, S + delta once a tile): they round about as little as a walk token by token
        auto step = [&](const Ops &f, int c) {
            const float4_t zero = {0.f, 0.f, 0.f, 0.f};
            float4_t ut[NT], dt[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                s_st[c & 1][wave][t][lane] = st[t];
                ut[t] = dt[t] = zero;
            }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < NT; ++t) ut[t] = dc_mfma(f.w[t][s], st[t][s], ut[t]);
#pragma unroll
            for (int t = 0; t < NT - 1; ++t) mfma_results_tie(ut[t]);
            mfma_results_ready<8>(ut[NT - 1]);
            float4_t u = ut[0];
#pragma unroll
            for (int t = 1; t < NT; ++t) u += ut[t];
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] += e == wave ? f.u0 : 0.f;      // (each wave brings one row of U0)
            s_u[c & 1][wave][lane] = u;
            __syncthreads();
            float4_t us[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) us[w] = s_u[c & 1][w][lane];
            u = (us[0] + us[1]) + (us[2] + us[3]);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < NT; ++t) dt[t] = dc_mfma(f.k[t][s], u[s], dt[t]);
#pragma unroll
            for (int t = 0; t < NT - 1; ++t) mfma_results_tie(dt[t]);
            mfma_results_ready<8>(dt[NT - 1]);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) st[t][e] = fmaf(st[t][e], f.total, dt[t][e]);
        };
        Ops ops[DEPTH];
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) fetch(ops[i]);
        for (int c = 0; c < ntiles; c += DEPTH) {
#pragma unroll
            for (int i = 0; i < DEPTH; ++i) {
                if (c + i < ntiles) {       // (uniform)
                    step(ops[i], c + i);
                    fetch(ops[i]);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) S[static_cast<int64_t>(base + 16 * t + 4 * g + e) * dv] = st[t][e];
        return;
    }
    // ---- the outputs, one barrier behind: diag(b) Q S over D / 4 rows of S, and step `wave` of A U ----------------------------------
    struct Ops {
        float4_t q[NT];
        float a, b;
    };
    const uint32_t a_off = 4 * (32 * D + 16 * dv + wave * 64 + lane), b_off = 4 * (32 * D + 16 * dv + 256 + 4 * g + (li & 3));
    uint32_t q_off = 4 * (li * qk + base + 4 * g);
    auto fetch = [&](Ops &f) {
        if (next == ntiles - 1) q_off = 4 * (min(li, (cnt - 1) & 15) * qk + base + 4 * g);
#pragma unroll
        for (int t = 0; t < NT; ++t) f.q[t] = dc_load4(rows, q_off + 64 * t);
        f.b = dc_load(pre, b_off);
        f.a = dc_load(pre, a_off);
        advance();
    };
    // the waves' shares of a tile's O, one accumulator row a wave
    float *orow = o + static_cast<int64_t>(row0 + 4 * g + wave) * hv + static_cast<int64_t>(h) * dv + col0 + li;
    const float *share = reinterpret_cast<const float *>(&s_o[0][0][lane]) + wave;
    auto put = [&](int c) {
        float v[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) v[w] = share[((c & 1) * 4 + w) * 256];
        if (16 * c + 4 * g + wave < cnt) orow[static_cast<int64_t>(16 * c) * hv] = (v[0] + v[1]) + (v[2] + v[3]);
    };
    auto step = [&](const Ops &f, int c) {
        const float4_t zero = {0.f, 0.f, 0.f, 0.f};
        __syncthreads();        // the tile's S and U's shares, and the previous tile's shares of O
        float4_t st[NT], ot[NT];
        float us[4];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            st[t] = s_st[c & 1][wave][t][lane];
            ot[t] = zero;
        }
        const float *up = reinterpret_cast<const float *>(&s_u[c & 1][0][lane]) + wave;
#pragma unroll
        for (int w = 0; w < 4; ++w) us[w] = up[w * 256];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int t = 0; t < NT; ++t) ot[t] = dc_mfma(f.q[t][s], st[t][s], ot[t]);
        float4_t own = dc_mfma(f.a, (us[0] + us[1]) + (us[2] + us[3]), zero);
        if (c > 0) put(c - 1);
#pragma unroll
        for (int t = 0; t < NT; ++t) mfma_results_tie(ot[t]);
        mfma_results_ready<8>(own);
#pragma unroll
        for (int t = 1; t < NT; ++t) ot[0] += ot[t];
        const float4_t b = quad_values(f.b);
#pragma unroll
        for (int e = 0; e < 4; ++e) own[e] = fmaf(ot[0][e], b[e], own[e]);
        s_o[c & 1][wave][lane] = own;
    };
    Ops ops[DEPTH];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) fetch(ops[i]);
    for (int c = 0; c < ntiles; c += DEPTH) {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) {
            if (c + i < ntiles) {       // (uniform)
                step(ops[i], c + i);
                fetch(ops[i]);
            }
        }
    }
    __syncthreads();
    put(ntiles - 1);
}

} // namespace swl

/* 1 when swl_delta_rule_tiles serves heads of dim x vdim. */
extern "C" int swl_delta_rule_tiles_supported(int32_t num_heads, int32_t num_qk_heads, int32_t dim, int32_t vdim) {
    return num_heads > 0 && num_heads <= 65535 && num_qk_heads > 0 && num_heads % num_qk_heads == 0 && (dim == 64 || dim == 128) && vdim > 0 &&
           vdim % 16 == 0 && vdim <= 1024;
}

extern "C" size_t swl_delta_rule_tiles_scratch_bytes(int64_t num_tiles, int32_t num_heads, int32_t dim, int32_t vdim) {
    return sizeof(float) * static_cast<size_t>(num_tiles * num_heads * swl::dc_floats(dim, vdim));
}

extern "C" int swl_delta_rule_tiles(float *o, const float *qn, const float *kn, const float *vv, const float *beta, const float *decay,
                                    float *state, int64_t slot_stride, int64_t s_off, const int32_t *seq_row0, const int32_t *seq_cnt,
                                    const int32_t *seq_tile0, const int32_t *tile_row0, const int32_t *tile_cnt, const int32_t *tok_pos,
                                    const int32_t *tok_state, int32_t num_seqs, int32_t num_tiles, int32_t num_heads,
                                    int32_t num_qk_heads, int32_t dim, int32_t vdim, float *scratch, swl_stream_t stream) {
    if (num_seqs < 0 || num_tiles < num_seqs) return SWL_ERR_BAD_ARG;
    if (!swl_delta_rule_tiles_supported(num_heads, num_qk_heads, dim, vdim)) return SWL_ERR_UNSUPPORTED;
    if (num_seqs == 0) return SWL_OK;
    if (!o || !qn || !kn || !vv || !beta || !decay || !state || !seq_row0 || !seq_cnt || !seq_tile0 || !tile_row0 || !tile_cnt || !tok_pos ||
        !tok_state || !scratch)
        return SWL_ERR_BAD_ARG;
    if (!swl::aligned16(qn) || !swl::aligned16(kn) || !swl::aligned16(scratch)) return SWL_ERR_BAD_ARG;
    const int64_t pairs = static_cast<int64_t>(num_seqs) * num_heads, blocks = (pairs + 7) / 8 * 8 * (vdim / 16);
    if (blocks > 0x7fffffffLL) return SWL_ERR_UNSUPPORTED;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 tiles(static_cast<unsigned>(num_tiles), static_cast<unsigned>(num_heads)), grid(static_cast<unsigned>(blocks));
#define SWL_DC_GO(DD)                                                                                                                       \
    hipLaunchKernelGGL((swl::delta_chunk_kernel<DD>), tiles, dim3(64), 0, s, scratch, qn, kn, vv, beta, decay, tile_row0, tile_cnt,          \
                       num_heads, num_qk_heads, vdim);                                                                                      \
    hipLaunchKernelGGL((swl::delta_walk_kernel<DD>), grid, dim3(512), 0, s, o, scratch, qn, state, slot_stride, s_off, seq_row0, seq_cnt, \
                       seq_tile0, tok_pos, tok_state, static_cast<int>(pairs), num_heads, num_qk_heads, vdim)
    if (dim == 64) {
        SWL_DC_GO(64);
    } else {
        SWL_DC_GO(128);
    }
#undef SWL_DC_GO
    return swl::check_launch();
}
