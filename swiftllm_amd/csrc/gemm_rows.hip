// gemm_rows.hip — the hidden-wide projections of a decode layer with K split INSIDE the workgroup and the residual add in
// the epilogue (gfx950, M <= 32 tokens, packed W).
//
// Replaces, for decode batches of <= 32 (o_proj) / <= 8 (down_proj) tokens in bfloat16, the pair
//     projection (reference swiftllm/worker/kernels/linear.py:3-12 at layers/transformer_layer.py:117 / :128)
//   + the residual-add half of fused_add_rmsnorm (kernels/rmsnorm.py:54-57 at transformer_layer.py:120 / the next layer's :46)
// which r01-r04 ran as a split-K GEMM (8 fp32 slabs, gemm_skinny.hip) followed by a consumer launch that does nothing
// but wait on memory: 9.6 + 5.0 us (o) per layer in the batch-32 trace (profiles/r04d_kernel_trace_configs2.md) for 33.6 MB
// of weights = 4.7 us of HBM time. The norm weight and the 1/rms are left to the projection that follows, which applies
// them while it stages the raw residual rows ("norm on the fly": gemm_skinny.hip, NF).
//
// Why a second in-workgroup scheme after r02's gemm_wgk (128 workgroups of 32 rows: 11.2 us, retired). What bounds such a
// kernel on this part is what ONE CU can pull through its L1: ~57 GB/s, L2 hit or HBM miss (DESIGN.md sections 4.6, 4.8). A
// workgroup that owns rows of W for all of K reads all of x[M, K]: bytes per CU = rows * K * e + M * K * e. With 32-row tiles
// only 128 CUs work and each moves 256 + 256 KiB (9.3 us); with SIXTEEN-row tiles all 256 CUs work and each moves
// 128 + 256 KiB (7 us) — and the op is one v_mfma_f32_16x16x32 per 1 KiB of W, so the tile height costs nothing:
//   * workgroup = 16 rows of W x all of K = 8 waves (2 per SIMD), wave w takes K/8 contiguous columns;
//   * W comes from the SAME packed copy the other decode kernels stream (swl_gemm_pack_weight: 32-row x 16-k fragments
//     of 1 KiB): the 16 x 32 A fragment of tile half h is lanes {16h..16h+15} and {32+16h..} of two consecutive
//     fragments — four 256-byte runs per wave-load, non-temporal; the sibling workgroup reads the other halves;
//   * x^T is the B operand, loaded straight into fragment layout (lane -> token l%16, 8 k): 64-byte runs of 16 rows,
//     L2-resident (every workgroup reads the same rows); rows >= M are clamped to row M-1 (L1 hits, never stored);
//   * EVERYTHING a wave needs is requested before its first MFMA: K = 4096 is 16 k-steps = 16 + 32 loads of 16 B per
//     lane (192 VGPRs), the whole workgroup 384 KiB in flight — the kernel is one memory round trip plus a drain at
//     the CU's own rate; longer K (down_proj: 14 chunks) refills a 4-deep ring of 4-step chunks behind exact counted waits;
//   * the 8 waves' 16 x 32 fp32 tiles meet in LDS (20 KiB), are added in wave order (= K order: deterministic), and the
//     512 threads finish one (token, column) each: residual += round(acc), the consumer launch's rounding points.
// r06b — x through a wave-private LDS tile (XLDS = true: from 9 tokens on). The fragment-shaped x loads above are 16 rows x 64 B
// per instruction: sixteen HALF cache lines per KiB delivered, and at 32 tokens x is 2/3 of what a CU pulls through its L1
// (the r05 "57 GB/s per CU, hit or miss" was measured through exactly that pattern). Here a wave requests its x chunk
// (32 tokens x 128 k) as FULL lines — lane -> (token 4i + lane/16, 16-byte piece lane%16): 4 rows x 256 contiguous bytes per
// instruction, the same register budget (8 loads per chunk at two token blocks) — and turns it into B fragments through an
// 8 KiB LDS tile of its own: ds_write_b128 at piece ^ (token & 15), ds_read_b128 of lane (r, kq) at (4j + kq) ^ r —
// conflict-free for the 8-lane write groups and for the irregular 16-lane groups of the b128 read.
// One wave's LDS operations execute in order: no barrier in the stream. Same MFMAs in the same order: the same bits.
// Plain results (swl_gemm_rows_store, optionally through a squared ReLU) serve the narrower matrices of the stepped designs, any
// number of rows: what such a launch costs is its start, one round trip and the 16 rows' share of x, where shares of K paid a second
// launch and 8 to 16 slabs. us at 32 tokens, cold bf16 weights, against the split ring kernel with its reduce launch (the
// library for 3088 rows): 1024 x 1024 6.3 -> 3.8, 2048 x 2048 7.7 -> 5.5, 3088 x 2048 11.5 -> 6.0, 8192 x 2048 12.8 -> 10.4
// (3.2 TB/s; 7.6 at one token: x is two thirds of what a CU reads). Where its line lies: kernels/linear.py, _rows_serves.
// No slabs, no second launch, no atomics, no cross-workgroup hand-off. (r05 also built an epilogue that wrote
// round(residual * w_norm) and one sum-of-squares partial per tile, with a SiLU-gate GEMM that added the 256 partials from
// LDS-DMA'd copies: correct, +2 us on the up/gate kernel, removed — last revision that has it: ca4e9a9, numbers in
// profiles/r05a_gemm_rows_micro_o_proj_pair.jsonl.)
#include <type_traits>

#include "swl_common.h"

namespace swl {

__device__ __forceinline__ float4_t rows_mfma(vec8_t<f16> a, vec8_t<f16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t rows_mfma(vec8_t<bf16> a, vec8_t<bf16> b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

constexpr int kRowsWaves = 8;     // K splits = waves per workgroup
constexpr int kRowsTile = 16;     // rows of W per workgroup
constexpr int kRowsCh = 4;        // k-steps (of 32) per ring chunk
constexpr int kRowsRing = 4;      // chunks in flight per wave, at most: 16 k-steps = 192 VGPRs at two token blocks
constexpr int kRowsKUnit = 32 * kRowsWaves * kRowsCh;
constexpr int kRowsRedPitch = 20; // floats per token row of a wave's tile image in LDS (80 B: 16-byte stores spread)

// What a workgroup does with its finished 16 columns:
//   kRowsAdd    residual += round(product)
//   kRowsStore  out = round(product)
//   kRowsRelu2  out = round(relu(round(product))^2): swl_relu_sq behind the stored product
//   kRowsSlab   out = product, fp32: one slab for a consumer that adds slabs into an fp32 stream (nothing is rounded on the way)
constexpr int kRowsAdd = 0, kRowsStore = 1, kRowsRelu2 = 2, kRowsSlab = 3;

struct RowsArgs {
    const void *x;
    const void *wp;
    void *residual;         // kRowsAdd: rows of N; otherwise the output, rows out_stride apart
    int64_t out_stride;
    int M, N, K;
    int64_t x_stride;
    // optional (r06c): ssq_out[M][N / 16] = sum of squares of the NEW residual values of (token, 16-column tile) — what an
    // EXACT rmsnorm of the updated rows needs before the next projection can stage them (swl_gemm_skinny_packed_*_nx)
    float *ssq_out;
};

constexpr int rows_waves_per_simd(int nch, int epi) { return epi != kRowsAdd && nch > 0 && nch <= 2 ? 4 : 2; }

// NCH > 0: the chunk count per wave is a compile-time constant <= kRowsRing — every load is issued up front, straight-line
// code with exact counted waits. NCH == 0: run-time chunk count, the ring refilled behind guards.
// Stores (EPI != kRowsAdd) take any N: the packed copy of a weight whose rows are no multiple of 32 ends with rows of zeros, and
// columns from N on are not stored. With one or two chunks a wave needs half the registers, and two workgroups share a CU.
template <typename T, int NCH, int MB, bool XLDS, int EPI>
__global__ __launch_bounds__(kRowsWaves * 64, rows_waves_per_simd(NCH, EPI)) void gemm_rows_kernel(RowsArgs a) {
    constexpr int kRing = NCH > 0 && NCH < kRowsRing ? NCH : kRowsRing;
    constexpr int XCK = 32 * kRowsCh;          // k per chunk (128): one 256-byte run per token
    constexpr int NXL = XLDS ? 4 * MB : kRowsCh * MB;   // x loads per chunk and lane (XLDS: 4 token rows each)
    // a wave's x tile; its tile image takes the same place once the wave has multiplied (its LDS operations run in order)
    constexpr int kXBytes = XLDS ? 16 * MB * XCK * 2 : 0, kRedBytes = 16 * MB * kRowsRedPitch * 4;
    constexpr int kWaveBytes = kXBytes > kRedBytes ? kXBytes : kRedBytes;
    __shared__ __attribute__((aligned(16))) char wave_lds[kRowsWaves][kWaveBytes];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int M = a.M, N = a.N, K = a.K;
    const int tile16 = blockIdx.x;
    const int n0 = tile16 * kRowsTile;
    const auto red = [&](int w) { return reinterpret_cast<float *>(&wave_lds[w][0]); };

    // ---- epilogue operands first: the oldest requests of the wave, no wait of the stream ever includes them ----
    const int et = threadIdx.x >> 4, en = threadIdx.x & 15; // (token, column n0 + en)
    const bool e_ok = et < M && (EPI == kRowsAdd || n0 + en < N);
    using O = std::conditional_t<EPI == kRowsSlab, float, T>;
    O *res_p = static_cast<O *>(a.residual) + static_cast<int64_t>(e_ok ? et : 0) * (EPI == kRowsAdd ? N : a.out_stride) + n0 + en;
    T rv{};
    if constexpr (EPI == kRowsAdd) rv = *res_p;

    // ---- the stream ----
    const int r = lane & 15, kq = lane >> 4;
    const int nsteps = K / 32 / kRowsWaves; // k-steps of this wave
    const int s0 = wave * nsteps;
    const int nch = NCH > 0 ? NCH : nsteps / kRowsCh;
    // packed W: fragment (tile32, kstep16) = 512 elements, lane L of it = row L%32, k = 16*kstep16 + 8*(L/32) .. +8.
    // 16x32 A fragment of step s, lane (r, kq): row 16*half + r, k = 32*s + 8*kq -> kstep16 = 2s + kq/2, L = 16*half + r + 32*(kq%2)
    const T *wsrc = static_cast<const T *>(a.wp) +
                    (static_cast<int64_t>(tile16 >> 1) * (K / 16) + 2 * s0 + (kq >> 1)) * 512 +
                    (16 * (tile16 & 1) + r + 32 * (kq & 1)) * 8;
    // fragment form: xsrc[mb] = row r + 16 mb at k = 8 kq; XLDS: xsrc[i] = row 4 i + lane/16 at piece lane%16 of the chunk
    const T *xsrc[XLDS ? NXL : MB];
    int xw_off[XLDS ? NXL : 1];                  // XLDS: where this lane's piece of load i goes in the tile (elements)
    int xr_off[XLDS ? kRowsCh : 1];              // XLDS: B fragment of k-step j of the chunk, token block 0 (elements)
    if constexpr (XLDS) {
        const int tsub = lane >> 4, pc = lane & 15;
#pragma unroll
        for (int i = 0; i < NXL; ++i) {
            const int tk = 4 * i + tsub;
            xsrc[i] = static_cast<const T *>(a.x) + static_cast<int64_t>(min(tk, M - 1)) * a.x_stride + 32 * s0 + 8 * pc;
            xw_off[i] = tk * XCK + ((pc ^ (tk & 15)) << 3);
        }
#pragma unroll
        for (int j = 0; j < kRowsCh; ++j) xr_off[j] = r * XCK + (((4 * j + kq) ^ r) << 3);
    } else {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
            xsrc[mb] = static_cast<const T *>(a.x) + static_cast<int64_t>(min(r + 16 * mb, M - 1)) * a.x_stride + 32 * s0 + 8 * kq;
    }
    T *xtw = reinterpret_cast<T *>(&wave_lds[wave][0]);

    vec8_t<T> wr[kRing][kRowsCh], xr[kRing][NXL];
    float4_t acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = float4_t{0.f, 0.f, 0.f, 0.f};
#define SWL_ROWS_ISSUE(slot, c)                                                                         \
    {                                                                                                   \
        if constexpr (XLDS) {   /* x first: the chunk's x is what the LDS pass waits for (loads return in order) */ \
            _Pragma("unroll") for (int i_ = 0; i_ < NXL; ++i_) xr[slot][i_] = load8(xsrc[i_] + (c) * XCK); \
        }                                                                                               \
        _Pragma("unroll") for (int j_ = 0; j_ < kRowsCh; ++j_) {                                        \
            const int s_ = (c) * kRowsCh + j_;                                                          \
            wr[slot][j_] = load8_nt(wsrc + static_cast<int64_t>(s_) * 1024);                            \
            if constexpr (!XLDS) {                                                                      \
                _Pragma("unroll") for (int mb_ = 0; mb_ < MB; ++mb_) xr[slot][j_ * MB + mb_] = load8(xsrc[mb_] + s_ * 32); \
            }                                                                                           \
        }                                                                                               \
    }
#define SWL_ROWS_PROCESS(slot)                                                                          \
    {                                                                                                   \
        if constexpr (XLDS) {                                                                           \
            _Pragma("unroll") for (int i_ = 0; i_ < NXL; ++i_)                                          \
                *reinterpret_cast<vec8_t<T> *>(xtw + xw_off[i_]) = xr[slot][i_];                        \
        }                                                                                               \
        _Pragma("unroll") for (int j_ = 0; j_ < kRowsCh; ++j_)                                          \
            _Pragma("unroll") for (int mb_ = 0; mb_ < MB; ++mb_) {                                      \
                vec8_t<T> b_;                                                                           \
                if constexpr (XLDS) b_ = *reinterpret_cast<const vec8_t<T> *>(xtw + xr_off[j_] + mb_ * 16 * XCK); \
                else b_ = xr[slot][j_ * MB + mb_];                                                      \
                acc[mb_] = rows_mfma(wr[slot][j_], b_, acc[mb_]);                                       \
            }                                                                                           \
    }
    if constexpr (NCH > 0) {
        // straight-line schedule, exact counted waits: the first min(NCH, ring) chunks are requested up front (K = 4096:
        // the whole K range of the wave), longer K (down_proj: 14 chunks) refills a slot as soon as it is multiplied
#pragma unroll
        for (int c = 0; c < kRing; ++c) SWL_ROWS_ISSUE(c, c);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            // pinned: left alone the scheduler sinks requests between the MFMAs of earlier chunks (fewer live registers,
            // and nothing in flight while the wave multiplies)
            __builtin_amdgcn_sched_barrier(0);
            SWL_ROWS_PROCESS(c % kRing);
            __builtin_amdgcn_sched_barrier(0);
            if (c + kRing < NCH) SWL_ROWS_ISSUE(c % kRing, c + kRing);
        }
    } else {
#pragma unroll
        for (int c = 0; c < kRing; ++c)
            if (c < nch) SWL_ROWS_ISSUE(c, c);
        for (int c0 = 0; c0 < nch; c0 += kRing) {
#pragma unroll
            for (int d = 0; d < kRing; ++d) {
                if (c0 + d < nch) {
                    __builtin_amdgcn_sched_barrier(0);
                    SWL_ROWS_PROCESS(d);
                    __builtin_amdgcn_sched_barrier(0);
                    if (c0 + d + kRing < nch) SWL_ROWS_ISSUE(d, c0 + d + kRing);
                }
            }
        }
    }
#undef SWL_ROWS_ISSUE
#undef SWL_ROWS_PROCESS

    // ---- in-workgroup reduction: acc[mb][j] = out^T[n = 4*kq + j][token = r + 16*mb] -> red[wave][token][n] ----
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) mfma_results_tie(acc[mb]);
    mfma_results_ready<4>(acc[MB - 1]); // stored by DS instructions next (swl_common.h)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
        *reinterpret_cast<float4_t *>(red(wave) + (r + 16 * mb) * kRowsRedPitch + 4 * kq) = acc[mb];
    __syncthreads();
    float s = 0.f;
    if (MB == 2 || et < 16) {
#pragma unroll
        for (int w = 0; w < kRowsWaves; ++w) s += red(w)[et * kRowsRedPitch + en]; // wave order = K order
    }
    if constexpr (EPI == kRowsSlab) {
        if (e_ok) *res_p = s;
    } else if constexpr (EPI == kRowsStore) {
        if (e_ok) *res_p = to_t<T>(s);
    } else if constexpr (EPI == kRowsRelu2) {
        const float v = fmaxf(to_f(to_t<T>(s)), 0.f);
        if (e_ok) *res_p = to_t<T>(v * v);
    } else {
        // splitk_add_scale_kernel's arithmetic (rmsnorm.hip) on this thread's element
        const T xn = add_t<T>(to_t<T>(s), rv); // the projection is rounded, then the sum (rmsnorm.py:54-57)
        if (e_ok) *res_p = xn;
        if (a.ssq_out != nullptr) {             // (wave-uniform) the 16 column lanes of a token: one DPP row reduction
            const float v = e_ok ? to_f(xn) : 0.f;
            const float t = group_allreduce_sum<16>(v * v);
            if (e_ok && en == 0) a.ssq_out[static_cast<int64_t>(et) * (N / kRowsTile) + tile16] = t;
        }
    }
}

static bool rows_shape_ok(int M, int N, int K) {
    return M > 0 && M <= 32 && N > 0 && N % 32 == 0 && K > 0 && K % kRowsKUnit == 0;
}

template <typename T, int MB, bool XLDS, int EPI>
static int launch_rows(const RowsArgs &a, hipStream_t stream) {
    const dim3 grid((a.N + kRowsTile - 1) / kRowsTile), block(kRowsWaves * 64);
    const int nch = a.K / (32 * kRowsWaves * kRowsCh);
    // K = 4096 (Llama-3-8B / Llama-2-7B hidden): 4 chunks, all in flight; 14336 (Llama-3-8B FFN): 14; 8192: 8
    if constexpr (EPI != kRowsAdd) {
        if (nch == 1) { hipLaunchKernelGGL((gemm_rows_kernel<T, 1, MB, XLDS, EPI>), grid, block, 0, stream, a); return check_launch(); }
        if (nch == 2) { hipLaunchKernelGGL((gemm_rows_kernel<T, 2, MB, XLDS, EPI>), grid, block, 0, stream, a); return check_launch(); }
    } else {
        if (nch == 14) { hipLaunchKernelGGL((gemm_rows_kernel<T, 14, MB, XLDS, EPI>), grid, block, 0, stream, a); return check_launch(); }
        if (nch == 8) { hipLaunchKernelGGL((gemm_rows_kernel<T, 8, MB, XLDS, EPI>), grid, block, 0, stream, a); return check_launch(); }
    }
    if (nch == 4) hipLaunchKernelGGL((gemm_rows_kernel<T, 4, MB, XLDS, EPI>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((gemm_rows_kernel<T, 0, MB, XLDS, EPI>), grid, block, 0, stream, a);
    return check_launch();
}

// x through LDS pays from 9 tokens on (graph-timed on MI355X, profiles/r06b_rows_kernel_us.jsonl: o_proj 32 tokens 11.7 ->
// 10.5 us, down_proj 16 / 32 tokens 25.0 -> 23.8 / 34.4 -> 28.4; at one token the LDS hop costs o_proj 0.45 us, at 16 the
// two forms tie). A/B switch for measurements: SWL_ROWS_X=frag / lds forces one form for every M (same bits either way).
static bool rows_x_through_lds(int M) {
    static const int forced = [] { const char *e = getenv("SWL_ROWS_X"); return !e ? 0 : e[0] == 'f' ? 1 : e[0] == 'l' ? 2 : 0; }();
    return forced ? forced == 2 : M > 8;
}

template <typename T, int EPI>
static int launch_rows_m(const RowsArgs &a, hipStream_t s) {
    if (rows_x_through_lds(a.M)) return a.M <= 16 ? launch_rows<T, 1, true, EPI>(a, s) : launch_rows<T, 2, true, EPI>(a, s);
    return a.M <= 16 ? launch_rows<T, 1, false, EPI>(a, s) : launch_rows<T, 2, false, EPI>(a, s);
}

} // namespace swl

extern "C" int swl_gemm_rows_supported(int32_t M, int32_t N, int32_t K) { return swl::rows_shape_ok(M, N, K) ? 1 : 0; }

static int rows_add_impl(void *residual, float *ssq_out, const void *x, const void *w_packed, int32_t M, int32_t N, int32_t K,
                         int64_t x_row_stride, int32_t dtype, swl_stream_t stream);

extern "C" int swl_gemm_rows_add(void *residual, const void *x, const void *w_packed, int32_t M, int32_t N, int32_t K,
                                 int64_t x_row_stride, int32_t dtype, swl_stream_t stream) {
    return rows_add_impl(residual, nullptr, x, w_packed, M, N, K, x_row_stride, dtype, stream);
}

/* swl_gemm_rows_add + ssq_out[M][N / 16] (fp32): per (token, 16-column tile) the sum of squares of the updated residual. */
extern "C" int swl_gemm_rows_add_ssq(void *residual, float *ssq_out, const void *x, const void *w_packed, int32_t M, int32_t N,
                                     int32_t K, int64_t x_row_stride, int32_t dtype, swl_stream_t stream) {
    if (M > 0 && (!ssq_out || (reinterpret_cast<uintptr_t>(ssq_out) & 3u))) return SWL_ERR_BAD_ARG;
    return rows_add_impl(residual, ssq_out, x, w_packed, M, N, K, x_row_stride, dtype, stream);
}

static int rows_add_impl(void *residual, float *ssq_out, const void *x, const void *w_packed, int32_t M, int32_t N, int32_t K,
                         int64_t x_row_stride, int32_t dtype, swl_stream_t stream) {
    if (M < 0 || N <= 0 || K <= 0) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!residual || !x || !w_packed) return SWL_ERR_BAD_ARG;
    if (!swl::rows_shape_ok(M, N, K)) return SWL_ERR_UNSUPPORTED;
    if (x_row_stride < K || (x_row_stride & 7)) return SWL_ERR_BAD_ARG;
    if (!swl::aligned16(x) || !swl::aligned16(w_packed) || (reinterpret_cast<uintptr_t>(residual) & 1u)) return SWL_ERR_BAD_ARG;
    swl::RowsArgs a = {};
    a.x = x; a.wp = w_packed; a.residual = residual;
    a.M = M; a.N = N; a.K = K; a.x_stride = x_row_stride; a.ssq_out = ssq_out;
    SWL_DISPATCH_DTYPE(dtype, T, {
        const hipStream_t s = static_cast<hipStream_t>(stream);
        return swl::launch_rows_m<T, swl::kRowsAdd>(a, s);
    });
}

template <bool SLAB>
static int rows_store_impl(void *out, const void *x, const void *w_packed, int32_t M, int32_t N, int32_t K, int64_t x_row_stride,
                           int64_t out_row_stride, bool relu2, int32_t dtype, swl_stream_t stream) {
    if (M < 0 || N <= 0 || K <= 0) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!out || !x || !w_packed) return SWL_ERR_BAD_ARG;
    if (M > 32 || K % swl::kRowsKUnit != 0) return SWL_ERR_UNSUPPORTED;
    if (x_row_stride < K || (x_row_stride & 7) || out_row_stride < N) return SWL_ERR_BAD_ARG;
    if (!swl::aligned16(x) || !swl::aligned16(w_packed) || (reinterpret_cast<uintptr_t>(out) & (SLAB ? 3u : 1u))) return SWL_ERR_BAD_ARG;
    swl::RowsArgs a = {};
    a.x = x; a.wp = w_packed; a.residual = out; a.out_stride = out_row_stride;
    a.M = M; a.N = N; a.K = K; a.x_stride = x_row_stride;
    SWL_DISPATCH_DTYPE(dtype, T, {
        const hipStream_t s = static_cast<hipStream_t>(stream);
        if constexpr (SLAB) return swl::launch_rows_m<T, swl::kRowsSlab>(a, s);
        else return relu2 ? swl::launch_rows_m<T, swl::kRowsRelu2>(a, s) : swl::launch_rows_m<T, swl::kRowsStore>(a, s);
    });
}

/* out[M, N] = round(x . W^T), or relu(that)^2 rounded again (relu2 = 1): any N, the packed copy holding whole tiles of 32 rows. */
extern "C" int swl_gemm_rows_store(void *out, const void *x, const void *w_packed, int32_t M, int32_t N, int32_t K,
                                   int64_t x_row_stride, int64_t out_row_stride, int32_t relu2, int32_t dtype, swl_stream_t stream) {
    if (relu2 < 0 || relu2 > 1) return SWL_ERR_BAD_ARG;
    return rows_store_impl<false>(out, x, w_packed, M, N, K, x_row_stride, out_row_stride, relu2 != 0, dtype, stream);
}

/* slab[M, N] = x . W^T, fp32: the sums that swl_gemm_rows_store rounds, for consumers of K shares (one slab). */
extern "C" int swl_gemm_rows_partial(float *slab, const void *x, const void *w_packed, int32_t M, int32_t N, int32_t K,
                                     int64_t x_row_stride, int64_t slab_row_stride, int32_t dtype, swl_stream_t stream) {
    return rows_store_impl<true>(slab, x, w_packed, M, N, K, x_row_stride, slab_row_stride, false, dtype, stream);
}
