// gemm_wide.hip — decode projections for LARGE batches (64 < M <= 256 tokens) on packed weights, gfx950.
//
// out[M, N] = x[M, K] . W[N, K]^T (reference: swiftllm/worker/kernels/linear.py:3-12, called from
// transformer_layer.py:54-56,117,126,128), for the batch sizes a 264 GB KV pool is sized for. Up to 32 tokens the
// product is pure weight streaming (gemm_skinny.hip); up to 64 two token blocks share every weight fragment
// (gemm_packed_mt_kernel). Beyond that hipBLASLt was the fallback, and its 256x256 tiles leave most of the chip idle on
// the narrow projections of a decode step (N = 4096 / 6144 at M = 256: 16-24 tiles on 256 CUs; qkv 36 us for 50 MB,
// down 48 us for 117 MB — profiles/r03_blas_m_sweep_decode_sizes.jsonl). At these M the op sits between streaming and
// a GEMM: W (N*K*e bytes) still has to come from HBM exactly once, but x (M*K*e) is re-read from L2 by every workgroup.
//
// What bounds it: what a CU can have on its way. Requests in flight seem to hold lines of its 32 KiB L1: a CU takes about 32 KiB a latency,
// whatever the depth of the ring behind it: at 120 tokens and 28672 x 4096 a workgroup takes 1 MiB of W and 1 MiB of x, and neither
// leaving out the products (48 us), nor reading x from L1 (48), nor W from L2 (44), nor 7 slices of W in flight instead of 4 (49) moves the
// 49 us by much; W alone, at 32 tokens, takes 38.5 (6.1 TB/s). Structure:
//   * W stays in MFMA-fragment order (swl_gemm_pack_weight): LDS-DMA, non-temporal, 4 KiB in a row; x comes row by row in whole 128-byte lines,
//     swizzled on the source side (16-byte slot = chunk ^ ((row >> 1) & 7): the fragment reads stay off each other's banks);
//   * 160 KiB of LDS hold 5 slices of 64 columns of both (4 beyond 128 tokens, 3 beyond 192). A step waits for the next slice alone: with
//     W in a register ring behind x, as before, the in-order counter made every wait for x drain the weights on their way too;
//   * four waves tile 128 rows of W x all tokens two by two (every fragment read feeds ceil(M/64) or 2 MFMAs); one barrier a slice;
//   * K is split across workgroups into fp32 slabs as far as that keeps <= 256 workgroups and K-chunks of >= 16 (8 beyond 128 tokens)
//     slices — gemm_wide_splits(); filling the chip beats the L2-resident slab round trip;
//   * SiLU-gate mode: a wave's two row blocks are up and gate of the same columns, so the gate is applied in registers; same rounding points
//     as linear -> silu_and_mul_inplace (silu_and_mul.py:16-23).
// Bits: every output is the fp32 sum over k in ascending 16-element steps inside a K-chunk, chunks added in slab
// order — the summation order of the M <= 64 kernels at the same split count.
// Measured (us, bf16, W cycled through 1.2 GB, this kernel alone: adding up K shares takes another 4 to 7; W through registers -> now; on other cards and
// in long runs up to a fifth more: 18.0 / 21.2 / 25.2, 15.6 / 17.6 / 20.9, 56 / 67 / 81, 31.5 / 38.9 / 46.7, 57 / 74 / 87), at 120 / 192 / 256 tokens: qkv 6144 x 4096 19.7 -> 17.1 /
// 24.0 -> 20.2 / 29.8 -> 25.1; o 4096 x 4096 17.5 -> 15.0 / 17.8 -> 16.5 / 22.2 -> 19.8; up/gate + SiLU 51.9 -> 47.3 / 65.4 -> 53.7 /
// 83.6 -> 67.6; down 4096 x 14336 28.6 -> 27.4 / 37.7 -> 32.7 / 45.2 -> 40.6; head 32000 x 4096 51.7 -> 47.5 / 66.7 -> 57.1 / 82.3 -> 73.6.
#include "swl_common.h"

extern "C" int swl_splitk_reduce(void *out, const float *slabs, int32_t k_splits, int32_t M, int32_t N,
                                 int64_t out_row_stride, int32_t dtype, swl_stream_t stream);

namespace swl {

__device__ __forceinline__ float16_t mfma_w(vec8_t<f16> a, vec8_t<f16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float16_t mfma_w(vec8_t<bf16> a, vec8_t<bf16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

constexpr int kWT = 64;      // k elements per slice
// slices in LDS (160 KiB): 5 of 32 KiB, 4 of 40 KiB, 3 of 48 KiB
constexpr int wide_ring(int mt) { return mt <= 4 ? 5 : mt <= 6 ? 4 : 3; }

enum WideMode { kWideDirect = 0, kWidePartial = 1, kWideSiluGate = 2 };

// A workgroup of four waves owns 128 rows of W (four packed 32-row blocks; SiLU-gate mode: up and gate blocks of 64 columns) x all tokens
// (MT blocks of 32), wave (wn, wm) two of the row blocks x half of the token blocks. RING slices of 64 columns of both operands are on
// their way or in LDS; a slice is asked for RING steps ahead, and what a step waits for is counted (vmcnt), so that every slice but the
// next one stays in flight.
template <typename T, int MT, int MODE>
__global__ __launch_bounds__(256, 1) void gemm_packed_wide_kernel(void *__restrict__ out_, const T *__restrict__ x, const T *__restrict__ wpk,
                                                                  int M, int N, int K, int kc, int64_t x_stride, int64_t out_stride) {
    constexpr int WB = 128 * kWT * 2, XB = MT * 32 * kWT * 2, BUF = WB + XB, RING = wide_ring(MT);      // bytes
    constexpr int TPW = MT / 2;                 // token blocks of a wave
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, hf = lane >> 5, wn = wave & 1, wm = wave >> 1;
    const int blocks = N / 32;                  // 32-row blocks of W (of each half in SiLU-gate mode)
    const int b0 = blockIdx.x * (MODE == kWideSiluGate ? 2 : 4);
    const int k_begin = blockIdx.y * kc, stages = kc / kWT;

    // ---- staging: wave w brings row block w (4 KiB in a row) and a quarter of the tokens, 8 rows of 128 bytes an instruction ---------
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    const int mine = MODE == kWideSiluGate ? min(b0 + (wave >> 1), blocks - 1) + (wave & 1) * blocks : min(b0 + wave, blocks - 1);
    const char *wsrc = reinterpret_cast<const char *>(wpk + (static_cast<int64_t>(mine) * (K / 16) + k_begin / 16) * 512);
    const char *xsrc = reinterpret_cast<const char *>(x + k_begin);
    const unsigned w_off = lane * 16;
    unsigned x_off[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int r = wave * 8 * MT + i * 8 + (lane >> 3);
        x_off[i] = static_cast<unsigned>(min(r, M - 1) * x_stride * 2 + ((lane & 7) ^ ((r >> 1) & 7)) * 16);
    }
    auto issue = [&](int st, unsigned buf) {
        const char *ws = wsrc + static_cast<int64_t>(st) * 4096, *xs = xsrc + static_cast<int64_t>(st) * kWT * 2;
        const unsigned to = lds0 + buf;
#pragma unroll
        for (int i = 0; i < 4; ++i) {           // (W is read once: non-temporal)
            unsigned keep;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
                         : "=&s"(keep) : "v"(w_off), "s"(ws + i * 1024), "s"(to + wave * 4096 + i * 1024) : "memory");
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            unsigned keep;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                         : "=&s"(keep) : "v"(x_off[i]), "s"(xs), "s"(to + WB + wave * (XB / 4) + i * 1024) : "memory");
        }
    };
    // x fragments: row l32 of a 32-row block, 16-byte unit 2 e + hf (swizzled as staged; rows 32 apart share the swizzle)
    unsigned frag[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) frag[e] = static_cast<unsigned>(WB + wm * (XB / 2) + l32 * 128 + (((2 * e + hf) ^ ((l32 >> 1) & 7)) * 16));
    const unsigned wfrag = static_cast<unsigned>(wn * 8192 + lane * 16);
    float16_t acc[2][TPW];                      // [row block][token block]
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < TPW; ++b) acc[a][b] = float16_t{};
    vec8_t<T> wf[2][2], xf[2][TPW];             // [set][block]: the fragments of 16 columns are requested in front of the products of the 16 before
    auto read = [&](unsigned buf, int e, int set) {
        const char *s = smem + buf;
#pragma unroll
        for (int a = 0; a < 2; ++a) wf[set][a] = *reinterpret_cast<const vec8_t<T> *>(s + a * 4096 + e * 1024 + wfrag);
#pragma unroll
        for (int b = 0; b < TPW; ++b) xf[set][b] = *reinterpret_cast<const vec8_t<T> *>(s + b * 4096 + frag[e]);
    };
    auto multiply = [&](int set) {
#pragma unroll
        for (int b = 0; b < TPW; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a) acc[a][b] = mfma_w(wf[set][a], xf[set][b], acc[a][b]);
    };
    auto step = [&](unsigned buf, int e, int set) {         // products of a set, the reads of the next spread between them
        __builtin_amdgcn_sched_barrier(0);
        read(buf, e, set ^ 1);
        multiply(set);
#pragma unroll
        for (int i = 0; i < 2 + TPW; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, TPW > 2 ? TPW - 2 : 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // this wave's pieces of the next slice have landed (`later` slices after it may be on their way), its reads of this one have returned;
    // then everyone's
    constexpr int DMA = 4 + MT;                 // staging instructions of a slice
    auto landed = [&](int later) {
        if (later >= RING - 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((RING - 2) * DMA) : "memory");
        else if (RING > 4 && later == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * DMA) : "memory");
        else if (RING > 3 && later == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(DMA) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
    };
#pragma unroll
    for (int i = 0; i < RING; ++i)
        if (i < stages) issue(i, i * BUF);
    if (stages >= RING) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 1) * DMA) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read(0, 0, 0);
    unsigned buf = 0;
    for (int st = 0; st + 1 < stages; ++st) {
        const unsigned next = buf == (RING - 1) * BUF ? 0 : buf + BUF;
        step(buf, 1, 0);
        step(buf, 2, 1);
        step(buf, 3, 0);
        landed(stages - 2 - st);
        if (st + RING < stages) issue(st + RING, buf);
        step(next, 0, 1);
        buf = next;
    }
    step(buf, 1, 0);
    step(buf, 2, 1);
    step(buf, 3, 0);
    multiply(1);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < TPW; ++b) mfma_results_tie(acc[a][b]);
    mfma_results_ready<8>(acc[1][TPW - 1]);     // acc comes straight out of the K loop (swl_common.h)

    // acc[a][b][r]: out^T[n = 32 * block + (r & 3) + 8 * (r >> 2) + 4 * hf][m = 32 * (wm * TPW + b) + l32]
    typedef T vec4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int b = 0; b < TPW; ++b) {
        const int m = 32 * (wm * TPW + b) + l32;
        if (m >= M) continue;
        if constexpr (MODE == kWideSiluGate) {  // a wave's blocks: up and gate of the same columns
            const int n = 32 * (b0 + wn) + 4 * hf;
            if (n >= N) continue;
            T *o = static_cast<T *>(out_) + static_cast<int64_t>(m) * out_stride + n;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                vec4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float g = to_f(to_t<T>(acc[1][b][4 * r4 + e]));
                    v[e] = mul_t<T>(to_t<T>(acc[0][b][4 * r4 + e]), to_t<T>(g / (1.0f + expf(-g))));
                }
                *reinterpret_cast<vec4 *>(o + 8 * r4) = v;
            }
        } else {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int n = 32 * (b0 + 2 * wn + a) + 4 * hf;
                if (n >= N) continue;
                if constexpr (MODE == kWidePartial) {
                    float *slab = static_cast<float *>(out_) + (static_cast<int64_t>(blockIdx.y) * M + m) * N + n;
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4) {
                        const float4_t v = {acc[a][b][4 * r4], acc[a][b][4 * r4 + 1], acc[a][b][4 * r4 + 2], acc[a][b][4 * r4 + 3]};
                        *reinterpret_cast<float4_t *>(slab + 8 * r4) = v;
                    }
                } else {
                    T *o = static_cast<T *>(out_) + static_cast<int64_t>(m) * out_stride + n;
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4) {
                        vec4 v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = to_t<T>(acc[a][b][4 * r4 + e]);
                        *reinterpret_cast<vec4 *>(o + 8 * r4) = v;
                    }
                }
            }
        }
    }
}

// K-split for (M, N, K): the largest power of two that keeps the launch at <= 256 workgroups and a chunk >= 16 slices (<= 128 tokens) / 8
// slices long.
static int gemm_wide_splits(int M, int N, int K) {
    const int wgs = (N / 32 + 3) / 4, min_chunk = (M <= 128 ? 16 : 8) * kWT;
    int ks = 1;
    while (ks < 16 && wgs * ks * 2 <= 256 && K % (kWT * ks * 2) == 0 && K / (ks * 2) >= min_chunk) ks *= 2;
    return ks;
}

template <typename T, int MT, int MODE>
static int launch_wide(dim3 grid, hipStream_t s, void *out, const T *x, const T *wp, int M, int N, int K, int kc, int64_t xs, int64_t os) {
    constexpr int lds = wide_ring(MT) * (128 + MT * 32) * kWT * 2;
    auto kernel = gemm_packed_wide_kernel<T, MT, MODE>;
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return SWL_ERR_LAUNCH;
    hipLaunchKernelGGL(kernel, grid, dim3(256), lds, s, out, x, wp, M, N, K, kc, xs, os);
    return check_launch();
}

template <typename T, int MODE>
static int launch_wide(dim3 grid, hipStream_t s, void *out, const T *x, const T *wp, int M, int N, int K, int kc, int64_t xs, int64_t os) {
    if (M <= 128) return launch_wide<T, 4, MODE>(grid, s, out, x, wp, M, N, K, kc, xs, os);
    if (M <= 192) return launch_wide<T, 6, MODE>(grid, s, out, x, wp, M, N, K, kc, xs, os);
    return launch_wide<T, 8, MODE>(grid, s, out, x, wp, M, N, K, kc, xs, os);
}

} // namespace swl

/* Workspace bytes swl_gemm_packed_wide needs for (M, N, K) with the library's own plan (0 = K is not split). */
extern "C" size_t swl_gemm_packed_wide_workspace_bytes(int32_t M, int32_t N, int32_t K) {
    if (M <= 0 || M > 256 || N <= 0 || K <= 0 || (N & 31) || (K & (swl::kWT - 1))) return 0;
    const int ks = swl::gemm_wide_splits(M, N, K);
    return ks > 1 ? static_cast<size_t>(ks) * M * N * sizeof(float) : 0;
}

/* out[M, N] = x . W^T for up to 256 tokens on a weight packed by swl_gemm_pack_weight. N % 32 == 0, K % 64 == 0.
 * waves_per_group: 0, 4 or 8 (one form serves all); k_splits: 0 = library's choice, else a power of two <= 16 with
 * K % (64 * k_splits) == 0. workspace >= k_splits * M * N * 4 bytes when K is split
 * (swl_gemm_packed_wide_workspace_bytes for the library's plan). */
extern "C" int swl_gemm_packed_wide(void *out, const void *x, const void *w_packed, void *workspace,
                                    size_t workspace_bytes, int32_t M, int32_t N, int32_t K, int64_t x_row_stride,
                                    int64_t out_row_stride, int32_t waves_per_group, int32_t k_splits, int32_t dtype,
                                    swl_stream_t stream) {
    if (M < 0 || N <= 0 || K <= 0) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!out || !x || !w_packed) return SWL_ERR_BAD_ARG;
    if (M > 256 || (N & 31) || (K & (swl::kWT - 1))) return SWL_ERR_UNSUPPORTED;
    if (x_row_stride < K || out_row_stride < N || (x_row_stride & 7) || (out_row_stride & 3)) return SWL_ERR_BAD_ARG;
    if (static_cast<int64_t>(M) * x_row_stride >= (1ll << 31)) return SWL_ERR_UNSUPPORTED;
    if (!swl::aligned16(x) || !swl::aligned16(w_packed) || (reinterpret_cast<uintptr_t>(out) & 7u) ||
        (workspace && !swl::aligned16(workspace)))
        return SWL_ERR_BAD_ARG;
    if (!(waves_per_group == 0 || waves_per_group == 4 || waves_per_group == 8)) return SWL_ERR_BAD_ARG;
    if (k_splits < 0 || k_splits > 16 || (k_splits & (k_splits - 1))) return SWL_ERR_BAD_ARG;
    const int ks = k_splits ? k_splits : swl::gemm_wide_splits(M, N, K);
    if (K % (swl::kWT * ks) != 0) return SWL_ERR_UNSUPPORTED;
    const int kc = K / ks;
    const dim3 grid((N / 32 + 3) / 4, ks);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (ks == 1) {
        SWL_DISPATCH_DTYPE(dtype, T, {
            return swl::launch_wide<T, swl::kWideDirect>(grid, s, out, static_cast<const T *>(x), static_cast<const T *>(w_packed), M, N, K,
                                                         kc, x_row_stride, out_row_stride);
        });
    }
    if (!workspace || workspace_bytes < static_cast<size_t>(ks) * M * N * sizeof(float)) return SWL_ERR_BAD_ARG;
    SWL_DISPATCH_DTYPE(dtype, T, {
        const int rc = swl::launch_wide<T, swl::kWidePartial>(grid, s, workspace, static_cast<const T *>(x), static_cast<const T *>(w_packed),
                                                              M, N, K, kc, x_row_stride, N);
        if (rc != SWL_OK) return rc;
    });
    return swl_splitk_reduce(out, static_cast<const float *>(workspace), ks, M, N, out_row_stride, dtype, stream);
}

/* The split count swl_gemm_packed_wide picks for k_splits = 0 (0 = shape unsupported). */
extern "C" int swl_gemm_packed_wide_choose_splits(int32_t M, int32_t N, int32_t K) {
    if (M <= 0 || M > 256 || N <= 0 || K <= 0 || (N & 31) || (K & (swl::kWT - 1))) return 0;
    return swl::gemm_wide_splits(M, N, K);
}

/* Partial slabs only (slabs[k_splits][M][N] fp32, k_splits >= 1: a power of two <= 16 with K % (64 * k_splits) == 0) for
 * the split-K consumers (swl_splitk_fused_add_rmsnorm, swl_splitk_rotary_store_kv_decode): swl_gemm_packed_wide minus its
 * reduce launch, same bits. */
extern "C" int swl_gemm_packed_wide_partial(float *slabs, size_t slabs_bytes, const void *x, const void *w_packed,
                                            int32_t M, int32_t N, int32_t K, int64_t x_row_stride,
                                            int32_t waves_per_group, int32_t k_splits, int32_t dtype,
                                            swl_stream_t stream) {
    if (M < 0 || N <= 0 || K <= 0) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!slabs || !x || !w_packed || k_splits < 1 || k_splits > 16 || (k_splits & (k_splits - 1))) return SWL_ERR_BAD_ARG;
    if (M > 256 || (N & 31) || (K & (swl::kWT - 1)) || K % (swl::kWT * k_splits)) return SWL_ERR_UNSUPPORTED;
    if (x_row_stride < K || (x_row_stride & 7) || !swl::aligned16(x) || !swl::aligned16(w_packed) || !swl::aligned16(slabs))
        return SWL_ERR_BAD_ARG;
    if (static_cast<int64_t>(M) * x_row_stride >= (1ll << 31)) return SWL_ERR_UNSUPPORTED;
    if (!(waves_per_group == 0 || waves_per_group == 4 || waves_per_group == 8)) return SWL_ERR_BAD_ARG;
    if (slabs_bytes < static_cast<size_t>(k_splits) * M * N * sizeof(float)) return SWL_ERR_BAD_ARG;
    const dim3 grid((N / 32 + 3) / 4, k_splits);
    SWL_DISPATCH_DTYPE(dtype, T, {
        return swl::launch_wide<T, swl::kWidePartial>(grid, static_cast<hipStream_t>(stream), slabs, static_cast<const T *>(x),
                                                      static_cast<const T *>(w_packed), M, N, K, K / k_splits, x_row_stride, N);
    });
}

/* out[M, I] = up * silu(gate) of x . [up ; gate]^T for up to 256 tokens on a packed weight (the large-batch twin of
 * swl_gemm_skinny_packed_silu_gate; same rounding points as linear + silu_and_mul). I % 32 == 0, K % 64 == 0.
 * waves_per_group: 0, 4 or 8 (one form serves all). */
extern "C" int swl_gemm_packed_wide_silu_gate(void *out, const void *x, const void *w_up_gate_packed, int32_t M,
                                              int32_t I, int32_t K, int64_t x_row_stride, int64_t out_row_stride,
                                              int32_t waves_per_group, int32_t dtype, swl_stream_t stream) {
    if (M < 0 || I <= 0 || K <= 0) return SWL_ERR_BAD_ARG;
    if (M == 0) return SWL_OK;
    if (!out || !x || !w_up_gate_packed) return SWL_ERR_BAD_ARG;
    if (M > 256 || (I & 31) || (K & (swl::kWT - 1))) return SWL_ERR_UNSUPPORTED;
    if (x_row_stride < K || out_row_stride < I || (x_row_stride & 7) || (out_row_stride & 3)) return SWL_ERR_BAD_ARG;
    if (static_cast<int64_t>(M) * x_row_stride >= (1ll << 31)) return SWL_ERR_UNSUPPORTED;
    if (!swl::aligned16(x) || !swl::aligned16(w_up_gate_packed) || (reinterpret_cast<uintptr_t>(out) & 7u))
        return SWL_ERR_BAD_ARG;
    if (!(waves_per_group == 0 || waves_per_group == 4 || waves_per_group == 8)) return SWL_ERR_BAD_ARG;
    const dim3 grid((I / 32 + 1) / 2, 1);
    SWL_DISPATCH_DTYPE(dtype, T, {
        return swl::launch_wide<T, swl::kWideSiluGate>(grid, static_cast<hipStream_t>(stream), out, static_cast<const T *>(x),
                                                       static_cast<const T *>(w_up_gate_packed), M, I, K, K, x_row_stride, out_row_stride);
    });
}
