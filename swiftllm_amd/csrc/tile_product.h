// tile_product.h — a tile of 128 x 128 results on the matrix cores, by a workgroup of four waves of 64 x 64 each (mfma 32x32x16, 2 x 2
// accumulators): what the expert products (moe_grouped.hip) and the expansion of latent rows (latent_expand.hip) share. 16-bit operands,
// fp32 sums.
//
// Both operands are rows with the reduction along them ("weights" W, "tokens" X), staged by LDS-DMA in 64-deep slices of whole 128-byte
// lines (half lines take 1.4 times as long): a slice is 128 rows of W, then 128 rows of X, a row's eight 16-byte units exchanged by
// bits 1 .. 3 of the row's number (tile_unit), on the source side, so that the fragment reads stay off each other's banks.
#pragma once

#include "swl_common.h"

namespace swl {

constexpr int kTile = 128, kTileDepth = 64, kTileSliceB = kTile * kTileDepth * 2;       // rows, depth, bytes of one operand's slice

__device__ __forceinline__ float16_t tile_mfma(vec8_t<f16> a, vec8_t<f16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float16_t tile_mfma(vec8_t<bf16> a, vec8_t<bf16> b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Staging: wave w asks for rows 32 w + 8 i .. + 7 of an operand with its instruction i = 0 .. 3, lane l for this row and this unit of it.
__device__ __forceinline__ int tile_row(int wave, int i, int lane) { return wave * 32 + i * 8 + (lane >> 3); }
__device__ __forceinline__ int tile_unit(int row, int lane) { return (lane & 7) ^ ((row >> 1) & 7); }
// 1 KiB (16 bytes a lane, from `base` + the lane's `off`) to the LDS address `to`
__device__ __forceinline__ void tile_ask(const char *base, unsigned off, unsigned to) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(off), "s"(base), "s"(to) : "memory");
}

// acc[a][b] = the tile's products over `stages` slices. TOKENS_FIRST false: element 4 q + r of acc[a][b] is (weight row 64 wn + 32 a + 8 q
// + 4 hf + r, token 64 wm + 32 b + l32), true: (token 64 wm + 32 a + 8 q + 4 hf + r, weight row 64 wn + 32 b + l32), with l32 = lane % 32,
// hf = lane / 32. issue(st): asks for slice st into buffer st % BUFS of smem (2 kTileSliceB each). BUFS 2: for two workgroups a CU, a
// slice on its way while one is multiplied; 1: for four workgroups a CU, which hide each other's waits, first and last slices too.
// The staged slices may still be read by other waves when it returns.
template <typename T, int BUFS, bool TOKENS_FIRST, typename Issue>
__device__ __forceinline__ void tile_product(const char *smem, int stages, int wn, int wm, int lane, float16_t (&acc)[2][2], Issue &&issue) {
    const int l32 = lane & 31, hf = lane >> 5;
    // fragments: row l32 of a 32-row piece, 16-byte unit 2 e + hf (exchanged as staged; rows 32 apart alike)
    unsigned frag[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) frag[e] = static_cast<unsigned>(l32 * 128 + (((2 * e + hf) ^ ((l32 >> 1) & 7)) * 16));
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = float16_t{};
    vec8_t<T> wf[2][2], xf[2][2];       // [set][piece]: the fragments of 16 columns are requested in front of the products of the 16 before
    auto read = [&](int st, int e, int set) {
        const char *ws = smem + (st & (BUFS - 1)) * 2 * kTileSliceB + wn * 64 * 128, *xs = smem + (st & (BUFS - 1)) * 2 * kTileSliceB + kTileSliceB + wm * 64 * 128;
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            wf[set][a] = *reinterpret_cast<const vec8_t<T> *>(ws + a * 32 * 128 + frag[e]);
            xf[set][a] = *reinterpret_cast<const vec8_t<T> *>(xs + a * 32 * 128 + frag[e]);
        }
    };
    auto multiply = [&](int set) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
                acc[a][b] = TOKENS_FIRST ? tile_mfma(xf[set][a], wf[set][b], acc[a][b]) : tile_mfma(wf[set][a], xf[set][b], acc[a][b]);
    };
    auto step = [&](int st, int e, int set) {       // products of a set, the reads of the next spread between them
        __builtin_amdgcn_sched_barrier(0);
        read(st, e, set ^ 1);
        multiply(set);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    issue(0);
    if constexpr (BUFS == 1) {
        for (int st = 0;; ++st) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // this wave's pieces of the slice have landed; then everyone's
            __builtin_amdgcn_s_barrier();
            read(st, 0, 0);
            step(st, 1, 0);
            step(st, 2, 1);
            step(st, 3, 0);
            multiply(1);        // (its operands were the last reads of the slice: all of them have returned; then everyone's)
            if (st + 1 == stages) break;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            issue(st + 1);
        }
    } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        if (stages > 1) issue(1);
        read(0, 0, 0);
        for (int st = 0; st + 1 < stages; ++st) {
            step(st, 1, 0);
            step(st, 2, 1);
            step(st, 3, 0);
            // this wave's pieces of the next slice have landed, its reads of this one have returned; then everyone's
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            if (st + 2 < stages) issue(st + 2);
            step(st + 1, 0, 1);
        }
        step(stages - 1, 1, 0);
        step(stages - 1, 2, 1);
        step(stages - 1, 3, 0);
        multiply(1);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
            if (a + b < 2) mfma_results_tie(acc[a][b]);
    mfma_results_ready<8>(acc[1][1]);
}

} // namespace swl
