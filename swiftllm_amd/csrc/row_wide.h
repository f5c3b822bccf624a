// row_wide.h — rows of a [tokens, width] stream held in registers: TPR threads of a 256-thread workgroup own a row (256 / TPR rows a workgroup),
// thread i the columns 4 (i + TPR j) .. + 3, j < NV. Every access is 16 bytes a lane of fp32 (8 of a 16-bit type), neighbouring lanes on
// neighbouring columns, and all of a row's loads are in flight together; a row that one wave owns needs no barrier.
#pragma once
#include "swl_common.h"

#include <type_traits>

namespace swl {

constexpr int kRowThreads = 256;

template <typename T>
__device__ __forceinline__ void row_load(float (&v)[4], const T *p) {
    if constexpr (sizeof(T) == 4) {
        const float4_t x = *reinterpret_cast<const float4_t *>(p);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = x[j];
    } else {
        const vec4_t<T> x = *reinterpret_cast<const vec4_t<T> *>(p);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = to_f(x[j]);
    }
}
template <typename T>
__device__ __forceinline__ void row_store(T *p, const float (&v)[4]) {
    vec4_t<T> x;
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = to_t<T>(v[j]);
    *reinterpret_cast<vec4_t<T> *>(p) = x;
}

// The same columns of `parts` fp32 slabs `stride` floats apart (a product whose K was split over workgroups), added in order: the slabs of
// a thread's columns are requested four (two, where a thread holds many columns; eight or sixteen, where a workgroup has a row) at a time, not one
// behind the other's sum.
template <int TPR, int NV>
__device__ __forceinline__ void row_load_parts(float (&v)[NV][4], const float *p, int c0, int width, int parts, int64_t stride) {
    if (parts == 1) {       // (the last slab stands in for the missing ones below: one slab would be read DEEP times)
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (c0 + 4 * TPR * j < width) row_load<float>(v[j], p + c0 + 4 * TPR * j);
        return;
    }
    auto add = [&](auto deep) {
        constexpr int DEEP = decltype(deep)::value;
        for (int k = 0; k < parts; k += DEEP) {
            float4_t b[DEEP][NV];
#pragma unroll
            for (int u = 0; u < DEEP; ++u)
#pragma unroll
                for (int j = 0; j < NV; ++j) {
                    b[u][j] = float4_t{0.f, 0.f, 0.f, 0.f};
                    if (c0 + 4 * TPR * j < width) b[u][j] = *reinterpret_cast<const float4_t *>(p + min(k + u, parts - 1) * stride + c0 + 4 * TPR * j);
                }
#pragma unroll
            for (int u = 0; u < DEEP; ++u) {
                if (k + u < parts) {
#pragma unroll
                    for (int j = 0; j < NV; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[j][e] = k + u ? v[j][e] + b[u][j][e] : b[u][j][e];
                }
            }
        }
    };
    // (a workgroup a row: steps of few rows, whose sums are a chain of waits. 32 rows of 2048 with 16 slabs 7.2 -> 6.4 us)
    if constexpr (TPR == 256 && NV <= 2) {
        if (parts > 8) return add(std::integral_constant<int, 16>{});
        if (parts > 4) return add(std::integral_constant<int, 8>{});
    }
    add(std::integral_constant<int, NV <= 2 ? 4 : 2>{});
}

// Sum over the threads of a row; `red`: one float per wave, its own for every sum of a kernel.
template <int TPR>
__device__ __forceinline__ float row_sum(float v, float *red) {
    v = wave_allreduce_sum(v);
    if constexpr (TPR > 64) {
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) red[wave] = v;
        __syncthreads();
        const int w0 = wave / (TPR / 64) * (TPR / 64);
        v = red[w0];
#pragma unroll
        for (int w = 1; w < TPR / 64; ++w) v += red[w0 + w];
    }
    return v;
}

template <typename T>
__host__ __device__ inline bool row_aligned(const void *p) { return (reinterpret_cast<uintptr_t>(p) & (4 * sizeof(T) - 1)) == 0; }

// Runs GO(TPR, NV) for a launch of `rows` rows: a wave (two) a row for many rows of up to 1024 (2048) columns, else a workgroup a row, which
// ends a step of few rows sooner.
#define SWL_ROW_SHAPE(rows, width, GO)                  \
    do {                                                \
        if ((rows) >= 1024 && (width) <= 1024) GO(64, 4); \
        else if ((rows) >= 1024 && (width) <= 2048) GO(128, 4); \
        else if ((width) <= 1024) GO(256, 1);           \
        else if ((width) <= 2048) GO(256, 2);           \
        else if ((width) <= 4096) GO(256, 4);           \
        else GO(256, 8);                                \
    } while (0)
constexpr int kRowMaxWidth = 8192;

} // namespace swl
