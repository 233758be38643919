// Sums and maxima over the lanes of a wave without LDS: halves and rows of 16 are swapped, lanes of a row rotated.  An exchange through LDS
// (ds_bpermute, what __shfl_xor is) takes some hundred cycles, and a sum over 64 lanes is six of them in line; these take a handful each.  The
// partners, and so the bits, are those of the exchanges over 32, 16, 8, 4, 2, 1: behind the first of them the partial results repeat every 8, 4, 2
// lanes, where rotating by that many meets the same value.  All lanes of the wave take part.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// Both values of lanes l and l ^ 32 (l ^ 16), in every lane the lower lane's first.
template <typename T> struct LanePair { T a, b; };
template <typename T> __device__ __forceinline__ LanePair<T> lane_halves(T v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t a = r[0], b = r[1];
    return LanePair<T>{__builtin_bit_cast(T, a), __builtin_bit_cast(T, b)};
}
template <typename T> __device__ __forceinline__ LanePair<T> lane_rows(T v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const uint32_t a = r[0], b = r[1];
    return LanePair<T>{__builtin_bit_cast(T, a), __builtin_bit_cast(T, b)};
}
// The value of the lane N places further round in the row of 16.
template <int N, typename T> __device__ __forceinline__ T lane_rotated(T v) {
    const int u = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(u, u, 0x120 | N, 0xf, 0xf, false));
}

template <typename T, class F> __device__ __forceinline__ T lanes_fold(T v, F f) {
    const LanePair<T> h = lane_halves(v);
    v = f(h.a, h.b);
    const LanePair<T> r = lane_rows(v);
    v = f(r.a, r.b);
    v = f(v, lane_rotated<8>(v));
    v = f(v, lane_rotated<4>(v));
    v = f(v, lane_rotated<2>(v));
    return f(v, lane_rotated<1>(v));
}
// Over the four lanes l, l ^ 16, l ^ 32, l ^ 48.
template <typename T, class F> __device__ __forceinline__ T rows_fold(T v, F f) {
    const LanePair<T> r = lane_rows(v);
    v = f(r.a, r.b);
    const LanePair<T> h = lane_halves(v);
    return f(h.a, h.b);
}
__device__ __forceinline__ float lanes_sum(float v) { return lanes_fold(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ float lanes_max(float v) { return lanes_fold(v, [](float a, float b) { return fmaxf(a, b); }); }
__device__ __forceinline__ int lanes_sum(int v) { return lanes_fold(v, [](int a, int b) { return a + b; }); }
__device__ __forceinline__ int lanes_max(int v) { return lanes_fold(v, [](int a, int b) { return a > b ? a : b; }); }
__device__ __forceinline__ float rows_sum(float v) { return rows_fold(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ float rows_max(float v) { return rows_fold(v, [](float a, float b) { return fmaxf(a, b); }); }
// The value of lane l ^ 32.
__device__ __forceinline__ float other_half(float v) {
    const LanePair<float> h = lane_halves(v);
    return (threadIdx.x & 32) ? h.a : h.b;
}
