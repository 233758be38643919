// Pieces of row kernels that run inside a wide product (Src of share_gemm_body): a workgroup of 512 threads holds whole rows of up to 4 096, two quads a
// thread (threadIdx.x and 512 further on).
#pragma once
#include "tile_common.h"

// 1 / rms of every row's v over the workgroup; each: LDS of [ROWS][8] of its own.
template <int ROWS>
__device__ __forceinline__ void rows_inverse(const f32x4 (&v)[ROWS][2], int width, int width_real, float eps, float* each, float (&inv)[ROWS]) {
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if ((int)threadIdx.x + 512 * j < width >> 2) s += v[r][j][0] * v[r][j][0] + v[r][j][1] * v[r][j][1] + v[r][j][2] * v[r][j][2] + v[r][j][3] * v[r][j][3];
        s = wave_sum64(s);
        if ((threadIdx.x & 63) == 0) each[8 * r + wave] = s;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        float s = each[8 * r];
#pragma unroll
        for (int k = 1; k < 8; ++k) s += each[8 * r + k];
        inv[r] = 1.0f / sqrtf(s / (float)width_real + eps);
    }
}

// xs [width / 8][rows][8] = v * inv * n
template <int ROWS>
__device__ __forceinline__ void rows_normed(const f32x4 (&v)[ROWS][2], const f32x4 (&n)[2], const float (&inv)[ROWS], int rows, int width, bf16* xs) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int q = threadIdx.x + 512 * j;
        if (q >= width >> 2) continue;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = v[r][j][e] * inv[r] * n[j][e];
            if (r < rows) store_quad(xs + ((q >> 1) * rows + r) * 8 + 4 * (q & 1), o);
        }
    }
}
