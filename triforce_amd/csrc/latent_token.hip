// The per-layer token input of a few decode rows in bfloat16: gelu(x . Wg^T) * table[ids] and its projection back to the width, as two launches that share
// the reduction.
#include "tile_common.h"
#include "../../include/triforce_latent.h"

// The gate's 16 panels (side dimension 256) are 16 CUs' work in one launch of panels: 128 KB of weights each, at what one CU pulls 2.5 us.  Here K is cut into
// parts over the grid and every part leaves its fp32 sums; the projection, which reads them next, adds them up in every workgroup (PARTS * 4 bytes per row
// and side element, from L2), takes gelu and the table's row and goes on with its own 16 outputs.  us of the two, 4 096 -> 256 -> 4 096, before -> now,
// 1 / 8 rows: 9.1 -> 7.4, 9.9 -> 9.35.
constexpr int PARTS = 8, WAVES = 8;

__global__ __launch_bounds__(64 * WAVES) void token_parts_kernel(const bf16* __restrict__ wp, const bf16* __restrict__ x, int64_t ld_x, int64_t x_oct, float* __restrict__ part,
                                                                 int rows, int n, int chunks) {
    __shared__ f32x4 sums[WAVES][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
    const int panel = blockIdx.x, p = blockIdx.y;
    const int c_beg = chunks * p / PARTS, c_end = chunks * (p + 1) / PARTS, per = (c_end - c_beg + WAVES - 1) / WAVES;
    const int beg = c_beg + wave * per, end = min(c_end, beg + per);
    const bf16* w_at = wp + ((int64_t)panel * chunks) * 512 + lane * 8;
    const bf16* x_at = x + (int64_t)min(i, rows - 1) * ld_x + g * x_oct;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 4;
    for (int c0 = beg; c0 < end; c0 += U) {
        bf16x8 w[U], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = min(c0 + u, end - 1);
            w[u] = load_frag_stream(w_at + (int64_t)c * 512);
            v[u] = load_frag(x_at + 4 * x_oct * c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u < end) acc = El<bf16>::mma(w[u], v[u], acc);
    }
    sums[wave][lane] = acc;
    __syncthreads();
    if (wave > 0 || i >= rows) return;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
        const f32x4 o = sums[w][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += o[e];
    }
    *reinterpret_cast<f32x4*>(part + ((int64_t)p * rows + i) * n + 16 * panel + 4 * g) = acc;
}

__global__ __launch_bounds__(64 * WAVES) void token_project_kernel(const bf16* __restrict__ wp, const float* __restrict__ part, const bf16* __restrict__ table, int64_t ld_tok,
                                                                   const int64_t* __restrict__ ids, int vocab, float* __restrict__ out, int64_t ld_out, int rows, int side,
                                                                   int side_real, int n_real) {
    __shared__ f32x4 sums[WAVES][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
    const int panel = blockIdx.x, chunks = side >> 5, row = min(i, rows - 1);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int64_t id = ids[row];
    id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    for (int c = wave; c < chunks; c += WAVES) {
        const bf16x8 w = load_frag_stream(wp + ((int64_t)panel * chunks + c) * 512 + lane * 8);
        const int k0 = 32 * c + 8 * g;
        f32x4 z[PARTS][2];
#pragma unroll
        for (int p = 0; p < PARTS; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h) z[p][h] = *reinterpret_cast<const f32x4*>(part + ((int64_t)p * rows + row) * side + k0 + 4 * h);
        bf16 e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = table[id * ld_tok + min(k0 + j, side_real - 1)];
        bf16x8 x;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float s = z[0][j >> 2][j & 3];
#pragma unroll
            for (int p = 1; p < PARTS; ++p) s += z[p][j >> 2][j & 3];
            x[j] = (bf16)(k0 + j < side_real ? gelu_tanh(s) * (float)e[j] : 0.f);
        }
        acc = El<bf16>::mma(w, x, acc);
    }
    sums[wave][lane] = acc;
    __syncthreads();
    if (wave > 0 || i >= rows) return;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
        const f32x4 o = sums[w][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += o[e];
    }
    float* y = out + (int64_t)i * ld_out + 16 * panel + 4 * g;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (16 * panel + 4 * g + e < n_real) y[e] = acc[e];
}

extern "C" int64_t tfl_token_side_ws_floats(int rows, int side) { return rows < 1 || side < 1 ? 0 : (int64_t)PARTS * rows * side; }

extern "C" int tfl_token_side(const void* gate_packed, const void* proj_packed, const void* x, int64_t ld_x, int64_t x_oct, const void* table, int64_t ld_tok, const int64_t* ids,
                              int vocab, float* out, int64_t ld_out, float* ws, int64_t ws_floats, int rows, int width, int side, int side_real, int n_real, void* stream) {
    if (!gate_packed || !proj_packed || !x || !table || !ids || !out || !ws || rows < 1 || rows > 16 || width < 32 || (width & 31) || width > (1 << 20) || side < 32 || (side & 31)
        || side > 4096 || side_real < 1 || side_real > side || n_real < 1 || n_real > width || vocab < 1 || ld_tok < side_real || ld_out < n_real || ld_x < 8 || (ld_x & 7)
        || x_oct < 8 || (x_oct & 7) || !at16(gate_packed, proj_packed, x, ws)) return TF_EINVAL;
    if (ws_floats < tfl_token_side_ws_floats(rows, side)) return TF_ENOSPC;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(token_parts_kernel, dim3(side / 16, PARTS), dim3(64 * WAVES), 0, st, (const bf16*)gate_packed, (const bf16*)x, ld_x, x_oct, ws, rows, side, width / 32);
    TFL_LAUNCH_CHECK();
    hipLaunchKernelGGL(token_project_kernel, dim3(width / 16), dim3(64 * WAVES), 0, st, (const bf16*)proj_packed, ws, (const bf16*)table, ld_tok, ids, vocab, out, ld_out, rows, side,
                       side_real, n_real);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}
