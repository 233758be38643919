// Row kernels of the latent-attention family: residual / norm steps between layers, the prefill half of the input projection
// (norms, rotation, cache append, gelu), the per-layer token gate, and the cache-row gather.
#include "tile_common.h"

extern "C" int tfl_abi_version(void) { return 2; }

// PREP: a step's first launch, with decode_prep_row() of all rows as one more workgroup (a launch of its own is 4.3 us of a step of one row of 516).
template <typename T, typename Y, bool PREP = false>
__global__ __launch_bounds__(256) void finish_kernel(const T* __restrict__ embed, const int64_t* __restrict__ ids, int vocab,
                                                     const Y* __restrict__ y, int64_t ld_y, const float* __restrict__ y_w,
                                                     const float* __restrict__ step, const float* __restrict__ norm_w,
                                                     float* __restrict__ x, T* __restrict__ h, int64_t ld_h, int64_t h_oct,
                                                     int width, int width_real, float eps, const TflDecodePrep prep) {
    if constexpr (PREP) {
        if ((int)blockIdx.x == prep.rows) {
            for (int m = threadIdx.x; m < prep.rows; m += 256) decode_prep_row(prep, m);
            return;
        }
    }
    __shared__ float red[4];
    const int row = blockIdx.x, nq = width >> 2;             // elements in groups of 4
    float* xr = x + (int64_t)row * width;
    const T* er = nullptr;
    if (embed) {
        int64_t id = ids[row];
        id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
        er = embed + id * (int64_t)width;
    }
    const Y* yr = y ? y + (int64_t)row * ld_y : nullptr;
    float yi = 0.f;
    if (yr) {
        float s = 0.f;
        for (int q = threadIdx.x; q < nq; q += 256) {
            const f32x4 v = load_quad(yr + 4 * q);
            s += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        s = block_sum<4>(s, red);
        yi = 1.0f / sqrtf(s / (float)width_real + eps);
    }
    float s = 0.f;
    for (int q = threadIdx.x; q < nq; q += 256) {
        f32x4 v = er ? load_quad(er + 4 * q) : *reinterpret_cast<const f32x4*>(xr + 4 * q);
        if (yr) {
            const f32x4 z = load_quad(yr + 4 * q), w = *reinterpret_cast<const f32x4*>(y_w + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += z[r] * yi * w[r];
        }
        if (step) {
            const f32x4 z = *reinterpret_cast<const f32x4*>(step + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += z[r];
        }
        s += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        if (er || yr || step) *reinterpret_cast<f32x4*>(xr + 4 * q) = v;
    }
    s = block_sum<4>(s, red);
    const float inv = 1.0f / sqrtf(s / (float)width_real + eps);
    for (int q = threadIdx.x; q < nq; q += 256) {             // (each thread re-reads what it wrote itself)
        f32x4 v = *reinterpret_cast<const f32x4*>(xr + 4 * q);
        const f32x4 w = *reinterpret_cast<const f32x4*>(norm_w + 4 * q);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = v[r] * inv * w[r];
        store_quad(h + (int64_t)row * ld_h + (q >> 1) * h_oct + 4 * (q & 1), v);
    }
}

// The same for rows that fit a workgroup's registers (HOLD quads per thread of NW waves): everything is asked for at once and nothing
// is read twice, where the form above makes three passes whose loads wait for each other.  A decode row is a latency chain:
// sixteen waves with one quad a thread; a prompt's rows are a stream: four waves with four.  Rows of 4 096: 1 row 5.1 ->
// 3.9 us, 32 rows 5.4 -> 4.1, 4 000 rows 40.6 -> 33.4 (5.9 TB/s).  Narrow rows take no more waves than they have quads (4 000 rows of 192 with four
// times four 8.6 us, with one wave 4.3, in the form above 6.7); 4 000 rows of 1 025 to 2 048, which leave half the four quads empty, are
// faster above (2 048 16.5 us and 18.6).
template <typename T, typename Y, int NW, int HOLD, bool PREP = false>
__global__ __launch_bounds__(64 * NW) void finish_row_kernel(const T* __restrict__ embed, const int64_t* __restrict__ ids, int vocab,
                                                             const Y* __restrict__ y, int64_t ld_y, const float* __restrict__ y_w,
                                                             const float* __restrict__ step, const float* __restrict__ norm_w,
                                                             float* __restrict__ x, T* __restrict__ h, int64_t ld_h, int64_t h_oct,
                                                             int width, int width_real, float eps, const TflDecodePrep prep) {
    if constexpr (PREP) {
        if ((int)blockIdx.x == prep.rows) {
            for (int m = threadIdx.x; m < prep.rows; m += 64 * NW) decode_prep_row(prep, m);
            return;
        }
    }
    __shared__ float red[NW];
    const int row = blockIdx.x, nq = width >> 2;
    float* xr = x + (int64_t)row * width;
    const T* er = nullptr;
    if (embed) {
        int64_t id = ids[row];
        id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
        er = embed + id * (int64_t)width;
    }
    const Y* yr = y ? y + (int64_t)row * ld_y : nullptr;
    f32x4 v[HOLD], z[HOLD], w[HOLD];
    // one quad a thread (few rows): nothing is left to be asked for behind a sum
    constexpr bool EARLY = HOLD == 1;
    f32x4 t0 = {0.f, 0.f, 0.f, 0.f}, n0 = {0.f, 0.f, 0.f, 0.f};
    if (EARLY && (int)threadIdx.x < nq) {
        if (step) t0 = *reinterpret_cast<const f32x4*>(step + 4 * threadIdx.x);
        n0 = *reinterpret_cast<const f32x4*>(norm_w + 4 * threadIdx.x);
    }
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < HOLD; ++j) {
        const int q = threadIdx.x + 64 * NW * j;
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        v[j] = z[j] = w[j] = zero;
        if (q < nq) {
            if (yr) z[j] = load_quad(yr + 4 * q);
            v[j] = er ? load_quad(er + 4 * q) : *reinterpret_cast<const f32x4*>(xr + 4 * q);
            if (yr) w[j] = *reinterpret_cast<const f32x4*>(y_w + 4 * q);
        }
    }
    float yi = 0.f;
    if (yr) {
#pragma unroll
        for (int j = 0; j < HOLD; ++j) s += z[j][0] * z[j][0] + z[j][1] * z[j][1] + z[j][2] * z[j][2] + z[j][3] * z[j][3];
        yi = 1.0f / sqrtf(block_sum<NW>(s, red) / (float)width_real + eps);
        s = 0.f;
    }
#pragma unroll
    for (int j = 0; j < HOLD; ++j) {
        const int q = threadIdx.x + 64 * NW * j;
        if (yr) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[j][r] += z[j][r] * yi * w[j][r];
        }
        if (q < nq) {
            if (step) {
                const f32x4 t = EARLY ? t0 : *reinterpret_cast<const f32x4*>(step + 4 * q);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[j][r] += t[r];
            }
            if (er || yr || step) *reinterpret_cast<f32x4*>(xr + 4 * q) = v[j];
            w[j] = EARLY ? n0 : *reinterpret_cast<const f32x4*>(norm_w + 4 * q);
        }
        s += v[j][0] * v[j][0] + v[j][1] * v[j][1] + v[j][2] * v[j][2] + v[j][3] * v[j][3];
    }
    const float inv = 1.0f / sqrtf(block_sum<NW>(s, red) / (float)width_real + eps);
#pragma unroll
    for (int j = 0; j < HOLD; ++j) {
        const int q = threadIdx.x + 64 * NW * j;
        if (q >= nq) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[j][r] = v[j][r] * inv * w[j][r];
        store_quad(h + (int64_t)row * ld_h + (q >> 1) * h_oct + 4 * (q & 1), v[j]);
    }
}

static int finish(const void* embed, const int64_t* ids, int vocab, const void* y, int y_f32, int64_t ld_y,
                          const float* y_w, const float* step, const float* norm_w, float* x, void* h, int64_t ld_h, int64_t h_oct,
                          int rows, int width, int width_real, float eps, const TflDecodePrep* prep, int dtype, void* stream) {
    if (!x || !h || !norm_w || rows < 1 || width < 8 || (width & 7) || ld_h < 8 || (ld_h & 7) || h_oct < 8 || (h_oct & 7) || width_real < 1 || width_real > width) return TF_EINVAL;
    if (embed && (!ids || vocab < 1)) return TF_EINVAL;
    if (y && (!y_w || ld_y < width || (ld_y & 3))) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const TflDecodePrep d = prep ? *prep : TflDecodePrep{};
#define ARGS(T, Y) 0, st, (const T*)embed, ids, vocab, (const Y*)y, ld_y, y_w, step, norm_w, x, (T*)h, ld_h, h_oct, width, width_real, eps, d
#define GO(T, Y, PREP)                                                                                                                              \
    do {                                                                                                                                      \
        if (width > 4096 || (width > 1024 && width <= 2048 && rows > 1024)) hipLaunchKernelGGL((finish_kernel<T, Y, PREP>), dim3(rows + PREP), dim3(256), ARGS(T, Y)); \
        else if (width <= 256) hipLaunchKernelGGL((finish_row_kernel<T, Y, 1, 1, PREP>), dim3(rows + PREP), dim3(64), ARGS(T, Y));                          \
        else if (width <= 1024) hipLaunchKernelGGL((finish_row_kernel<T, Y, 4, 1, PREP>), dim3(rows + PREP), dim3(256), ARGS(T, Y));                        \
        else if (rows <= 256) hipLaunchKernelGGL((finish_row_kernel<T, Y, 16, 1, PREP>), dim3(rows + PREP), dim3(1024), ARGS(T, Y));  /* a row per CU */    \
        else hipLaunchKernelGGL((finish_row_kernel<T, Y, 4, 4, PREP>), dim3(rows + PREP), dim3(256), ARGS(T, Y));                                          \
    } while (0)
    if (prep) { if (dtype == 0) GO(bf16, bf16, true); else if (dtype == 1) GO(float, float, true); else return TF_EINVAL; }
    else if (dtype == 0) { if (y_f32) GO(bf16, float, false); else GO(bf16, bf16, false); }
    else if (dtype == 1) GO(float, float, false);
    else return TF_EINVAL;
#undef GO
#undef ARGS
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tfl_finish(const void* embed, const int64_t* ids, int vocab, const void* y, int y_f32, int64_t ld_y,
                          const float* y_w, const float* step, const float* norm_w, float* x, void* h, int64_t ld_h, int64_t h_oct,
                          int rows, int width, int width_real, float eps, int dtype, void* stream) {
    return finish(embed, ids, vocab, y, y_f32, ld_y, y_w, step, norm_w, x, h, ld_h, h_oct, rows, width, width_real, eps, nullptr, dtype, stream);
}

extern "C" int tfl_finish_first(const void* embed, const int64_t* ids, int vocab, const float* step, const float* norm_w, float* x, void* h, int64_t ld_h, int64_t h_oct,
                                int rows, int width, int width_real, float eps, const TflDecodePrep* prep, int dtype, void* stream) {
    if (!embed || !decode_prep_ok(prep, rows)) return TF_EINVAL;
    return finish(embed, ids, vocab, nullptr, 0, 0, nullptr, step, norm_w, x, h, ld_h, h_oct, rows, width, width_real, eps, prep, dtype, stream);
}

template <typename T>
__global__ __launch_bounds__(256) void residual_kernel(const T* __restrict__ d, float* __restrict__ x, T* __restrict__ xt,
                                                       int64_t nq) {
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < nq; q += (int64_t)gridDim.x * 256) {
        f32x4 v = *reinterpret_cast<const f32x4*>(x + 4 * q);
        const f32x4 z = load_quad(d + 4 * q);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += z[r];
        *reinterpret_cast<f32x4*>(x + 4 * q) = v;
        if (xt) store_quad(xt + 4 * q, v);
    }
}

extern "C" int tfl_residual(const void* d, float* x, void* xt, int64_t n, int dtype, void* stream) {
    if (!d || !x || n < 4 || (n & 3)) return TF_EINVAL;
    const int64_t nq = n / 4;
    const unsigned gx = (unsigned)((nq + 255) / 256 < 4096 ? (nq + 255) / 256 : 4096);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == 0) hipLaunchKernelGGL((residual_kernel<bf16>), dim3(gx), dim3(256), 0, st, (const bf16*)d, x, (bf16*)xt, nq);
    else if (dtype == 1) hipLaunchKernelGGL((residual_kernel<float>), dim3(gx), dim3(256), 0, st, (const float*)d, x, (float*)xt, nq);
    else return TF_EINVAL;
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

template <typename T>
__global__ __launch_bounds__(256) void token_gate_kernel(const T* __restrict__ s, int64_t ld_s, const T* __restrict__ table,
                                                         int64_t ld_tok, const int64_t* __restrict__ ids, int vocab,
                                                         T* __restrict__ out, int n, int n_real) {
    const int row = blockIdx.x;
    int64_t id = ids[row];
    id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    for (int c = threadIdx.x; c < n; c += 256)
        out[(int64_t)row * n + c] = c < n_real ? (T)(gelu_tanh((float)s[(int64_t)row * ld_s + c]) * (float)table[id * ld_tok + c]) : (T)0.f;
}

extern "C" int tfl_token_gate(const void* s, int64_t ld_s, const void* table, int64_t ld_tok, const int64_t* ids, int vocab,
                              void* out, int rows, int n, int n_real, int dtype, void* stream) {
    if (!s || !table || !ids || !out || rows < 1 || n < 1 || n_real < 1 || n_real > n || ld_s < n || ld_tok < n_real || vocab < 1)
        return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
#define GO(T) hipLaunchKernelGGL((token_gate_kernel<T>), dim3(rows), dim3(256), 0, st, (const T*)s, ld_s, (const T*)table, ld_tok, \
                                 ids, vocab, (T*)out, n, n_real)
    if (dtype == 0) GO(bf16);
    else if (dtype == 1) GO(float);
    else return TF_EINVAL;
#undef GO
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// One workgroup per new token.
// Workgroups (row, 0) do the two norms, the rotation and the cache row - a chain of two reductions -, (row, 1) the gelu of the row's
// feed-forward part, a stream of 16-byte pieces: one after the other in one workgroup, with expf and a division per element, 4 000
// rows of 1 536 | 512 | 64 | 11 008 took 53.6 us, now 39.9 (214 MB: 5.4 TB/s).
template <typename T, int EPP>
__global__ __launch_bounds__(256) void prepare_kernel(const T* __restrict__ y, int64_t ld_y, int q, int q_real, int C, int c_real,
                                                      int R, int up_off, int n_up, const float* __restrict__ q_norm,
                                                      const float* __restrict__ kv_norm, float eps, const float* __restrict__ cosb,
                                                      const float* __restrict__ sinb, int half, int max_pos,
                                                      const int32_t* __restrict__ pos, const int32_t* __restrict__ slot,
                                                      T* __restrict__ cache, int cache_rows, T* __restrict__ cq, T* __restrict__ ck,
                                                      T* __restrict__ act, int64_t ld_act) {
    __shared__ float red[4];
    const int row = blockIdx.x;
    const T* yr = y + (int64_t)row * ld_y;
    if (blockIdx.y == 1) {
        typedef T Piece __attribute__((ext_vector_type(EPP)));
        const T* src = yr + up_off;
        T* dst = act + (int64_t)row * ld_act;
#pragma unroll 4
        for (int c = threadIdx.x; c < n_up / EPP; c += 256) {
            Piece v = *reinterpret_cast<const Piece*>(src + EPP * c);
#pragma unroll
            for (int e = 0; e < EPP; ++e) v[e] = (T)gelu_of<T>((float)v[e]);
            *reinterpret_cast<Piece*>(dst + EPP * c) = v;
        }
        return;
    }
    float s = 0.f;
    for (int c = threadIdx.x; c < q / 4; c += 256) {
        const f32x4 v = load_quad(yr + 4 * c);
        s += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    s = block_sum<4>(s, red);
    const float inv = 1.0f / sqrtf(s / (float)q_real + eps);
    for (int c = threadIdx.x; c < q / 4; c += 256) {
        f32x4 v = load_quad(yr + 4 * c);
        const f32x4 w = *reinterpret_cast<const f32x4*>(q_norm + 4 * c);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = v[r] * inv * w[r];
        store_quad(cq + (int64_t)row * q + 4 * c, v);
    }
    int p = pos[row];
    p = p < 0 ? 0 : (p >= max_pos ? max_pos - 1 : p);
    const int sl = slot[row], W = C + R;
    const T* kv = yr + q;
    cache_row<T, 4>([kv](int c) { return (float)kv[c]; }, C, c_real, R, kv_norm, eps, cosb + (int64_t)p * half,
                     sinb + (int64_t)p * half, half, sl >= 0 && sl < cache_rows ? cache + (int64_t)sl * W : (T*)nullptr,
                     ck ? ck + (int64_t)row * W : (T*)nullptr, red);
}

extern "C" int tfl_prepare(const void* y, int64_t ld_y, int q, int q_real, int C, int c_real, int R, int up_off, int n_up,
                           const float* q_norm, const float* kv_norm, float eps, const float* cosb, const float* sinb, int half,
                           int max_pos, const int32_t* pos, const int32_t* slot, void* cache, int cache_rows, void* cq, void* ck,
                           void* act, int64_t ld_act, int rows, int dtype, void* stream) {
    if (!y || !q_norm || !kv_norm || !pos || !slot || !cache || !cq || rows < 1 || cache_rows < 1) return TF_EINVAL;
    if (q < 4 || (q & 3) || q_real < 1 || q_real > q || C < 4 || (C & 3) || c_real < 1 || c_real > C || R < 0 || (R & 3)) return TF_EINVAL;
    if (ld_y < q + C + R || (ld_y & 3) || half < 0 || 2 * half > R || max_pos < 1 || (half && (!cosb || !sinb))) return TF_EINVAL;
    if (n_up < 0 || (n_up & 3) || (n_up && (!act || (ld_act & 3) || ld_act < n_up || (up_off & 3) || up_off < q + C + R || ld_y < up_off + n_up)))
        return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
#define GO(T, EPP) hipLaunchKernelGGL((prepare_kernel<T, EPP>), dim3(rows, n_up ? 2 : 1), dim3(256), 0, st, (const T*)y, ld_y, q, q_real, C,  \
                                      c_real, R, up_off, n_up, q_norm, kv_norm, eps, cosb, sinb, half, max_pos, pos, slot, (T*)cache,    \
                                      cache_rows, (T*)cq, (T*)ck, (T*)act, ld_act)
    // 16-byte pieces where every row's part starts on one
    const bool octets = !((n_up | up_off | ld_y | ld_act) & 7) && !(((uintptr_t)y | (uintptr_t)act) & 15);
    if (dtype == 0) { if (octets) GO(bf16, 8); else GO(bf16, 4); }
    else if (dtype == 1) GO(float, 4);
    else return TF_EINVAL;
#undef GO
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// 16-byte pieces; a row is ppr of them.
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint4* __restrict__ cache, int cache_rows,
                                                          const int32_t* __restrict__ src, uint4* __restrict__ dst, int rows, int ppr) {
    const int64_t total = (int64_t)rows * ppr;
    for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < total; p += (int64_t)gridDim.x * 256) {
        const int64_t r = p / ppr;
        int s = src[r];
        s = s < 0 ? 0 : (s >= cache_rows ? cache_rows - 1 : s);
        dst[p] = cache[(int64_t)s * ppr + (p - r * ppr)];
    }
}

extern "C" int tfl_gather_rows(const void* cache, int cache_rows, const int32_t* src, void* dst, int rows, int W, int dtype, void* stream) {
    if (!cache || !src || !dst || rows < 1 || cache_rows < 1 || W < 8 || (W & 7) || (dtype != 0 && dtype != 1)) return TF_EINVAL;
    const int ppr = W * (dtype ? 4 : 2) / 16;
    const int64_t total = (int64_t)rows * ppr;
    const unsigned gx = (unsigned)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192);
    hipLaunchKernelGGL(gather_rows_kernel, dim3(gx), dim3(256), 0, (hipStream_t)stream, (const uint4*)cache, cache_rows, src,
                       (uint4*)dst, rows, ppr);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}
