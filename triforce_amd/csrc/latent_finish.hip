// Residual bookkeeping and norm of a few decode rows inside the wide product that reads them (bfloat16).
#include "tile_common.h"
#include "share_gemm.h"
#include "share_shape.h"
#include "row_source.h"
#include "../../include/triforce_latent.h"

// The row step between two layers (finish_row_kernel in latent_ops.hip) as a product's source of x: rows of up to 4 096, two quads a thread.
// A launch of its own is 4.2 us of round trips in which memory idles; here they run under the first 160 KB of weights of every CU, in every workgroup for
// itself.  17 216 x 4 096, one row, apart -> together: 4.2 + 24.8 -> 26.4 us; eight steps of six layer runs, 1 / 2 rows 4 403 -> 4 279, 4 607 -> 4 521; with 3 and 4
// rows it takes longer than the launch that it saves (4 704 -> 4 761, 4 756 -> 4 834).
template <int ROWS>
struct FinishSource {
    static constexpr bool INSIDE = true, SCALED = false, TILE = false, ALSO = false;
    const TflFinish& f;
    bf16* xs;                                                 // [width / 8][rows][8]
    float* red;                                               // [2][ROWS][8]
    int rows, groups;
    f32x4 x[ROWS][2], y[ROWS][2], w[2], t[2], n[2];

    __device__ __forceinline__ FinishSource(const TflFinish& f_, bf16* xs_, float* red_, int rows_, int groups_)
        : f(f_), xs(xs_), red(red_), rows(rows_), groups(groups_) {}
    __device__ __forceinline__ int quad(int j) const { return min((int)threadIdx.x + 512 * j, (f.width >> 2) - 1); }
    __device__ __forceinline__ void ask() {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = 4 * quad(j);
#pragma unroll
            for (int r = 0; r < ROWS; ++r) y[r][j] = *reinterpret_cast<const f32x4*>(f.y + min(r, rows - 1) * f.ld_y + q);
#pragma unroll
            for (int r = 0; r < ROWS; ++r) x[r][j] = *reinterpret_cast<const f32x4*>(f.x + (int64_t)min(r, rows - 1) * f.width + q);
            w[j] = *reinterpret_cast<const f32x4*>(f.y_w + q);
            t[j] = f.step ? *reinterpret_cast<const f32x4*>(f.step + q) : f32x4{0.f, 0.f, 0.f, 0.f};
            n[j] = *reinterpret_cast<const f32x4*>(f.norm_w + q);
        }
    }
    __device__ __forceinline__ const bf16* make(int cu) {
        float inv[ROWS];
        rows_inverse<ROWS>(y, f.width, f.width_real, f.eps, red, inv);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = threadIdx.x + 512 * j;
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[r][j][e] += y[r][j][e] * inv[r] * w[j][e];
                if (f.step)
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[r][j][e] += t[j][e];
                if (q < f.width >> 2 && q % groups == cu && r < rows) *reinterpret_cast<f32x4*>(f.x_out + (int64_t)r * f.width + 4 * q) = x[r][j];
            }
        }
        rows_inverse<ROWS>(x, f.width, f.width_real, f.eps, red + 8 * ROWS, inv);
        rows_normed<ROWS>(x, n, inv, rows, f.width, xs);
        __syncthreads();
        return xs;
    }
};

template <int EPI, int P, bool TAIL, int ROWS, int U>
__global__ __launch_bounds__(512, 2) void finish_gemm_kernel(const TflFinish f, const TflGemm a, const int tail_rows, const int tail_per) {
    extern __shared__ __align__(16) char smem[];
    constexpr int PARTS = 8 * (P + (TAIL ? 1 : 0)) * 64 * (int)sizeof(f32x4);
    float* red = reinterpret_cast<float*>(smem + PARTS);
    bf16* xs = reinterpret_cast<bf16*>(red + 16 * ROWS);
    share_gemm_body<bf16, EPI, P, TAIL, 1, U, FinishSource<ROWS>>(a, tail_rows, tail_per, blockIdx.x, 0, smem,
                                                                  FinishSource<ROWS>(f, xs, red, a.rows, gridDim.x));
}

template <int EPI, int P, bool TAIL, int ROWS>
static int launch_finish_rows(const TflFinish& f, const TflGemm& a, const ShareShape& s, hipStream_t st) {
    constexpr int NP = P + (TAIL ? 1 : 0), U = 2, PARTS = 8 * NP * 64 * (int)sizeof(f32x4);
    const int lds = PARTS + 16 * ROWS * (int)sizeof(float) + 2 * a.rows * f.width;
    auto* k = finish_gemm_kernel<EPI, P, TAIL, ROWS, U>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(k, dim3(TAIL ? 256 : ((a.n >> 4) + P - 1) / P), dim3(512), lds, st, f, a, s.left, s.rest);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

template <int EPI, int P, bool TAIL>
static int launch_finish(const TflFinish& f, const TflGemm& a, const ShareShape& s, hipStream_t st) {
    return a.rows == 1 ? launch_finish_rows<EPI, P, TAIL, 1>(f, a, s, st) : launch_finish_rows<EPI, P, TAIL, 2>(f, a, s, st);
}

static ShareShape finish_shape(int rows, int width, int n, int k, int epi, int n_raw) {
    if (rows < 1 || rows > 2 || width < 2048 || width > 4096 || (width & 31) || k != width || n < 16 || (n & 15) || n > (1 << 20)
        || (epi != TFL_EPI_IN && epi != TFL_EPI_F32)) return {0, 0, 0};
    const ShareShape s = share_shape(n >> 4, false, epi == TFL_EPI_IN ? n_raw : 0, rows);
    return s.each >= 3 ? s : ShareShape{0, 0, 0};             // (a shorter stream does not cover the rows)
}

template <int EPI>
static int finish_gemm(const TflFinish& f, const TflGemm& a, hipStream_t st) {
    const ShareShape s = finish_shape(a.rows, f.width, a.n, a.k, EPI, a.n_raw);
    if (s.rest) switch (s.each) {
        case 3: return launch_finish<EPI, 3, true>(f, a, s, st);
        case 4: return launch_finish<EPI, 4, true>(f, a, s, st);
        case 5: return launch_finish<EPI, 5, true>(f, a, s, st);
        case 6: return launch_finish<EPI, 6, true>(f, a, s, st);
        case 7: return launch_finish<EPI, 7, true>(f, a, s, st);
        default: return TF_ERANGE;
    }
    switch (s.each) {
        case 3: return launch_finish<EPI, 3, false>(f, a, s, st);
        case 4: return launch_finish<EPI, 4, false>(f, a, s, st);
        case 5: return launch_finish<EPI, 5, false>(f, a, s, st);
        case 6: return launch_finish<EPI, 6, false>(f, a, s, st);
        case 7: return launch_finish<EPI, 7, false>(f, a, s, st);
        case 8: return launch_finish<EPI, 8, false>(f, a, s, st);
        default: return TF_ERANGE;
    }
}

extern "C" int tfl_finish_gemm_takes(int rows, int width, int n, int k, int epilogue, int n_raw) {
    return finish_shape(rows, width, n, k, epilogue, n_raw).each > 0 ? 1 : 0;
}

extern "C" int tfl_finish_gemm(const TflFinish* pf, const TflGemm* pa, int epilogue, void* stream) {
    if (!pf || !pa || !pa->wp || !pf->y || !pf->y_w || !pf->norm_w || !pf->x || !pf->x_out || pf->x == pf->x_out) return TF_EINVAL;
    const TflFinish f = *pf;
    const TflGemm a = *pa;
    if (a.rows < 1 || a.groups != 1 || a.chunk_major != 1 || f.width < 4 || (f.width & 3) || f.width_real < 1 || f.width_real > f.width || f.ld_y < f.width
        || (f.ld_y & 3) || !a.out_f || (a.n & 15) || a.n < 16 || !at16(a.wp, f.y, f.y_w, f.step, f.norm_w, f.x, f.x_out)) return TF_EINVAL;
    if (epilogue == TFL_EPI_F32) {
        if (a.n_real < 1 || a.n_real > a.n || a.ld_f < a.n_real) return TF_EINVAL;
        return finish_gemm<TFL_EPI_F32>(f, a, (hipStream_t)stream);
    }
    if (epilogue != TFL_EPI_IN || !a.ss_out || !at16(a.out_f, a.out_t, a.out_t2, a.norm_w) || a.n_raw < 16 || (a.n_raw & 15) || a.n_raw > a.n || a.ld_f < a.n_raw || (a.ld_f & 3) || a.ss_ld < a.n_raw / 16
        || a.n_scaled < 0 || (a.n_scaled & 15) || a.n_scaled > a.n_raw || (a.n_scaled && (!a.norm_w || !a.out_t2))
        || (a.n_raw < a.n && (!a.out_t || a.t_oct < 8 || (a.t_oct & 7) || (a.ld_t & 7) || a.ld_t < 8))) return TF_EINVAL;
    return finish_gemm<TFL_EPI_IN>(f, a, (hipStream_t)stream);
}
