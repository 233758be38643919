// Residual streams and norm of a few decode rows inside the wide product that reads them (bfloat16).
#include "hybrid_common.h"
#include "share_gemm.h"
#include "share_shape.h"
#include "row_source.h"

// connect_kernel (hybrid_ops.hip) between two sublayers as a product's source of x: up to S streams of a row of up to 4 096.  It serves widths whose last products
// are not whole panels of every CU, 2 048 to 4 064 (4 096 is, see hybrid_streams.hip).
// A launch of its own is 5 us of round trips in which memory idles; here they run under the first 160 KB of weights of every CU.  One row, twelve layers of a parallel
// mixer and a gated unit, four streams, a step apart -> together: width 2 048 704 -> 688 us, 2 560 863 -> 829, 3 072 1 028 -> 981, 3 584 1 218 -> 1 185; one stream of
// 3 072 1 015 -> 970.  Two rows of four streams are 160 KB for every workgroup and take longer than the launch that they save.
template <int S>
struct ConnectSource {
    static constexpr bool INSIDE = true, SCALED = false, TILE = false, ALSO = false;
    static constexpr int ROWS = 1;
    const TfhConnect& f;
    bf16* xs;                                                 // [width / 8][rows][8]
    float* red;                                               // [ROWS][8]
    int rows, groups;
    f32x4 x[ROWS][S][2], u[ROWS][2], n[2];                    // (u: the sublayer's result, then the next one's input)

    __device__ __forceinline__ ConnectSource(const TfhConnect& f_, bf16* xs_, float* red_, int rows_, int groups_)
        : f(f_), xs(xs_), red(red_), rows(rows_), groups(groups_) {}
    __device__ __forceinline__ void ask() {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = 4 * min((int)threadIdx.x + 512 * j, (f.width >> 2) - 1);
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const int row = min(r, rows - 1);
#pragma unroll
                for (int s = 0; s < S; ++s) x[r][s][j] = *reinterpret_cast<const f32x4*>(f.x + ((int64_t)row * f.streams + min(s, f.streams - 1)) * f.width + q);
                u[r][j] = *reinterpret_cast<const f32x4*>(f.y + row * f.ld_y + q);
            }
            n[j] = *reinterpret_cast<const f32x4*>(f.norm_w + q);
        }
    }
    __device__ __forceinline__ const bf16* make(int cu) {
        float mix[S][S], out[S], in[S];
#pragma unroll
        for (int t = 0; t < S; ++t) {
            const int ct = min(t, f.streams - 1);
            out[t] = t < f.streams ? f.out[ct] : 0.f;
            in[t] = t < f.streams ? f.in[ct] : 0.f;
#pragma unroll
            for (int s = 0; s < S; ++s) mix[s][t] = s < f.streams && t < f.streams ? f.mix[min(s, f.streams - 1) * f.streams + ct] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = threadIdx.x + 512 * j;
            const bool mine = f.x_out && q < f.width >> 2 && q % groups == cu;
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const f32x4 y = u[r][j];
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < S; ++t) {
                    f32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = out[t] * y[e];
#pragma unroll
                    for (int s = 0; s < S; ++s)
                        if (s < f.streams)                    // (what stands for a stream that is not there may be anything)
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[e] = fmaf(mix[s][t], x[r][s][j][e], v[e]);
                    if (mine && r < rows && t < f.streams) *reinterpret_cast<f32x4*>(f.x_out + ((int64_t)r * f.streams + t) * f.width + 4 * q) = v;
                    if (t < f.streams)
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum[e] = fmaf(in[t], v[e], sum[e]);
                }
                u[r][j] = sum;
            }
        }
        float inv[ROWS];
        rows_inverse<ROWS>(u, f.width, f.width_real, f.eps, red, inv);
        rows_normed<ROWS>(u, n, inv, rows, f.width, xs);
        __syncthreads();
        return xs;
    }
};

template <int EPI, int P, bool TAIL>
__global__ __launch_bounds__(512, 2) void connect_gemm_kernel(const TfhConnect f, const TflGemm a, const int tail_rows, const int tail_per) {
    extern __shared__ __align__(16) char smem[];
    constexpr int PARTS = 8 * (P + (TAIL ? 1 : 0)) * 64 * (int)sizeof(f32x4);
    float* red = reinterpret_cast<float*>(smem + PARTS);
    bf16* xs = reinterpret_cast<bf16*>(red + 8);
    share_gemm_body<bf16, EPI, P, TAIL, 1, 2, ConnectSource<4>>(a, tail_rows, tail_per, blockIdx.x, 0, smem,
                                                                      ConnectSource<4>(f, xs, red, a.rows, gridDim.x));
}

template <int EPI, int P, bool TAIL>
static int launch_connect(const TfhConnect& f, const TflGemm& a, const ShareShape& s, hipStream_t st) {
    constexpr int PARTS = 8 * (P + (TAIL ? 1 : 0)) * 64 * (int)sizeof(f32x4);
    const int lds = PARTS + 8 * (int)sizeof(float) + 2 * f.width;
    auto* k = connect_gemm_kernel<EPI, P, TAIL>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(k, dim3(TAIL ? 256 : ((a.n >> 4) + P - 1) / P), dim3(512), lds, st, f, a, s.left, s.rest);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

static ShareShape connect_shape(int rows, int streams, int width, int n, int k, int epi) {
    if (rows != 1 || streams < 1 || streams > 4 || width < 2048 || width > 4096 || (width & 31) || k != width || n < 16 || (n & 15) || n > (1 << 20)
        || (epi != TFL_EPI_GLU && epi != TFL_EPI_F32)) return {0, 0, 0};
    const ShareShape s = share_shape(n >> 4, epi == TFL_EPI_GLU, 0, rows);
    return s.each >= 3 ? s : ShareShape{0, 0, 0};             // (a shorter stream does not cover the rows)
}

template <int EPI>
static int connect_gemm(const TfhConnect& f, const TflGemm& a, hipStream_t st) {
    const ShareShape s = connect_shape(a.rows, f.streams, f.width, a.n, a.k, EPI);
    if (s.rest) switch (s.each) {
        case 3: return launch_connect<EPI, 3, true>(f, a, s, st);
        case 4: return launch_connect<EPI, 4, true>(f, a, s, st);
        case 5: return launch_connect<EPI, 5, true>(f, a, s, st);
        case 6: return launch_connect<EPI, 6, true>(f, a, s, st);
        case 7: return launch_connect<EPI, 7, true>(f, a, s, st);
        default: return TF_ERANGE;
    }
    switch (s.each) {
        case 3: return launch_connect<EPI, 3, false>(f, a, s, st);
        case 4: return launch_connect<EPI, 4, false>(f, a, s, st);
        case 5: return launch_connect<EPI, 5, false>(f, a, s, st);
        case 6: return launch_connect<EPI, 6, false>(f, a, s, st);
        case 7: return launch_connect<EPI, 7, false>(f, a, s, st);
        case 8: return launch_connect<EPI, 8, false>(f, a, s, st);
        default: return TF_ERANGE;
    }
}

extern "C" int tfh_connect_gemm_takes(int rows, int streams, int width, int n, int k, int epilogue) {
    return connect_shape(rows, streams, width, n, k, epilogue).each > 0 ? 1 : 0;
}

extern "C" int tfh_connect_gemm(const TfhConnect* pf, const TflGemm* pa, int epilogue, void* stream) {
    if (!pf || !pa || !pa->wp || !pf->y || !pf->out || !pf->mix || !pf->in || !pf->norm_w || !pf->x || pf->x == pf->x_out) return TF_EINVAL;
    const TfhConnect f = *pf;
    const TflGemm a = *pa;
    if (a.rows < 1 || a.groups != 1 || a.chunk_major != 1 || f.width < 4 || (f.width & 3) || f.width_real < 1 || f.width_real > f.width || f.ld_y < f.width
        || (f.ld_y & 3) || (a.n & 15) || a.n < 16 || !at16(a.wp, f.y, f.norm_w, f.x, f.x_out)) return TF_EINVAL;
    if (epilogue == TFL_EPI_F32) {
        if (!a.out_f || a.n_real < 1 || a.n_real > a.n || a.ld_f < a.n_real) return TF_EINVAL;
        return connect_gemm<TFL_EPI_F32>(f, a, (hipStream_t)stream);
    }
    if (epilogue != TFL_EPI_GLU || !a.out_t || !at16(a.out_t) || a.ld_t < 8 || (a.ld_t & 7) || a.t_oct < 8 || (a.t_oct & 7)) return TF_EINVAL;
    return connect_gemm<TFL_EPI_GLU>(f, a, (hipStream_t)stream);
}
