// Residual streams between two sublayers of a decode step without a launch of their own (bfloat16): the product that makes a sublayer's result brings the streams
// on, and leaves the next sublayer's input without its norm's scale and the sums of squares of which the next product makes that.
#include "hybrid_common.h"
#include "share_gemm.h"
#include "share_shape.h"

// What connect_kernel (hybrid_ops.hip) does to four outputs of a row, in the epilogue of the product: the streams there are asked for in front of the weights.
// A launch between two products is 4 to 5 us of round trips in which memory idles, whatever the rows; here its loads come under the weights, its stores are the
// product's own, and the row's scale, the one thing that needs all of the row, waits until behind the next product (the input's rounding to bfloat16 is
// relative, so it may come before the scale).  us of eight steps of four layers of 4 096 x 4 streams, apart -> so: 1 row (made inside the readers, see
// hybrid_connect.hip) 3 670 -> 3 609, 2 3 906 -> 3 680, 4 3 943 -> 3 716, 8 4 891 -> 4 603, 16 5 429 -> 5 147, 32 6 940 -> 6 641, 48 9 574 -> 9 445, 64 10 019 -> 9 893.
template <int S>
struct StreamsTile {
    static constexpr bool INSIDE = false, SCALED = false, TILE = true, ALSO = false;
    const TfhConnect& f;
    const TflGemm& a;
    f32x4 x[S], w;
    float mix[S][S], out[S], in[S];

    __device__ __forceinline__ StreamsTile(const TfhConnect& f_, const TflGemm& a_) : f(f_), a(a_) {}
    __device__ __forceinline__ const float* at(int m, int n, int s) const { return f.x + ((int64_t)m * f.streams + s) * f.width + n; }
    __device__ __forceinline__ void ask_tile(int m, int n) {
        n = min(n, f.width - 4);
#pragma unroll
        for (int s = 0; s < S; ++s) x[s] = *reinterpret_cast<const f32x4*>(at(m, n, min(s, f.streams - 1)));
        w = *reinterpret_cast<const f32x4*>(f.norm_w + n);
#pragma unroll
        for (int t = 0; t < S; ++t) {
            const int ct = min(t, f.streams - 1);
            out[t] = f.out[ct];
            in[t] = f.in[ct];
#pragma unroll
            for (int s = 0; s < S; ++s) mix[s][t] = f.mix[min(s, f.streams - 1) * f.streams + ct];
        }
    }
    __device__ __forceinline__ void put_tile(int m, bool live, int panel, int panels, int g, f32x4 y) {
        if (panel >= panels) return;
        const int n = 16 * panel + 4 * g;
        f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < S; ++t) {
            if (t >= f.streams) continue;
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = out[t] * y[e];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                if (s >= f.streams) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = fmaf(mix[s][t], x[s][e], v[e]);
            }
            if (live && f.x_out) *reinterpret_cast<f32x4*>(f.x_out + ((int64_t)m * f.streams + t) * f.width + n) = v;
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] = fmaf(in[t], v[e], u[e]);
        }
        float q = u[0] * u[0] + u[1] * u[1] + u[2] * u[2] + u[3] * u[3];
        q = rows_sum(q);
        if (!live) return;
        if (g == 0) a.ss_out[(int64_t)m * a.ss_ld + panel] = q;
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] *= w[e];
        store_quad((bf16*)a.out_t + (int64_t)m * a.ld_t + (n >> 3) * a.t_oct + (n & 7), u);
    }
};

template <int P, int MT>
__global__ __launch_bounds__(512, 2) void streams_gemm_kernel(const TfhConnect f, const TflGemm a) {
    extern __shared__ __align__(16) char smem[];
    share_gemm_body<bf16, TFL_EPI_F32, P, false, MT, P == 1 ? 4 : 2, StreamsTile<4>>(a, 0, 0, blockIdx.x, blockIdx.y, smem, StreamsTile<4>(f, a));
}

template <int EPI, int P, bool TAIL, int MT, int U>
__global__ __launch_bounds__(512, 2) void scaled_gemm_kernel(const TflGemm a, const int tail_rows, const int tail_per) {
    extern __shared__ __align__(16) char smem[];
    share_gemm_body<bf16, EPI, P, TAIL, MT, U, FromMemoryScaled>(a, tail_rows, tail_per, blockIdx.x, blockIdx.y, smem);
}

template <int P, int MT>
static int launch_streams(const TfhConnect& f, const TflGemm& a, hipStream_t st) {
    constexpr int LDS = 8 * P * MT * 64 * (int)sizeof(f32x4);
    hipLaunchKernelGGL((streams_gemm_kernel<P, MT>), dim3(((a.n >> 4) + P - 1) / P, (a.rows + 16 * MT - 1) / (16 * MT)), dim3(512), LDS, st, f, a);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

template <int EPI, int P, bool TAIL, int MT>
static int launch_scaled(const TflGemm& a, const ShareShape& s, hipStream_t st) {
    constexpr int NP = P + (TAIL ? 1 : 0), LDS = 8 * NP * MT * 64 * (int)sizeof(f32x4) + 16 * MT * (int)sizeof(float);
    constexpr int U = NP == 1 ? 4 : NP * MT <= 14 ? 2 : 1;    // (as launch_share_rows in tile_gemm.hip)
    auto* k = scaled_gemm_kernel<EPI, P, TAIL, MT, U>;
    if (LDS > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(k, dim3(TAIL ? 256 : ((a.n >> 4) + P - 1) / P, (a.rows + 16 * MT - 1) / (16 * MT)), dim3(512), LDS, st, a, s.left, s.rest);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

template <int EPI>
static int scaled_gemm(const TflGemm& a, hipStream_t st) {
    const ShareShape s = share_shape(a.n >> 4, EPI == TFL_EPI_GLU, 0, a.rows);
#define GO(P, TAIL) return a.rows <= 16 ? launch_scaled<EPI, P, TAIL, 1>(a, s, st) : launch_scaled<EPI, P, TAIL, 2>(a, s, st)
    if (s.rest) switch (s.each) {
        case 1: GO(1, true);
        case 2: GO(2, true);
        case 3: GO(3, true);
        case 4: GO(4, true);
        case 5: GO(5, true);
        case 6: GO(6, true);
        case 7: GO(7, true);
        default: return TF_ERANGE;
    }
    switch (s.each) {
        case 1: GO(1, false);
        case 2: GO(2, false);
        case 3: GO(3, false);
        case 4: GO(4, false);
        case 5: GO(5, false);
        case 6: GO(6, false);
        case 7: GO(7, false);
        case 8: GO(8, false);
        default: return TF_ERANGE;
    }
#undef GO
}

// Whole panels: of rows that are left over no workgroup has the sums of squares.  n in 64s: their readers take four sums at a time.
static int streams_panels(int rows, int streams, int n, int k) {
    if (rows < 1 || rows > (1 << 20) || streams < 1 || streams > 4 || n < 4096 || n > 8192 || (n & 63) || k < 32 || (k & 31)) return 0;
    const ShareShape s = share_shape(n >> 4, false, n, rows);
    return s.rest == 0 && s.each <= 2 ? s.each : 0;
}

extern "C" int tfh_streams_gemm_takes(int rows, int streams, int n, int k) { return streams_panels(rows, streams, n, k) > 0 ? 1 : 0; }

extern "C" int tfh_scaled_gemm_takes(int rows, int n, int epilogue) {
    if (rows < 1 || rows > (1 << 20) || n < 16 || (n & 15) || n > (1 << 20) || (epilogue != TFL_EPI_GLU && epilogue != TFL_EPI_F32)) return 0;
    return share_shape(n >> 4, epilogue == TFL_EPI_GLU, 0, rows).each > 0 ? 1 : 0;
}

extern "C" int tfh_streams_gemm(const TfhConnect* pf, const TflGemm* pa, void* stream) {
    if (!pf || !pa || !pa->wp || !pa->x || !pf->out || !pf->mix || !pf->in || !pf->norm_w || !pf->x) return TF_EINVAL;
    const TfhConnect f = *pf;
    const TflGemm a = *pa;
    if (a.rows < 1 || a.groups != 1 || a.chunk_major != 1 || a.n != f.width || (a.n & 15) || a.n < 16 || a.k < 32 || (a.k & 31) || a.ld_x < 8 || (a.ld_x & 7) || a.x_oct < 8
        || (a.x_oct & 7) || !a.out_t || a.ld_t < 8 || (a.ld_t & 7) || a.t_oct < 8 || (a.t_oct & 7) || !a.ss_out || a.ss_ld < a.n >> 4
        || !at16(a.wp, a.x, a.out_t, f.norm_w, f.x, f.x_out)) return TF_EINVAL;
    const int each = streams_panels(a.rows, f.streams, a.n, a.k);
    hipStream_t st = (hipStream_t)stream;
    if (each == 1) return a.rows <= 16 ? launch_streams<1, 1>(f, a, st) : launch_streams<1, 2>(f, a, st);
    if (each == 2) return a.rows <= 16 ? launch_streams<2, 1>(f, a, st) : launch_streams<2, 2>(f, a, st);
    return TF_ERANGE;
}

extern "C" int tfh_scaled_gemm(const TflGemm* pa, int epilogue, void* stream) {
    if (!pa || !pa->wp || !pa->x || !pa->ss_in) return TF_EINVAL;
    const TflGemm a = *pa;
    if (a.rows < 1 || a.groups != 1 || a.chunk_major != 1 || (a.n & 15) || a.n < 16 || a.k < 32 || (a.k & 31) || a.ld_x < 8 || (a.ld_x & 7) || a.x_oct < 8 || (a.x_oct & 7)
        || a.ss_n < 4 || (a.ss_n & 3) || a.ss_n > 512 || a.ss_ld < a.ss_n || (a.ss_ld & 3) || a.k_real < 1 || !at16(a.wp, a.x, a.ss_in)) return TF_EINVAL;
    if (epilogue == TFL_EPI_F32) {
        if (!a.out_f || a.n_real < 1 || a.n_real > a.n || a.ld_f < a.n_real) return TF_EINVAL;
    } else if (epilogue != TFL_EPI_GLU || !a.out_t || !at16(a.out_t) || a.ld_t < 8 || (a.ld_t & 7) || a.t_oct < 8 || (a.t_oct & 7)) {
        return TF_EINVAL;
    }
    if (!tfh_scaled_gemm_takes(a.rows, a.n, epilogue)) return TF_ERANGE;
    return epilogue == TFL_EPI_F32 ? scaled_gemm<TFL_EPI_F32>(a, (hipStream_t)stream) : scaled_gemm<TFL_EPI_GLU>(a, (hipStream_t)stream);
}
