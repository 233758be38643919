// The skinny GEMM of gemv.hip for wide weights, one workgroup per CU: y[M, N] = x[M, K] . W[N, K]^T, M <= 32, fp16, with the same rounding points and the
// same epilogues (residual and sums of squares, SwiGLU, rotation and KV append, fp32 logits) and the RMSNorm of the operand in front.
#include "gemv_common.h"
#include "share_shape.h"

// Bound by the weight stream.  A workgroup per panel (gemv.hip) leaves a few CUs with a panel more than the rest, reads x once per panel and begins with one
// batch of weights a wave.  Here all CUs have the same share (share_shape.h) and read x once.
// us in a graph over weights that come from memory, panel by panel -> here, 7 / 17 rows, k-octet-major x (a read of the same bytes):
//   q|k|v   12 288 x  4 096  21.2 -> 17.5, 26.6 -> 20.8 (16.5)      15 360 x 5 120  27.7 -> 27.4, 33.4 -> 29.3 (24.8)
//   o        4 096 x  4 096   8.5 ->  7.8,  9.8 ->  9.0 (6.7)
//   gate|up 22 016 x  4 096  32.1 -> 31.1, 40.2 -> 33.2 (28.1)      27 648 x 5 120  49.6 -> 45.1, 53.3 -> 46.9 (43.1)
//   down     4 096 x 11 008  17.6 -> 16.9, 21.0 -> 18.7 (15.0)
//   logits  32 000 x  4 096  48.4 -> 42.0, 53.3 -> 43.3 (40.1)      32 000 x 5 120  52.9 -> 52.0, 64.2 -> 53.1 (49.6)
//
// The bits are those of the panel form: WAVES parts of K, as many as that form has for these sizes (8 for o and down, 4 for the others), each summed chunk by
// chunk, and the parts in their order.  (Eight parts everywhere and another order of the chunks: q|k|v 16.9, o 7.7, gate|up 30.9, down 16.5, but which tokens
// top-p keeps depends on last digits of the logits.)
// Weights are packed chunk-major, [K/32][N/16][64][8], so that the chip reads one moving window per wave index; as the waves' ranges of K start a power of
// two apart, the chunks of wave w's range lie turned by 2 w in it (o 8.4 us without, 8.0 with).  A wave asks for two batches of chunks (weights,
// operand, norm weights) before anything waits, the norm's sums of squares in front of them, so that the fold of those runs under the stream; after
// that a batch is asked for whenever one has been used.
template <int MODE, bool NORM, int P, bool TAIL, int MT, int U, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void gemv_wide_kernel(const h16* __restrict__ wp, const h16* __restrict__ x, const float* __restrict__ ss_in,
                                                           const h16* __restrict__ ln_w, int K, int M, int x_sm, int x_sk, float eps, int N,
                                                           const h16* resid, SgAct ra, void* yv, SgAct ya, SgRope rp, float* __restrict__ ss_out,
                                                           int tail_rows, int tail_per) {
    constexpr int NP = P + (TAIL ? 1 : 0), CUS = 256, G = 4 * WAVES, SSB = 256 / G;
    static_assert(!TAIL || MODE == SG_F32 || MODE == SG_GATEUP, "rotation and sums of squares need whole panels");
    extern __shared__ __align__(16) char wide_smem[];
    f32x4 (*part)[NP * MT][64] = reinterpret_cast<f32x4 (*)[NP * MT][64]>(wide_smem);
    __shared__ float red[NORM ? MT : 1][G][16];             // (G: groups of 16 threads)
    const int cu = blockIdx.x, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int npan = N >> 4, panel0 = cu * P, chunks = K >> 5;
    const int per = (chunks + WAVES - 1) / WAVES, c_beg = wave * per, n_own = min(chunks, c_beg + per) - c_beg;
    const int rot = n_own > 0 ? 2 * wave % n_own : 0;
    const int64_t wstep = (int64_t)npan * 512, xstep = 4 * (int64_t)x_sk;
    const h16* w_at[NP];
#pragma unroll
    for (int p = 0; p < P; ++p) w_at[p] = wp + (int64_t)min(panel0 + p, npan - 1) * 512 + lane * 8;
    const int tail0 = ((cu & ~31) | (cu & 7) << 2 | (cu >> 3 & 3)) * tail_per;          // (neighbours on one XCD, as in share_gemm.h)
    if constexpr (TAIL) {
        const int row = min(min(tail0 + i, tail0 + tail_per - 1), tail_rows - 1);
        int slot = row & 15;
        if constexpr (MODE == SG_GATEUP) slot = ((slot >> 2) << 1) + (slot & 1) + ((slot & 2) << 2);
        w_at[P] = wp + (int64_t)(CUS * P + (row >> 4)) * 512 + g * 128 + slot * 8;
    }
    const h16* x_at[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) x_at[t] = x + (int64_t)min(16 * t + i, M - 1) * x_sm + (int64_t)g * x_sk;
    struct Batch { half8 w[U][NP], x[U][MT], ln[NORM ? U : 1]; };
    auto load = [&](Batch& b, int c0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int o = min(c0 + u, n_own - 1), c = c_beg + o, at = c_beg + (o + rot >= n_own ? o + rot - n_own : o + rot);
#pragma unroll
            for (int t = 0; t < MT; ++t) b.x[u][t] = load_half8(x_at[t] + xstep * c);
            if constexpr (NORM) b.ln[u] = load_half8(ln_w + 32 * c + 8 * g);
#pragma unroll
            for (int p = 0; p < NP; ++p) b.w[u][p] = load_half8_stream(w_at[p] + wstep * at);
        }
    };
    float inv[MT];
    f32x4 acc[NP][MT];
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[p][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Batch& b, int c0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u < n_own) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    half8 v = b.x[u][t];
                    if constexpr (NORM) v = sg_normalise(v, b.ln[u], inv[t]);
#pragma unroll
                    for (int p = 0; p < NP; ++p) acc[p][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b.w[u][p], v, acc[p][t], 0, 0, 0);
                }
            }
    };

    // ---- what the sums of squares, and the epilogue of a wave's first result tile, read ----
    const int nparts = K >> 4, pg = tid >> 4, m16 = tid & 15;
    float ssv[MT][SSB];
    if constexpr (NORM) {
        const float* from = ss_in ? ss_in : reinterpret_cast<const float*>(wp);          // (no branch around loads; not used then)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int j = 0; j < SSB; ++j) ssv[t][j] = from[(int64_t)min(pg + j * G, nparts - 1) * 32 + 16 * t + m16];
    }
    const int t_end = wave % MT, panel_end = min(panel0 + wave / MT, npan - 1), m_end = min(16 * t_end + i, M - 1);
    int64_t pos_end = 0;
    int slot0 = 0;
    half4 with = {0, 0, 0, 0};
    if constexpr (MODE == SG_QKV) {
        pos_end = rp.positions[m_end];
        slot0 = rp.slot0_dev ? *rp.slot0_dev : rp.slot0;
    }
    auto residual = [&](int panel, int m) {
        const h16* r = resid + (int64_t)m * ra.sm + (int64_t)(2 * panel + (g >> 1)) * ra.sk + 4 * (g & 1);
        return *reinterpret_cast<const half4*>(r);
    };
    if constexpr (MODE == SG_PLAIN) {
        if (resid) with = residual(panel_end, m_end);
    }
    asm volatile("" ::: "memory");
    Batch a, b;
    load(a, 0);
    load(b, U);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    // ---- 1 / rms of the rows ----
    if constexpr (NORM) {
        if (ss_in) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                float s = 0.f;
#pragma unroll
                for (int j = 0; j < SSB; ++j) s += pg + j * G < nparts ? ssv[t][j] : 0.f;
                for (int p = pg + SSB * G; p < nparts; p += G) s += ss_in[(int64_t)p * 32 + 16 * t + m16];
                red[t][pg][m16] = s;
            }
        } else {                                              // (first layer: of the rows themselves)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                float s = 0.f;
                for (int c = c_beg; c < c_beg + n_own; ++c) {
                    const half8 v = load_half8(x_at[t] + xstep * c);
#pragma unroll
                    for (int e = 0; e < 8; ++e) s = fmaf((float)v[e], (float)v[e], s);
                }
                s = rows_sum(s);
                if (g == 0) red[t][wave][i] = s;
            }
        }
        __syncthreads();
        const int groups = ss_in ? G : WAVES;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            float s = 0.f;
            for (int k = 0; k < groups; ++k) s += red[t][k][i];
            inv[t] = 1.0f / sqrtf(s / (float)K + eps);
        }
    }
    half4 cs_end = {0, 0, 0, 0}, sn_end = {0, 0, 0, 0};
    auto turn = [&](int panel, int64_t pos, half4& cs, half4& sn) {
        const int pph = rp.D >> 4, sec = panel / (rp.H * pph), d = 8 * (panel % pph) + 4 * (g & 1) + (g >= 2 ? rp.D >> 1 : 0);
        if (sec == 0 || (sec == 1 && rp.rotate_k)) {
            cs = *reinterpret_cast<const half4*>(rp.cosb + pos * rp.D + d);
            sn = *reinterpret_cast<const half4*>(rp.sinb + pos * rp.D + d);
        }
    };
    if constexpr (MODE == SG_QKV) {
        if (wave < NP * MT) turn(panel_end, pos_end, cs_end, sn_end);
    }

    int c0 = 0;
    for (; c0 + 2 * U < n_own; c0 += 2 * U) {
        multiply(a, c0);
        load(a, c0 + 2 * U);
        multiply(b, c0 + U);
        load(b, c0 + 3 * U);
    }
    multiply(a, c0);
    multiply(b, c0 + U);

    // ---- the waves' sums, in wave order; lane (g, i): outputs 4g .. 4g+3 of the tile, row i ----
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int t = 0; t < MT; ++t) part[wave][p * MT + t][lane] = acc[p][t];
    __syncthreads();
    for (int j = wave; j < NP * MT; j += WAVES) {
        const int p = j / MT, t = j - p * MT, m = 16 * t + i;
        f32x4 s = part[0][j][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) {
            const f32x4 o = part[w][j][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] += o[r];
        }
        const bool live = m < M;
        if (TAIL && p == P) {
            const int row = tail0 + 4 * g;                   // first of this lane's four left-over rows
            if (!live || 4 * g >= tail_per || row >= tail_rows) continue;
            const int panel = CUS * P + (row >> 4);
            if constexpr (MODE == SG_GATEUP) {               // gate, gate, up, up of outputs 2q, 2q + 1 of a panel's octet
                typedef h16 half2v __attribute__((ext_vector_type(2)));
                half2v o;
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const float gf = (float)(h16)s[r];
                    o[r] = hmul_rn((h16)(gf / (1.0f + expf(-gf))), (h16)s[2 + r]);
                }
                *reinterpret_cast<half2v*>((h16*)yv + (int64_t)m * ya.sm + (int64_t)panel * ya.sk + ((row & 15) >> 1)) = o;
            } else {
                float* dst = (float*)yv + (int64_t)m * ya.sm + 16 * panel + (row & 15);
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[r] = (float)(h16)s[r];
            }
            continue;
        }
        const int panel = panel0 + p;
        if (panel >= npan) continue;
        if constexpr (MODE == SG_GATEUP) {                   // lanes g < 2 hold gate rows, g + 2 the same outputs' up rows
            f32x4 up;
#pragma unroll
            for (int r = 0; r < 4; ++r) up[r] = other_half(s[r]);
            if (!live || g >= 2) continue;
            half4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float gf = (float)(h16)s[r];
                o[r] = hmul_rn((h16)(gf / (1.0f + expf(-gf))), (h16)up[r]);
            }
            *reinterpret_cast<half4*>((h16*)yv + (int64_t)m * ya.sm + (int64_t)panel * ya.sk + 4 * g) = o;
        } else if constexpr (MODE == SG_F32) {
            if (!live) continue;
            float* dst = (float*)yv + (int64_t)m * ya.sm + 16 * panel + 4 * g;
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[r] = (float)(h16)s[r];
        } else if constexpr (MODE == SG_PLAIN) {
            half4 o;
            float y[4];
            if (resid && j != wave) with = residual(panel, min(m, M - 1));
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                o[r] = (h16)s[r];
                if (resid) o[r] = hadd_rn(with[r], o[r]);
                y[r] = live ? (float)o[r] : 0.f;
            }
            if (live) *reinterpret_cast<half4*>((h16*)yv + (int64_t)m * ya.sm + (int64_t)(2 * panel + (g >> 1)) * ya.sk + 4 * (g & 1)) = o;
            if (ss_out) {                                    // this panel's share of sum(y^2) per row, for the next norm
                const float q = rows_sum(y[0] * y[0] + y[1] * y[1] + y[2] * y[2] + y[3] * y[3]);
                if (g == 0) ss_out[(int64_t)panel * 32 + m] = q;
            }
        } else {                                             // q and k panels hold rows d0..d0+7 | d0+D/2..d0+D/2+7 of a head
            const int H = rp.H, D = rp.D, pph = D >> 4, sec = panel / (H * pph), hd = panel / pph % H, pp = panel % pph;
            h16 val[4], oth[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                val[r] = (h16)s[r];
                oth[r] = (h16)other_half((float)val[r]);     // rotary partner (exact)
            }
            if (!live) continue;
            half4 out, cs = cs_end, sn = sn_end;
            if (j != wave) turn(panel, rp.positions[m], cs, sn);
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = val[r];
            if (sec == 2) {
                *reinterpret_cast<half4*>(rp.v_cache + (int64_t)(slot0 + m) * rp.stride_t + (int64_t)hd * rp.stride_h + 16 * pp + 4 * g) = out;
                continue;
            }
            const bool hi = g >= 2;
            if (sec == 0 || rp.rotate_k) {                   // (x*cos) + (rotate_half(x)*sin) in fp16
#pragma unroll
                for (int r = 0; r < 4; ++r) out[r] = hadd_rn(hmul_rn(val[r], cs[r]), hmul_rn(hi ? oth[r] : (h16)(-(float)oth[r]), sn[r]));
            }
            const int d = 8 * pp + 4 * (g & 1) + (hi ? D >> 1 : 0);
            h16* dst = sec == 0 ? rp.q_out + ((int64_t)m * H + hd) * D + d
                                : rp.k_cache + (int64_t)(slot0 + m) * rp.stride_t + (int64_t)hd * rp.stride_h + d;
            *reinterpret_cast<half4*>(dst) = out;
        }
    }
}

struct WideArgs {
    const void *wp, *x, *ln_w, *resid;
    void* y;
    SgAct xa, ra, ya;
    float eps;
    int M, N, K;
    const float* ss_in;
    float* ss_out;
    SgRope rp;
};

// The shape of a product in this form; each == 0: gemv.hip's.  Rotation and sums of squares come in whole panels: there a share of a panel more is taken
// where it leaves no more than an eighth of the CUs without work.  Which form a weight has is settled when it is packed, for all rows, so the sizes that are slower
// at few of them stay panels; us, panels -> here, at 1 / 2 / 7 / 17 rows:
//   gate | up below two panels a CU: 4 352 x 2 048 7.6 / 7.7 / 8.0 / 9.5 -> 8.8 / 8.9 / 8.8 / 10.7, 5 120 x 4 096 11.9 / 12.0 / 12.3 / 15.0 -> 11.7 / 11.7 / 12.0 / 14.9 (32 rows
//     15.6 -> 15.9), 6 144 x 2 048 8.2 / 8.2 / 8.6 / 9.9 -> 8.3 / 8.3 / 8.4 / 10.1; from there on 8 192 x 2 048 9.3 / 9.0 / 9.3 / 11.3 -> 9.1 / 9.1 / 9.1 / 10.5;
//   logits with one panel and up to four rows: 4 352 x 2 048 8.0 / 8.0 / 8.5 / 12.9 -> 8.6 / 8.6 / 8.4 / 10.3; 5 120 x 2 048 is 8.2 / 8.2 / 8.7 / 13.1 -> 7.4 / 7.4 / 7.5 / 9.4;
//   o and down on a part of the CUs over a short K: 7 424 x 2 560 8.9 / 8.6 / 9.8 / 11.2 -> 9.1 / 9.2 / 9.3 / 10.0, 7 168 x 4 096 12.2 / 11.7 / 12.6 / 14.6 -> 12.0 / 12.1 / 12.1 / 12.5;
//     7 168 x 7 168 is 19.3 / 18.3 / 20.2 / 23.8 -> 18.5 / 18.5 / 18.3 / 19.7, 7 680 x 7 680 22.5 / 21.9 / 22.9 / 26.3 -> 20.2 / 20.1 / 20.0 / 20.9.
// Taken although slower at up to four rows, beside gate | up of the same layer: q|k|v 15 360 x 5 120 26.3 / 26.6 / 27.3 / 32.1 -> 27.2 / 27.4 / 26.8 / 29.6 (27 648 x 5 120 49.6 /
// 48.1 / 48.6 / 51.8 -> 45.5 / 44.6 / 43.6 / 45.5).
static ShareShape wide_shape(int mode, int N, int K) {
    if (K < 2048 || K > (1 << 20) || (K % 32) || N < 4096 || (N % 16) || N > (1 << 20)) return {0, 0, 0};
    const int panels = N / 16;
    if (mode == SG_PLAIN || mode == SG_QKV) {
        const int each = (panels + 255) / 256;
        if (mode == SG_PLAIN && panels != each * 256 && K < 7168) return {0, 0, 0};
        return each <= (mode == SG_QKV ? 6 : 2) && panels * 8 >= each * 256 * 7 ? ShareShape{each, 0, 0} : ShareShape{0, 0, 0};
    }
    const ShareShape s = share_shape(panels, mode == SG_GATEUP, 0, 32);
    return (mode == SG_GATEUP && panels < 512) || (s.each == 1 && s.rest == 4) ? ShareShape{0, 0, 0} : s;
}

template <int MODE, bool NORM, int P, bool TAIL, int MT>
static int launch_wide_rows(const WideArgs& a, const ShareShape& f, hipStream_t st) {
    constexpr int WAVES = MODE == SG_PLAIN ? 8 : 4;
    constexpr int NP = P + (TAIL ? 1 : 0), LDS = WAVES * NP * MT * 64 * (int)sizeof(f32x4);
    // Chunks of a batch.  More gain nothing (q|k|v, three panels, six chunks 17.5 -> 18.3 us; gate | up, six tiles, three 31.1 -> 31.8).
    constexpr int U = WAVES == 8 ? 4 : NP <= 2 ? 8 : NP <= 4 ? 4 : 2;
    static_assert(LDS <= 152 * 1024, "one workgroup's partial tiles");
    auto* k = gemv_wide_kernel<MODE, NORM, P, TAIL, MT, U, WAVES>;
    if (LDS > 60 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(k, dim3(TAIL ? 256 : (a.N / 16 + P - 1) / P), dim3(64 * WAVES), LDS, st, (const h16*)a.wp, (const h16*)a.x, a.ss_in,
                       (const h16*)a.ln_w, a.K, a.M, (int)a.xa.sm, (int)a.xa.sk, a.eps, a.N, (const h16*)a.resid, a.ra, a.y, a.ya, a.rp, a.ss_out, f.left,
                       f.rest);
    TF_LAUNCH_CHECK();
    return TF_OK;
}

template <int MODE, bool NORM, int P, bool TAIL>
static int launch_wide(const WideArgs& a, const ShareShape& f, hipStream_t st) {
    return a.M <= 16 ? launch_wide_rows<MODE, NORM, P, TAIL, 1>(a, f, st) : launch_wide_rows<MODE, NORM, P, TAIL, 2>(a, f, st);
}

template <int MODE, bool NORM>
static int wide(const WideArgs& a, hipStream_t st) {
    const ShareShape f = wide_shape(MODE, a.N, a.K);
#define WIDE(P) case P: return launch_wide<MODE, NORM, P, false>(a, f, st)
#define WIDE_TAIL(P) case P: return launch_wide<MODE, NORM, P, true>(a, f, st)
    if constexpr (MODE == SG_PLAIN) {
        switch (f.each) { WIDE(1); WIDE(2); }
    } else if constexpr (MODE == SG_QKV) {
        switch (f.each) { WIDE(1); WIDE(2); WIDE(3); WIDE(4); WIDE(5); WIDE(6); }
    } else {
        if constexpr (MODE == SG_F32) {
            if (f.each == 1) return f.rest ? launch_wide<MODE, NORM, 1, true>(a, f, st) : launch_wide<MODE, NORM, 1, false>(a, f, st);
        }
        if (f.rest) switch (f.each) { WIDE_TAIL(2); WIDE_TAIL(3); WIDE_TAIL(4); WIDE_TAIL(5); WIDE_TAIL(6); WIDE_TAIL(7); }
        else switch (f.each) { WIDE(2); WIDE(3); WIDE(4); WIDE(5); WIDE(6); WIDE(7); WIDE(8); }
    }
#undef WIDE
#undef WIDE_TAIL
    return TF_ERANGE;
}

extern "C" int tf_wide_gemm_takes(int mode, int N, int K) {
    if (mode < SG_PLAIN || mode > SG_QKV || N < 16 || (N % 16) || K < 32 || (K % 32)) return TF_EINVAL;
    return wide_shape(mode, N, K).each > 0 ? 1 : 0;
}

static bool quads(const SgAct& s, const void* p) { return s.sm > 0 && s.sk > 0 && !(s.sm % 4) && !(s.sk % 4) && !(reinterpret_cast<uintptr_t>(p) % 8); }

extern "C" int tf_wide_gemm_act(const void* w_packed, const void* x, int64_t xs_m, int64_t xs_k, const void* ln_w, float eps, const float* ss_in,
                                const void* resid, int64_t rs_m, int64_t rs_k, float* ss_out, void* y, int64_t ys_m, int64_t ys_k, int M, int N, int K,
                                int out_f32, void* stream) {
    WideArgs a = {};
    a.wp = w_packed, a.x = x, a.ln_w = ln_w, a.resid = resid, a.y = y, a.eps = eps, a.M = M, a.N = N, a.K = K, a.ss_in = ss_in, a.ss_out = ss_out;
    a.xa = SgAct{xs_m, xs_k}, a.ra = SgAct{rs_m, rs_k}, a.ya = SgAct{ys_m, ys_k};
    if (!w_packed || !x || !y || !sg_shape_ok(M, N, K, a.xa) || (reinterpret_cast<uintptr_t>(x) % 16)) return TF_EINVAL;
    if ((out_f32 && (resid || ss_out)) || (ss_in && !ln_w) || (!out_f32 && ln_w) || ys_m <= 0) return TF_EINVAL;
    if (!out_f32 && (!quads(a.ya, y) || (resid && !quads(a.ra, resid)))) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    if (out_f32) return ln_w ? wide<SG_F32, true>(a, st) : wide<SG_F32, false>(a, st);
    return wide<SG_PLAIN, false>(a, st);
}

extern "C" int tf_wide_gemm_swiglu_act(const void* gate_up_packed, const void* x, int64_t xs_m, int64_t xs_k, const void* ln_w, float eps,
                                       const float* ss_in, void* act, int64_t ys_m, int64_t ys_k, int M, int I, int K, void* stream) {
    WideArgs a = {};
    a.wp = gate_up_packed, a.x = x, a.ln_w = ln_w, a.y = act, a.eps = eps, a.M = M, a.N = 2 * I, a.K = K, a.ss_in = ss_in;
    a.xa = SgAct{xs_m, xs_k}, a.ya = SgAct{ys_m, ys_k};
    if (!gate_up_packed || !x || !act || !ln_w || I < 8 || (I % 8) || I > (1 << 20) || !sg_shape_ok(M, a.N, K, a.xa) || (reinterpret_cast<uintptr_t>(x) % 16)
        || !quads(a.ya, act)) return TF_EINVAL;
    return wide<SG_GATEUP, true>(a, (hipStream_t)stream);
}

extern "C" int tf_wide_qkv_rope_act(const void* wqkv_packed, const void* x, int64_t xs_m, int64_t xs_k, const void* ln_w, float eps, const float* ss_in,
                                    const void* cosb, const void* sinb, const int64_t* positions, void* q_out, void* k_cache, void* v_cache,
                                    int64_t stride_t, int64_t stride_h, int slot0, const int32_t* slot0_dev, int M, int H, int D, int K, int rotate_k,
                                    void* stream) {
    if (!wqkv_packed || !x || !ln_w || !cosb || !sinb || !positions || !q_out || !k_cache || !v_cache) return TF_EINVAL;
    if (H < 1 || H > 4096 || D < 32 || D > 4096 || (D % 32) || (stride_t % 4) || (stride_h % 4)) return TF_EINVAL;
    WideArgs a = {};
    a.wp = wqkv_packed, a.x = x, a.ln_w = ln_w, a.eps = eps, a.M = M, a.N = 3 * H * D, a.K = K, a.ss_in = ss_in;
    a.xa = SgAct{xs_m, xs_k};
    if (!sg_shape_ok(M, a.N, K, a.xa) || (reinterpret_cast<uintptr_t>(x) % 16)) return TF_EINVAL;
    a.rp.cosb = (const h16*)cosb, a.rp.sinb = (const h16*)sinb, a.rp.positions = positions, a.rp.q_out = (h16*)q_out, a.rp.k_cache = (h16*)k_cache;
    a.rp.v_cache = (h16*)v_cache, a.rp.stride_t = stride_t, a.rp.stride_h = stride_h, a.rp.slot0_dev = slot0_dev, a.rp.slot0 = slot0;
    a.rp.H = H, a.rp.D = D, a.rp.rotate_k = rotate_k;
    return wide<SG_QKV, true>(a, (hipStream_t)stream);
}
