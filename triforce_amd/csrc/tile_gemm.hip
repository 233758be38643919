// Skinny GEMM of the batch-served model families: y[m, n] = x[m, :] . W[n, :], one 16-row weight panel per workgroup, the panel's
// K range split over the workgroup's waves, batch rows in blocks of 16 * MT.  Same weight packing and wave structure as
// csrc/gemv.hip (a wave's weight load is one contiguous run per 16x32 tile, partial tiles meet in LDS), with the element type
// a template parameter and these epilogues:
//   IN        the four projections that read the layer's one norm (query latent, key latent | key, gate, feed-forward up):
//             raw fp32 outputs plus per-panel sums of squares, the query latent also times its norm weight as the next operand
//             (its row scale is applied behind the next product), gelu on the last part
//   QUERY     row scale from the sums of squares, heads written as unrotated | rotated; spare workgroups of the same launch
//             normalise, rotate and store the cache rows
//   LATENT    per head: query through the transposed key up-projection, next to the rotated part
//   GATED     per head: value up-projection of the attended latent, times the output gate
//   RESIDUAL  attention output and feed-forward down in one matrix, added to the fp32 residual
//             (and the sum again as the next operand)
//   TOKEN     per-layer token input: gelu times the token's row of a table
//   GLU       panels of 8 gate | 8 up rows: gelu(gate) * up
//   F32       the sums themselves
#include "tile_common.h"
#include "share_gemm.h"
#include "share_shape.h"

#ifndef TFL_PAIR_MIN
#define TFL_PAIR_MIN 420     // panel pairs from which two panels share a workgroup
#endif

// P panels per workgroup (they share the operand rows), MT 16-row blocks, U tiles of 32 per batch; AHEAD: the next batch's weights
// are requested before the current one is used (long K), otherwise a wave's whole K range should fit one or two batches.
// bx, rb of blocks: this workgroup's place (a WAVES-wide half of one may stand for it, tid within it), part: its LDS.
template <typename T, int EPI, int P, int MT, int WAVES, int U, bool AHEAD>
__device__ __forceinline__ void latent_gemm_body(const TflGemm& a, const int tid, const int bx, const int blocks, const int rb, f32x4 (*part)[P * MT][64]) {
    typedef typename El<T>::Frag Frag;
    static_assert(P * MT <= WAVES, "one wave finishes one 16x16 tile");
    const int ppg = a.n >> 4, npan = ppg * a.groups;
    if constexpr (EPI == TFL_EPI_QUERY) {
        if (bx >= npan) {                                    // the cache row of one batch row
            const int m = rb * (blocks - npan) + bx - npan;
            if (m >= a.rows) return;
            const int slot = a.slot[m];
            if (slot < 0 || slot >= a.cache_rows) return;
            int p = a.pos[m];
            p = p < 0 ? 0 : (p >= a.max_pos ? a.max_pos - 1 : p);
            const float* src = a.kv_raw + (int64_t)m * a.ld_kv;
            cache_row<T, WAVES>([src](int c) { return src[c]; }, a.C, a.c_real, a.R, a.kv_norm_w, a.eps, a.cos + (int64_t)p * a.half,
                                a.sin + (int64_t)p * a.half, a.half, (T*)a.cache + (int64_t)slot * (a.C + a.R), (T*)nullptr,
                                (float*)&part[0][0][0]);
            return;
        }
    }
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int panel0 = bx * P, grp = panel0 / ppg;            // (several groups: their panels come in whole P)
    const int m0 = rb * 16 * MT;
    const int chunks = a.k >> 5;
    const int per = (chunks + WAVES - 1) / WAVES;
    const int c_beg = wave * per, c_end = min(chunks, c_beg + per), last = c_end - 1;
    const T* wp[P];
#pragma unroll
    for (int p = 0; p < P; ++p) wp[p] = (const T*)a.wp + (int64_t)min(panel0 + p, npan - 1) * (a.chunk_major ? 512 : chunks * 512) + lane * 8;
    const int64_t wstep = a.chunk_major ? (int64_t)npan * 512 : 512;
    int64_t xoff[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
        xoff[t] = (int64_t)min(m0 + 16 * t + i, a.rows - 1) * a.ld_x + (int64_t)grp * a.x_group + g * a.x_oct;
    const int64_t xstep = 4 * a.x_oct;
    auto load_w = [&](Frag (&w)[P][U], int c0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (AHEAD || c0 + u < c_end) {                    // (AHEAD: straight-line code, the tail repeats the last tile)
#pragma unroll
                for (int p = 0; p < P; ++p) w[p][u] = load_frag_stream(wp[p] + wstep * min(c0 + u, last));
            }
    };
    f32x4 acc[P][MT];
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[p][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // What the epilogue reads is asked for in front of the weights by the wave that finishes a tile, not behind the products, where nothing is
    // left to hide it (us: QUERY at one row 6.85 -> 6.62; at 32 rows TOKEN 8.97 -> 8.50, GATED 5.62 -> 5.21).
    const int t_end = wave % MT, panel_end = panel0 + wave / MT, pin_end = panel_end - grp * ppg;
    const int m_end = min(m0 + 16 * t_end + i, a.rows - 1), n_end = 16 * pin_end + 4 * g;
    const bool ends = wave < P * MT && panel_end < npan;
    [[maybe_unused]] f32x4 with = {0.f, 0.f, 0.f, 0.f};
    [[maybe_unused]] float cs[2] = {}, sn[2] = {};
    [[maybe_unused]] T row4[4] = {};
    [[maybe_unused]] int64_t id = 0;
    [[maybe_unused]] int p_end = 0;
    if (ends) {
        if constexpr (EPI == TFL_EPI_IN) {
            if (16 * pin_end < a.n_raw && n_end < a.n_scaled) with = *reinterpret_cast<const f32x4*>(a.norm_w + n_end);
        }
        if constexpr (EPI == TFL_EPI_GATED) with = *reinterpret_cast<const f32x4*>(a.gate + (int64_t)m_end * a.ld_gate + grp * a.n + n_end);
        if constexpr (EPI == TFL_EPI_RESIDUAL) with = *reinterpret_cast<const f32x4*>(a.out_f + (int64_t)m_end * a.ld_f + n_end);
        if constexpr (EPI == TFL_EPI_TOKEN) id = a.ids[m_end];
        if constexpr (EPI == TFL_EPI_QUERY) p_end = a.pos[m_end];
    }
    asm volatile("" ::: "memory");
    auto second = [&] {                                       // what depends on the first
        if (!ends) return;
        if constexpr (EPI == TFL_EPI_TOKEN) {
            id = id < 0 ? 0 : (id >= a.vocab ? a.vocab - 1 : id);
            const T* e = (const T*)a.tok_table + id * a.ld_tok;
#pragma unroll
            for (int r = 0; r < 4; ++r) row4[r] = e[min(n_end + r, a.n_real - 1)];
        }
        if constexpr (EPI == TFL_EPI_QUERY) {
            const int d = n_end % (a.N + a.R) - a.N, p = p_end < 0 ? 0 : (p_end >= a.max_pos ? a.max_pos - 1 : p_end);
            if (d >= 0 && a.half > 0) {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const int64_t at = (int64_t)p * a.half + min((d >> 1) + r, a.half - 1);
                    cs[r] = a.cos[at];
                    sn[r] = a.sin[at];
                }
            }
        }
    };
    // QUERY: the producer's sums of squares are asked for here and added behind the products
    constexpr int SSU = EPI == TFL_EPI_QUERY ? 12 : 1;
    [[maybe_unused]] float2 sums[SSU];
    [[maybe_unused]] const float2* ss = nullptr;
    if constexpr (EPI == TFL_EPI_QUERY) {
        if (wave < MT) {
            ss = reinterpret_cast<const float2*>(a.ss_in + (int64_t)min(m0 + 16 * wave + i, a.rows - 1) * a.ss_ld);
#pragma unroll
            for (int u = 0; u < SSU; ++u) sums[u] = ss[min(g + 4 * u, a.ss_n / 2 - 1)];
        }
        asm volatile("" ::: "memory");
    }
    // float32: where the loads of a batch stand is no longer the scheduler's choice, which put those of its second operand behind the first one's products and
    // changed with the code around (up to 20 % either way).  One row block: the next weights in front of this batch's products too, two: among them.  us at 1 /
    // 16 / 17 / 32 rows, scheduled -> so: 4 096 x 15 104 61.4 / 64.7 / 88.9 / 93.7 -> 45.9 / 54.9 / 60.6 / 66.1, 17 216 x 4 096 63.8 / 81.3 / 94.8 / 111.5 -> 63.1 / 76.2 / 83.6 / 92.1,
    // gate | up of 4 096 x 4 096 19.3 / 20.2 / 26.7 / 27.9 -> 16.5 / 19.2 / 19.2 / 20.2.  (LATENT, a chunk or two a wave, is slower for either: 32 rows 8.8 -> 9.4.)
    constexpr bool HOLD = AHEAD && sizeof(T) == 4 && EPI != TFL_EPI_LATENT;
    if (c_beg < c_end) {
        Frag w[P][U], wn[P][U];
        load_w(w, c_beg);
        for (int c0 = c_beg; c0 < c_end; c0 += U) {
            Frag x[U][MT];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (AHEAD || c0 + u < c_end) {
#pragma unroll
                    for (int t = 0; t < MT; ++t) x[u][t] = load_frag((const T*)a.x + xoff[t] + xstep * min(c0 + u, last));
                }
            if constexpr (HOLD && MT > 1) __builtin_amdgcn_sched_barrier(0);
            if constexpr (AHEAD) load_w(wn, c0 + U);
            if constexpr (HOLD && MT == 1) __builtin_amdgcn_sched_barrier(0);
            if constexpr (EPI == TFL_EPI_QUERY) {
                if (c0 == c_beg) second();
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (c0 + u < c_end) {
#pragma unroll
                    for (int t = 0; t < MT; ++t)
#pragma unroll
                        for (int p = 0; p < P; ++p) acc[p][t] = El<T>::mma(w[p][u], x[u][t], acc[p][t]);
                }
            if constexpr (AHEAD) {
#pragma unroll
                for (int p = 0; p < P; ++p)
#pragma unroll
                    for (int u = 0; u < U; ++u) w[p][u] = wn[p][u];
            } else if (c0 + U < c_end) {
                load_w(w, c0 + U);
            }
        }
    } else if constexpr (EPI == TFL_EPI_QUERY) {
        second();                                             // (a wave without a part of a short K)
    }
    if constexpr (EPI == TFL_EPI_TOKEN) second();             // (under the waves' meeting; inside the loop 32 rows 9.0 -> 9.25 us)
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int t = 0; t < MT; ++t) part[wave][p * MT + t][lane] = acc[p][t];
    float inv = 1.f;
    if constexpr (EPI == TFL_EPI_QUERY) {                    // scale of row m from the producer's per-panel sums of squares
        if (wave < MT) {
            float q = 0.f;
#pragma unroll
            for (int u = 0; u < SSU; ++u)
                if (g + 4 * u < a.ss_n / 2) q += sums[u].x + sums[u].y;
#pragma unroll 4
            for (int p = g + 4 * SSU; p < a.ss_n / 2; p += 4) {
                const float2 v = ss[p];
                q += v.x + v.y;
            }
            q = rows_sum(q);
            inv = 1.0f / sqrtf(q / (float)a.k_real + a.eps);
        }
    }
    __syncthreads();
    if (wave >= P * MT) return;                              // wave p * MT + t finishes row block t of panel p
    const int t = wave % MT, panel = panel0 + wave / MT, pin = panel - grp * ppg;
    if (panel >= npan) return;
    f32x4 s = part[0][wave][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
        const f32x4 o = part[w][wave][lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] += o[r];
    }
    const int m = m0 + 16 * t + i;                           // this lane: outputs n .. n+3 of row m
    const bool live = m < a.rows;
    const int n = 16 * pin + 4 * g;
    if constexpr (EPI == TFL_EPI_IN) {
        if (16 * pin < a.n_raw) {
            float q = s[0] * s[0] + s[1] * s[1] + s[2] * s[2] + s[3] * s[3];
            q = rows_sum(q);
            if (live) {
                *reinterpret_cast<f32x4*>(a.out_f + (int64_t)m * a.ld_f + n) = s;
                if (n < a.n_scaled) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[r] *= with[r];
                    store_quad((T*)a.out_t2 + (int64_t)m * 8 + (n >> 3) * (8 * (int64_t)a.rows) + (n & 7), s);
                }
                if (g == 0) a.ss_out[(int64_t)m * a.ss_ld + pin] = q;
            }
        } else if (live) {
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = gelu_tanh(s[r]);
            const int k = n - a.n_raw;
            store_quad((T*)a.out_t + (int64_t)m * a.ld_t + (k >> 3) * a.t_oct + (k & 7), s);
        }
        return;
    }
    if constexpr (EPI == TFL_EPI_GLU) {                      // lanes g < 2 hold gate rows, g + 2 the same outputs' up rows
        f32x4 up;
#pragma unroll
        for (int r = 0; r < 4; ++r) up[r] = other_half(s[r]);
        if (live && g < 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = gelu_tanh(s[r]) * up[r];
            store_quad((T*)a.out_t + (int64_t)m * a.ld_t + pin * a.t_oct + 4 * g, s);
        }
        return;
    }
    if (!live) return;
    if constexpr (EPI == TFL_EPI_F32) {
        float* y = a.out_f + (int64_t)m * a.ld_f + n;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < a.n_real) y[r] = s[r];
    } else if constexpr (EPI == TFL_EPI_QUERY) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] *= inv;
        const int per_head = a.N + a.R, h = n / per_head, e = n - h * per_head;
        const int64_t row = (int64_t)m * a.H + h;
        if (e < a.N) {
            store_quad((T*)a.out_t2 + row * a.N + e, s);
        } else {
            const int d = e - a.N;
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const int pr = (d + r) >> 1;
                if (pr < a.half) {
                    const float u = s[r], v = s[r + 1];
                    s[r] = u * cs[r / 2] - v * sn[r / 2];
                    s[r + 1] = v * cs[r / 2] + u * sn[r / 2];
                }
            }
            store_quad((T*)a.out_t + row * (a.C + a.R) + a.C + d, s);
        }
    } else if constexpr (EPI == TFL_EPI_LATENT) {
        store_quad((T*)a.out_t + ((int64_t)m * a.H + grp) * (a.C + a.R) + n, s);
    } else if constexpr (EPI == TFL_EPI_GATED) {
        const int col = grp * a.n + n;
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] *= sigmoid(with[r]);
        store_quad((T*)a.out_t + (int64_t)m * a.ld_t + (col >> 3) * a.t_oct + (col & 7), s);
    } else if constexpr (EPI == TFL_EPI_RESIDUAL) {
        f32x4* y = reinterpret_cast<f32x4*>(a.out_f + (int64_t)m * a.ld_f + n);
        f32x4 o = with;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] += s[r];
        *y = o;
        if (a.out_t) store_quad((T*)a.out_t + (int64_t)m * a.ld_t + (n >> 3) * a.t_oct + (n & 7), o);
    } else if constexpr (EPI == TFL_EPI_TOKEN) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] = n + r < a.n_real ? gelu_tanh(s[r]) * (float)row4[r] : 0.f;
        store_quad((T*)a.out_t + (int64_t)m * a.ld_t + n, s);
    }
}

template <typename T, int EPI, int P, int MT, int WAVES, int U, bool AHEAD>
__global__ __launch_bounds__(WAVES * 64) void latent_gemm_kernel(const TflGemm a) {
    __shared__ f32x4 part[WAVES][P * MT][64];
    latent_gemm_body<T, EPI, P, MT, WAVES, U, AHEAD>(a, threadIdx.x, blockIdx.x, gridDim.x, blockIdx.y, part);
}

// LATENT of up to 16 rows, and in front of it, on workgroups of their own, panels of another product that waits for nothing of it: out_f += x . W^T.
// The decode step's query to latent is 4 MB of weights in a launch of 4.9 us, most of which is the launch's own start and end, while the feed-forward's down
// product (90 MB) runs on half of the CUs beside the attention.  With 33 MB of it in here this launch takes 8.5 us, 0.6 more than those alone would, and
// the attention's 14.4 instead of 20.0 (one row of 4 000 keys).  As many columns as tfl_latent_carry says.  Both workgroups are 512 threads of up
// to 128 registers, so that every CU holds one of each; the carried ones are the longer and come first.  Half a workgroup is a workgroup of
// latent_gemm_kernel: the same sums in the same order.
__global__ __launch_bounds__(512, 4) void latent_carry_kernel(const TflGemm a, const TflGemm g, const int carried, const int blocks) {
    __shared__ __align__(16) f32x4 part[8][2][64];
    if ((int)blockIdx.x < carried) {
        share_gemm_body<bf16, TFL_EPI_RESIDUAL, 1, false, 1, 4>(g, 0, 0, blockIdx.x, 0, (char*)part);
        return;
    }
    const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    latent_gemm_body<bf16, TFL_EPI_LATENT, 2, 1, 4, 8, false>(a, threadIdx.x & 255, 2 * ((int)blockIdx.x - carried) + half, blocks, 0, part + 4 * half);
}

template <typename T, int EPI, int P, bool TAIL, int MT, int U, class Src = FromMemory>
__global__ __launch_bounds__(512, 2) void share_gemm_kernel(const TflGemm a, const int tail_rows, const int tail_per) {
    extern __shared__ __align__(16) char share_smem[];
    share_gemm_body<T, EPI, P, TAIL, MT, U, Src>(a, tail_rows, tail_per, blockIdx.x, blockIdx.y, share_smem);
}

template <typename T, int EPI, int P, bool TAIL, int MT, class Src = FromMemory>
static int launch_share_rows(const TflGemm& a, int tail_rows, int tail_per, hipStream_t st) {
    constexpr int NP = P + (TAIL ? 1 : 0), LDS = 8 * NP * MT * 64 * (int)sizeof(f32x4);
    // Chunks asked for ahead: what the registers hold (seven panels and two row blocks 221; with one chunk ahead 1 792 panels of 4 096 took 51.8
    // us at 32 rows, more than 2 048 do, and 41.1 with two; eight panels and two row blocks would spill).
    constexpr int U = NP == 1 ? 4 : NP * MT <= 14 ? 2 : 1;
    static_assert(LDS <= 160 * 1024, "one workgroup's partial tiles");
    if (LDS > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)share_gemm_kernel<T, EPI, P, TAIL, MT, U, Src>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        if (e != hipSuccess) return (int)e;
    }
    const int panels = a.n >> 4;
    const dim3 grid(TAIL ? 256 : (panels + P - 1) / P, (a.rows + 16 * MT - 1) / (16 * MT));
    hipLaunchKernelGGL((share_gemm_kernel<T, EPI, P, TAIL, MT, U, Src>), grid, dim3(512), LDS, st, a, tail_rows, tail_per);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

template <typename T, int EPI, int P, bool TAIL>
static int launch_share(const TflGemm& a, int tail_rows, int tail_per, hipStream_t st) {
    if constexpr (EPI == TFL_EPI_RESIDUAL && sizeof(T) == 2) { // (forms of their own: asked about in these, one row, six layer runs, eight steps 4 134 -> 4 162 us)
        if (a.n_also > 0) return launch_share_rows<T, EPI, P, TAIL, 2, FromMemoryAlso>(a, tail_rows, tail_per, st);
    }
    return a.rows <= 16 ? launch_share_rows<T, EPI, P, TAIL, 1>(a, tail_rows, tail_per, st)
                        : launch_share_rows<T, EPI, P, TAIL, 2>(a, tail_rows, tail_per, st);
}

// TF_ERANGE: not a shape of this form.
template <typename T, int EPI>
static int share_gemm(const TflGemm& a, hipStream_t st) {
    if (!a.chunk_major) return TF_ERANGE;
    const ShareShape f = share_shape(a.n >> 4, EPI == TFL_EPI_GLU, EPI == TFL_EPI_IN ? a.n_raw : 0, a.rows);
    const int left = f.left, per = f.rest;
    if (per == 0) switch (f.each) {
        case 1: return launch_share<T, EPI, 1, false>(a, 0, 0, st);
        case 2: return launch_share<T, EPI, 2, false>(a, 0, 0, st);
        case 3: return launch_share<T, EPI, 3, false>(a, 0, 0, st);
        case 4: return launch_share<T, EPI, 4, false>(a, 0, 0, st);
        case 5: return launch_share<T, EPI, 5, false>(a, 0, 0, st);
        case 6: return launch_share<T, EPI, 6, false>(a, 0, 0, st);
        case 7: return launch_share<T, EPI, 7, false>(a, 0, 0, st);
        case 8: return launch_share<T, EPI, 8, false>(a, 0, 0, st);
        default: return TF_ERANGE;
    }
    switch (f.each) {
        case 1: return launch_share<T, EPI, 1, true>(a, left, per, st);
        case 2: return launch_share<T, EPI, 2, true>(a, left, per, st);
        case 3: return launch_share<T, EPI, 3, true>(a, left, per, st);
        case 4: return launch_share<T, EPI, 4, true>(a, left, per, st);
        case 5: return launch_share<T, EPI, 5, true>(a, left, per, st);
        case 6: return launch_share<T, EPI, 6, true>(a, left, per, st);
        case 7: return launch_share<T, EPI, 7, true>(a, left, per, st);
        default: return TF_ERANGE;
    }
}

template <typename T, int EPI, int P, int WAVES, int U, bool AHEAD>
static int launch_form(const TflGemm& a, hipStream_t st) {
    const int panels = (a.n >> 4) * a.groups;
    // Two row blocks of 16 share a workgroup's weights, and take its CU's time for twice the rows of x.  Up to 64 rows they go to workgroups of their own as long as
    // there is a CU for each.  us, bfloat16 | float32, together -> apart: TOKEN at 17 / 32 / 64 rows, 256 x 4 096 7.1 / 7.6 / 7.4 -> 6.0 / 6.3 / 6.1 | 23.1 / 23.7 / 21.3 -> 11.9 /
    // 12.9 / 12.1, 256 x 8 192 11.7 / 13.8 / 12.8 -> 9.0 / 9.7 / 9.3; GATED of 64 panels 3.5 / 3.8 / 3.8 -> 3.4 / 3.4 / 3.4 | 5.4 / 5.9 / 5.6 -> 4.4 / 4.4 / 4.3, of 128 at 17 / 32 rows
    // 3.6 / 3.9 -> 3.5 / 3.5 | 5.6 / 6.0 -> 4.5 / 4.6.  With fewer CUs than workgroups GATED is slower for it: 128 panels at 33 / 64 rows 3.9 / 4.0 -> 5.4 / 5.4 | 5.6 / 5.9 -> 6.1 / 6.7,
    // 256 at 17 / 64 3.7 / 6.1 -> 3.7 / 6.2 | 6.1 / 12.0 -> 7.0 / 15.0.  QUERY of 384 panels and LATENT of 1 024 too (befidra decode 32 6 519 -> 6 578, 6 571).
    const bool apart = a.rows <= 64 && ((EPI == TFL_EPI_TOKEN && panels <= 64) || (EPI == TFL_EPI_GATED && panels * ((a.rows + 15) / 16) <= 256));
    const int mt = a.rows <= 16 || apart ? 1 : 2, rb = (a.rows + 16 * mt - 1) / (16 * mt);
    const int extra = EPI == TFL_EPI_QUERY && a.kv_raw ? (a.rows + rb - 1) / rb : 0;
    const dim3 grid((panels + P - 1) / P + extra, rb), block(64 * WAVES);
    if (mt == 1) hipLaunchKernelGGL((latent_gemm_kernel<T, EPI, P, 1, WAVES, U, AHEAD>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((latent_gemm_kernel<T, EPI, P, 2, WAVES, U, AHEAD>), grid, block, 0, st, a);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// Waves per panel by panel count (few panels: more waves keep the weight stream deep enough); wide outputs of more than 16 rows
// take two panels per workgroup.  The small products issue a wave's whole K range at once.
template <typename T, int EPI>
static int launch_gemm(const TflGemm& a, hipStream_t st) {
    const int panels = (a.n >> 4) * a.groups;
    if constexpr (sizeof(T) == 4) {
        return launch_form<T, EPI, 1, 8, 2, true>(a, st);
    } else if constexpr (EPI == TFL_EPI_IN || EPI == TFL_EPI_F32 || EPI == TFL_EPI_RESIDUAL || EPI == TFL_EPI_GLU) {
        const int rc = share_gemm<T, EPI>(a, st);
        if (rc != TF_ERANGE) return rc;
        if (panels >= 2 * TFL_PAIR_MIN && a.rows > 16) return launch_form<T, EPI, 2, 4, 4, true>(a, st);
        if (panels > 512) return launch_form<T, EPI, 1, 4, 4, true>(a, st);
        if (panels > 128) return launch_form<T, EPI, 1, 8, 4, true>(a, st);
        return launch_form<T, EPI, 1, 16, 4, true>(a, st);
    } else {
        if (panels > 512) return launch_form<T, EPI, 1, 4, 8, false>(a, st);
        if (panels > 128) return launch_form<T, EPI, 1, 8, 8, false>(a, st);
        return launch_form<T, EPI, 1, 16, 8, false>(a, st);
    }
}

template <typename T>
static int dispatch_gemm(const TflGemm& a, int epi, hipStream_t st) {
    switch (epi) {
        case TFL_EPI_F32: return launch_gemm<T, TFL_EPI_F32>(a, st);
        case TFL_EPI_IN: return launch_gemm<T, TFL_EPI_IN>(a, st);
        case TFL_EPI_QUERY: return launch_gemm<T, TFL_EPI_QUERY>(a, st);
        case TFL_EPI_LATENT: return launch_gemm<T, TFL_EPI_LATENT>(a, st);
        case TFL_EPI_GATED: return launch_gemm<T, TFL_EPI_GATED>(a, st);
        case TFL_EPI_RESIDUAL: return launch_gemm<T, TFL_EPI_RESIDUAL>(a, st);
        case TFL_EPI_TOKEN: return launch_gemm<T, TFL_EPI_TOKEN>(a, st);
        case TFL_EPI_GLU: return launch_gemm<T, TFL_EPI_GLU>(a, st);
    }
    return TF_EINVAL;
}

// What an epilogue asks of its operands.
static int check_gemm(const TflGemm& a, int dtype, int epi) {
    if (a.n_also && (epi != TFL_EPI_RESIDUAL || dtype != 0)) return TF_EINVAL;
    switch (epi) {
        case TFL_EPI_F32:
            if (!a.out_f || a.groups != 1 || a.n_real < 1 || a.n_real > a.n || a.ld_f < a.n_real) return TF_EINVAL;
            break;
        case TFL_EPI_IN:
            if (!a.out_f || !a.ss_out || a.groups != 1 || a.n_raw < 16 || (a.n_raw & 15) || a.n_raw > a.n || a.ld_f < a.n_raw
                || (a.ld_f & 3) || a.ss_ld < a.n_raw / 16 || a.n_scaled < 0
                || (a.n_scaled & 15) || a.n_scaled > a.n_raw || (a.n_scaled && (!a.norm_w || !a.out_t2))) return TF_EINVAL;
            if (a.n_raw < a.n && (!a.out_t || (a.ld_t & 7) || a.ld_t < 8)) return TF_EINVAL;
            break;
        case TFL_EPI_QUERY:
            if (!a.out_t || !a.out_t2 || !a.pos || a.groups != 1 || a.H < 1 || a.N < 16 || a.R < 0 || a.C < 16) return TF_EINVAL;
            if ((a.N & 15) || (a.R & 15) || (a.C & 15) || a.n != a.H * (a.N + a.R)) return TF_EINVAL;
            if (!a.ss_in || a.ss_n < 2 || (a.ss_n & 1) || (a.ss_ld & 1) || a.ss_ld < a.ss_n || a.k_real < 1 || a.k_real > a.k) return TF_EINVAL;
            if (a.half < 0 || 2 * a.half > a.R || a.max_pos < 1 || (a.half && (!a.cos || !a.sin))) return TF_EINVAL;
            if (a.kv_raw && (!a.kv_norm_w || !a.cache || !a.slot || a.ld_kv < a.C + a.R || a.c_real < 1 || a.c_real > a.C
                             || a.cache_rows < 1)) return TF_EINVAL;
            break;
        case TFL_EPI_LATENT:
            if (!a.out_t || a.groups != a.H || a.C != a.n || a.R < 0 || (a.R & 3)) return TF_EINVAL;
            break;
        case TFL_EPI_GATED:
            if (!a.out_t || !a.gate || a.ld_t < 8 || a.ld_gate < (int64_t)a.groups * a.n || (a.ld_t & 7) || (a.ld_gate & 3)) return TF_EINVAL;
            break;
        case TFL_EPI_RESIDUAL:
            if (a.n_also < 0 || a.n_also > 4 || (a.n_also && (a.rows <= 16 || !a.also || !at16(a.also) || !a.chunk_major || share_shape(a.n >> 4, false, 0, a.rows).each == 0))) return TF_EINVAL;
            if (!a.out_f || a.groups != 1 || a.ld_f < a.n || (a.ld_f & 3) || (a.out_t && (a.ld_t < 8 || (a.ld_t & 7)))) return TF_EINVAL;
            break;
        case TFL_EPI_TOKEN:
            if (!a.out_t || !a.ids || !a.tok_table || a.groups != 1 || a.n_real < 1 || a.n_real > a.n || a.ld_tok < a.n_real
                || a.ld_t < a.n || (a.ld_t & 3) || a.vocab < 1) return TF_EINVAL;
            break;
        case TFL_EPI_GLU:
            if (!a.out_t || a.groups != 1 || a.ld_t < 8 || (a.ld_t & 7)) return TF_EINVAL;
            break;
        default:
            return TF_EINVAL;
    }
    return TF_OK;
}

extern "C" int tfl_gemm(const TflGemm* p, int dtype, int epi, void* stream) {
    if (!p || !p->wp || !p->x) return TF_EINVAL;
    const TflGemm a = *p;
    if (a.rows < 1 || a.rows > (1 << 20) || a.n < 16 || (a.n & 15) || a.k < 32 || (a.k & 31) || a.groups < 1) return TF_EINVAL;
    if ((a.ld_x & 7) || (a.x_group & 7) || a.x_oct < 8 || (a.x_oct & 7) || a.ld_x < 8) return TF_EINVAL;
    if (a.chunk_major != 0 && (a.chunk_major != 1 || a.groups != 1)) return TF_EINVAL;
    if (a.out_t && (a.t_oct < 8 || (a.t_oct & 7))) return TF_EINVAL;
    if (dtype != 0 && dtype != 1) return TF_EINVAL;
    const int rc = check_gemm(a, dtype, epi);
    if (rc != TF_OK) return rc;
    return dtype == 0 ? dispatch_gemm<bf16>(a, epi, (hipStream_t)stream) : dispatch_gemm<float>(a, epi, (hipStream_t)stream);
}

extern "C" int tfl_gemm_carry(const TflGemm* p, const TflGemm* carried, void* stream) {
    if (!p || !p->wp || !p->x || !carried) return TF_EINVAL;
    const TflGemm a = *p, g = *carried;
    if (a.rows < 1 || a.rows > 16 || a.n < 64 || (a.n & 63) || a.n > (1 << 16) || a.k < 32 || (a.k & 31) || a.groups < 1 || a.groups > 4096 || a.chunk_major != 0
        || (a.ld_x & 7) || (a.x_group & 7) || a.x_oct < 8 || (a.x_oct & 7) || a.ld_x < 8) return TF_EINVAL;
    if (!g.wp || !g.x || !g.out_f || g.out_t || g.rows != a.rows || g.n < 16 || (g.n & 15) || g.n > (1 << 16) || g.k < 32 || (g.k & 31) || g.groups != 1 || g.chunk_major != 1
        || (g.ld_x & 7) || g.ld_x < 8 || g.x_oct < 8 || (g.x_oct & 7) || g.ld_f < g.n || (g.ld_f & 3)) return TF_EINVAL;
    const int rc = check_gemm(a, 0, TFL_EPI_LATENT);
    if (rc != TF_OK) return rc;
    const int blocks = (a.n >> 5) * a.groups, carry = g.n >> 4;            // (an even number of pairs of panels: n in 64s)
    hipLaunchKernelGGL(latent_carry_kernel, dim3(carry + blocks / 2), dim3(512), 0, (hipStream_t)stream, a, g, carry, blocks);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}
