// One-workgroup-per-CU form of the skinny GEMM and the epilogues of four outputs a lane: for the launches of tile_gemm.hip, and for launches
// that have CUs to spare beside other work.
#pragma once
#include "tile_common.h"

// What one lane does with four finished outputs n .. n+3 of batch row m (`s`); panel-wide parts (sums of squares, gate | up pairs) are
// its caller's.
// old: RESIDUAL's fp32 residual there.
template <typename T, int EPI>
__device__ __forceinline__ void finish_quad(const TflGemm& a, int m, int n, f32x4 s, f32x4 old) {
    if constexpr (EPI == TFL_EPI_F32) {
        float* y = a.out_f + (int64_t)m * a.ld_f + n;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < a.n_real) y[r] = s[r];
    } else if constexpr (EPI == TFL_EPI_RESIDUAL) {
        f32x4 o = old;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] += s[r];
        *reinterpret_cast<f32x4*>(a.out_f + (int64_t)m * a.ld_f + n) = o;
        if (a.out_t) store_quad((T*)a.out_t + (int64_t)m * a.ld_t + (n >> 3) * a.t_oct + (n & 7), o);
    } else {                                                 // IN behind its raw part
        static_assert(EPI == TFL_EPI_IN, "quad epilogues");
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] = gelu_tanh(s[r]);
        const int k = n - a.n_raw;
        store_quad((T*)a.out_t + (int64_t)m * a.ld_t + (k >> 3) * a.t_oct + (k & 7), s);
    }
}

// IN's raw part: outputs n .. n+3 of a panel that all lanes of the wave hold (g = quad of the panel, i = row); w: their norm weights.
template <typename T>
__device__ __forceinline__ void finish_raw(const TflGemm& a, int m, bool live, int pin, int n, int g, f32x4 s, f32x4 w) {
    float q = s[0] * s[0] + s[1] * s[1] + s[2] * s[2] + s[3] * s[3];
    q = rows_sum(q);
    if (!live) return;
    *reinterpret_cast<f32x4*>(a.out_f + (int64_t)m * a.ld_f + n) = s;
    if (n < a.n_scaled) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] *= w[r];
        store_quad((T*)a.out_t2 + (int64_t)m * 8 + (n >> 3) * (8 * (int64_t)a.rows) + (n & 7), s);
    }
    if (g == 0) a.ss_out[(int64_t)m * a.ss_ld + pin] = q;
}

// The wide outputs: one workgroup per CU, each with P whole panels and tail_per more rows (0, 4, 8 or 12) of what 256 workgroups
// leave over, over weights packed chunk-major.  Bound by the weight stream.  Three things held the workgroup-per-panel form back:
//   * a few CUs with one panel more than the rest: 1 028 panels of 4 096 took 1.9 us (1 row) to 6.7 us (32 rows) longer than 1 024.
//     Here all CUs have the same share to within four rows; the rows left over are MFMA tiles whose upper rows repeat the
//     last one (the same addresses, no traffic), for gate | up panels dealt in quads of two gate and the same two up rows;
//   * every workgroup read all of x (256 KB at 32 rows: twice the weights' bytes, from L2) and asked for it right before its use: here
//     once per CU, and U chunks ahead like the weights;
//   * one private stream per wave, panels a power of two apart: chunk-major, the chip reads one moving window per wave index.  (The same
//     kernel on panel-major weights is slower than the old form up to 8 rows: 28.4 us at 1 076 panels.)
// us before -> now at 1 / 8 / 32 rows, K 4 096: 256 panels 10.5 / 10.4 / 11.9 -> 7.8 / 8.1 / 10.7, 512: 13.9 / 14.8 / 20.5 -> 12.9 / 12.8 /
// 15.6, 1 076: 27.9 / 29.2 / 39.5 -> 24.5 / 24.3 / 26.6, 1 376: 34.2 / 34.7 / 41.9 -> 30.5 / 29.6 / 31.5, 2 000: 44.6 / 45.9 / 56.5 -> 43.4 /
// 43.6 / 46.1 (6.0 TB/s); 256 panels of 15 104: 26.9 / 28.7 / 36.5 -> 21.2 / 22.2 / 32.9 (5.8 TB/s).
// cu: this workgroup's place among those that share the panels, mb: its block of rows.
// Src: where x comes from.  FromMemory: a.x, asked for with the weights.  Otherwise (INSIDE, one block of rows) the workgroup makes it itself under the first
// two batches of weights: src.ask() issues its loads in front of them, src.make() leaves x in LDS, octet-major, and ends with a barrier.
// SCALED: row m of the result is a.x's times 1 / sqrt(sum(a.ss_in[m]) / a.k_real + a.eps) before anything else is done with it; what is asked for in front of
// the weights is added up while the first of them come.  TILE: src.ask_tile() and src.put_tile() in the place of an epilogue (one tile a wave, whole panels).
// ALSO: RESIDUAL adds a.n_also further parts of the sum.
struct FromMemory { static constexpr bool INSIDE = false, SCALED = false, TILE = false, ALSO = false; };
struct FromMemoryScaled { static constexpr bool INSIDE = false, SCALED = true, TILE = false, ALSO = false; };
struct FromMemoryAlso { static constexpr bool INSIDE = false, SCALED = false, TILE = false, ALSO = true; };
template <typename T, int EPI, int P, bool TAIL, int MT, int U, class Src = FromMemory>
__device__ __forceinline__ void share_gemm_body(const TflGemm& a, const int tail_rows, const int tail_per, const int cu, const int mb, char* share_smem,
                                                Src src = Src()) {
    typedef typename El<T>::Frag Frag;
    constexpr int WAVES = 8, NP = P + (TAIL ? 1 : 0), CUS = 256;
    f32x4 (*part)[NP * MT][64] = reinterpret_cast<f32x4 (*)[NP * MT][64]>(share_smem);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int npan = a.n >> 4, panel0 = cu * P, m0 = mb * 16 * MT;
    const int chunks = a.k >> 5, per = (chunks + WAVES - 1) / WAVES;
    const int c_beg = wave * per, n_own = min(chunks, c_beg + per) - c_beg;
    // (the waves' ranges start K/8 chunks apart, a power of two for most K: in step they would ask the same few channels)
    const int rot = n_own > 0 ? 2 * wave % n_own : 0;
    const int64_t wstep = (int64_t)npan * 512;               // one chunk of all panels
    const T* wp[NP];
#pragma unroll
    for (int p = 0; p < P; ++p) wp[p] = (const T*)a.wp + min(panel0 + p, npan - 1) * 512 + lane * 8;
    // The rows left over are dealt in fours of workgroups on one XCD: four rows are 64 bytes of a chunk's 256, and a cache line that two XCDs ask for is
    // fetched twice.  us at 1 / 8 / 32 rows, workgroup by workgroup -> here, K 4 096: 1 076 panels 25.1 / 24.9 / 26.9 -> 24.5 / 24.3 / 26.6, 1 172 25.8 /
    // 26.1 / 28.4 -> 25.0 / 25.3 / 28.0, gate | up of 1 376 31.9 / 31.0 / 32.3 -> 30.5 / 29.6 / 31.5 (5.9 to 6.1 TB/s).
    const int tail0 = ((cu & ~31) | (cu & 7) << 2 | (cu >> 3 & 3)) * tail_per;
    if constexpr (TAIL) {
        const int row = min(min(tail0 + i, tail0 + tail_per - 1), tail_rows - 1);
        int slot = row & 15;
        if constexpr (EPI == TFL_EPI_GLU) slot = ((slot >> 2) << 1) + (slot & 1) + ((slot & 2) << 2);
        wp[P] = (const T*)a.wp + (CUS * P + (row >> 4)) * 512 + g * 128 + slot * 8;
    }
    const T* xp[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xp[t] = (const T*)a.x + (int64_t)min(m0 + 16 * t + i, a.rows - 1) * a.ld_x + g * a.x_oct;
    const int64_t xstep = 4 * a.x_oct;
    f32x4 acc[NP][MT];
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[p][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto chunk = [&](int o) {                                // (past the end: the last chunk again, not used)
        const int c = min(o, n_own - 1) + rot;
        return c_beg + (c >= n_own ? c - n_own : c);
    };
    auto load = [&](Frag (&w)[U][NP], Frag (&x)[U][MT], int c0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = chunk(c0 + u);
#pragma unroll
            for (int p = 0; p < NP; ++p) w[u][p] = load_frag_stream(wp[p] + wstep * c);
            if constexpr (!Src::INSIDE) {
#pragma unroll
                for (int t = 0; t < MT; ++t) x[u][t] = load_frag(xp[t] + xstep * c);
            }
        }
    };
    auto multiply = [&](const Frag (&w)[U][NP], const Frag (&x)[U][MT], int c0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c0 + u < n_own) {
#pragma unroll
                for (int p = 0; p < NP; ++p)
#pragma unroll
                    for (int t = 0; t < MT; ++t) acc[p][t] = El<T>::mma(w[u][p], x[u][t], acc[p][t]);
            }
    };
    // What the epilogue of result tile j (row block t of panel or left-over tile p) reads: of a wave's first one asked for in front of the weights,
    // not behind the products, where nothing is left to hide it (4 096 x 4 096 onto the residual, 1 / 32 rows: 7.90 -> 7.43 us, 11.83 -> 11.34).
    auto beside = [&](int j) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if constexpr (EPI == TFL_EPI_RESIDUAL || EPI == TFL_EPI_IN) {
            const int p = j / MT, m = m0 + 16 * (j - p * MT) + i, row = tail0 + 4 * g;
            const bool whole = !TAIL || p < P;
            const int n = whole ? 16 * (panel0 + p) + 4 * g : 16 * CUS * P + row;
            if (j < NP * MT && (whole ? panel0 + p < npan : 4 * g < tail_per && row < tail_rows)) {
                if constexpr (EPI == TFL_EPI_IN) {
                    if (whole && n < a.n_scaled) v = *reinterpret_cast<const f32x4*>(a.norm_w + n);
                } else {
                    v = *reinterpret_cast<const f32x4*>(a.out_f + (int64_t)min(m, a.rows - 1) * a.ld_f + n);
                }
            }
        }
        return v;
    };
    const f32x4 first = beside(wave);
    [[maybe_unused]] f32x4 more[4];                           // ALSO: of the wave's first tile
    [[maybe_unused]] auto also_at = [&](int j, int q) {
        const int p = j / MT, m = m0 + 16 * (j - p * MT) + i;
        const int n = !TAIL || p < P ? min(16 * (panel0 + p) + 4 * g, a.n - 4) : min(16 * CUS * P + tail0 + 4 * g, a.n - 4);
        return *reinterpret_cast<const f32x4*>(a.also + ((int64_t)q * a.rows + min(m, a.rows - 1)) * a.n + n);
    };
    if constexpr (Src::ALSO) {
        static_assert(EPI == TFL_EPI_RESIDUAL, "sums to be added");
        if (wave < NP * MT) {
#pragma unroll
            for (int q = 0; q < 4; ++q) more[q] = also_at(wave, min(q, a.n_also - 1));
        }
    }
    if constexpr (Src::TILE)
        if (wave < NP * MT) src.ask_tile(min(m0 + 16 * (wave % MT) + i, a.rows - 1), 16 * (panel0 + min(wave / MT, NP - 1)) + 4 * g);
    constexpr int TPR = 512 / (16 * MT), SQ = 128 / TPR;      // SCALED: threads a row, quads of its sums of squares each (512 sums)
    [[maybe_unused]] f32x4 sq[SQ];
    [[maybe_unused]] float* const scale = reinterpret_cast<float*>(share_smem + sizeof(f32x4) * WAVES * NP * MT * 64);
    if constexpr (Src::SCALED) {
        const float* ss = a.ss_in + (int64_t)min(m0 + tid / TPR, a.rows - 1) * a.ss_ld;
#pragma unroll
        for (int u = 0; u < SQ; ++u) sq[u] = *reinterpret_cast<const f32x4*>(ss + 4 * min(tid % TPR + u * TPR, (a.ss_n >> 2) - 1));
    }
    [[maybe_unused]] auto row_scales = [&] {
        float q = 0.f;
#pragma unroll
        for (int u = 0; u < SQ; ++u)
            if (tid % TPR + u * TPR < a.ss_n >> 2) q += (sq[u][0] + sq[u][1]) + (sq[u][2] + sq[u][3]);
        q += lane_rotated<8>(q);
        q += lane_rotated<4>(q);
        q += lane_rotated<2>(q);
        q += lane_rotated<1>(q);
        if constexpr (TPR == 32) {
            const LanePair<float> r = lane_rows(q);
            q = r.a + r.b;
        }
        if (tid % TPR == 0) scale[tid / TPR] = 1.0f / sqrtf(q / (float)a.k_real + a.eps);
    };
    asm volatile("" ::: "memory");
    if constexpr (Src::INSIDE) {
        static_assert(MT == 1, "one block of rows");
        Frag wa[U][NP], wb[U][NP], x[U][MT];
        src.ask();
        asm volatile("" ::: "memory");
        if (n_own > 0) {
            load(wa, x, 0);
            load(wb, x, U);
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const T* xs = src.make(cu) + (g * a.rows + min(i, a.rows - 1)) * 8;
        auto take = [&](int c0) {
#pragma unroll
            for (int u = 0; u < U; ++u) x[u][0] = load_frag(xs + chunk(c0 + u) * 32 * a.rows);
        };
        if (n_own > 0) {
            int c0 = 0;
            for (; c0 + 2 * U < n_own; c0 += 2 * U) {
                take(c0);
                multiply(wa, x, c0);
                load(wa, x, c0 + 2 * U);
                take(c0 + U);
                multiply(wb, x, c0 + U);
                load(wb, x, c0 + 3 * U);
            }
            take(c0);
            multiply(wa, x, c0);
            take(c0 + U);
            multiply(wb, x, c0 + U);
        }
    } else {
        Frag wa[U][NP], xa[U][MT], wb[U][NP], xb[U][MT];
        if (n_own > 0) load(wa, xa, 0);
        if constexpr (Src::SCALED) {
            __builtin_amdgcn_sched_barrier(0);
            row_scales();
        }
        for (int c0 = 0; c0 < n_own; c0 += 2 * U) {
            load(wb, xb, c0 + U);
            multiply(wa, xa, c0);
            if (c0 + U >= n_own) break;
            load(wa, xa, c0 + 2 * U);
            multiply(wb, xb, c0 + U);
        }
    }
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int t = 0; t < MT; ++t) part[wave][p * MT + t][lane] = acc[p][t];
    __syncthreads();
    for (int j = wave; j < NP * MT; j += WAVES) {            // row block t of tile p: the waves' sums, in wave order
        const int p = j / MT, t = j - p * MT, m = m0 + 16 * t + i;
        f32x4 s = part[0][j][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) {
            const f32x4 o = part[w][j][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] += o[r];
        }
        if constexpr (Src::SCALED) {
            const float by = scale[16 * t + i];
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] *= by;
        }
        const bool live = m < a.rows;
        if constexpr (Src::TILE) {
            static_assert(!TAIL && NP * MT <= WAVES, "one tile a wave");
            src.put_tile(m, live, panel0 + p, npan, g, s);
            continue;
        }
        const f32x4 with = j == wave ? first : beside(j);
        if constexpr (Src::ALSO) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (q < a.n_also) {
                    const f32x4 o = j == wave ? more[q] : also_at(j, q);
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[r] += o[r];
                }
        }
        if (!TAIL || p < P) {
            const int panel = panel0 + p, n = 16 * panel + 4 * g;
            if (panel >= npan) continue;
            if constexpr (EPI == TFL_EPI_GLU) {              // lanes g < 2 hold gate rows, g + 2 the same outputs' up rows
                f32x4 up;
#pragma unroll
                for (int r = 0; r < 4; ++r) up[r] = other_half(s[r]);
                if (live && g < 2) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[r] = gelu_tanh(s[r]) * up[r];
                    store_quad((T*)a.out_t + (int64_t)m * a.ld_t + panel * a.t_oct + 4 * g, s);
                }
            } else {
                if constexpr (EPI == TFL_EPI_IN) {
                    if (16 * panel < a.n_raw) {
                        finish_raw<T>(a, m, live, panel, n, g, s, with);
                        continue;
                    }
                }
                if (live) finish_quad<T, EPI>(a, m, n, s, with);
            }
        } else {
            const int row = tail0 + 4 * g;   // first of this lane's four left-over rows
            if (!live || 4 * g >= tail_per || row >= tail_rows) continue;
            if constexpr (EPI == TFL_EPI_GLU) {              // gate, gate, up, up of outputs 2q, 2q + 1 of a panel's octet
                typedef T Pair __attribute__((ext_vector_type(2)));
                const Pair y = {(T)(gelu_tanh(s[0]) * s[2]), (T)(gelu_tanh(s[1]) * s[3])};
                *reinterpret_cast<Pair*>((T*)a.out_t + (int64_t)m * a.ld_t + (CUS * P + (row >> 4)) * a.t_oct + ((row & 15) >> 1)) = y;
            } else {
                finish_quad<T, EPI>(a, m, 16 * CUS * P + row, s, with);
            }
        }
    }
}
