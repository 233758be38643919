// Prefill attention of contexts that come from memory: 256 query rows per workgroup, 64 per wave and one wave per SIMD, heads of 128 in fp16.
//
// The loop of attn_prefill_ahead_body reads every key and value fragment from LDS for 32 query rows; here one read serves 64, and a workgroup's tile
// comes in once for 256 rows instead of 128.  Past the Infinity Cache that loop is bound by what the matrix cores, LDS and memory draw
// together, and what they draw less the clock makes up: 32 heads, 4 096 rows x 65 536 keys 4 118 -> 3 847 us (1.11 PFLOP/s), x 124 928
// 8 012 -> 7 300.  (All data zero, at full clock: 3 310 and 3 390.)
// One wave has to hide everything itself: every product is followed by two operations at most (a wave issues one in five cycles, a product
// takes sixteen), in an order fixed here, half a tile of 32 keys at a time: scores of the next half beside the exponentials of this one, then its
// values beside the maxima of the next.  K and V come in by LDS-DMA, four tiles deep, the waves meet once per tile.  Sums and scores are written
// in place by inline asm, which the compiler would copy; a rescale of 128 sums is one block of asm with its own branches for the same reason.
#pragma once
#include "common.h"
#include "lds_dma.h"

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef h16 half2v __attribute__((ext_vector_type(2)));

struct PrefillWide {
    typedef half8 Frag;
    typedef __attribute__((address_space(3))) const char* Lds;
    static constexpr int KT = 64, QT = 4, NC = 4, NT = 8, D = 128, ROWS = 256, SLOTS = 4, TILE = 2 * KT * D, LDS = 2 * SLOTS * TILE;
    struct Tile { const h16 *k, *v; int last; };              // first rows of a tile, and the last row that may be read
    Frag q[QT][NC];
    f32x4 acc[QT][NT];
    float l[QT];

    template <int N> struct Num { static constexpr int value = N; };
    template <int N, int B = 0, class F> static __device__ __forceinline__ void each(F&& f) {
        if constexpr (B < N) {
            f(Num<B>{});
            each<N, B + 1>(f);
        }
    }
    static __device__ __forceinline__ void first(Frag a, Frag b, f32x4& c) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=&v"(c) : "a"(a), "a"(b)); }
    static __device__ __forceinline__ void more(Frag a, Frag b, f32x4& c) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "a"(a), "a"(b)); }
    static __device__ __forceinline__ void value(Frag a, uint4v b, f32x4& c) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "a"(a), "v"(b)); }
    static __device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
    template <int LEFT> static __device__ __forceinline__ void meet() { meet_dma<LEFT, false>(); }

    // tile(t): the Tile; whole(k0): every row of the wave sees all 32 keys from k0 on (wave-uniform); otherwise query u sees lo[u] .. hi[u].
    // load() fills q, lo and hi.  k_ld: elements from row to row (63 rows stay below 2^32 bytes).
    // A wave multiplies the tiles up to t_own, its last row's (wave-uniform), and brings in its part of the others: a hidden weight of 0 times a value that
    // is not finite is no number, so what a row does not see must end with its wave's 64 rows and not with the workgroup's 256.
    template <class Load, class Src, class Whole>
    __device__ __forceinline__ void run(char* smem, int t_beg, int t_own, int t_end, uint32_t k_ld, float scale, const int (&lo)[QT], const int (&hi)[QT], Load&& load,
                                        Src&& tile, Whole&& whole) {
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, i = lane & 15;
        const float sc = scale * 1.4426950408889634f;
        const int lr = tid >> 4, lc = tid & 15;
        const uint32_t row = 2 * k_ld, lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
        const uint32_t piece = 16 * (lc ^ ((lr & 3) | (((lr >> 3) & 3) << 2)));
        uint32_t k_off[4], v_off[4];                          // this lane's bytes from a tile's first row, 16 rows a pass
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            k_off[p] = (lr + 16 * p) * row + (piece ^ ((p & 1) * 128));
            v_off[p] = (lr + 16 * p) * row + 16 * ((((lc >> 1) ^ ((lr & 3) | (((lr >> 3) & 1) << 2))) << 1) | (lc & 1));
        }
        auto dma = [&](const uint4v& src, uint32_t off, uint32_t dst) __attribute__((always_inline)) {
            const uint32_t at = __builtin_amdgcn_readfirstlane(dst);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(at), "v"(off), "s"(src) : "memory", "m0");
        };
        // a tile as a buffer that ends with its last row: what lies behind comes in as zeros
        auto source = [&](const h16* base, int last) __attribute__((always_inline)) {
            const uint64_t a = (uint64_t)base;
            return uint4v{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)last * row + 2 * D, 0x00020000};
        };
        auto at_tile = [&](int t) __attribute__((always_inline)) { return tile(min(t, t_end - 1)); };
        const uint32_t mine = lds + 1024 * wave;
        auto fetch_k = [&](const uint4v& src, uint32_t slot, int p) __attribute__((always_inline)) { dma(src, k_off[p], mine + slot + p * 4096); };
        auto fetch_v = [&](const uint4v& src, uint32_t slot, int p) __attribute__((always_inline)) { dma(src, v_off[p], mine + SLOTS * TILE + slot + p * 4096); };
        const int row_a = 8 * (i >> 2) + (i & 3);
        uint32_t kp = lds + row_a * 256 + 16 * (g ^ i), vp = lds + SLOTS * TILE + 2 * ((8 * g + (i >> 2)) * D + 4 * (i & 3) + 16 * ((i >> 2) | ((g & 1) << 2)));
        constexpr int KA = 2, VA = 4;
        Frag ka[KA + 1], kb[KA + 1], vf[NT];
        auto read_k = [&](int h, int n) __attribute__((always_inline)) {
            const Lds src = (Lds)(uintptr_t)(kp ^ (64 * n)) + h * 8192;
            ka[(4 * h + n) % (KA + 1)] = *(const __attribute__((address_space(3))) Frag*)src;
            kb[(4 * h + n) % (KA + 1)] = *(const __attribute__((address_space(3))) Frag*)(src + 1024);
        };
        auto read_v = [&](int h, int t) __attribute__((always_inline)) {
            const Lds src = (Lds)(uintptr_t)(vp ^ (32 * t)) + h * 8192;
            const half4 x = lds_read_tr4((const h16*)src), y = lds_read_tr4((const h16*)(src + 1024));
            vf[t] = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        float top[QT], raw[QT], m[QT], sum[QT];               // raw: the largest score of a row so far, m: the reference of its weights
        auto largest = [&](const f32x4 (&x)[2][QT], int u, int n) __attribute__((always_inline)) {
            if (n == 0) top[u] = vmax3_raw(x[0][u][0], x[0][u][1], x[0][u][2]);
            if (n == 1) top[u] = vmax3_raw(top[u], x[0][u][3], x[1][u][0]);
            if (n == 2) top[u] = vmax3_raw(top[u], x[1][u][1], x[1][u][2]);
            if (n == 3) top[u] = vmax_raw(top[u], x[1][u][3]);
        };
        auto hide = [&](f32x4 (&x)[2][QT], int k0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < QT; ++u) {
                const int first = lo[u] - k0 - 8 * g, last = hi[u] - k0 - 8 * g;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    if (k > last || k < first) x[k >> 2][u][k & 3] = -__builtin_inff();
                    fence();
                }
            }
        };
        auto score = [&](f32x4 (&x)[2][QT], int h, int e) __attribute__((always_inline)) {
            const int n = e / 8, u = e % 8 / 2, z = e % 2;
            if (e % 8 == 0) asm volatile("" : "+a"(ka[(4 * h + n) % (KA + 1)]), "+a"(kb[(4 * h + n) % (KA + 1)]));       // one wait for both
            const Frag a = z ? kb[(4 * h + n) % (KA + 1)] : ka[(4 * h + n) % (KA + 1)];
            if (n == 0) first(a, q[u][0], x[z][u]);
            else more(a, q[u][n], x[z][u]);
        };
        auto across = [&](float x) __attribute__((always_inline)) {
            const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
            x = vmax_raw(__uint_as_float(a[0]), __uint_as_float(a[1]));
            const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
            return vmax_raw(__uint_as_float(b[0]), __uint_as_float(b[1]));
        };
        auto half_step = [&](f32x4 (&s)[2][QT], f32x4 (&next)[2][QT], auto half, int t, uint32_t slot) __attribute__((always_inline)) {
            constexpr int h = decltype(half)::value;
            uint4v p[QT];
            auto weight = [&](int e) __attribute__((always_inline)) {
                if (e < 32) {
                    const int u = e / 8, z = e % 8 / 4, r = e % 4;
                    float y = __builtin_amdgcn_exp2f(fmaf(s[z][u][r], sc, -m[u]));
                    s[z][u][r] = y;
                }
                if (e > 0) {
                    const int f = e - 1, u = f / 8, z = f % 8 / 4, r = f % 4;
                    if (h == 0 && f % 8 == 0) sum[u] = s[z][u][r];
                    else sum[u] += s[z][u][r];
                    if (f % 2) p[u][f % 8 / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{s[z][u][r - 1], s[z][u][r]}), half2v));
                }
            };
            each<32>([&](auto num) __attribute__((always_inline)) {
                constexpr int e = decltype(num)::value;
                score(next, h ^ 1, e);
                fence();
                if (e % 8 == 0 && e / 8 + KA < 4) read_k(h ^ 1, e / 8 + KA);
                if (e % 4 != 3) weight(e / 4 * 3 + e % 4);
                if (e >= 20 && e % 3 == 2) read_v(h, (e - 20) / 3);
                fence();
            });
            uint4v src;
            each<32>([&](auto num) __attribute__((always_inline)) {
                constexpr int e = decltype(num)::value, t_ = e % 16 / 2, u = e / 16 * 2 + e % 2;
                if (e < 16 && e % 4 == 0) asm volatile("" : "+a"(vf[t_]), "+a"(vf[t_ + 1]));
                value(vf[t_], p[u], acc[u][t_]);
                fence();
                if (e % 4 == 0 && e / 2 + VA < NT) { read_v(h, e / 2 + VA); read_v(h, e / 2 + VA + 1); }
                if (e <= 8) weight(24 + e);
                if (e == 9) {                                 // (nothing of the above into what follows the branch)
#pragma unroll
                    for (int w = 0; w < QT; ++w) asm volatile("" : "+v"(sum[w]), "+v"(p[w]));
                }
                if (e == 9 && !whole(t * KT + 32 * (h + 1))) hide(next, t * KT + 32 * (h + 1));
                if (e >= 10 && e < 26) largest(next, (e - 10) % 4, (e - 10) / 4);
                if (h == 0 && e == 12) {
                    meet<8>();                                // K[t + 1], V[t + 1]
                    kp += slot == 3 * TILE ? -3 * TILE : TILE;
                }
                if (e == 13) {
                    const Tile a = at_tile(t + 3);
                    src = source(h ? a.v : a.k, a.last);
                }
                if (h == 0 && e >= 14 && e < 30 && e % 4 == 2) fetch_k(src, (slot + 3 * TILE) & (3 * TILE), (e - 14) / 4);
                if (h == 1 && e >= 14 && e < 30 && e % 4 == 2) fetch_v(src, (slot + 3 * TILE) & (3 * TILE), (e - 14) / 4);
                if (e == 26 || e == 29) read_k(h, (e - 26) / 3);
                fence();
            });
            if (h == 1) {
                vp += slot == 3 * TILE ? -3 * TILE : TILE;
#pragma unroll
                for (int u = 0; u < QT; ++u) l[u] += sum[u];
            }
        };
        // a row with a new largest score gets a new reference
        auto refer = [&](bool both) __attribute__((always_inline)) {
            uint64_t far[QT];
#pragma unroll
            for (int u = 0; u < QT; ++u) far[u] = __builtin_amdgcn_ballot_w64(top[u] > raw[u]);
            const uint64_t any = far[0] | far[1] | far[2] | far[3];
            float w[QT] = {1.f, 1.f, 1.f, 1.f};
            if (any) {
#pragma unroll
                for (int u = 0; u < QT; ++u) {
                    raw[u] = fmaxf(raw[u], across(top[u]));
                    const float to = fmaxf(m[u], raw[u] * sc);
                    w[u] = __builtin_amdgcn_exp2f(m[u] - to);
                    m[u] = to;
                    l[u] *= w[u];
                    if (both) sum[u] *= w[u];
                }
            }
            float x[QT][NT][4];
#pragma unroll
            for (int u = 0; u < QT; ++u)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[u][t][r] = acc[u][t][r];
            fence();
#define W1(n, w) "v_mul_f32 %" #n ", %[" w "], %" #n "\n\t"
#define W8(a, b, c, d, e, f, g, h, w) W1(a, w) W1(b, w) W1(c, w) W1(d, w) W1(e, w) W1(f, w) W1(g, w) W1(h, w)
#define W32A(w) W8(0, 1, 2, 3, 4, 5, 6, 7, w) W8(8, 9, 10, 11, 12, 13, 14, 15, w) W8(16, 17, 18, 19, 20, 21, 22, 23, w) W8(24, 25, 26, 27, 28, 29, 30, 31, w)
#define W32B(w) W8(32, 33, 34, 35, 36, 37, 38, 39, w) W8(40, 41, 42, 43, 44, 45, 46, 47, w) W8(48, 49, 50, 51, 52, 53, 54, 55, w) W8(56, 57, 58, 59, 60, 61, 62, 63, w)
#define V4(u, t) "+v"(x[u][t][0]), "+v"(x[u][t][1]), "+v"(x[u][t][2]), "+v"(x[u][t][3])
#define V32(u) V4(u, 0), V4(u, 1), V4(u, 2), V4(u, 3), V4(u, 4), V4(u, 5), V4(u, 6), V4(u, 7)
#define RESCALE(u, v)                                                                                                              \
    asm volatile("s_cmp_eq_u64 %[any], 0\n\ts_cbranch_scc1 .Lall%=\n\ts_nop 11\n\t"                                               \
                 "s_cmp_eq_u64 %[fa], 0\n\ts_cbranch_scc1 .La%=\n\t" W32A("wa") ".La%=:\n\t"                                     \
                 "s_cmp_eq_u64 %[fb], 0\n\ts_cbranch_scc1 .Lb%=\n\t" W32B("wb") ".Lb%=:\n\t.Lall%=:"                              \
                 : V32(u), V32(v)                                                                                                  \
                 : [any] "s"(any), [fa] "s"(far[u]), [wa] "v"(w[u]), [fb] "s"(far[v]), [wb] "v"(w[v])                              \
                 : "scc")
            RESCALE(0, 1);
            RESCALE(2, 3);
#undef RESCALE
#undef V32
#undef V4
#undef W32B
#undef W32A
#undef W8
#undef W1
            fence();
#pragma unroll
            for (int u = 0; u < QT; ++u)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[u][t][r] = x[u][t][r];
        };

        load();
        {
            const Tile a = at_tile(t_beg);
            const uint4v k0 = source(a.k, a.last), v0 = source(a.v, a.last);
#pragma unroll
            for (int p = 0; p < 4; ++p) fetch_k(k0, 0, p);
#pragma unroll
            for (int u = 0; u < QT; ++u) {
#pragma unroll
                for (int c = 0; c < NC; ++c) asm volatile("" : "+a"(q[u][c]));
                m[u] = raw[u] = -__FLT_MAX__;
                l[u] = 0.f;
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            meet<0>();
#pragma unroll
            for (int p = 0; p < 4; ++p) fetch_v(v0, 0, p);
#pragma unroll
            for (int x = 1; x < 3; ++x) {
                const Tile b = at_tile(t_beg + x);
                const uint4v kx = source(b.k, b.last), vx = source(b.v, b.last);
#pragma unroll
                for (int p = 0; p < 4; ++p) fetch_k(kx, x * TILE, p);
#pragma unroll
                for (int p = 0; p < 4; ++p) fetch_v(vx, x * TILE, p);
            }
        }
        f32x4 sa[2][QT], sb[2][QT];
#pragma unroll
        for (int n = 0; n < KA; ++n) read_k(0, n);
        fence();
        each<32>([&](auto num) __attribute__((always_inline)) {
            constexpr int e = decltype(num)::value;
            score(sa, 0, e);
            fence();
            if (e % 8 == 0 && e / 8 + KA < 4) read_k(0, e / 8 + KA);
            if (e == 24 || e == 28) read_k(1, (e - 24) / 4);
            fence();
        });
        hold_sums();
        if (!whole(t_beg * KT)) hide(sa, t_beg * KT);
#pragma unroll
        for (int u = 0; u < QT; ++u) {
#pragma unroll
            for (int n = 0; n < 4; ++n) largest(sa, u, n);
            raw[u] = fmaxf(raw[u], across(top[u]));
            m[u] = fmaxf(m[u], raw[u] * sc);
        }
        meet<16>();                                           // V[0]
        uint32_t slot = 0;
        for (int t = t_beg; t < t_own; ++t) {
            half_step(sa, sb, Num<0>{}, t, slot);
            refer(true);
            half_step(sb, sa, Num<1>{}, t, slot);
            refer(false);
            slot = (slot + TILE) & (3 * TILE);
        }
        hold_sums();
#pragma unroll
        for (int u = 0; u < QT; ++u)
#pragma unroll
            for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(acc[u][t]));
        for (int t = t_own; t < t_end; ++t) {
            meet<8>();
            const Tile a = at_tile(t + 3);
            const uint4v k0 = source(a.k, a.last), v0 = source(a.v, a.last);
#pragma unroll
            for (int p = 0; p < 4; ++p) fetch_k(k0, (slot + 3 * TILE) & (3 * TILE), p);
#pragma unroll
            for (int p = 0; p < 4; ++p) fetch_v(v0, (slot + 3 * TILE) & (3 * TILE), p);
            slot = (slot + TILE) & (3 * TILE);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);                   // no load is under way when the LDS is given back
    }
    __device__ __forceinline__ float weight(int u) const {
        return rows_sum(l[u]);
    }
};

