// Products of many rows (prefill) in 16 bits: y = x . W^T, x [rows, k] and W [n, k] row-major, sums in fp32.
//
// Four waves per workgroup, one per SIMD, 16 MT rows x 16 NT outputs each; a step is 64 of k.  Operands come in by LDS-DMA in whole lines of 128
// bytes, the XOR that keeps the fragments' reads free of bank conflicts (measured: none) applied where the DMA reads from.  A half step's
// fragments are in registers before its first product, those of the next half are read beside its products, one read to three products, one
// DMA load to eight: in bursts they hold the products up (4 096 x 4 096 x 11 008, all loads behind a step's first products 315 us, one to
// four products in one half of the step 280, one to eight in both halves 266).  For the latter x has a step more in LDS than W: its loads
// may then begin before the waves have met.  No branch lies between the products of two steps (a test for the end of the tile there: 266 ->
// 250), so steps are counted in runs, and the loads run on into the next tile while this one is finished.
//
// Bound by power: at 8 000 x 12 288 x 4 096 the matrix cores are busy 77 % of the cycles at 1.79 GHz (the library's kernel: 81 % at 1.71, 0.97 to 1.0
// of the time), and other orders of reads, loads and meeting points give the same time to 1 %.  Four waves of 128 x 128 instead of eight of 128 x 64
// read a third less from LDS: as fast, and cooler.  Against the library's product (us, weights from memory; plan() picks tile and parts):
//   22 016 x 4 096:  130 rows 51 -> 55, 700 140 -> 141, 1 500 294 -> 236, 3 100 547 -> 425, 4 096 654 -> 556, 8 000 1 152 -> 1 027
//   4 096 x 11 008:  130 rows 49 -> 34, 700  89 ->  71, 1 500 129 -> 122, 3 100 221 -> 210, 4 096 243 -> 247, 8 000   480 -> 487
//   4 096 x 4 096:   130 rows 18 -> 13, 700  31 ->  33, 1 500  50 ->  50, 3 100  84 ->  80, 4 096  94 ->  99, 8 000   185 -> 191
// Where the library is still the faster one, and where it is taken: library_is_faster() of ops_rows.py.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace rg {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// add_in_place(): the same without the compiler's say in where the sum goes.  Of 192 to 256 registers of sums it moves some forty through others
// in every step, or spills them.  It does not see then what the matrix core still has to read or write either: see hold().
template <typename T> struct El;
template <> struct El<_Float16> {
    typedef _Float16 Frag __attribute__((ext_vector_type(8)));
    typedef _Float16 Pair __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ void add(Frag a, Frag b, f32x4& c) { c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ void add_in_place(Frag a, Frag b, f32x4& c) { asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
};
template <> struct El<__bf16> {
    typedef __bf16 Frag __attribute__((ext_vector_type(8)));
    typedef __bf16 Pair __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ void add(Frag a, Frag b, f32x4& c) { c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ void add_in_place(Frag a, Frag b, f32x4& c) { asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }
};
// Twelve wait states between products and what else touches their sums: behind a 16 x 16 x 32 product (eight passes) eleven are needed.  Behind the
// products of a step, inside their loop, so that no copy of a sum can come first.
__device__ __forceinline__ void hold() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 11" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// What becomes of the products: themselves; silu(gate) * up of W = [gate rows | up rows]; gelu(gate) * up of W in blocks of 8 gate | 8 up rows.
enum Form { PLAIN = 0, SILU_HALVES = 1, GELU_EIGHTS = 2 };

struct Args {
    const void *x, *w;
    void* out;
    float* ws;                                                // [splits][rows][n]
    int64_t ld_x, ld_out;
    int rows, n, k, splits;
};

template <typename T> __device__ __forceinline__ float rounded(float v) { return (float)(T)v; }
template <typename T> __device__ __forceinline__ uint32_t pack(float a, float b) {
    typename El<T>::Pair p = {(T)a, (T)b};
    return __builtin_bit_cast(uint32_t, p);
}
// As the decode forms of both units compute them: the silu of values rounded to T, the gelu of the sums.  exp2 and reciprocal of the hardware
// (1 ulp of fp32 each, in front of a rounding to T).
template <typename T, int FORM> __device__ __forceinline__ float glu(float gate, float up) {
    if constexpr (FORM == SILU_HALVES) {
        const float z = rounded<T>(gate), u = rounded<T>(up);
        return rounded<T>(z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z))) * u;
    }
    const float v = 0.7978845608028654f * (gate + 0.044715f * gate * gate * gate);
    return gate * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.0f * 1.4426950408889634f * v)) * up;
}

// All but the LEFT youngest loads of this wave have landed, its reads of LDS are done, and so are every other wave's; no access crosses.
template <int LEFT> __device__ __forceinline__ void meet() {
    static_assert(LEFT < 64, "six bits");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (LEFT & 15) | (LEFT >> 4 << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One part of a tile's k: where its steps of 64 begin, how many they are.
struct Item { int mt, nt, split, c_beg, steps; };
template <int BM, int BN> __device__ __forceinline__ Item item_of(const Args& a, int id) {
    const int mts = (a.rows + BM - 1) / BM, nts = (a.n + BN - 1) / BN, tiles = mts * nts;
    const int groups = (mts + 7) / 8, gs = (mts + groups - 1) / groups, nk = a.k >> 6, per = (nk + a.splits - 1) / a.splits;
    const int split = id / tiles, t = id - split * tiles, grp = t / (gs * nts), in = t - grp * gs * nts, gh = min(gs, mts - grp * gs);
    return Item{grp * gs + in % gh, in / gh, split, split * per, min(nk, (split + 1) * per) - split * per};
}

// NB steps of weights and one more of x are in LDS: x comes in during the first half of a step, weights during the second.
template <int MT, int NT, int NB> constexpr int lds_bytes() { return (4 * MT * (NB + 1) + 4 * NT * NB) * 1024; }

// 32 MT rows x 32 NT outputs per tile, four waves of 16 MT x 16 NT.
template <typename T, int MT, int NT, int NB, int FORM, int OCC>
__global__ __launch_bounds__(256, OCC) void rows_gemm_kernel(const Args a) {
    typedef typename El<T>::Frag Frag;
    constexpr int BM = 32 * MT, BN = 32 * NT, XG = 4 * MT, PER = MT + NT, XS = 4096 * MT, WS = 4096 * NT, NX = NB + 1, S = MT * NT;
    constexpr bool IN_PLACE = S >= 48;
    constexpr int RS = S / (PER + 2) > 0 ? S / (PER + 2) : 1, LAST = (PER - 1) * RS;       // reads of a half step: one in RS products
    constexpr int XLAST = NT * (MT - 1) + NT / 2, FIRST = (LAST > XLAST ? LAST : XLAST) + 1, MEET = FIRST > S - 2 ? FIRST : S - 2;      // where the waves meet
    static_assert(MEET <= S, "reads and loads of a step have to fit between its products");
    extern __shared__ __align__(16) char smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int wn = wave & 1, wm = wave >> 1;
    const int items = (a.rows + BM - 1) / BM * ((a.n + BN - 1) / BN) * a.splits, xcd = blockIdx.x & 7, stride = gridDim.x >> 3;
    const int id_end = (int)((int64_t)items * (xcd + 1) >> 3);
    int id = (int)((int64_t)items * xcd >> 3) + (int)(blockIdx.x >> 3);
    if (id >= id_end) return;
    Item now = item_of<BM, BN>(a, id), load = now;
    uint32_t off[PER];                                        // this lane's places in its loads: bytes from the step's scalar pointers
    const char *xp, *wp;
    auto point = [&] {                                        // at the first step of `load`
        const int r8 = lane >> 3;
        const uint32_t piece = 16 * ((lane & 7) ^ r8);
#pragma unroll
        for (int f = 0; f < PER; ++f) {
            const int grp8 = wave + 4 * f;
            if (f < MT) {
                off[f] = (uint32_t)min(load.mt * BM + 8 * grp8 + r8, a.rows - 1) * (uint32_t)(2 * a.ld_x) + piece;
            } else {
                const int r = 8 * (grp8 - XG) + r8, p = load.nt * 2 * NT + (r >> 4);
                const int row = FORM == SILU_HALVES ? (p & 1) * (a.n >> 1) + min(16 * (p >> 1) + (r & 15), (a.n >> 1) - 1) : min(16 * p + (r & 15), a.n - 1);
                off[f] = (uint32_t)row * (uint32_t)(2 * a.k) + piece;
            }
        }
        xp = (const char*)a.x + (int64_t)load.c_beg * 128;
        wp = (const char*)a.w + (int64_t)load.c_beg * 128;
    };
    point();
    int load_id = id, to_come = load.steps - 1;
    auto dma = [&](int buf, int f) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((f < MT ? xp : wp) + off[f]),
                                         (__attribute__((address_space(3))) void*)(smem + (f < MT ? buf * XS : NX * XS + buf * WS - XG * 1024) + (wave + 4 * f) * 1024), 16, 0, 0);
    };
    auto forward = [&](int steps) {                           // the loads are that many steps further on
        to_come -= steps;
        if (to_come >= 0) return;
        if (load_id + stride < id_end) {                      // at the next item
            load_id += stride;
            load = item_of<BM, BN>(a, load_id);
            to_come = load.steps - 1;
            point();
        } else {                                              // past the last one: its last step again, not used
            xp -= 128;
            wp -= 128;
            to_come = 0;
        }
    };
    const uint32_t x_at = (wm * MT * 16 + i) * 128 + ((g ^ (i & 7)) * 16), w_at = NX * XS + (wn * NT * 16 + i) * 128 + ((g ^ (i & 7)) * 16);
    Frag x0[MT], w0[NT], x1[MT], w1[NT];
    f32x4 acc[NT][MT];
    auto add = [&](Frag w, Frag x, f32x4& c) {
        if constexpr (IN_PLACE) El<T>::add_in_place(w, x, c);
        else El<T>::add(w, x, c);
    };
    auto keep = [&](f32x4& c) {                               // to be read where it is needed: read ahead, the sums of a tile take all registers
        if constexpr (IN_PLACE) asm volatile("" : "+a"(c));
    };
    // the n-th fragment of a half step of 32: weights first, they are all needed at once
    auto read = [&](Frag (&x)[MT], Frag (&w)[NT], int bx, int bw, int kk, int n) {
        if (n < NT) w[n] = *reinterpret_cast<const Frag*>(smem + bw * WS + (w_at ^ (64 * kk)) + 2048 * n);
        else x[n - NT] = *reinterpret_cast<const Frag*>(smem + bx * XS + (x_at ^ (64 * kk)) + 2048 * (n - NT));
    };
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int f = 0; f < PER; ++f) dma(b, f);
        xp += 128;
        wp += 128;
        forward(1);
    }
    meet<(NB - 1) * PER>();
#pragma unroll
    for (int n = 0; n < PER; ++n) read(x0, w0, 0, 0, 0, n);
    int bx = 0, bw = 0;
    for (;;) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (IN_PLACE) hold();
        for (int left = now.steps, run; left; left -= run, forward(run)) {
            run = min(left, to_come + 1);                     // no branch between the products of two steps
            for (int c = run; c; --c) {
            const int next_x = bx + 1 == NX ? 0 : bx + 1, free_x = bx ? bx - 1 : NX - 1, next_w = bw + 1 == NB ? 0 : bw + 1;
#pragma unroll
            for (int f = 0; f < PER; ++f) asm("" : "+v"(off[f]));
            asm("" : "+s"(xp), "+s"(wp));                     // (opaque: sums of scalar and lane offsets, made ahead, would cost a register pair each)
#pragma unroll
            for (int s = 0; s < S; ++s) {
                if (s == MEET) meet<(NB - 2) * PER + MT>();   // the next step is in LDS, and this one's weights have been read
                add(w0[s % NT], x0[s / NT], acc[s % NT][s / NT]);
                __builtin_amdgcn_sched_barrier(0);
                if (s % RS == 0 && s / RS < PER) {
                    read(x1, w1, bx, bw, 1, s / RS);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (s % NT == NT / 2) {
                    dma(free_x, s / NT);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (MEET == S) meet<(NB - 2) * PER + MT>();
#pragma unroll
            for (int s = 0; s < S; ++s) {
                add(w1[s % NT], x1[s / NT], acc[s % NT][s / NT]);
                __builtin_amdgcn_sched_barrier(0);
                if (s % RS == 0 && s / RS < PER) {
                    read(x0, w0, next_x, next_w, 0, s / RS);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (s % MT == MT / 2) {
                    dma(bw, MT + s / MT);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (IN_PLACE) hold();
            xp += 128;
            wp += 128;
            bx = next_x;
            bw = next_w;
            }
        }
        const int row0 = (now.mt * 2 + wm) * 16 * MT, p0 = (now.nt * 2 + wn) * NT;       // this wave's first row and panel
        const bool whole = now.mt * BM + BM <= a.rows && now.nt * BN + BN <= a.n;
        if (a.splits > 1) {
            const uint32_t at = 4 * ((uint32_t)i * (uint32_t)a.n + 4 * g);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                __builtin_amdgcn_sched_barrier(0);
                char* y = (char*)(a.ws + ((int64_t)now.split * a.rows + row0 + 16 * m) * a.n);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    keep(acc[t][m]);
                    const int p = p0 + t, n0 = FORM == SILU_HALVES ? (p & 1) * (a.n >> 1) + 16 * (p >> 1) : 16 * p;
                    if (whole || (row0 + 16 * m + i < a.rows && 16 * p < a.n)) *reinterpret_cast<f32x4*>(y + 4 * n0 + at) = acc[t][m];
                }
            }
        } else {
            constexpr int NQ = FORM == PLAIN ? NT : NT / 2;   // panels of 16 results
            const int q0 = FORM == PLAIN ? p0 : p0 >> 1, n_out = FORM == PLAIN ? a.n : a.n >> 1, side = 16 * (g & 1) + 8 * (g >> 1);
            const uint32_t at = 2 * ((uint32_t)i * (uint32_t)a.ld_out + side);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    keep(acc[t][m]);
                }
                u32x2 q[NQ];
#pragma unroll
                for (int t = 0; t < NQ; ++t) {
                    f32x4 v;
                    if constexpr (FORM == PLAIN) {
                        v = acc[t][m];
                    } else {
                        f32x4 z = acc[2 * t][m], u = acc[2 * t + 1][m];
                        if constexpr (FORM == GELU_EIGHTS)    // lanes 0 .. 31 hold gates, the others ups: those of two panels side by side
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float ze = z[e], ue = u[e];
                                const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, ze), __builtin_bit_cast(uint32_t, ue), false, false);
                                const uint32_t r0 = r[0], r1 = r[1];
                                z[e] = __builtin_bit_cast(float, r0);
                                u[e] = __builtin_bit_cast(float, r1);
                            }
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = glu<T, FORM>(z[e], u[e]);
                    }
                    q[t] = u32x2{pack<T>(v[0], v[1]), pack<T>(v[2], v[3])};
                }
                char* y = (char*)((T*)a.out + (int64_t)(row0 + 16 * m) * a.ld_out + 16 * q0);
                // a lane has results 4 g .. 4 g + 3 of every panel: of two panels it keeps 8 of one
#pragma unroll
                for (int t = 0; t + 1 < NQ; t += 2) {
                    const auto lo = __builtin_amdgcn_permlane16_swap(q[t][0], q[t + 1][0], false, false);
                    const auto hi = __builtin_amdgcn_permlane16_swap(q[t][1], q[t + 1][1], false, false);
                    if (whole || (row0 + 16 * m + i < a.rows && 16 * (q0 + t) + side < n_out)) *reinterpret_cast<u32x4*>(y + 32 * t + at) = u32x4{lo[0], hi[0], lo[1], hi[1]};
                }
                if constexpr (NQ & 1)
                    if (whole || (row0 + 16 * m + i < a.rows && 16 * (q0 + NQ - 1) < n_out))
                        *reinterpret_cast<u32x2*>(y + 32 * (NQ - 1) + at + 2 * (4 * g - side)) = q[NQ - 1];
            }
        }
        id += stride;
        if (id >= id_end) break;
        now = item_of<BM, BN>(a, id);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);                       // no load is under way when the workgroup's LDS is given back
}

// The parts of a split k, summed in order, and their form: eight results a thread.
template <typename T, int FORM> __global__ __launch_bounds__(256) void rows_sum_kernel(const Args a) {
    const int n_out = FORM == PLAIN ? a.n : a.n >> 1, octets = n_out >> 3;
    const int64_t total = (int64_t)a.rows * octets, part = (int64_t)a.rows * a.n;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int64_t row = e / octets;
        const int c = 8 * (int)(e - row * octets);
        constexpr int Q = FORM == PLAIN ? 2 : 4;              // fours of sums: gates, then ups
        const float* src = a.ws + row * a.n + (FORM == GELU_EIGHTS ? 2 * c : c);
        const int up = FORM == SILU_HALVES ? n_out : 8;
        f32x4 v[Q] = {};
        for (int z = 0; z < a.splits; ++z)
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const f32x4 p = *reinterpret_cast<const f32x4*>(src + z * part + (q & 1) * 4 + (q >> 1) * up);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[q][j] += p[j];
            }
        u32x4 o;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (FORM != PLAIN)
#pragma unroll
                for (int j = 0; j < 4; ++j) v[h][j] = glu<T, FORM>(v[h][j], v[2 + h][j]);
            o[2 * h] = pack<T>(v[h][0], v[h][1]);
            o[2 * h + 1] = pack<T>(v[h][2], v[h][3]);
        }
        *reinterpret_cast<u32x4*>((T*)a.out + row * a.ld_out + c) = o;
    }
}

// Tiles: rows, outputs, workgroups that share a CU, and in us what a step costs where a CU is full and at least, and what a tile costs besides.
// Fitted to 24 products of 256 .. 32 000 outputs and 256 .. 15 104 columns at 57 counts of rows from 33 to 8 000, weights from memory, every tile with
// 1 to 16 parts of each timed: the one picked is 1.006 of the best on average, more than 1.05 in one of 18.  (Tiles of 160 x 64, 96 x 128 and 128 x 128 were
// the best of all nowhere by more than 1 %.)
struct Shape { int rows, cols, per_cu; float step, least, tile; };
constexpr Shape SHAPES[] = {{256, 256, 1, 1.268f, 0.60f, 7.1f}, {224, 256, 1, 1.173f, 0.60f, 4.5f}, {192, 256, 1, 1.108f, 0.60f, 4.6f}, {160, 256, 1, 1.044f, 0.60f, 2.4f},
                            {128, 256, 1, 0.542f, 0.79f, 2.8f}, {64, 128, 2, 0.323f, 0.28f, 0.07f}, {96, 64, 2, 0.241f, 0.07f, 0.18f}, {64, 64, 2, 0.179f, 0.03f, 0.17f}};
constexpr int N_SHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);

struct Plan { int shape, splits; };

// The bytes each operand needs at 7.1 TB/s; the steps of a CU's tiles, one or two at a time; parts of k are written and read at 4 TB/s by
// another launch.  XCDs take an eighth of the tiles each, and their 32 CUs whole ones.  Small tiles in number are bound by what they read from L2,
// 20 TB/s (12 288 x 4 096: 190 rows 47 -> 41 us by another tile, 255 rows 53 -> 47, 350 rows 62 -> 57; 4 096 x 11 008, 255 rows 51 -> 42).
inline Plan plan(int rows, int n, int k) {
    const int nk = k >> 6;
    const double mem = (2.0 * n * k + 2.0 * rows * k + 2.0 * rows * n) / 7.1e6;
    Plan best{0, 1};
    double least = 0;
    for (int s = 0; s < N_SHAPES; ++s) {
        const Shape& h = SHAPES[s];
        const int64_t tiles = (int64_t)((rows + h.rows - 1) / h.rows) * ((n + h.cols - 1) / h.cols);
        const double l2 = h.per_cu > 1 ? (double)tiles * nk * (h.rows + h.cols) * 128 / 20e6 : 0.0;
        for (int z = 1; z <= 16; ++z) {
            const int per = (nk + z - 1) / z;
            if (z > 1 && ((z - 1) * per >= nk || per < 4 || tiles * z > 410 * h.per_cu || (int64_t)z * rows * n > (int64_t)1 << 28)) continue;
            const int64_t a_cu = ((tiles * z + 7) / 8 + 31) / 32, full = a_cu / h.per_cu;
            const double fully = per * (double)fmaxf(h.per_cu * h.step, h.least) + h.per_cu * h.tile;
            const double work = full * fully + (a_cu > full * h.per_cu ? per * (double)fmaxf(h.step, h.least) + h.tile : 0.0);
            const double t = cbrt(work * work * work + mem * mem * mem + l2 * l2 * l2) + (z > 1 ? 2.55 + z * (0.18 + 4.0 * rows * n / 4.2e6) : 0.0);
            if ((s == 0 && z == 1) || t < least) { least = t; best = Plan{s, z}; }
        }
    }
    return best;
}

// Operands that the kernel takes: whole steps of k, whole panels of outputs (pairs of them for a gated unit), rows and pointers of 16 bytes,
// offsets within 32 bits.
inline bool takes(int64_t ld_x, int64_t ld_out, int rows, int n, int k, int form) {
    const int n_out = form == PLAIN ? n : n / 2;
    return rows >= 1 && n >= 16 && k >= 64 && (n & (form == PLAIN ? 15 : 31)) == 0 && (k & 63) == 0 && ld_x >= k && (ld_x & 7) == 0 && ld_out >= n_out
        && (ld_out & 7) == 0 && ld_out < 1 << 26 && n < 1 << 26 && (int64_t)rows * ld_x < (int64_t)1 << 31 && (int64_t)n * k < (int64_t)1 << 31
        && (int64_t)((rows + 63) / 64) * ((n + 63) / 64) < (int64_t)1 << 26;
}

inline int64_t ws_floats(int rows, int n, int splits) { return splits > 1 ? (int64_t)splits * rows * n : 0; }

template <typename T, int MT, int NT, int NB, int FORM, int OCC> int launch_tile(const Args& a, hipStream_t st) {
    constexpr int LDS = lds_bytes<MT, NT, NB>();
    static_assert(LDS * OCC <= 160 * 1024, "LDS of a CU");
    const auto kernel = rows_gemm_kernel<T, MT, NT, NB, FORM, OCC>;
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return (int)e;
    const int64_t items = (int64_t)((a.rows + 32 * MT - 1) / (32 * MT)) * ((a.n + 32 * NT - 1) / (32 * NT)) * a.splits;
    const int per_xcd = (int)((items + 7) / 8 < 32 * OCC ? (items + 7) / 8 : 32 * OCC);
    hipLaunchKernelGGL(kernel, dim3(8 * per_xcd), dim3(256), LDS, st, a);
    return (int)hipGetLastError();
}

template <typename T, int FORM> int launch(const Args& a, int shape, hipStream_t st) {
    int e;
    switch (shape) {
        case 0: e = launch_tile<T, 8, 8, 2, FORM, 1>(a, st); break;
        case 1: e = launch_tile<T, 7, 8, 2, FORM, 1>(a, st); break;
        case 2: e = launch_tile<T, 6, 8, 2, FORM, 1>(a, st); break;
        case 3: e = launch_tile<T, 5, 8, 2, FORM, 1>(a, st); break;
        case 4: e = launch_tile<T, 4, 8, 3, FORM, 1>(a, st); break;
        case 5: e = launch_tile<T, 2, 4, 3, FORM, 2>(a, st); break;
        case 6: e = launch_tile<T, 3, 2, 3, FORM, 2>(a, st); break;
        default: e = launch_tile<T, 2, 2, 4, FORM, 2>(a, st);
    }
    if (e || a.splits == 1) return e;
    const int64_t octets = (int64_t)a.rows * (FORM == PLAIN ? a.n : a.n / 2) / 8, blocks = (octets + 255) / 256;
    hipLaunchKernelGGL((rows_sum_kernel<T, FORM>), dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

// The entry point of a library: OTHER is the gated unit that it has.  Codes as the header says.
template <typename T, int OTHER> int entry(const void* x, int64_t ld_x, const void* w, void* out, int64_t ld_out, float* ws, int64_t ws_have, int rows, int n,
                                           int k, int form, int shape, int splits, void* stream) {
    if (!x || !w || !out || (form != PLAIN && form != OTHER) || !takes(ld_x, ld_out, rows, n, k, form) || shape < 0 || shape >= N_SHAPES || splits < 1) return TF_EINVAL;
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)ws) & 15) return TF_EINVAL;
    const int nk = k >> 6;
    if (splits > 64 || (splits - 1) * ((nk + splits - 1) / splits) >= nk) return TF_EINVAL;           // every part has a step
    if (splits > 1 && (!ws || ws_have < ws_floats(rows, n, splits))) return TF_ENOSPC;
    const Args a = {x, w, out, ws, ld_x, ld_out, rows, n, k, splits};
    return form == PLAIN ? launch<T, PLAIN>(a, shape, (hipStream_t)stream) : launch<T, OTHER>(a, shape, (hipStream_t)stream);
}
inline int64_t entry_plan(int rows, int n, int k, int32_t* shape, int32_t* splits) {
    if (!shape || !splits || rows < 1 || n < 1 || k < 64) return TF_EINVAL;
    const Plan p = plan(rows, n, k);
    *shape = p.shape;
    *splits = p.splits;
    return ws_floats(rows, n, p.splits);
}

}  // namespace rg
