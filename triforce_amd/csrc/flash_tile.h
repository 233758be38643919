// The loop over key tiles of a bfloat16 prefill attention: 128 query rows per workgroup (four waves of 2 x 16), tiles of 64 keys, values of
// 128, keys of 128 (KR = 0) or 128 + 64 in two places (KR = 2).
//
// The chain of a tile is QK^T -> softmax -> PV: matrix core, VALU, matrix core.  K[t] is dead once its scores are there, so with two K and two
// V tiles in LDS the loop holds K one tile ahead of V: step t runs QK^T(t + 1) beside the exponentials of tile t, then PV(t).  One barrier
// per step.  K and V come in by LDS-DMA (no staging registers, no ds_write); the XOR swizzle that keeps the fragments' reads free of bank
// conflicts is applied where the DMA reads from.  Two workgroups per CU fill each other's waits.
// Bound by what the products and the VALU work between them (exponentials, addresses) draw together: the matrix cores are busy less than half
// of the cycles, at the clock of a GEMM.  So: tile pointers are scalar, a lane adds 32-bit
// offsets; fragments are reached by one XOR; masked and unmasked tiles take one path; fragments are read 4 (K) and 8 (V) steps ahead in a
// fixed order (left to itself the scheduler moves all reads to the front and spills).
#pragma once
#include "tile_common.h"

// Which (sequence, head, query block) the workgroup at (at, row) takes of a grid of width (sequences times heads) x blocks.  Row by row, all
// sequences and heads of a row side by side; by_seq: in the same linear order sequence by sequence, then block by block, heads side by side.
struct SeqBlock { int seq, head, block; };
__device__ __forceinline__ SeqBlock seq_block(int at, int width, int heads, int row, int blocks, bool by_seq) {
    if (!by_seq) return SeqBlock{at / heads, at % heads, row};
    const int l = row * width + at, rest = l / heads;
    return SeqBlock{rest / blocks, l % heads, rest % blocks};
}

template <int KR, int NWV> struct FlashTile {
    static constexpr int KT = 64, QT = 2, NC = 4 + KR, NT = 8, D = 128, ROWS = 32 * NWV, STEP = 4 * NWV;
    static constexpr int K_ELEMS = KT * D, R_ELEMS = KT * 32 * KR, LDS = 2 * (2 * K_ELEMS + R_ELEMS) * 2;      // bytes
    struct Tile { const bf16 *k, *r, *v; int last; };         // first rows (of this head) and the last row that may be read
    bf16x8 q[QT][NC];
    f32x4 acc[QT][NT];
    float m[QT], l[QT];                                       // running maximum (of score * scale * log2 e) and this lane's part of the sum

    // tile(t): the Tile; whole(k0): every row of the wave sees all 64 keys from k0 on (wave-uniform); otherwise query u sees lo[u] .. hi[u].
    // k_ld / r_ld: elements from row to row (63 rows stay below 2^32 bytes).  load() fills q, lo and hi while the first tiles are on their way.
    template <class Load, class Src, class Whole>
    __device__ __forceinline__ void run(char* smem, int t_beg, int t_end, uint32_t k_ld, uint32_t r_ld, float scale, const int (&lo)[QT],
                                        const int (&hi)[QT], Load&& load, Src&& tile, Whole&& whole) {
        bf16* sk = (bf16*)smem;
        bf16* sv = sk + 2 * K_ELEMS;
        bf16* sr = sv + 2 * K_ELEMS;
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, i = lane & 15;
        const float sc = scale * 1.4426950408889634f;
#pragma unroll
        for (int u = 0; u < QT; ++u) {
            m[u] = -__FLT_MAX__;
            l[u] = 0.f;
#pragma unroll
            for (int d = 0; d < NT; ++d) acc[u][d] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // 16 pieces of 16 bytes per row of 128: pass p of a tile brings rows 16 p .. + 15 (a wave 4 of them, 1 KiB in lane order)
        const int lr = tid >> 4, lc = tid & 15, rr = tid >> 3, rc = tid & 7;
        const uint32_t k_row = 2 * k_ld, r_row = 2 * r_ld;
        uint32_t row_off = lr * k_row, rope_off = rr * r_row;
        uint32_t piece_k = 16 * (lc ^ ((lr & 3) | (((lr >> 3) & 3) << 2)));              // odd passes: XOR 8 pieces
        uint32_t piece_v = 16 * ((((lc >> 1) ^ ((lr & 3) | (((lr >> 3) & 1) << 2))) << 1) | (lc & 1));
        uint32_t piece_r = 16 * (rc ^ (((rr >> 1) & 1) | (((rr >> 3) & 3) << 1)));
        auto dma = [&](const bf16* first, uint32_t off, bf16* dst) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((const char*)first + off),
                                             (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
        };
        auto fetch_k = [&](int t, int buf) {
            const Tile a = tile(t);
            const uint32_t last = (uint32_t)a.last * k_row;
#pragma unroll
            for (int p = 0; p < KT / STEP; ++p)
                dma(a.k, min(row_off + (uint32_t)(STEP * p) * k_row, last) + (NWV == 4 ? piece_k ^ ((p & 1) * 128) : piece_k), sk + buf * K_ELEMS + (STEP * p + 4 * wave) * D);
#pragma unroll
            for (int p = 0; p < (KR ? KT / (2 * STEP) : 0); ++p)
                dma(a.r, min(rope_off + (uint32_t)(2 * STEP * p) * r_row, (uint32_t)a.last * r_row) + piece_r, sr + buf * R_ELEMS + (2 * STEP * p + 8 * wave) * 64);
        };
        auto fetch_v = [&](int t, int buf) {
            const Tile a = tile(t);
            const uint32_t last = (uint32_t)a.last * k_row;
#pragma unroll
            for (int p = 0; p < KT / STEP; ++p)
                dma(a.v, min(row_off + (uint32_t)(STEP * p) * k_row, last) + piece_v, sv + buf * K_ELEMS + (STEP * p + 4 * wave) * D);
        };
        // fragment places: result rows 4 g .. 4 g + 3 of the two products of a half are keys 8 g .. 8 g + 7, the value operand's order
        const int row_a = 8 * (i >> 2) + (i & 3);
        int k_at = row_a * D + 8 * (g ^ i);
        int r_at = row_a * 64 + 8 * (g ^ (((row_a >> 1) & 1) | (((row_a >> 3) & 3) << 1)));
        int v_at = (8 * g + (i >> 2)) * D + 4 * (i & 3) + 16 * ((i >> 2) | ((g & 1) << 2));
        typedef __attribute__((address_space(3))) bf16x4* lds4;
        auto scores = [&](int buf, f32x4 (&s)[4][QT], auto&& beside) {
            constexpr int STEPS = 2 * NC, AHEAD = 4;
            const int kb = k_at + buf * K_ELEMS, rb = r_at + buf * R_ELEMS;
            bf16x8 a[AHEAD + 1], b[AHEAD + 1];
            auto read = [&](int n) {
                const int c = n % NC;
                const bf16* src = c < 4 ? sk + (kb ^ (32 * c)) + (n / NC) * 32 * D : sr + (rb ^ (32 * (c - 4))) + (n / NC) * 32 * 64;
                a[n % (AHEAD + 1)] = load_frag(src);
                b[n % (AHEAD + 1)] = load_frag(src + 4 * (c < 4 ? D : 64));
            };
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int u = 0; u < QT; ++u) s[x][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int n = 0; n < AHEAD; ++n) read(n);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < STEPS; ++n) {
                if (n + AHEAD < STEPS) read(n + AHEAD);
#pragma unroll
                for (int u = 0; u < QT; ++u) {
                    f32x4 &x = s[2 * (n / NC)][u], &y = s[2 * (n / NC) + 1][u];
                    x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n % (AHEAD + 1)], q[u][n % NC], x, 0, 0, 0);
                    y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[n % (AHEAD + 1)], q[u][n % NC], y, 0, 0, 0);
                }
                beside(n);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto values = [&](int buf, const bf16x8 (&p)[2][QT]) {
            constexpr int STEPS = 2 * NT, AHEAD = 8;
            const int vb = v_at + buf * K_ELEMS;
            bf16x4 x[AHEAD + 1], y[AHEAD + 1];
            auto read = [&](int n) {
                const bf16* src = sv + (vb ^ (16 * (n % NT))) + (n / NT) * 32 * D;
                x[n % (AHEAD + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4)src);
                y[n % (AHEAD + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4)(src + 4 * D));
            };
#pragma unroll
            for (int n = 0; n < AHEAD; ++n) read(n);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < STEPS; ++n) {
                if (n + AHEAD < STEPS) read(n + AHEAD);
                const bf16x8 v = __builtin_shufflevector(x[n % (AHEAD + 1)], y[n % (AHEAD + 1)], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int u = 0; u < QT; ++u) acc[u][n % NT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, p[n / NT][u], acc[u][n % NT], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        f32x4 s[4][QT];                                       // scores of the current tile
        fetch_k(t_beg, 0);
        fetch_v(t_beg, 0);
        if (t_beg + 1 < t_end) fetch_k(t_beg + 1, 1);
        load();
        __builtin_amdgcn_s_waitcnt(0x0F70);                   // vmcnt(0): queries and the first tiles have landed
        __syncthreads();
        scores(0, s, [](int) {});
        __syncthreads();                                      // every wave is done with K[t_beg] before step 0 overwrites it
        for (int t = t_beg; t < t_end; ++t) {
            const int buf = (t - t_beg) & 1, k0 = t * KT;
            // (opaque once per step: sums and XORs on these are one instruction each, hoisted they would take the scores' registers)
            asm("" : "+v"(row_off), "+v"(rope_off), "+v"(piece_k), "+v"(piece_v), "+v"(piece_r));
            asm("" : "+v"(k_at), "+v"(r_at), "+v"(v_at));
            if (t + 2 < t_end) fetch_k(t + 2, buf);           // over K[t], dead since the previous barrier
            if (t + 1 < t_end) fetch_v(t + 1, buf ^ 1);       // over V[t - 1]
            if (!whole(k0)) {
#pragma unroll
                for (int u = 0; u < QT; ++u) {
                    const int first = lo[u] - k0 - 8 * g, last = hi[u] - k0 - 8 * g;
#pragma unroll
                    for (int x = 0; x < 4; ++x)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {         // exp2 of -inf minus any finite maximum is 0
                            const int k = 32 * (x >> 1) + 4 * (x & 1) + r;
                            if (k > last || k < first) s[x][u][r] = -__builtin_inff();
                        }
                }
            }
            float top[QT];
#pragma unroll
            for (int u = 0; u < QT; ++u) {
                float mx = s[0][u][0];
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(fmaxf(fmaxf(mx, s[0][u][r]), fmaxf(s[1][u][r], s[2][u][r])), s[3][u][r]);
                mx = rows_max(mx);
                top[u] = fmaxf(m[u], mx * sc);
                if (__builtin_amdgcn_ballot_w64(top[u] != m[u])) {                       // (most tiles leave every maximum where it was)
                    const float alpha = __builtin_amdgcn_exp2f(m[u] - top[u]);
                    l[u] *= alpha;
#pragma unroll
                    for (int d = 0; d < NT; ++d)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[u][d][r] *= alpha;
                    m[u] = top[u];
                }
            }
            f32x4 next[4][QT];
            bf16x8 p[2][QT];
            float sum[QT] = {};
            scores(buf ^ 1, next, [&](int n) {                // (past the end: finite or not, never used)
                if (n >= 8) return;
                const int u = n / 4, x = n % 4;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = __builtin_amdgcn_exp2f(fmaf(s[x][u][r], sc, -top[u]));
                    sum[u] += e;
                    p[x >> 1][u][4 * (x & 1) + r] = (bf16)e;
                }
            });
            values(buf, p);
#pragma unroll
            for (int u = 0; u < QT; ++u) {
                l[u] += sum[u];
#pragma unroll
                for (int x = 0; x < 4; ++x) s[x][u] = next[x][u];
            }
            __builtin_amdgcn_s_waitcnt(0x0F70);               // vmcnt(0): this wave's DMA is in LDS before the barrier
            __syncthreads();
        }
    }

    // Sum of the weights of query u (over the four lanes that hold its keys).
    __device__ __forceinline__ float weight(int u) const {
        float s = l[u];
        s = rows_sum(s);
        return s;
    }
};
