// float32 products of many rows (prefill) on the bfloat16 matrix cores: y = x . W^T.
//
// The products of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations"
// (ARITH 2019): a float32 is exactly the sum of three bfloat16 h + m + l, each the nearest to what is left (|m| <= 2^-8 and |l| <= 2^-17 of the
// value, of either sign), and six of the nine products of two such sums, hh + hm + mh + mm + hl + lh, leave out at most 2^-24 of a product
// (ml + lm, 2^-25 each, and ll), without a preferred sign.  Products of bfloat16 are exact in the matrix core and the sums are fp32, hh in
// an accumulator of its own: beside a large sum the five small products of a step would fall below its last place, step after step, and
// with parts that are cut instead of rounded always towards zero.
// Error against 64 bits, relative 2-norm, fp32 instruction -> cut parts in one accumulator -> this:
//   700 rows of k = 4 096   normals 1.1e-6 -> 7.1e-7 -> 2.7e-7, their absolute values 9.9e-7 -> 3.2e-6 -> 1.8e-7;
//   700 rows of k = 15 104  normals 2.1e-6 -> 9.2e-7 -> 3.4e-7, absolute values 1.7e-6 -> 5.8e-6 -> 1.2e-7, normals of mean 1
//   1.5e-6 -> 4.7e-6 -> 1.4e-7, uniform in 1 .. 2 1.6e-6 -> 8.4e-6 -> 1.4e-7.
// (Rounded parts in one accumulator: 9.1e-7, 2.2e-7, 2.5e-7, 2.3e-7.  The accuracy costs 1 to 2 % where a CU has many steps, up to 6 % in short parts: 22 016 x 4 096 at 700
// rows 730 -> 740 us.)
// Six bf16 instructions take 3/8 of the cycles of the eight fp32 ones that cover the same 16 x 16 x 32.
//
// 256 outputs x 128 rows per workgroup, four waves of 64 x 128, one per SIMD: per step of 32 a wave reads 36 KB from LDS for 192 products (3 170
// cycles), a third of what LDS delivers.  x is cut once by a kernel in front, into planes in MFMA order ([rows/16][k/32][3][64 lanes][8]: a fragment is one
// contiguous KiB that goes to LDS by DMA); a weight is used by one workgroup per 128 rows and is cut on its way to LDS, between the products.
// (Cut at load time
// into planes, weights cost 6 bytes beside the 4 and gain 3 to 8 %.)  A wave issues one operation in five cycles and a product takes sixteen, so two
// operations behind every product cost nothing and five behind every third product do: the cut goes in eighths, 128 of them behind 144 products
// (in thirds 2 048 rows of 22 016 1 565 -> 1 665 us, two products at a time 1 645).  Weights asked for in whole lines of 128 bytes, an eighth of the
// rows a load, need twice the stores to LDS: 1 565 -> 1 577; asked for four steps ahead into L2 as well, 1 644.
//
// Bound by the power of the matrix cores (1.6 to 1.7 GHz under these products, as bf16 GEMMs; all operands zero, at full clock, 22 016 x 4 096 at 700
// rows takes 536 us), by what a step costs beside its products and by rounds of tiles.  A matrix core draws less where a product goes to the sum
// that the one before it went to (registers alone, bf16 normals: 2 110 TFLOP/s with another sum each time, 2 226 in twos, 2 350 in fours, 2 395 in
// eights), so the five small products of a result follow each other.  700 rows, each product to another sum in eight waves of 64 x 64 -> in fives -> four
// waves: 22 016 x 4 096 665 -> 613 -> 588 us, 18 784 x 4 096 567 -> 537 -> 512, 4 096 x 15 104 481 -> 456 -> 427, 4 096 x 8 192 266 -> 256 -> 247; 2 048
// rows of 22 016 1 719 -> 1 632 -> 1 563 (236 TFLOP/s); 256 rows of 12 320 158 -> 156 -> 149.
// The fp32 instruction, x's cut and the sum of parts included: 700 rows, 22 016 x 4 096 940 us, 18 784 x 4 096 900, 4 096 x 15 104 680; 2 048 rows,
// 22 016 x 4 096 2 600.
//
// Range: both operands are cut at 2^24 times their value, so the last bit of the smallest float32 (2^-149) is still a normal bfloat16 and no
// product of parts that counts leaves fp32's range below; results are multiplied by 2^-48.  Above, a factor from 2^104 or a sum from 2^80
// on becomes infinite on the way; such a result, and one that is not finite because a factor is not (an infinity times a zero part is NaN),
// is computed again in plain fp32, the 16 x 16 tile that it lies in by its wave on the fp32 instruction; rows of x with a NaN, which is what
// an infinity leaves behind in a model, are marked when they are cut and keep their NaN results.  One infinite row of 700 in front of
// 22 016 x 4 096 costs 600 -> 1 070 us, of 300 in front of 4 096 x 15 104 236 -> 665 (by a thread per result 4 200 and 9 900).  The kernel stores all
// sums first and walks through a wave's tiles again where one was odd: thirty-two walks in line cost every launch 4 %.  (The scaling is 16 of some 200 VALU operations per step: 22 016 x 4 096 at 700 rows 740 -> 752 us.)
#include "lds_dma.h"
#include "tile_common.h"
#include <type_traits>

#define SPLIT_KC 512                   // columns of x that one workgroup cuts
#define SPLIT_SCALE 0x1p24f            // of either operand

__device__ __forceinline__ void cut_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    typedef bf16 Pair __attribute__((ext_vector_type(2)));
    a *= SPLIT_SCALE;
    b *= SPLIT_SCALE;
    h = __builtin_bit_cast(uint32_t, Pair{(bf16)a, (bf16)b});
    a -= __builtin_bit_cast(float, h << 16);
    b -= __builtin_bit_cast(float, h & 0xFFFF0000u);
    m = __builtin_bit_cast(uint32_t, Pair{(bf16)a, (bf16)b});
    a -= __builtin_bit_cast(float, m << 16);
    b -= __builtin_bit_cast(float, m & 0xFFFF0000u);
    l = __builtin_bit_cast(uint32_t, Pair{(bf16)a, (bf16)b});
}

// Eight values into the three planes of a fragment.
__device__ __forceinline__ void cut_store(const f32x4 (&v)[2], bf16* dst) {
    u32x4 out[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t h, m, l;
        cut_pair(v[e >> 1][2 * (e & 1)], v[e >> 1][2 * (e & 1) + 1], h, m, l);
        out[0][e] = h;
        out[1][e] = m;
        out[2][e] = l;
    }
#pragma unroll
    for (int z = 0; z < 3; ++z) *reinterpret_cast<u32x4*>(dst + 512 * z) = out[z];
}

// A product without the compiler's say in where its sum goes: it moves some of 256 registers of sums through others in every step.  It does not
// see then what the matrix core still has to read or write: hold_sums() stands behind the products of a step, inside their loop, so that no copy of a
// sum can come first.
__device__ __forceinline__ void add_in_place(bf16x8 a, bf16x8 b, f32x4& c) { asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }

// One workgroup: 16 rows, SPLIT_KC columns.  nans[row][part]: the row has a NaN in this part of k.
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ x, int64_t ld, int rows, int k, bf16* __restrict__ planes,
                                                         int32_t* __restrict__ nans) {
    __shared__ int found[4][16];
    const int panel = blockIdx.x, tid = threadIdx.x, lane = tid & 63, chunks = k >> 5, row = 16 * panel + (lane & 15);
    const int c_end = min(chunks, (int)(blockIdx.y + 1) * (SPLIT_KC / 32));
    int nan = 0;
    for (int c = blockIdx.y * (SPLIT_KC / 32) + (tid >> 6); c < c_end; c += 4) {
        f32x4 v[2] = {};
        if (row < rows) {
            const f32x4* src = reinterpret_cast<const f32x4*>(x + (int64_t)row * ld + 32 * c + 8 * (lane >> 4));
            v[0] = src[0];
            v[1] = src[1];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) nan |= v[e >> 2][e & 3] != v[e >> 2][e & 3];
        cut_store(v, planes + ((int64_t)panel * chunks + c) * 1536 + lane * 8);
    }
    nan |= __shfl_xor(nan, 16, 64);
    nan |= __shfl_xor(nan, 32, 64);
    if (lane < 16) found[tid >> 6][lane] = nan;
    __syncthreads();
    if (tid < 16 && row < rows) nans[(int64_t)row * gridDim.y + blockIdx.y] = found[0][tid] | found[1][tid] | found[2][tid] | found[3][tid];
}

struct SplitGemm {
    const float* w;
    const bf16* xp;
    const float* x;
    float* out;
    float* ws;                                                // [8 XCDs][slots][128 rows][256 outputs]
    const int32_t* nans;
    int64_t ld_x, ld_out;
    int rows, n, k;
    int whole, splits, sharers, slots;                        // see Share; slots of an XCD
    int fold;                                                 // steps that are added up in registers
};

// An XCD's tiles (an eighth of all): the first `whole` of them have a workgroup each.  The steps of the others stand in a line, which is cut among
// the XCD's `sharers` evenly, at eights of steps, or, without sharers, tile by tile into `splits` parts.  A sharer has a part of one tile or of
// two; the parts in their order along the line are numbered by sharer + tile, the slots of ws by part.
struct Share {
    int first, own, rest, sharers, chunks, parts;             // of one XCD: its tiles, those of one workgroup, the others, who shares them; parts of a tile or 0
    __device__ __forceinline__ int cut(int q) const {         // (32 sharers of up to 2^24 steps)
        const uint32_t s = q, n = sharers, p = parts;
        if (parts) return (int)(s / p * chunks + s % p * chunks / p);
        return s < n ? (int)(s * (uint32_t)(rest * chunks) / n & ~7u) : rest * chunks;
    }
};
__device__ __forceinline__ Share share_of(int tiles, int chunks, int whole, int splits, int sharers, int xcd) {
    const int first = (int)((int64_t)tiles * xcd >> 3), all = (int)((int64_t)tiles * (xcd + 1) >> 3) - first, own = min(all, whole), rest = all - own;
    const int parts = min(splits, chunks);                    // (a step at least to each part, an eight to each sharer)
    return Share{first, own, rest, sharers > 0 ? min(sharers, rest * chunks >> 3) : rest * parts, chunks, sharers > 0 ? 0 : parts};
}
constexpr int SLOT = 128 * 256;                               // floats of a part in ws
static int split_tiles(int rows, int n) { return (n + 255) / 256 * ((rows + 127) / 128); }
// Slots of an XCD.
static int split_slots(int tiles, int whole, int splits, int sharers) {
    const int rest = (tiles + 7) / 8 - whole;
    return rest > 0 ? (sharers > 0 ? sharers : rest * splits) + rest - 1 : 0;
}

__host__ __device__ __forceinline__ int split_parts(int k) { return (k + SPLIT_KC - 1) / SPLIT_KC; }

// Results row0 + i, n0 + 4 g .. + 3 of a wave's 16 x 16 tile: those that are not finite, again on the fp32 instruction (whole tile, one wave).
__device__ __forceinline__ void mend(const SplitGemm& a, int row0, int n0, f32x4& v) {
    const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
    bool lost[4], any = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        lost[e] = row0 + i < a.rows && !(__builtin_fabsf(v[e]) < __builtin_inff());
        any = any || lost[e];
    }
    if (!__any(any)) return;
    if (any) {
        const int parts = split_parts(a.k);
        int nan = 0;
        for (int z = 0; z < parts; ++z) nan |= a.nans[(int64_t)(row0 + i) * parts + z];
        any = nan == 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) lost[e] = lost[e] && any;
    }
    if (!__any(any)) return;
    const float* x = a.x + (int64_t)min(row0 + i, a.rows - 1) * a.ld_x + 4 * g;
    const float* w = a.w + (int64_t)(n0 + i) * a.k + 4 * g;
    f32x4 p = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = 8;                                      // steps of 16 asked for at once: the loads are the chain
    for (int c = 0; c < a.k; c += 16 * U) {
        f32x4 xc[U], wc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {                         // (k in any order, the same for both; past the end: the last step again, not used)
            xc[u] = *reinterpret_cast<const f32x4*>(x + min(c + 16 * u, a.k - 16));
            wc[u] = *reinterpret_cast<const f32x4*>(w + min(c + 16 * u, a.k - 16));
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (c + 16 * u < a.k) {
#pragma unroll
                for (int e = 0; e < 4; ++e) p = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[u][e], xc[u][e], p, 0, 0, 0);
            }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = lost[e] ? p[e] : v[e];
}

// f(0), f(1), .. f(N - 1), their arguments known to the compiler.
template <int N, int I = 0, class F> __device__ __forceinline__ void upto(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        upto<N, I + 1>(f);
    }
}

// Waves: 4 x 64 outputs, one per SIMD, each with all 128 rows.  FOLDS: a.fold is below a tile's steps.
template <bool FOLDS>
__global__ __launch_bounds__(256, 1) void split_gemm_kernel(const SplitGemm a) {
    constexpr int MT = 8, NP = 16, PER = 3 * MT / 4, BUF = 3 * (NP + MT) * 512;
    extern __shared__ __align__(16) bf16 tiles[];             // [2][NP + MT][3][512]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int chunks = a.k >> 5;
    // workgroups go round-robin over the 8 XCDs: each takes an eighth of the tiles, the row tiles of one column tile one after the other, which
    // share its weights in L2
    const int mts = (a.rows + 16 * MT - 1) / (16 * MT), xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    const Share share = share_of((a.n + 255) / 256 * mts, chunks, a.whole, a.splits, a.sharers, xcd);
    int q = j - share.own;
    if (q >= share.sharers) return;
    if (q >= 0 && a.sharers == 0) q = q % share.rest * share.parts + q / share.rest;     // (the same part of all tiles together)
    int beg = 0, end = chunks;                                // of the line of shared tiles, or of this workgroup's own tile
    if (q >= 0) {
        beg = share.cut(q);
        end = share.cut(q + 1);
    }
    const int xpan = (a.rows + 15) >> 4;
    const bf16* src[PER];                                     // this wave's fragments of x: scalar pointers to their first chunk
    const float* wsrc[4];                                     // this lane's eight weights of four panels
    f32x4 staged[4][2];
    auto fetch_x = [&](int f, int c, int buf) {
        lds_dma((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)(tiles + buf * BUF + (3 * NP + wave * PER + f) * 512), 16u * lane, src[f] + (int64_t)c * 1536);
    };
    auto fetch_w = [&](int f, int c) {
#pragma unroll
        for (int h = 0; h < 2; ++h) staged[f][h] = *reinterpret_cast<const f32x4*>(wsrc[f] + 32 * c + 4 * h);
    };
    bf16x8 w[4][3], x[2][3];
    auto read_w = [&](int t, int z, int buf) { w[t][z] = load_frag(tiles + buf * BUF + (3 * (4 * wave + t) + z) * 512 + lane * 8); };
    auto read_x = [&](int m, int z, int buf) { x[m & 1][z] = load_frag(tiles + buf * BUF + (3 * (NP + m) + z) * 512 + lane * 8); };
    // What makes a step's tiles visible to the other waves: this wave's DMA has landed (nothing may be in flight but weights asked for behind
    // it, which stay in flight over the barrier), its LDS stores are done, and no access crosses the barrier.  Both are compiler fences too: an access
    // to LDS may not move over them, whatever order the scheduler likes.
    auto landed = [&] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    auto meet = [&] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    f32x4 acc[4][MT], low[4][MT];                             // hh and the five small products
    auto clear = [&] {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[t][m] = low[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    do {
    const int r = beg / chunks, c_beg = beg - r * chunks, c_end = min(chunks, c_beg + end - beg), id = share.first + (q < 0 ? j : share.own + r);
    const int nt = id / mts, mt0 = id % mts;
#pragma unroll
    for (int f = 0; f < PER; ++f) {
        const int p = (wave * PER + f) / 3, z = (wave * PER + f) % 3;
        src[f] = a.xp + (int64_t)min(mt0 * MT + p, xpan - 1) * chunks * 1536 + z * 512;
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) wsrc[f] = a.w + (int64_t)min(nt * 256 + 16 * (wave + 4 * f) + i, a.n - 1) * a.k + 8 * g;
    float* part = q < 0 ? nullptr : a.ws + ((int64_t)xcd * a.slots + q + r) * SLOT;           // a row of 256 behind the other
    clear();
    const int lines = q < 0 ? a.rows : 1 << 30, panels = min(4, (a.n - nt * 256 - 64 * wave) >> 4);
    float odd = 0.f;                                          // NaN behind a result that is not finite
    // this lane's places in row 0 of the result, or of the part's slot, and of the row tiles behind it
    float* y0 = (q < 0 ? a.out + nt * 256 : part) + 64 * wave;
    const int64_t ld = q < 0 ? a.ld_out : 256;
    auto place = [&](int m, int at) { return reinterpret_cast<f32x4*>(y0 + ((q < 0 ? mt0 * 16 * MT : 0) + 16 * m + (at & 15)) * ld + 4 * (at >> 4)); };
    // Sums go to the result, or to a part's slot, and to what is there.
    auto put = [&](bool more) __attribute__((always_inline)) {
        int at = lane;
        asm volatile("" : "+v"(at));                          // (places made ahead of the steps would take registers from them)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int row0 = mt0 * 16 * MT + 16 * m;
            asm volatile("" ::: "memory");                    // (sums and places of all rows, read ahead, would take all registers)
            __builtin_amdgcn_sched_barrier(0);
            if (row0 >= a.rows) break;
            f32x4* y = place(m, at);
            const bool live = row0 + (at & 15) < lines;
            f32x4 have[4] = {};
            if (FOLDS && more && live)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (t < panels) have[t] = y[4 * t];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                asm volatile("" : "+a"(acc[t][m]), "+a"(low[t][m]));
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = (acc[t][m][e] + low[t][m][e]) * (1.f / (SPLIT_SCALE * SPLIT_SCALE));
                    if constexpr (FOLDS) v[e] += have[t][e];
                    odd = fmaf(v[e], 0.f, odd);
                }
                if (t < panels && live) y[4 * t] = v;
            }
        }
    };
    // Steps c .. stop - 1 over the first LIVE row tiles.  While step c is multiplied the weights of c + 1 are cut, between its products, and those of
    // c + 2 asked for, as soon as x of c + 1 has landed.  The waves meet in front of the last row tile, whose x is in registers: from there on x of c + 2
    // may come in over this step's, and w and x of c + 1 are read behind their last use.
    auto run = [&](auto live, int& c, int stop) __attribute__((always_inline)) {
        constexpr int LIVE = decltype(live)::value, CUTS = 4 * (LIVE - 2);     // (cut behind the first CUTS results)
        for (; c < stop; ++c) {
            const int buf = (c - c_beg) & 1;
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_nop 1" ::: "memory");             // (between zeros and copies, which the loop may begin with, and the products that read them)
            __builtin_amdgcn_sched_barrier(0);
            float va = 0.f, vb = 0.f;
            u32x4 out[3];
            // an eighth of the cut of a pair: two operations at most, what the matrix core leaves room for behind a product
            uint32_t ha, hb;
            auto cut = [&](auto at) __attribute__((always_inline)) {
                constexpr int p = decltype(at)::value / 8, f = p / 4, e = p % 4, z = decltype(at)::value % 8;
                if constexpr (z == 0) {
                    va = staged[f][e >> 1][2 * (e & 1)] * SPLIT_SCALE;
                    vb = staged[f][e >> 1][2 * (e & 1) + 1] * SPLIT_SCALE;
                    asm volatile("" ::"v"(va), "v"(vb));
                } else if constexpr (z == 1 || z == 4 || z == 7) {
                    typedef bf16 Pair __attribute__((ext_vector_type(2)));
                    constexpr int y = z / 3;
                    uint32_t v = __builtin_bit_cast(uint32_t, Pair{(bf16)va, (bf16)vb});
                    asm("" : "+v"(v));
                    out[y][e] = v;
                    if constexpr (e == 3) *reinterpret_cast<u32x4*>(tiles + (buf ^ 1) * BUF + (wave + 4 * f) * 1536 + 512 * y + lane * 8) = out[y];
                    if constexpr (f == 0 && e == 3 && y == 2) landed();                  // (x of the next step, asked for behind the last barrier)
                    if constexpr (e == 3 && y == 2) fetch_w(f, min(c + 2, c_end - 1));
                } else if constexpr (z == 2 || z == 5) {
                    ha = out[z / 3][e] << 16;
                    hb = out[z / 3][e] & 0xFFFF0000u;
                    asm volatile("" ::"v"(ha), "v"(hb));
                } else {
                    va -= __builtin_bit_cast(float, ha);
                    vb -= __builtin_bit_cast(float, hb);
                    asm volatile("" ::"v"(va), "v"(vb));
                }
            };
            upto<24 * LIVE>([&](auto at) __attribute__((always_inline)) {
                constexpr int s = decltype(at)::value % 6, t = decltype(at)::value / 6 % 4, m = decltype(at)::value / 24;
                constexpr int WZ[6] = {2, 0, 1, 1, 0, 0}, XZ[6] = {0, 2, 1, 0, 1, 0};          // smallest first
                constexpr int P = decltype(at)::value, FIRST = P < 6 * CUTS ? 128 * P / (6 * CUTS) : 0, N = P < 6 * CUTS ? 128 * (P + 1) / (6 * CUTS) - FIRST : 0;
                if constexpr (m == LIVE - 1 && t == 0 && s == 0) meet();
                if constexpr (s < 5) add_in_place(w[t][WZ[s]], x[m & 1][XZ[s]], low[t][m]);
                else add_in_place(w[t][WZ[s]], x[m & 1][XZ[s]], acc[t][m]);
                __builtin_amdgcn_sched_barrier(0);
                upto<N>([&](auto n) __attribute__((always_inline)) { cut(std::integral_constant<int, FIRST + decltype(n)::value>()); });
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (t < 3 && s == 0) read_x(m + 1 < LIVE ? m + 1 : 0, t, m + 1 < LIVE ? buf : buf ^ 1);
                if constexpr (m + 1 == LIVE && t > 0 && (s & 1) == 0) read_w(t - 1, s / 2, buf ^ 1);
                if constexpr (m + 1 == LIVE && t == 0) fetch_x(s, min(c + 2, c_end - 1), buf);
                __builtin_amdgcn_sched_barrier(0);
            });
#pragma unroll
            for (int z = 0; z < 3; ++z) read_w(3, z, buf ^ 1);
            hold_sums();
        }
    };
    const bool half = xpan - mt0 * MT <= MT / 2;
    if (c_beg < c_end) {
#pragma unroll
        for (int f = 0; f < PER; ++f) fetch_x(f, c_beg, 0);
#pragma unroll
        for (int f = 0; f < 4; ++f) fetch_w(f, c_beg);
#pragma unroll
        for (int f = 0; f < 4; ++f) cut_store(staged[f], tiles + (wave + 4 * f) * 1536 + lane * 8);
        landed();
#pragma unroll
        for (int f = 0; f < 4; ++f) fetch_w(f, min(c_beg + 1, c_end - 1));
        meet();
#pragma unroll
        for (int f = 0; f < PER; ++f) fetch_x(f, min(c_beg + 1, c_end - 1), 1);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int z = 0; z < 3; ++z) read_w(t, z, 0);
#pragma unroll
        for (int z = 0; z < 3; ++z) read_x(0, z, 0);
    }
    for (int c = c_beg;;) {
    const int stop = FOLDS ? min(c_end, c + a.fold) : c_end;
    if (half) run(std::integral_constant<int, MT / 2>(), c, stop);
    else run(std::integral_constant<int, MT>(), c, stop);
    put(c > c_beg + a.fold);
    if (!FOLDS || c >= c_end) break;
    clear();
    }
    landed();
    meet();                                                   // nothing is on its way to LDS, and nobody reads it
    if (q < 0 && __any(odd != 0.f))
#pragma unroll 1
        for (int e = 0; e < 4 * MT; ++e) {
            const int row0 = mt0 * 16 * MT + 16 * (e >> 2), t = e & 3;
            if (row0 >= a.rows || t >= panels) continue;
            f32x4 *y = place(e >> 2, lane) + 4 * t, v = {0.f, 0.f, 0.f, 0.f};
            if (row0 + i < lines) v = *y;
            mend(a, row0, nt * 256 + 64 * wave + 16 * t, v);
            if (row0 + i < lines) *y = v;
        }
    beg += c_end - c_beg;
    } while (beg < end);
}

// The parts of shared tiles, summed in order: a wave takes a 16 x 16 tile, a workgroup four side by side.
__global__ __launch_bounds__(256) void split_sum_kernel(const SplitGemm a) {
    const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15, mts = (a.rows + 127) / 128, tiles = (a.n + 255) / 256 * mts;
    const int xcd = blockIdx.x & 7, r = blockIdx.x >> 8, at = blockIdx.x >> 3 & 31;          // (32 pieces of a tile)
    const Share share = share_of(tiles, a.k >> 5, a.whole, a.splits, a.sharers, xcd);
    if (r >= share.rest) return;
    const int id = share.first + share.own + r, in_row = 16 * (at >> 2), in_n = 64 * (at & 3) + 16 * (threadIdx.x >> 6);
    const int row0 = id % mts * 128 + in_row, n0 = id / mts * 256 + in_n;
    if (row0 >= a.rows || n0 >= a.n) return;
    int q = r * share.parts, parts = share.parts;
    if (!parts) {
        q = r * share.sharers / share.rest;                   // its first part begins in it, or reaches into it from the tile before
        while (q > 0 && share.cut(q) > r * share.chunks) --q;
        while (share.cut(q + 1) <= r * share.chunks) ++q;
        for (parts = 1; q + parts < share.sharers && share.cut(q + parts) < (r + 1) * share.chunks;) ++parts;
    }
    const float* src = a.ws + ((int64_t)xcd * a.slots + q + r) * SLOT + 256 * (in_row + i) + in_n + 4 * g;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < parts; ++z) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(src + (int64_t)z * SLOT);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += v[e];
    }
    mend(a, row0, n0, s);
    if (row0 + i < a.rows) *reinterpret_cast<f32x4*>(a.out + (int64_t)(row0 + i) * a.ld_out + n0 + 4 * g) = s;
}

static int launch_split_gemm(const SplitGemm& a, hipStream_t st) {
    constexpr int LDS = 2 * 3 * (16 + 8) * 1024;              // two buffers of 16 panels of weights and 8 of x, in three parts
    const auto kernel = a.fold < a.k >> 5 ? split_gemm_kernel<true> : split_gemm_kernel<false>;
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return (int)e;
    const int each = (split_tiles(a.rows, a.n) + 7) / 8, own = each < a.whole ? each : a.whole, rest = each - own;
    hipLaunchKernelGGL(kernel, dim3(8 * (own + (rest == 0 ? 0 : a.sharers > 0 ? a.sharers : rest * a.splits))), dim3(256), LDS, st, a);
    TFL_LAUNCH_CHECK();
    if (rest > 0) {
        hipLaunchKernelGGL(split_sum_kernel, dim3((unsigned)rest * 256), dim3(256), 0, st, a);
        TFL_LAUNCH_CHECK();
    }
    return TF_OK;
}

// In floats: x's planes, and one mark per row and part of k (16-byte pieces).
static int64_t split_planes(int rows, int k) { return (int64_t)((rows + 15) / 16) * (k / 32) * 1536 * 2 / 4; }
static int64_t split_marks(int rows, int k) { return ((int64_t)rows * split_parts(k) + 3) / 4 * 4; }

struct Parts { int whole, splits, sharers, fold; };

// How k is cut: rounds of workgroups, each with the fill of its pipe (4 steps of 32), against what the parts cost on their way through memory
// (a written and read 128 x 256 part as much as 8 steps).  Rounds are an XCD's: it has 32 CUs and its eighth of the tiles, rounded up (36 tiles in
// seven parts are 252 workgroups, but 35 on some XCDs: 700 rows, 1 536 x 6 144 in seven 126 us, in six 92).  256 rows, 12 320 x 4 096: 240 us
// without parts, 148 with two, 164 with four; 700 rows, 4 096 x 8 192: 468, 274 with two, 250 with five, 256 with eight.
// From 32 tiles an XCD on: whole rounds of whole tiles, and the steps of the others shared by all CUs, 8 or more to each.  Whole tiles alone | the best of
// two to eight parts of all tiles | this: 700 rows of 22 016 x 4 096 757 | 692 | 605 us, of 12 320 499 | 402 | 364, 1 000 rows of them 523 | 531 | 466,
// 300 rows of 22 016 414 | 349 | 309, 1 500 1 331 | 1 324 | 1 193.  Below, sharing gains nothing over whole tiles on fewer CUs, which run at a higher clock (256
// rows of 22 016, 172 tiles, with eight waves: 317 us alone, 327 shared).  The constants were fitted to eight waves of 64 x 64 and hold for these four: over 19
// sizes of 256 to 2 048 rows what they pick takes 1.03 of the best number of parts at most.
// A running sum of all steps is further off than the parts that k would be in otherwise (absolute values, 4 096 columns: 3.5e-7, two parts 1.8e-7,
// three 1.1e-7), so it goes to the result as often (`fold`), at 4 steps' cost each (eight waves, 700 rows of 22 016: 637 -> 665 us), error as in two parts.
static Parts pick_parts(int rows, int n, int k) {
    const int tiles = split_tiles(rows, n), per_xcd = (tiles + 7) / 8;
    const double chunks = k / 32;
    Parts best{0, 1, 0, k / 32};
    double least = 0;
    for (int s = 1; s <= 8 && (s == 1 || s * 512 <= k); ++s) {
        const double t = (double)(((int64_t)per_xcd * s + 31) / 32) * (1.0 / s + 4.0 / chunks) + (s > 1 ? 8.0 * (double)s * tiles / 256 / chunks : 0);
        if (s == 1 || t < least) { best.splits = s; least = t; }
    }
    const int parts = best.splits, fold = (k / 32 + parts - 1) / parts;
    for (int w = per_xcd >> 5; w > 0 && w >= (per_xcd >> 5) - 1; --w) {
        const int rest = per_xcd - 32 * w;
        const int64_t line = (int64_t)rest * (k / 32);
        if (rest == 0 || line < 16 || line > 1 << 24) continue;
        const int sharers = (int)(line / 8 < 32 ? line / 8 : 32);
        const double t = w * (1.0 + 4.0 * parts / chunks) + rest / (double)sharers + (rest > 1 ? 8.0 : 4.0) / chunks + 8.0 * (sharers + rest) / 32 / chunks + 3.0 / chunks;
        if (t < least) { best = Parts{32 * w, 1, sharers, fold}; least = t; }
    }
    if (best.sharers == 0 && best.splits == 1) best.whole = 1 << 28;
    return best;
}

static Parts given_parts(int rows, int n, int k, int splits) {
    return splits == 0 ? pick_parts(rows, n, k) : Parts{splits == 1 ? 1 << 28 : 0, splits, 0, k / 32};
}

extern "C" int64_t tfl_split_gemm_ws_floats(int rows, int n, int k, int splits) {
    if (rows < 1 || rows > (1 << 24) || n < 16 || k < 32 || splits < 0 || splits > 64) return 0;
    const Parts p = given_parts(rows, n, k, splits);
    return split_planes(rows, k) + split_marks(rows, k) + (int64_t)8 * split_slots(split_tiles(rows, n), p.whole, p.splits, p.sharers) * SLOT;
}

extern "C" int tfl_split_gemm(const float* w, const float* x, int64_t ld_x, float* out, int64_t ld_out, float* ws, int64_t ws_floats, int rows, int n,
                              int k, int splits, void* stream) {
    if (!w || !x || !out || !ws || rows < 1 || rows > (1 << 24) || n < 16 || (n & 15) || k < 32 || (k & 31) || ld_x < k || (ld_x & 3) || ld_out < n
        || (ld_out & 3) || splits < 0 || splits > 64) return TF_EINVAL;
    if (((uintptr_t)w | (uintptr_t)x | (uintptr_t)out | (uintptr_t)ws) & 15) return TF_EINVAL;
    const Parts p = given_parts(rows, n, k, splits);
    if (ws_floats < tfl_split_gemm_ws_floats(rows, n, k, splits)) return TF_ENOSPC;
    int32_t* nans = (int32_t*)(ws + split_planes(rows, k));
    hipLaunchKernelGGL(split_rows_kernel, dim3((rows + 15) / 16, split_parts(k)), dim3(256), 0, (hipStream_t)stream, x, ld_x, rows, k, (bf16*)ws, nans);
    TFL_LAUNCH_CHECK();
    const SplitGemm a = {w, (const bf16*)ws, x, out, ws + split_planes(rows, k) + split_marks(rows, k), nans, ld_x, ld_out, rows, n, k, p.whole, p.splits, p.sharers,
                         split_slots(split_tiles(rows, n), p.whole, p.splits, p.sharers), p.fold};
    return launch_split_gemm(a, (hipStream_t)stream);
}
