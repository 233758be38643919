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
// 256 outputs x 128 rows per workgroup, eight waves of 64 x 64: per step of 32 a wave reads 24 KB from LDS for 96 products (1 536 cycles),
// half of what LDS delivers.  x is cut once by a kernel in front, into planes in MFMA order ([rows/16][k/32][3][64 lanes][8]: a fragment is one
// contiguous KiB that goes to LDS by DMA); a weight is used by one workgroup per 128 rows and is cut on its way to LDS, beside the products.
// (Cut at load time
// into planes, weights cost 6 bytes beside the 4 and gain 3 to 8 %: 22 016 x 4 096 at 700 rows 706 us against 730.  The cut between the
// products instead of behind them waits for x's DMA before each store to LDS: 22 016 x 4 096 at 2 048 rows 1 830 -> 2 230 us.)
//
// Bound by the power of the matrix cores (1.6 to 1.7 GHz under these products, as bf16 GEMMs), by what a step costs beside its products (all
// operands zero, at full clock: 22 016 x 4 096 at 700 rows 613 -> 567 us) and by rounds of tiles.  A matrix core draws less where a product goes to the sum
// that the one before it went to (registers alone, bf16 normals: 2 110 TFLOP/s with another sum each time, 2 226 in twos, 2 350 in fours, 2 395 in
// eights), so the five small products of a result follow each other, and a row tile's parts are read during the products of the one before: 700 rows,
// 22 016 x 4 096 665 -> 613 us, 18 784 x 4 096 567 -> 537, 4 096 x 15 104 481 -> 460, 4 096 x 8 192 266 -> 256; 2 048 rows of 22 016 1 719 -> 1 642
// (225 TFLOP/s); 256 rows of 12 320 158 -> 156.  (In two halves, four waves cutting their weights in front of the products and four behind: nothing.)
// The fp32 instruction, x's cut and the sum of parts included: 700 rows, 22 016 x 4 096 940 us, 18 784 x 4 096 900, 4 096 x 15 104 680; 2 048 rows,
// 22 016 x 4 096 2 600.
//
// Range: both operands are cut at 2^24 times their value, so the last bit of the smallest float32 (2^-149) is still a normal bfloat16 and no
// product of parts that counts leaves fp32's range below; results are multiplied by 2^-48.  Above, a factor from 2^104 or a sum from 2^80
// on becomes infinite on the way; such a result, and one that is not finite because a factor is not (an infinity times a zero part is NaN),
// is computed again in plain fp32, the 16 x 16 tile that it lies in by its wave on the fp32 instruction; rows of x with a NaN, which is what
// an infinity leaves behind in a model, are marked when they are cut and keep their NaN results.  One infinite row of 700 in front of
// 22 016 x 4 096 costs 770 -> 1 040 us, of 300 in front of 4 096 x 15 104 265 -> 530 (by a thread per result 4 200 and 9 900).  (The scaling is 16 of some 200 VALU operations per step: 22 016 x 4 096 at 700 rows 740 -> 752 us.)
#include "tile_common.h"

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

// Waves: 4 x 64 outputs, 2 x 64 rows (MT 16-row tiles of x each); every wave brings PER fragments of x in.  FOLDS: a.fold is below a tile's steps.
template <bool FOLDS>
__global__ __launch_bounds__(512, 2) void split_gemm_kernel(const SplitGemm a) {
    constexpr int MT = 4, NP = 16, XP = 2 * MT, PER = 3 * XP / 8, BUF = 3 * (NP + XP) * 512;
    extern __shared__ __align__(16) bf16 tiles[];             // [2][NP + XP][3][512]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int wn = wave & 3, wm = wave >> 2, chunks = a.k >> 5;
    // workgroups go round-robin over the 8 XCDs: each takes an eighth of the tiles, the row tiles of one column tile one after the other, which
    // share its weights in L2
    const int mts = (a.rows + 32 * MT - 1) / (32 * MT), xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
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
    const float* wsrc[2];                                     // this lane's eight weights of two panels
    f32x4 staged[2][2];
    auto fetch_x = [&](int c, int buf) {
#pragma unroll
        for (int f = 0; f < PER; ++f)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[f] + (int64_t)c * 1536 + lane * 8),
                                             (__attribute__((address_space(3))) void*)(tiles + buf * BUF + (3 * NP + wave * PER + f) * 512), 16, 0, 0);
    };
    auto fetch_w = [&](int c) {
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int h = 0; h < 2; ++h) staged[f][h] = *reinterpret_cast<const f32x4*>(wsrc[f] + 32 * c + 4 * h);
    };
    auto put_w = [&](int buf) {
#pragma unroll
        for (int f = 0; f < 2; ++f) cut_store(staged[f], tiles + buf * BUF + (wave + 8 * f) * 1536 + lane * 8);
    };
    // What makes a step's tiles visible to the other waves: this wave's DMA has landed (nothing may be in flight but the weights asked for
    // behind it, which stay in flight over the barrier), its LDS stores are done, and no access crosses the barrier.  Both are compiler
    // fences too: an access to LDS may not move over them, whatever order the scheduler likes.
    auto landed = [&] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    auto meet = [&] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    do {
    const int r = beg / chunks, c_beg = beg - r * chunks, c_end = min(chunks, c_beg + end - beg), id = share.first + (q < 0 ? j : share.own + r);
    const int nt = id / mts, mt0 = id % mts;
#pragma unroll
    for (int f = 0; f < PER; ++f) {
        const int p = (wave * PER + f) / 3, z = (wave * PER + f) % 3;
        src[f] = a.xp + (int64_t)min(mt0 * XP + p, xpan - 1) * chunks * 1536 + z * 512;
    }
#pragma unroll
    for (int f = 0; f < 2; ++f) wsrc[f] = a.w + (int64_t)min(nt * 256 + 16 * (wave + 8 * f) + i, a.n - 1) * a.k + 8 * g;
    const bool live = mt0 * XP + wm * MT < xpan;              // a wave without rows leaves the matrix core to its neighbour
    float* part = q < 0 ? nullptr : a.ws + ((int64_t)xcd * a.slots + q + r) * SLOT;           // a row of 256 behind the other
    f32x4 acc[4][MT], low[4][MT];                             // hh and the five small products
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = low[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    // f of this lane's places in the result, or in the part's slot
    const int lines = q < 0 ? a.rows : 1 << 30;
    bool lost = false;                                        // a result that is not finite
    auto each = [&](auto&& f) {
        int at = lane;
        if constexpr (FOLDS) asm volatile("" : "+v"(at));     // (places made ahead of the steps would take registers from them)
        const int g = at >> 4, i = at & 15;
        float* y = q < 0 ? a.out : part;
        const int64_t ld = q < 0 ? a.ld_out : 256;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int in_row = 16 * (wm * MT + m), row0 = mt0 * 32 * MT + in_row;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int in_n = 64 * wn + 16 * t;
                if constexpr (FOLDS) {                        // one after the other: what is there would take a step's registers
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (row0 >= a.rows || nt * 256 + in_n >= a.n) continue;
                f(m, t, reinterpret_cast<f32x4*>(y + (q < 0 ? row0 + i : in_row + i) * ld + (q < 0 ? nt * 256 : 0) + in_n + 4 * g), row0, i);
            }
        }
    };
    if (c_beg < c_end) {
        fetch_x(c_beg, 0);
        fetch_w(c_beg);
        put_w(0);
        landed();
        fetch_w(min(c_beg + 1, c_end - 1));
        meet();
    }
    for (int c = c_beg;;) {
    for (const int stop = FOLDS ? min(c_end, c + a.fold) : c_end; c < stop; ++c) {
        const int buf = (c - c_beg) & 1;
        fetch_x(min(c + 1, c_end - 1), buf ^ 1);              // in flight under this step's products
        if (live) {
            const bf16* wt = tiles + buf * BUF + wn * 4 * 1536 + lane * 8;
            const bf16* xt = tiles + buf * BUF + (NP + wm * MT) * 1536 + lane * 8;
            bf16x8 w[4][3];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int z = 0; z < 3; ++z) w[t][z] = load_frag(wt + (3 * t + z) * 512);
            bf16x8 x[2][3];
            auto read_x = [&](int m) {
#pragma unroll
                for (int z = 0; z < 3; ++z) x[m & 1][z] = load_frag(xt + (3 * m + z) * 512);
            };
            read_x(0);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                constexpr int WZ[6] = {2, 0, 1, 1, 0, 0}, XZ[6] = {0, 2, 1, 0, 1, 0};          // smallest first
                if (m + 1 < MT) read_x(m + 1);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int q = 0; q < 6; ++q) {
                        f32x4& s = q < 5 ? low[t][m] : acc[t][m];
                        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][WZ[q]], x[m & 1][XZ[q]], s, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);    // (left to itself the scheduler deals them out among the sums)
                    }
            }
        }
        put_w(buf ^ 1);
        landed();
        fetch_w(min(c + 2, c_end - 1));
        meet();
    }
    if constexpr (!FOLDS) break;
    each([&](int m, int t, f32x4* y, int row0, int i) {       // sums go to the result, or to a part's slot, and to what is there
        f32x4 v, have = {0.f, 0.f, 0.f, 0.f};
        if (c > c_beg + a.fold && row0 + i < lines) have = *y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = (acc[t][m][e] + low[t][m][e]) * (1.f / (SPLIT_SCALE * SPLIT_SCALE)) + have[e];
            lost = lost || !(__builtin_fabsf(v[e]) < __builtin_inff());
        }
        acc[t][m] = low[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (row0 + i < lines) *y = v;
    });
    if (c >= c_end) break;
    }
    if (!FOLDS || (q < 0 && __any(lost)))
        each([&](int m, int t, f32x4* y, int row0, int i) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            if constexpr (!FOLDS) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = (acc[t][m][e] + low[t][m][e]) * (1.f / (SPLIT_SCALE * SPLIT_SCALE));
            } else if (row0 + i < lines) {
                v = *y;
            }
            if (q < 0) mend(a, row0, nt * 256 + 64 * wn + 16 * t, v);
            if (row0 + i < lines) *y = v;
        });
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
    hipLaunchKernelGGL(kernel, dim3(8 * (own + (rest == 0 ? 0 : a.sharers > 0 ? a.sharers : rest * a.splits))), dim3(512), LDS, st, a);
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
// seven parts are 252 workgroups, but 35 on some XCDs: 700 rows, 1 536 x 6 144 in seven 119 us, in six 95).  256 rows, 12 320 x 4 096: 267 us
// without parts, 159 with two, 171 with four; 700 rows, 4 096 x 8 192: 514, 296 with two, 262 with five, 265 with eight.
// From 32 tiles an XCD on: whole rounds of whole tiles, and the steps of the others shared by all CUs, 8 or more to each.  A last round of few tiles,
// or parts of all tiles instead (516 tiles of 22 016 x 4 096 at 700 rows in two parts, 2.5 rounds and 250 MB of parts): 755 -> 665 us; 12 320
// outputs 425 -> 402, 1 000 rows of them 565 -> 509, 300 rows of 22 016 402 -> 365, 1 500 1 437 -> 1 288.  Below, sharing gains nothing over whole
// tiles on fewer CUs, which run at a higher clock (256 rows of 22 016, 172 tiles: 317 us alone, 327 shared).
// A running sum of all steps is further off than the parts that k would be in otherwise (absolute values, 4 096 columns: 3.5e-7, two parts 1.8e-7,
// three 1.1e-7), so it goes to the result as often (`fold`), at 4 steps' cost each: 700 rows of 22 016 637 -> 665 us, error as in two parts.
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
