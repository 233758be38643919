// Attention of the latent family for gfx950.
//
// Decode: the query has been taken through the key up-projection, so the cached row itself is the key ([latent | rotated]) and its latent part the
// value, for every head: one KV stream shared by all heads.  Scores are computed transposed (S^T = K Q^T: rows keys, columns heads), so that a lane
// owns one head's statistics; the weights go to LDS as [head][key] and every wave accumulates its share of the latent columns, O^T = C^T P^T, with the
// transposed operand read straight from the key-major page (ds_read_b64_tr_b16).  In bfloat16 of 512 + 64 (attn_latent_sized_body) half of a workgroup's
// waves score a half page of 32 keys while the other half multiplies the one before; other sizes (attn_latent_kernel) take whole pages, staged in LDS,
// wave w keys 16w .. 16w+15.
//
// Prefill (attn_prefill_kernel): keys and values up-projected once per chunk, flash attention with 16 query rows per wave (2 x 16 in
// attn_prefill_sized_kernel), the waves of a workgroup sharing the key / value tile.  Also transposed: the S^T result registers of two 16-key tiles ARE the P operand of
// one PV product (the value operand is read with the matching key order), so the weights never leave the registers.
#include "flash_tile.h"
#include "lds_dma.h"
#include "share_gemm.h"

#define NEG_INF (-__builtin_inff())
#define LOG2E 1.4426950408889634f

// ---------------------------------------------------------------------------------------------------------------- decode
// Weights as two bfloat16 (value and remainder): the PV product then sees them to 16 bits like the fp32 softmax made them.
template <typename T> struct DecodeCfg { static constexpr int PARTS = sizeof(T) == 2 ? 2 : 1; };

// Any sizes up to the LDS limit.
template <typename T, int NW, int HT, int NTW>
__global__ __launch_bounds__(NW * 64, 1) void attn_latent_kernel(const T* __restrict__ q, const T* __restrict__ cache, int n_pages,
                                                              const int32_t* __restrict__ table, int table_ld,
                                                              const int32_t* __restrict__ len, T* __restrict__ out,
                                                              float* __restrict__ ws, int H, int C, int R, float scale,
                                                              int nsplit, int rows) {
    typedef typename El<T>::Frag Frag;
    constexpr int KT = 16 * NW, NT = NW * 64, EPV = 16 / sizeof(T), PADE = EPV;
    constexpr int PARTS = DecodeCfg<T>::PARTS;
    extern __shared__ __align__(16) char smem[];
    const int W = C + R, wc = W >> 5, ldk = W + PADE, ldp = KT + PADE;
    T* Kt = (T*)smem;                                         // [KT][ldk]
    T* Qs = Kt + KT * ldk;                                    // [16 HT][ldk]
    T* Ps = Qs + 16 * HT * ldk;                               // [PARTS][16 HT][ldp]
    float* red = (float*)(Ps + PARTS * 16 * HT * ldp);        // [NW][16 HT]
    const int split = blockIdx.x, h0 = blockIdx.y * 16 * HT, row = blockIdx.z;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int n = len[row];
    const int ntiles = n > 0 ? (n + KT - 1) / KT : 0;
    const int per = (ntiles + nsplit - 1) / nsplit;
    const int t_beg = min(split * per, ntiles), t_end = min(ntiles, t_beg + per);
    const int ppr = W / EPV;                 // 16-byte pieces per row
    const int32_t* tab = table + (int64_t)row * table_ld;

    for (int p = tid; p < 16 * HT * ppr; p += NT) {           // queries of this head group (heads past H: zeros)
        const int r = p / ppr, c = p - r * ppr;
        u32x4 v = {0, 0, 0, 0};
        if (h0 + r < H) v = *reinterpret_cast<const u32x4*>(q + ((int64_t)row * H + h0 + r) * W + EPV * c);
        *reinterpret_cast<u32x4*>(Qs + r * ldk + EPV * c) = v;
    }
    auto page_base = [&](int t) {
        const int k0 = t * KT;
        int pg = tab[k0 / TFL_PAGE];
        pg = pg < 0 ? 0 : (pg >= n_pages ? n_pages - 1 : pg);
        return (int64_t)pg * TFL_PAGE + (k0 & (TFL_PAGE - 1));
    };
    f32x4 o[HT][NTW];
    float m_run[HT], l_run[HT];
#pragma unroll
    for (int h = 0; h < HT; ++h) {
        m_run[h] = NEG_INF;
        l_run[h] = 0.f;
#pragma unroll
        for (int t = 0; t < NTW; ++t) o[h][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int t = t_beg; t < t_end; ++t) {
        const int k0 = t * KT;
        const T* base = cache + page_base(t) * W;
        for (int p = tid; p < KT * ppr; p += NT) {
            const int r = p / ppr, c = p - r * ppr;
            u32x4 v = {0, 0, 0, 0};
            if (k0 + r < n) v = *reinterpret_cast<const u32x4*>(base + (int64_t)r * W + EPV * c);
            *reinterpret_cast<u32x4*>(Kt + r * ldk + EPV * c) = v;
        }
        __syncthreads();
        f32x4 s[HT];
#pragma unroll
        for (int h = 0; h < HT; ++h) s[h] = f32x4{0.f, 0.f, 0.f, 0.f};
        const T* kp = Kt + (16 * wave + i) * ldk + 8 * g;
        const T* qp = Qs + i * ldk + 8 * g;
        auto chunk = [&](int c) {
            const Frag a = load_frag(kp + 32 * c);
#pragma unroll
            for (int h = 0; h < HT; ++h) s[h] = El<T>::mma(a, load_frag(qp + h * 16 * ldk + 32 * c), s[h]);
        };
        for (int c = 0; c < wc; ++c) chunk(c);
#pragma unroll
        for (int h = 0; h < HT; ++h) {
            float mx = NEG_INF;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[h][r] = k0 + 16 * wave + 4 * g + r < n ? s[h][r] * scale : NEG_INF;
                mx = fmaxf(mx, s[h][r]);
            }
            mx = rows_max(mx);
            if (g == 0) red[wave * 16 * HT + 16 * h + i] = mx;
        }
        __syncthreads();
        float alpha[HT];
#pragma unroll
        for (int h = 0; h < HT; ++h) {
            float mx = m_run[h];
#pragma unroll
            for (int w = 0; w < NW; ++w) mx = fmaxf(mx, red[w * 16 * HT + 16 * h + i]);
            alpha[h] = exp2f((m_run[h] - mx) * LOG2E);        // (the tile's first key is visible: mx is finite)
            m_run[h] = mx;
            f32x4 p, lo;
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] = exp2f((s[h][r] - mx) * LOG2E);
                sum += p[r];
                lo[r] = p[r] - (float)(T)p[r];
            }
            l_run[h] = l_run[h] * alpha[h] + sum;
            T* dst = Ps + (16 * h + i) * ldp + 16 * wave + 4 * g;
            store_quad(dst, p);
            if constexpr (PARTS == 2) store_quad(dst + 16 * HT * ldp, lo);
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < HT; ++h)
#pragma unroll
            for (int x = 0; x < NTW; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[h][x][r] *= alpha[h];
#pragma unroll
        for (int c = 0; c < KT / 32; ++c) {
            Frag b[HT][PARTS];
#pragma unroll
            for (int h = 0; h < HT; ++h)
#pragma unroll
                for (int z = 0; z < PARTS; ++z) b[h][z] = load_frag(Ps + (z * 16 * HT + 16 * h + i) * ldp + 32 * c + 8 * g);
#pragma unroll
            for (int x = 0; x < NTW; ++x) {
                const int col = 16 * (wave * NTW + x);
                if (col < C) {
                    const Frag a = load_frag_t(Kt, ldk, 32 * c + 8 * g, 32 * c + 8 * g + 4, col, i);
#pragma unroll
                    for (int h = 0; h < HT; ++h)
#pragma unroll
                        for (int z = 0; z < PARTS; ++z) o[h][x] = El<T>::mma(a, b[h][z], o[h][x]);
                }
            }
        }
        __syncthreads();
    }
    // sum of the weights: lane groups hold different keys, waves too
#pragma unroll
    for (int h = 0; h < HT; ++h) {
        float l = l_run[h];
        l = rows_sum(l);
        if (g == 0) red[wave * 16 * HT + 16 * h + i] = l;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < HT; ++h) {
        const int head = h0 + 16 * h + i;
        if (head >= H) continue;
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) l += red[w * 16 * HT + 16 * h + i];
        if (nsplit == 1) {
            const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
            for (int x = 0; x < NTW; ++x) {
                const int col = 16 * (wave * NTW + x) + 4 * g;
                if (col < C) {
                    f32x4 v = o[h][x];
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] *= inv;
                    store_quad(out + ((int64_t)row * H + head) * C + col, v);
                }
            }
        } else {
            const int64_t at = ((int64_t)row * H + head) * nsplit + split;
            float* wo = ws + at * C;
#pragma unroll
            for (int x = 0; x < NTW; ++x) {
                const int col = 16 * (wave * NTW + x) + 4 * g;
                if (col < C && l > 0.f) *reinterpret_cast<f32x4*>(wo + col) = o[h][x];   // (empty splits are not read either)
            }
            if (wave == 0 && g == 0) {
                float* ml = ws + (int64_t)rows * H * nsplit * C + at * 2;
                ml[0] = m_run[h];
                ml[1] = l;
            }
        }
    }
}

// Merge of the splits: one workgroup per (64 latent columns, head, row); 16 threads across the columns, 16 over the splits.
template <typename T>
__global__ __launch_bounds__(256) void latent_merge_kernel(const float* __restrict__ ws, T* __restrict__ out, int rows, int H,
                                                           int C, int nsplit) {
    __shared__ float wgt[256];
    __shared__ float red[8];
    __shared__ f32x4 acc[256];
    const int head = blockIdx.y, row = blockIdx.z, tid = threadIdx.x;
    const int64_t at = ((int64_t)row * H + head) * nsplit;
    const float* ml = ws + (int64_t)rows * H * nsplit * C + at * 2;
    const int col = 64 * blockIdx.x + 4 * (tid & 15), grp = tid >> 4;
    const float* src = ws + at * C + min(col, C - 4);
    // Bound by round trips: the first partial rows are asked for together with the statistics, whose two halves come at once (1 row of 4 000 keys,
    // 32 heads, 4.7 -> 4.0 us).
    constexpr int U = 4;
    f32x4 z0[U];
#pragma unroll
    for (int u = 0; u < U; ++u) z0[u] = *reinterpret_cast<const f32x4*>(src + (int64_t)min(grp + 16 * u, nsplit - 1) * C);
    // thread s owns the statistics of split s (nsplit <= 256); an empty split has weight 0 and its partial row is never used
    const float m_have = ml[2 * min(tid, nsplit - 1)], l_have = ml[2 * min(tid, nsplit - 1) + 1];
    const float ls = tid < nsplit ? l_have : 0.f, ms = ls > 0.f ? m_have : NEG_INF;
    float m = ms;
    m = lanes_max(m);
    if ((tid & 63) == 0) red[4 + (tid >> 6)] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7]));
    const float w = ls > 0.f ? exp2f((ms - m) * LOG2E) : 0.f;
    const float l = block_sum<4>(w * ls, red);
    wgt[tid] = l > 0.f ? w / l : 0.f;
    __syncthreads();
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (col < C) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = grp + 16 * u;
            const float f = s < nsplit ? wgt[s] : 0.f;
            if (f > 0.f) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = fmaf(z0[u][r], f, v[r]);
            }
        }
#pragma unroll 4
        for (int s = grp + 16 * U; s < nsplit; s += 16) {
            const float ws_ = wgt[s];
            if (ws_ > 0.f) {
                const f32x4 z = *reinterpret_cast<const f32x4*>(src + (int64_t)s * C);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = fmaf(z[r], ws_, v[r]);
            }
        }
    }
    acc[tid] = v;
    __syncthreads();
    if (grp == 0 && col < C) {
#pragma unroll
        for (int k = 1; k < 16; ++k) {
            const f32x4 z = acc[16 * k + tid];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += z[r];
        }
        store_quad(out + ((int64_t)row * H + head) * C + col, v);
    }
}

// The merge for at most 64 splits and whole 128-column blocks: one wave per (128 latent columns, head, row), lane s holding the statistics
// of split s, so there is no LDS and no barrier; two columns per lane, 16 partial rows asked for at once.  The form above spends
// a workgroup with four barriers on 64 columns: 32 rows x 32 heads x 8 splits of 512 11.8 -> 5.5 us; one row (128 waves) stays with
// it.
template <typename T>
__global__ __launch_bounds__(256) void latent_merge_waves_kernel(const float* __restrict__ ws, T* __restrict__ out, int rows, int H, int C, int nsplit) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef T Pair __attribute__((ext_vector_type(2)));
    constexpr int U = 16;
    const int blocks = C >> 7, lane = threadIdx.x & 63;
    const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), pair = unit / blocks;          // pair = row * H + head
    if (pair >= (int64_t)rows * H) return;
    const int col = 128 * (int)(unit - pair * blocks) + 2 * lane;
    const float* ml = ws + (int64_t)rows * H * nsplit * C + pair * nsplit * 2;
    const float m_have = ml[2 * min(lane, nsplit - 1)], l_have = ml[2 * min(lane, nsplit - 1) + 1];      // (both at once)
    const float ls = lane < nsplit ? l_have : 0.f, ms = ls > 0.f ? m_have : NEG_INF;
    const float* src = ws + pair * nsplit * C + col;
    f32x2 v = {0.f, 0.f};
    float w = 0.f;
    for (int s0 = 0; s0 < nsplit; s0 += U) {
        f32x2 z[U];
#pragma unroll
        for (int u = 0; u < U; ++u) z[u] = *reinterpret_cast<const f32x2*>(src + (int64_t)min(s0 + u, nsplit - 1) * C);
        if (s0 == 0) {                                        // (the statistics arrive under the first partial rows)
            float m = ms;
            m = lanes_max(m);
            w = ls > 0.f ? exp2f((ms - m) * LOG2E) : 0.f;
            const float l = wave_sum64(w * ls);
            w = l > 0.f ? w / l : 0.f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float f = __shfl(w, min(s0 + u, 63), 64);
            if (s0 + u < nsplit && f > 0.f) {                 // (an empty split's partial row was never written)
                v[0] = fmaf(z[u][0], f, v[0]);
                v[1] = fmaf(z[u][1], f, v[1]);
            }
        }
    }
    *reinterpret_cast<Pair*>(out + pair * C + col) = Pair{(T)v[0], (T)v[1]};
}

template <typename T>
static int launch_merge(const float* ws, void* out, int rows, int H, int C, int nsplit, hipStream_t st) {
    if (nsplit <= 64 && (C & 127) == 0 && rows * H >= 128) {
        const int64_t waves = (int64_t)rows * H * (C >> 7);
        hipLaunchKernelGGL((latent_merge_waves_kernel<T>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, ws, (T*)out, rows, H, C, nsplit);
    } else {
        hipLaunchKernelGGL((latent_merge_kernel<T>), dim3((C + 63) / 64, H, rows), dim3(256), 0, st, ws, (T*)out, rows, H, C, nsplit);
    }
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// The same attention for rows of 512 + 64 in bfloat16, up to 32 heads per workgroup.  Half pages (32 keys) stream through four places in LDS,
// where LDS-DMA brings them two ahead of their use.  Waves 0 .. 3 score a half page (16 keys x 16 heads each, queries in registers) while waves
// 4 .. 7 multiply the one before it with its weights (128 of the latent columns each, all heads): one barrier a half page.
// The weights' reference lies ROOM above a head's largest score of the first half page, and stays until a score passes it; then it moves ROOM above that
// one and the sums are scaled.  So no weight is above 1, and sums of large latents overflow where they do with a running maximum, not before.  The largest
// weight is at least 2^-8 behind a reference that has just moved: weights go in as value and remainder, whose precision does not depend on the scale,
// and 8 places leave the smallest normal latents' sums (2^-126 of them, in denormals of 2^-149) more places than the result has.
// A place holds rows of 1 152 bytes; inside every 128 bytes the pieces of 16 are XORed by swap(row), which leaves the row reads of the scores and
// the transposing reads of the values without bank conflicts.
// 5.5 TB/s behind some 9 us of start and end, with one half page under way: where a page is looked up the compiler waits for the loads before it.  With
// that wait in the branch that asks for more ids, and so two under way, 1 204 sizes are the same to 1 % (apart 0.99 to 1.00, beside a product 1.00).
// Eight waves that took a page together, scored it, met, weighed it, met and multiplied it needed 2.6 us a page from L2 and 3.8 from memory, with the
// maxima and the scaling in every page; this 2.05 and 3.4.  us with the merge, 32 heads, keys from memory, before -> now: 32 rows of 24 / 48 / 96 pages
// 28.2 / 40.0 / 62.7 -> 25.5 / 34.8 / 55.1, 8 of 48 / 192 22.3 / 38.3 -> 19.3 / 34.3, one of 64 / 512 18.1 / 28.3 -> 14.3 / 25.7.  More loads under way (one
// word of each line, 4 to 8 half pages ahead): 62 -> 71 to 77.
struct LatentTile {
    static constexpr int KT = 32, W = 576, C = 512, H = 32, BYTES = KT * W * 2, RING = 4, LDP = KT + 8, PARTS = 2;
    static constexpr int P_ELEMS = PARTS * H * LDP, RED = RING * BYTES + 2 * P_ELEMS * 2, LDS = RED + 4 * (2 * H + H + 2);
};
static_assert(LatentTile::LDS <= 160 * 1024, "LDS");

template <int LEFT> __device__ __forceinline__ void meet() { meet_dma<LEFT, true>(); }

// (everything but the pointers is the same in all lanes)
__device__ __forceinline__ void attn_latent_sized_body(const bf16* __restrict__ q, const bf16* __restrict__ cache, int n_pages, const int32_t* __restrict__ tab,
                                                       int n, bf16* __restrict__ out, float* __restrict__ ws, int H, float scale, int nsplit, int rows,
                                                       int row, int h0, int split, int t_beg, int t_end, char* smem) {
    typedef LatentTile Z;
    constexpr int W = Z::W, C = Z::C, LDP = Z::LDP, ROW = 2 * W, PIECES = W / 8, LOADS = Z::BYTES / 4096;
    constexpr float ROOM = 8.0f / LOG2E;
    typedef __attribute__((address_space(3))) const char* Lds;
    typedef __attribute__((address_space(3))) bf16x4* Lds4;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15, part = wave & 3;
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    bf16* Ps = (bf16*)(smem + Z::RING * Z::BYTES);            // [2 half pages][2 (value, remainder)][32 heads][LDP]
    float* red = (float*)(smem + Z::RED);                     // [2][32]: by 16 keys
    float* ref = red + 2 * Z::H;                              // [32]
    volatile int* grow = (volatile int*)(ref + Z::H);         // [2 half pages]: (a fast wave may set the next one's before a slow one has read this one's)
    const int keys = max(0, min(n, 64 * t_end) - 64 * t_beg), nt = (keys + Z::KT - 1) / Z::KT;         // of this split
    auto swap = [](int r) { return (r >> 2 & 1) | (r >> 1 & 1) << 1 | (r >> 3 & 1) << 2; };

    if (wave < 4) {                                           // ---- scores and weights
        const int ks = part & 1, head = 16 * (part >> 1) + i; // this wave's keys, a lane's head
        float* ml = ws + (int64_t)rows * H * nsplit * C + (((int64_t)row * H + h0 + head) * nsplit + split) * 2;
        const bool writes = nsplit > 1 && ks == 0 && g == 0 && h0 + head < H;
        if (nt == 0) {
            if (writes) {
                ml[0] = NEG_INF;
                ml[1] = 0.f;
            }
            return;
        }
        // loads: pieces tid + 256 u of a half page; the ids of 64 pages at a time in the lanes
        uint32_t off[LOADS];
        int ids = 0, window = 0;
        auto place = [&](int u, int last) {
            const int p = tid + 256 * u, r = p / PIECES, c = p - PIECES * r;
            return (uint32_t)min(r, last) * ROW + 16 * ((c & ~7) | ((c ^ swap(r)) & 7));
        };
        auto page_ids = [&] { ids = t_beg + 64 * window + lane < t_end ? tab[t_beg + 64 * window + lane] : 0; };
        auto fetch = [&](int j) {                             // (past the end: the last one again, not used)
            const int c = min(j, nt - 1), t = c >> 1, left = keys - 1 - Z::KT * c;
            if (t >> 6 != window) {
                window = t >> 6;
                page_ids();
            }
            const int pg = __builtin_amdgcn_readlane(ids, t & 63);
            const char* src = (const char*)(cache + (int64_t)(pg < 0 ? 0 : (pg >= n_pages ? n_pages - 1 : pg)) * (64 * W)) + (c & 1) * Z::BYTES;
            const uint32_t dst = lds + (j & 3) * Z::BYTES + 1024 * part;
#pragma unroll
            for (int u = 0; u < LOADS; ++u) lds_dma(__builtin_amdgcn_readfirstlane(dst + 4096 * u), left >= Z::KT - 1 ? off[u] : place(u, left), src);
        };
        page_ids();
#pragma unroll
        for (int u = 0; u < LOADS; ++u) off[u] = place(u, Z::KT - 1);
        fetch(0);
        fetch(1);
        fetch(2);
        bf16x8 qf[W / 32];
        f32x4 s = {0.f, 0.f, 0.f, 0.f};                       // scores of the half page whose weights are not used yet
        float m, l = 0.f, sum = 0.f;                          // sum: of those weights
        auto frag = [&](uint32_t at, int c) { return *(const __attribute__((address_space(3))) bf16x8*)((Lds)(uintptr_t)(at ^ (64 * (c & 1))) + 128 * (c >> 1)); };
        const uint32_t k_at = lds + (16 * ks + i) * ROW + 16 * (g ^ swap(i));
        auto scores = [&](int j) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
            const uint32_t at = k_at + (j & 3) * Z::BYTES;
#pragma unroll
            for (int c = 0; c < W / 32; c += 2) {
                a = El<bf16>::mma(frag(at, c), qf[c], a);
                b = El<bf16>::mma(frag(at, c + 1), qf[c + 1], b);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = Z::KT * j + 16 * ks + 4 * g + r < keys ? (a[r] + b[r]) * scale : NEG_INF;
        };
        auto largest = [&] {                                  // of these 16 keys, into red
            float x = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
            x = rows_max(x);
            if (g == 0) red[Z::H * ks + head] = x;
        };
        auto weights = [&](int j) {
            f32x4 p, lo;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] = __builtin_amdgcn_exp2f((s[r] - m) * LOG2E);
                lo[r] = p[r] - (float)(bf16)p[r];
            }
            sum = (p[0] + p[1]) + (p[2] + p[3]);
            bf16* dst = Ps + (j & 1) * Z::P_ELEMS + head * LDP + 16 * ks + 4 * g;
            store_quad(dst, p);
            store_quad(dst + Z::H * LDP, lo);
        };
        meet<2 * LOADS>();                                    // the first half page, and the queries in the last place
        const uint32_t q_at = lds + 3 * Z::BYTES + head * ROW + 16 * (g ^ swap(head));
#pragma unroll
        for (int c = 0; c < W / 32; ++c) qf[c] = frag(q_at, c);
        scores(0);
        largest();
        meet<63>();
        m = fmaxf(red[head], red[Z::H + head]) + ROOM;        // (the first key is visible: finite)
        if (ks == 0 && g == 0) ref[head] = m;
        weights(0);
        meet<LOADS>();
        for (int j = 1; j <= nt; ++j) {
            const int grown = grow[(j - 1) & 1];
            if (j < nt) fetch(j + 2);
            if (__builtin_amdgcn_readfirstlane(grown)) {      // the half page before this one needs another reference
                largest();
                meet<63>();
                const float to = fmaxf(m, fmaxf(red[head], red[Z::H + head]) + ROOM);
                l *= __builtin_amdgcn_exp2f((m - to) * LOG2E);
                m = to;
                weights(j - 1);
                meet<63>();
                if (ks == 0 && g == 0) ref[head] = m;
            }
            l += sum;
            if (j < nt) {
                scores(j);
                const float top = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
                if (__builtin_amdgcn_ballot_w64(top > m)) {
                    if (lane == 0) grow[j & 1] = 1;
                }
                weights(j);
            }
            meet<LOADS>();
        }
        l = rows_sum(l);
        if (g == 0) red[Z::H * ks + head] = l;
        meet<0>();                                            // (no load is under way when the LDS is given back)
        if (writes) {
            ml[0] = m;
            ml[1] = red[head] + red[Z::H + head];
        }
        return;
    }

    // ---- values
    constexpr int HT = 2, NTW = 8;                            // head tiles, a wave's 16-wide tiles of the latent
    f32x4 o[HT][NTW];
#pragma unroll
    for (int h = 0; h < HT; ++h)
#pragma unroll
        for (int x = 0; x < NTW; ++x) o[h][x] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (nt > 0) {
        const int t4 = tid - 256;
        u32x4 z[LOADS];
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const int p = t4 + 256 * u, r = p / PIECES, c = p - PIECES * r;
            z[u] = *reinterpret_cast<const u32x4*>(q + ((int64_t)row * H + min(h0 + r, H - 1)) * W + 8 * c);
            if (h0 + r >= H) z[u] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < LOADS; ++u) {
            const int p = t4 + 256 * u, r = p / PIECES, c = p - PIECES * r;
            *reinterpret_cast<u32x4*>(smem + 3 * Z::BYTES + r * ROW + 16 * ((c & ~7) | ((c ^ swap(r)) & 7))) = z[u];
        }
        if (t4 < 2) grow[t4] = 0;
        const int vrow = 8 * g + (i >> 2);
        const uint32_t v_at = lds + vrow * ROW + 256 * part + 16 * (((i & 3) >> 1) ^ swap(vrow)) + 8 * (i & 1);
        meet<63>();
        meet<63>();
        meet<63>();
        for (int j = 1; j <= nt; ++j) {
            const int grown = grow[(j - 1) & 1];
            bf16x8 b[HT][2];
            auto read_p = [&] {
                const bf16* src = Ps + ((j - 1) & 1) * Z::P_ELEMS + i * LDP + 8 * g;
#pragma unroll
                for (int h = 0; h < HT; ++h)
#pragma unroll
                    for (int y = 0; y < 2; ++y) b[h][y] = load_frag(src + (Z::H * y + 16 * h) * LDP);
            };
            read_p();
            if (__builtin_amdgcn_readfirstlane(grown)) {
                meet<63>();
#pragma unroll
                for (int h = 0; h < HT; ++h) {
                    const float was = ref[16 * h + i], to = fmaxf(was, fmaxf(red[16 * h + i], red[Z::H + 16 * h + i]) + ROOM);
                    const float f = __builtin_amdgcn_exp2f((was - to) * LOG2E);
#pragma unroll
                    for (int x = 0; x < NTW; ++x)
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[h][x][r] *= f;
                }
                if (t4 == 0) grow[(j - 1) & 1] = 0;
                meet<63>();
                read_p();
            }
            const uint32_t base = v_at + ((j - 1) & 3) * Z::BYTES;
#pragma unroll
            for (int x = 0; x < NTW; ++x) {                   // keys 8 g .. + 3 and + 4 .. + 7 of 16 columns
                const uint32_t at = base ^ (32 * (x & 3));
                const bf16x4 u = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((Lds4)(uintptr_t)(at + 128 * (x >> 2)));
                const bf16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((Lds4)(uintptr_t)((at ^ 16) + 128 * (x >> 2) + 4 * ROW));
                const bf16x8 a = __builtin_shufflevector(u, v, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int y = 0; y < 2; ++y)
#pragma unroll
                    for (int h = 0; h < HT; ++h) o[h][x] = El<bf16>::mma(a, b[h][y], o[h][x]);
            }
            meet<63>();
        }
        meet<63>();
    }
#pragma unroll
    for (int h = 0; h < HT; ++h) {
        const int head = h0 + 16 * h + i;
        if (head >= H) continue;
        const float l = nt > 0 ? red[16 * h + i] + red[Z::H + 16 * h + i] : 0.f;
        if (nsplit == 1) {
            const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
            for (int x = 0; x < NTW; ++x) {
                f32x4 v = o[h][x];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= inv;
                store_quad(out + ((int64_t)row * H + head) * C + 128 * part + 16 * x + 4 * g, v);
            }
        } else if (l > 0.f) {                                 // (the partial row of an empty split is not read either)
            float* dst = ws + (((int64_t)row * H + head) * nsplit + split) * C + 128 * part + 4 * g;
#pragma unroll
            for (int x = 0; x < NTW; ++x) *reinterpret_cast<f32x4*>(dst + 16 * x) = o[h][x];
        }
    }
}

__global__ __launch_bounds__(512, 2) void attn_latent_sized_kernel(const bf16* __restrict__ q, const bf16* __restrict__ cache, int n_pages,
                                                                   const int32_t* __restrict__ table, int table_ld, const int32_t* __restrict__ len,
                                                                   bf16* __restrict__ out, float* __restrict__ ws, int H, float scale, int nsplit, int rows) {
    extern __shared__ __align__(16) char smem[];
    const int split = blockIdx.x, row = blockIdx.z, n = len[row];
    const int ntiles = n > 0 ? (n + 63) / 64 : 0;
    const int per = (ntiles + nsplit - 1) / nsplit;
    const int t_beg = min(split * per, ntiles), t_end = min(ntiles, t_beg + per);
    attn_latent_sized_body(q, cache, n_pages, table + (int64_t)row * table_ld, n, out, ws, H, scale, nsplit, rows, row, blockIdx.y * 32, split, t_beg,
                           t_end, smem);
}

// The same attention on the first `workers` workgroups, and a product that waits for nothing of it on the others: out_f += x . W^T, P panels of
// W each.  A workgroup of either kind has a CU to itself (two pages in LDS), so the two share the chip by CUs: attention draws up to 35 bytes a ns
// and CU behind 8 us of start, the product up to 50.
// Splits are dealt: as many pages each, 2 at least where a row has more than 16, as make the splits of all rows fit the workers; a row has
// nsplit at most, with as many pages each as that takes.  Statistics of splits that a row does not have are zero, which the merge skips.
// us, 32 heads, attention, merge, value and the output product (shorter by 11 008 of its 15 104), apart -> so: a row of 64 pages 38.5 -> 33.6, 32 rows
// with 1 167 pages 68.0 -> 60.1 (more beside beside_plan).
// SPLIT: the product's workgroups take P panels over one of `parts` ranges of k each and leave the range's sums in g.out_f [parts][rows][n], for the output
// product to add.  Above 16 rows a workgroup reads as much of x as of the weights where it has two panels of all of k (704 KB each of 32 rows and k
// 11 008), and is the longer side for it (figures at tfl_beside_parts).
template <int P, int MT, bool SPLIT>
__global__ __launch_bounds__(512, 2) void attn_latent_beside_kernel(const bf16* __restrict__ q, const bf16* __restrict__ cache, int n_pages,
                                                                    const int32_t* __restrict__ table, int table_ld, const int32_t* __restrict__ len,
                                                                    float* __restrict__ ws, int H, float scale, int nsplit, int rows, int workers,
                                                                    const TflGemm g, const int parts) {
    extern __shared__ __align__(16) char smem[];
    // which of the two start first: on 128 CUs the product is the longer side up to 1 200 pages (one row of 64 pages 33.4 -> 33.2 us with it first, 32
    // rows of 1 568 61.6 -> 61.2), on 86 and 64 it is slower for it (40.0 -> 41.5, 45.1 -> 45.7)
    constexpr bool FIRST = P == 2;
    const int me = (int)blockIdx.x - (FIRST ? (int)gridDim.x - workers : 0), group = (int)blockIdx.x - (FIRST ? 0 : workers);
    if constexpr (SPLIT) {
        if (group >= 0) {
            const int npan = g.n >> 4, groups = (npan + P - 1) / P, part = group / groups, chunks = g.k >> 5;
            const int c_beg = chunks * part / parts, c_end = chunks * (part + 1) / parts;
            TflGemm own = g;
            own.wp = (const bf16*)g.wp + (int64_t)c_beg * npan * 512;
            own.x = (const bf16*)g.x + 4 * g.x_oct * c_beg;
            own.k = 32 * (c_end - c_beg);
            own.out_f = g.out_f + (int64_t)part * g.rows * g.n;
            share_gemm_body<bf16, TFL_EPI_F32, P, false, MT, 1>(own, 0, 0, group - part * groups, 0, smem);
            return;
        }
    } else if (FIRST ? me < 0 : group >= 0) {
        share_gemm_body<bf16, TFL_EPI_RESIDUAL, P, false, MT, 2>(g, 0, 0, group, 0, smem);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int pages = lane < rows ? max(1, (len[min(lane, rows - 1)] + 63) >> 6) : 0;        // (a row without keys has one empty split)
    const int total = lanes_sum(pages), most = lanes_max(pages);
    int per = max((total + workers - 1) / workers, most > 16 ? 2 : 1), mine, end;
    for (;; ++per) {                                          // (with `most` pages a split there are as many splits as rows)
        mine = lane < rows ? min(nsplit, (pages + per - 1) / per) : 0;
        end = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
            if (o < rows) {                                   // (lanes from `rows` on are not looked at)
                const int v = __shfl_up(end, o, 64);
                if (lane >= o) end += v;
            }
        if (per >= most || __builtin_amdgcn_readlane(end, rows - 1) <= workers) break;
    }
    const uint64_t before = __builtin_amdgcn_ballot_w64(lane < rows && end <= me);
    const int row = __popcll(before);
    if (row >= rows) return;
    const int have = __builtin_amdgcn_readlane(mine, row), split = me - (__builtin_amdgcn_readlane(end, row) - have), n = len[row];
    const int ntiles = n > 0 ? (n + 63) >> 6 : 0, each = (ntiles + have - 1) / have;
    const int t_beg = min(split * each, ntiles), t_end = min(ntiles, t_beg + each);
    if (split == have - 1)
        for (int s = have + (int)threadIdx.x / 32; s < nsplit; s += 16) {
            const int head = threadIdx.x & 31;
            if (head < H) ws[(int64_t)rows * H * nsplit * 512 + (((int64_t)row * H + head) * nsplit + s) * 2 + 1] = 0.f;
        }
    attn_latent_sized_body(q, cache, n_pages, table + (int64_t)row * table_ld, n, nullptr, ws, H, scale, nsplit, rows, row, 0, split, t_beg,
                                      t_end, smem);
}

#define TFL_MAX_SPLIT 256

extern "C" int64_t tfl_attn_decode_ws_floats(int rows, int H, int C, int nsplit) {
    if (rows < 1 || H < 1 || C < 1 || nsplit < 1) return 0;
    return nsplit == 1 ? 0 : (int64_t)rows * H * nsplit * (C + 2);
}

// One workgroup per CU (256) as long as a split keeps at least two pages of keys, or one of up to 16.  us of the attention with its merge, latent to value
// and an output product of k 6 144, 32 heads, pairs -> single pages: one row of 8 pages 26.0 -> 24.1, of 16 26.2 -> 24.7; of 64 27.2 -> 26.3, of 128
// 28.1 -> 30.0; 4 rows of 64 30.6 -> 30.8, 8 of 48 31.9 -> 39.2 (more than the CUs).  So the line would lie at 17 to 64 pages for one or two rows
// (17 pages 26.3 -> 24.7; 16 heads, 32 pages 23.0 -> 21.1), which this rule leaves at pairs, as it does three to eight pages of 32 rows and more at
// one a split, where one split of all costs less (64 rows of three pages 51.4 -> 46.8, 64 heads 78.1 -> 67.1): over 568 points of 1 to 64 rows, 1 to 512
// pages and 16 to 64 heads it takes 1.011 of the best, in the worst 1.16.  Two pages are one split where the second one costs less than the merge: always in
// the form of known sizes (one row 24.0 us in two, 22.8 in one, 64 rows 50.7 and 44.9).  The other forms, attention and merge alone: bfloat16 from 65
// workgroups of 16 heads on (256 | 32, 16 heads, 96 rows 11.5 against 12.4; 32 rows 11.5 against 10.6), never in float32 (55 against 35).  Float32
// takes 16 heads per workgroup, one to a CU: single pages only where they are no more rounds of 256 than pairs would be (32 heads, 12 rows of 12 pages
// 86.5 us against 92.8).
extern "C" int tfl_attn_decode_splits(int rows, int H, int C, int R, int max_len, int dtype) {
    if (rows < 1 || H < 1 || max_len < 1) return 1;
    const int groups = H <= 16 ? 1 : (H + 31) / 32, pages = (max_len + TFL_PAGE - 1) / TFL_PAGE, pairs = (pages + 1) / 2;
    const int64_t tiles = (int64_t)rows * ((H + 15) / 16);
    const int room = (int)(256 / ((int64_t)rows * groups));
    int n = pages < room ? pages : room;
    const bool twice = dtype == 1 && tiles * n > 256 && tiles * pairs <= 256;
    const bool merge = pages == 2 && dtype == 0 && ((C == 512 && R == 64) || tiles > 64);
    if ((pages > 16 || twice || merge) && n > pairs) n = pairs;
    if (n > TFL_MAX_SPLIT) n = TFL_MAX_SPLIT;
    return n < 1 ? 1 : n;
}

// The same for the form of known sizes.
extern "C" int tfl_attn_decode_pick_nsplit(int rows, int H, int max_len) { return tfl_attn_decode_splits(rows, H, 512, 64, max_len, 0); }

template <typename T, int NW, int HT, int NTW>
static int launch_latent(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len,
                         void* out, float* ws, int rows, int H, int C, int R, float scale, int nsplit, hipStream_t st) {
    const int W = C + R, pad = 16 / (int)sizeof(T), KT = 16 * NW;
    const size_t lds = sizeof(T) * ((size_t)(KT + 16 * HT) * (W + pad) + (size_t)DecodeCfg<T>::PARTS * 16 * HT * (KT + pad))
                     + sizeof(float) * NW * 16 * HT;
    if (lds > 160 * 1024) return TF_ERANGE;
    auto k = attn_latent_kernel<T, NW, HT, NTW>;
    static bool attr = false;
    if (!attr) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        attr = true;
    }
    hipLaunchKernelGGL(k, dim3(nsplit, (H + 16 * HT - 1) / (16 * HT), rows), dim3(NW * 64), lds, st, (const T*)q, (const T*)cache,
                       n_pages, table, table_ld, len, (T*)out, ws, H, C, R, scale, nsplit, rows);
    TFL_LAUNCH_CHECK();
    return nsplit > 1 ? launch_merge<T>(ws, out, rows, H, C, nsplit, st) : TF_OK;
}

static int launch_latent_sized(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len, void* out, float* ws,
                               int rows, int H, float scale, int nsplit, hipStream_t st) {
    const hipError_t e = hipFuncSetAttribute((const void*)attn_latent_sized_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LatentTile::LDS);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(attn_latent_sized_kernel, dim3(nsplit, (H + 31) / 32, rows), dim3(512), LatentTile::LDS, st, (const bf16*)q, (const bf16*)cache,
                       n_pages, table, table_ld, len, (bf16*)out, ws, H, scale, nsplit, rows);
    TFL_LAUNCH_CHECK();
    return nsplit > 1 ? launch_merge<bf16>(ws, out, rows, H, LatentTile::C, nsplit, st) : TF_OK;
}

extern "C" int tfl_attn_decode(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len,
                               void* out, float* ws, int64_t ws_floats, int rows, int H, int C, int R, float scale, int nsplit,
                               int dtype, void* stream) {
    if (!q || !cache || !table || !len || !out || rows < 1 || rows > 65535 || H < 1 || n_pages < 1 || table_ld < 1) return TF_EINVAL;
    if (C < 32 || (C & 31) || R < 0 || (R & 31) || nsplit < 1 || nsplit > TFL_MAX_SPLIT) return TF_EINVAL;
    if (nsplit > 1 && (!ws || ws_floats < tfl_attn_decode_ws_floats(rows, H, C, nsplit))) return TF_ENOSPC;
    hipStream_t st = (hipStream_t)stream;
#define GO(T, NW, HT, NTW) \
    return launch_latent<T, NW, HT, NTW>(q, cache, n_pages, table, table_ld, len, out, ws, rows, H, C, R, scale, nsplit, st)
    if (dtype == 0) {
        if (C == 512 && R == 64) return launch_latent_sized(q, cache, n_pages, table, table_ld, len, out, ws, rows, H, scale, nsplit, st);
        if (C <= 128) { if (H <= 16) GO(bf16, 4, 1, 2); GO(bf16, 4, 2, 2); }
        if (C <= 512) { if (H <= 16) GO(bf16, 4, 1, 8); GO(bf16, 4, 2, 8); }
        if (C <= 1024) GO(bf16, 2, 1, 32);
        return TF_ERANGE;
    }
    if (dtype == 1) {
        if (C <= 128) { if (H <= 16) GO(float, 4, 1, 2); GO(float, 4, 2, 2); }
        if (C <= 512) GO(float, 2, 1, 16);
        return TF_ERANGE;
    }
#undef GO
    return TF_EINVAL;
}

// How the CUs are shared between the attention of `pages` pages in all, `longest` of them in one row, and a product of n outputs of k, or 0 workers
// where the two are better one after the other.  The product takes up to half of the CUs, which draw all that memory gives (38 bytes a ns each).
// us of a graph of the attention, its merge, latent to value and the whole output product (32 heads, n 4096, k 11 008 of 15 104, rows half to all as long
// as the longest, weights and keys from memory), apart -> beside with the product on 128 CUs | 86 | 64:
//   pages in all   one each                 ~60                  ~200                  ~590                 ~1 160                 ~1 550                 ~2 320
//    1 row    32.0->32.3|41.0|45.0   38.5->33.6|42.2|46.0   41.7->37.7|45.4|49.4   47.3->41.1|47.3|51.0 (512)
//    4 rows   35.6->36.6|44.3|49.0   39.8->38.3|45.1|49.5   41.9->40.5|48.0|51.9   46.8->44.0|49.8|54.3                          62.2->63.0|56.8|61.6
//    8 rows   36.7->38.7|46.1|51.3   39.2->40.2|47.1|52.7   41.5->42.6|49.6|54.5   46.2->44.4|51.7|56.9   56.4->54.9|56.7|61.6   61.8->61.9|57.6|64.4
//   16 rows   41.0->41.3|49.9|55.6   41.6->42.9|50.5|56.6   44.3->45.9|52.4|58.4   49.6->48.0|54.7|60.3   59.3->55.1|59.2|66.0   64.8->61.9|61.9|68.2   75.9->78.4|70.5|72.4
//   32 rows   52.2->52.3|59.5|66.0   52.5->52.9|59.9|66.4   53.8->54.5|61.3|67.7   58.6->55.3|63.4|69.8   68.0->60.1|68.0|75.5   74.4->67.1|70.4|77.4   84.6->83.0|74.5|81.2
// The constants are fitted to 1 862 such points: 20 to 32 heads, 1 to 32 rows, 1 to 4 096 pages, n 4 096 to 8 192, k 2 048 to 16 384; rows half to all as
// long as the longest, all alike, and one eight times as long as the others, whose pages too few splits then share (32 rows with 503 pages, 100 of
// them in one row: 76.3 apart, 57.3 beside).  What they pick takes 1.008 of the best on average and at most 1.10.  Half of that is short contexts,
// which stay beside where that costs a tenth at most: apart, the splits follow the cache's room, beside, what is in it.  (Not at k above 12 288, where the
// product's half of the CUs is by far the longer side.)
struct BesideTime { int workers; double product, attention, all; };
static BesideTime beside_time(int rows, int H, int64_t pages, int64_t longest, int n, int k, int p) {
    const int g = ((n >> 4) + p - 1) / p, a = 256 - g, most = 2 * a / rows < 128 ? 2 * a / rows : 128;
    if (g > 128) return {0, 0., 0., 0.};
    const double heads = H / 32.0, each = fmax((double)pages / a, (double)((longest + most - 1) / most));
    const double product = 26.33 * 2e-6 * n * k / g + 0.527 * rows * k / 11008.0, attention = 3.22 + 2.7475 * each + 0.945 * p;
    return {a, product, attention, fmax(product, attention) + 0.25 * heads * rows + 0.0068 * heads * (double)(pages < a ? pages : a) - 1.892 * (rows < 5 ? 5 - rows : 0)};
}

// The two one after the other.
static double apart_time(int rows, int H, int64_t pages, int64_t longest, int n, int k) {
    const int ns = tfl_attn_decode_splits(rows, H, 512, 64, (int)(pages < 16 ? 16 : pages) * TFL_PAGE, 0);        // (a cache of what is there, or more)
    const double mb = 2e-6 * n * k, heads = H / 32.0, x = rows * k / 11008.0;
    return 3.345 + 0.1237 * mb + 0.1656 * rows + 0.4873 * x + 0.0083 * heads * rows * ns + 0.0026 * pages + 2.245 * (double)((longest + ns - 1) / ns);
}

static int beside_plan(int rows, int H, int64_t pages, int64_t longest, int n, int k, int* panels_each) {
    const int panels = n >> 4;
    if (rows < 1 || rows > 32 || H <= 16 || H > 32 || pages < 1 || pages > (1 << 20) || longest < 1 || panels < 256 || panels > 512 || k < 2048) return 0;
    double least = apart_time(rows, H, pages, longest, n, k);
    if (pages < 32 * rows && k <= 12288) least *= 1.0 / 0.9;
    int workers = 0;
    for (int p = 2; p <= 4; ++p) {
        const BesideTime b = beside_time(rows, H, pages, longest, n, k, p);
        if (b.workers > 0 && b.all < least) { least = b.all; workers = b.workers; *panels_each = p; }
    }
    return workers;
}

extern "C" int tfl_attn_beside_plan_of(int rows, int H, int C, int R, int64_t pages, int64_t longest, int n, int k, int32_t* panels_each, int32_t* nsplit,
                                       int32_t* parts) {
    if (!panels_each || !nsplit || !parts || C != 512 || R != 64) return 0;
    int p = 0;
    const int a = beside_plan(rows, H, pages, longest, n, k, &p);
    *panels_each = p;
    *nsplit = rows < 1 ? 0 : 2 * a / rows < 128 ? 2 * a / rows : 128;
    *parts = 0;
    if (a > 0) {                                              // (as the kernel deals them when all rows have as many pages)
        const int64_t per = (pages + a - 1) / a, least = pages > 16 * rows ? 2 : 1, all = (pages + rows) / (per > least ? per : least) + rows;
        *parts = (int32_t)(all < a ? all : a);
    }
    return a;
}

// Columns of that product's k, from the last on, that the query to latent product in front of the attention carries (latent_carry_kernel in tile_gemm.hip): one
// amount for a product's k, or none.  An amount that followed the context would be a captured step of its own in each of its ranges, 65 to 110 ms of
// capture while an answer grows (8 rows changed it at 2 048, 3 072 and 4 032 tokens), for up to 1 us a layer run: us of query to latent, attention, value and
// output product (32 heads, n 4 096, k 11 008), none | 4 096 | 5 120 | 6 144 columns, the longest row of 300, 2 000, 4 000, 9 000, 16 000 keys:
//    1 row   34.7|33.7|33.4|33.0  35.2|34.4|34.2|34.5  36.1|35.3|35.0|35.4  39.0|38.0|37.8|38.2  41.7|40.3|40.5|40.9, of 20 000 41.7|40.9|41.7|42.6
//    4 rows  39.5|38.5|38.1|37.6  41.0|39.7|39.2|39.5  43.0|41.3|41.0|41.1  45.4|44.8|45.6|45.0
//    8 rows  42.1|40.6|39.8|39.2  45.3|42.7|42.0|41.9  45.9|44.1|44.9|45.8
//   16 rows  46.5|44.0|43.4|42.8  49.0|46.3|45.9|47.1  51.9|55.1|54.6|55.4
// Carried as long as the fitted times save 0.8 us by it, also where the two without it would go one after the other: 131 of 218 points (1 to 16 rows, 300 to
// 28 000 keys, 20 to 32 heads, n 4 096 and 6 144), 1.6 us or 3.8 % faster on average, one of them slower (0.12 us).
// Up to 16 rows: of 32 rows a carried panel reads twice its weights' bytes of x (6 664 us of eight steps -> 6 924).
extern "C" int tfl_latent_carry(int rows, int H, int C, int R, int64_t pages, int64_t longest, int n, int k) {
    const int columns = k >= 5120 + 2048 ? 5120 : 4096;       // (4 096: a carried panel of less costs its start more than the other one saves)
    if (C != 512 || R != 64 || rows < 1 || rows > 16 || longest < 1 || k > (1 << 20) || k - columns < 2048) return 0;
    int p = 0, q = 0;
    if (beside_plan(rows, H, pages, longest, n, k - columns, &q) == 0) return 0;
    const double without = beside_plan(rows, H, pages, longest, n, k, &p) ? beside_time(rows, H, pages, longest, n, k, p).all : apart_time(rows, H, pages, longest, n, k);
    const double with = beside_time(rows, H, pages, longest, n, k - columns, q).all + 0.55 + 3.2e-7 * columns * n + 0.11 * rows;
    return without - with > 0.8 && (p == 0 || p == q) ? columns : 0;
}

// Ranges of k (4, or 3 where the attention would be left with too few CUs; 0: none) into which 17 to 32 rows' product is cut where that is faster than
// beside_plan's division or the two apart.  The times of query to latent, attention, value and output product as fitted to 720 measured ones (17, 20, 24, 28, 32 rows
// of 300 to 6 000 keys; 17, 20, 24, 32 heads; n 4 096 to 8 192, k 4 096 to 14 336): 2.5 % off on average, so 2 % have to be in it.  Every division is a captured step of
// its own, 65 to 110 ms of capture while an answer grows, so there is the one cut of short contexts and no other between it and whole panels (three
// ranges besides: 0.3 % on average).  Of 226 other points (17 to 32 rows, 20 to 32 heads, k 8 192 to 14 336) it is 1.85 % faster on average than without, 2 are more than 1 %
// slower (1.5 %).  us, 32 heads, n 4 096, k 11 008, rows half to all as long as the longest, 2 | 3 whole panels, 3 | 4 ranges, * the pick:
//   17 rows of   300 49.6|56.6|52.2|46.8*  2 000 51.5|59.6|54.7|49.3*  3 500 53.9|62.7|58.5|53.6*  5 000 56.6*|65.3|60.5|58.4   6 000 61.4*|65.9|61.8|62.9
//   24 rows of   300 53.3|59.1|53.8|49.7*  2 000 55.1|63.3|56.7|52.5*  3 500 57.5*|67.3|61.7|59.0  5 000 66.1*|67.8|64.3|68.1   6 000 73.0|70.2*|69.0|74.9
//   32 rows of   300 56.5|64.5|57.2|51.7*  2 000 60.9|69.7|61.7|57.2*  3 000 63.0*|70.7|64.5|64.8  4 000 69.6*|72.6|67.9|71.8   5 000 79.1|74.3*|74.5|81.0
// Up to 16 rows it is never faster (16 rows of 300 43.2 -> 48.6 in three ranges, 46.3 in four), nor in one or two ranges, which leave the product too few CUs.
extern "C" int tfl_beside_parts(int rows, int H, int C, int R, int64_t pages, int64_t longest, int n, int k, int32_t* workers, int32_t* nsplit) {
    if (!workers || !nsplit || C != 512 || R != 64 || rows < 17 || rows > 32 || H <= 16 || H > 32 || pages < 1 || pages > (1 << 20) || longest < 1 || n < 4096 || n > 8192 || (n & 15)
        || k < 4096 || k > 14336) return 0;
    const double mb = 2e-6 * n * k, x = rows * k / 11008.0, heads = rows * H / 32.0, out = 2.56e-4 * n * H;
    auto load = [&](int a) {                                  // pages of the busiest worker
        const int most = 2 * a / rows < 128 ? 2 * a / rows : 128;
        return fmax((double)pages / a, (double)((longest + most - 1) / most));
    };
    const int eights = (n + 127) / 128;
    const bool four = 256 - 4 * eights >= 64 && 256 - 4 * eights >= 2 * rows;
    int p = 0;
    double least;
    if (beside_plan(rows, H, pages, longest, n, k, &p)) {
        const int g = ((n >> 4) + p - 1) / p;
        const double product = 24.79 * mb / g + 0.190 * x, attention = 2.44 + 2.477 * load(256 - g);
        least = fmax(product, attention) + 0.295 * fmin(product, attention) + 0.320 * heads + 0.163 * out + 17.15;
    } else {
        least = 0.4464 * mb - 1.623 * rows + 0.6034 * x * n / 4096.0 + 0.017 * pages + 1.276 * heads - 0.279 * out;
    }
    const int c = four ? 4 : 3, g = c * eights, a = 256 - g;
    if (a < 64 || a < 2 * rows) return 0;
    const double product = 22.23 * mb / g + (0.0332 * c - 0.0462) * x, attention = 2.31 + 2.568 * load(a);
    if (fmax(product, attention) + 0.417 * fmin(product, attention) + 0.320 * heads + 0.163 * out + 17.15 >= 0.98 * least) return 0;
    *workers = a;
    *nsplit = 2 * a / rows < 128 ? 2 * a / rows : 128;
    return c;
}

// The same where nobody knows the longest row: rows half to all as long as it.
extern "C" int tfl_attn_beside_plan(int rows, int H, int C, int R, int64_t pages, int n, int k, int32_t* panels_each, int32_t* nsplit, int32_t* parts) {
    const int64_t longest = rows < 1 || pages < rows ? 1 : (4 * pages - 1) / (3 * (int64_t)rows) + 1;
    return tfl_attn_beside_plan_of(rows, H, C, R, pages, rows == 1 ? pages : longest, n, k, panels_each, nsplit, parts);
}

template <int P, int MT, bool SPLIT = false>
static int launch_beside(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len, float* ws, int rows, int H,
                         float scale, int nsplit, int workers, const TflGemm& g, hipStream_t st, int parts = 1) {
    constexpr int LDS = LatentTile::LDS;
    static_assert(8 * P * MT * 64 * (int)sizeof(f32x4) <= LDS, "LDS");
    const hipError_t e = hipFuncSetAttribute((const void*)attn_latent_beside_kernel<P, MT, SPLIT>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((attn_latent_beside_kernel<P, MT, SPLIT>), dim3(workers + ((g.n >> 4) + P - 1) / P * parts), dim3(512), LDS, st, (const bf16*)q, (const bf16*)cache,
                       n_pages, table, table_ld, len, ws, H, scale, nsplit, rows, workers, g, parts);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

static int attn_decode_beside(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len, void* out,
                              float* ws, int64_t ws_floats, int rows, int H, float scale, int nsplit, int workers, int panels_each,
                                      int parts, const TflGemm* product, void* stream) {
    if (!q || !cache || !table || !len || !ws || !product || rows < 1 || rows > 32 || H <= 16 || H > 32 || n_pages < 1 || table_ld < 1) return TF_EINVAL;
    if (nsplit < 2 || nsplit > 128 || workers < 2 * rows || workers > 255) return TF_EINVAL;
    if (ws_floats < tfl_attn_decode_ws_floats(rows, H, 512, nsplit)) return TF_ENOSPC;
    const TflGemm g = *product;
    if (!g.wp || !g.x || !g.out_f || g.out_t || g.rows != rows || g.n < 16 || (g.n & 15) || g.k < 32 || (g.k & 31) || g.groups != 1 || g.chunk_major != 1
        || (g.ld_x & 7) || g.ld_x < 8 || g.x_oct < 8 || (g.x_oct & 7) || g.ld_f < g.n || (g.ld_f & 3)) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    int rc = TF_EINVAL;
#define GO(P) rc = rows <= 16 ? launch_beside<P, 1>(q, cache, n_pages, table, table_ld, len, ws, rows, H, scale, nsplit, workers, g, st) \
                              : launch_beside<P, 2>(q, cache, n_pages, table, table_ld, len, ws, rows, H, scale, nsplit, workers, g, st)
    if (parts > 0) {
        if (panels_each == 8 && parts <= 4 && rows > 16 && g.k >= 32 * parts && g.ld_f == g.n)
            rc = launch_beside<8, 2, true>(q, cache, n_pages, table, table_ld, len, ws, rows, H, scale, nsplit, workers, g, st, parts);
    } else switch (panels_each) {
        case 2: GO(2); break;
        case 3: GO(3); break;
        case 4: GO(4); break;
    }
#undef GO
    return rc == TF_OK && out ? launch_merge<bf16>(ws, out, rows, H, 512, nsplit, st) : rc;
}

extern "C" int tfl_attn_decode_beside(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len, void* out,
                                      float* ws, int64_t ws_floats, int rows, int H, float scale, int nsplit, int workers, int panels_each,
                                      const TflGemm* product, void* stream) {
    return attn_decode_beside(q, cache, n_pages, table, table_ld, len, out, ws, ws_floats, rows, H, scale, nsplit, workers, panels_each, 0, product, stream);
}

extern "C" int tfl_attn_decode_beside_parts(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len, void* out,
                                            float* ws, int64_t ws_floats, int rows, int H, float scale, int nsplit, int workers, int parts,
                                            const TflGemm* product, void* stream) {
    if (parts < 1 || !product || product->n_real != product->n) return TF_EINVAL;
    return attn_decode_beside(q, cache, n_pages, table, table_ld, len, out, ws, ws_floats, rows, H, scale, nsplit, workers, 8, parts, product, stream);
}

// The merge of the splits in front of latent to value: out = (merged . W_head^T) * sigmoid(gate) for up to 4 rows of 512 latents, one panel of
// values to a workgroup.  Each of a head's workgroups merges for itself, from L2: that costs less than a launch between the two as long as the
// splits are few.  The panel's weights and gates come in under it.  One row of 4 000 keys (32 splits): merge 4.7 and product 4.5 -> 5.8 us, eight
// steps of six layer runs 4 666 -> 4 568.  us of a graph of the attention beside its product and this, merge launched -> here (splits of all rows): 1 row
// 26.5 -> 24.9 (16), 27.2 -> 25.2 (32), 29.7 -> 28.9 (80); 2 rows 27.4 -> 26.9 (32), 28.7 -> 28.0 (64), 30.8 -> 31.2 (100); 4 rows 31.9 -> 30.6 (64);
// 8 rows 32.0 -> 35.5 (64).
constexpr int VALUE_ROWS = 4;
__global__ __launch_bounds__(512) void latent_value_kernel(const float* __restrict__ ws, int nsplit, const TflGemm a) {
    __shared__ float weight[VALUE_ROWS][128];
    __shared__ int count[VALUE_ROWS];
    __shared__ __align__(16) float sums[4][VALUE_ROWS][512];
    __shared__ __align__(16) bf16 merged[VALUE_ROWS][512 + 8];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int ppg = a.n >> 4, head = (blockIdx.x & 7) + 8 * ((blockIdx.x >> 3) / ppg), panel = (blockIdx.x >> 3) % ppg;        // (a head on one XCD)
    if (head >= a.groups) return;
    const int col = head * a.n + 16 * panel + 4 * g, quad = tid & 127, grp = tid >> 7;
    const float* src = ws + (int64_t)head * nsplit * 512 + 4 * quad;
    const int64_t row_step = (int64_t)a.groups * nsplit * 512;
    bf16x8 w[2];
    f32x4 z[8];                                               // splits grp, grp + 4, .. of the first row: asked for before it is known which there are
#pragma unroll
    for (int u = 0; u < 8; ++u) z[u] = *reinterpret_cast<const f32x4*>(src + (int64_t)min(grp + 4 * u, nsplit - 1) * 512);
#pragma unroll
    for (int u = 0; u < 2; ++u) w[u] = load_frag_stream((const bf16*)a.wp + ((int64_t)(head * ppg + panel) * 16 + 2 * wave + u) * 512 + lane * 8);
    f32x4 gate = {0.f, 0.f, 0.f, 0.f};
    if (wave == 0 && i < a.rows) gate = *reinterpret_cast<const f32x4*>(a.gate + (int64_t)i * a.ld_gate + col);
    if (wave < a.rows) {
        const float* ml = ws + (int64_t)a.rows * a.groups * nsplit * 512 + ((int64_t)wave * a.groups + head) * nsplit * 2;
        float l[2], m[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int s = lane + 64 * h;
            const float m_have = ml[2 * min(s, nsplit - 1)], l_have = ml[2 * min(s, nsplit - 1) + 1];         // (both at once)
            l[h] = s < nsplit ? l_have : 0.f;
            m[h] = l[h] > 0.f ? m_have : NEG_INF;             // (an empty split: its partial row is not read either)
        }
        float most = fmaxf(m[0], m[1]), all = 0.f;
        most = lanes_max(most);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            m[h] = l[h] > 0.f ? exp2f((m[h] - most) * LOG2E) : 0.f;
            all += m[h] * l[h];
        }
        all = lanes_sum(all);
#pragma unroll
        for (int h = 0; h < 2; ++h) weight[wave][lane + 64 * h] = all > 0.f ? m[h] / all : 0.f;
        const uint64_t low = __builtin_amdgcn_ballot_w64(l[0] > 0.f), high = __builtin_amdgcn_ballot_w64(l[1] > 0.f);
        if (lane == 0) count[wave] = high ? 128 - __builtin_clzll(high) : low ? 64 - __builtin_clzll(low) : 0;
    }
    __syncthreads();
    for (int r = 0; r < a.rows; ++r) {
        const int n = count[r], next = r + 1 < a.rows ? count[r + 1] : 0;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = grp;; s0 += 32) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float x = s0 + 4 * u < n ? weight[r][s0 + 4 * u] : 0.f;
                if (x > 0.f)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = fmaf(z[u][e], x, v[e]);
            }
            if (s0 + 32 >= n) break;
#pragma unroll
            for (int u = 0; u < 8; ++u) z[u] = *reinterpret_cast<const f32x4*>(src + r * row_step + (int64_t)min(s0 + 32 + 4 * u, n - 1) * 512);
        }
        if (next > 0)
#pragma unroll
            for (int u = 0; u < 8; ++u) z[u] = *reinterpret_cast<const f32x4*>(src + (r + 1) * row_step + (int64_t)min(grp + 4 * u, next - 1) * 512);
        *reinterpret_cast<f32x4*>(&sums[grp][r][4 * quad]) = v;
    }
    __syncthreads();
    for (int r = 0; r < a.rows; ++r) merged[r][tid] = (bf16)(sums[0][r][tid] + sums[1][r][tid] + sums[2][r][tid] + sums[3][r][tid]);
    __syncthreads();
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        bf16x8 x = {};
        if (i < a.rows) x = load_frag(&merged[i][32 * (2 * wave + u) + 8 * g]);
        acc = El<bf16>::mma(w[u], x, acc);
    }
    f32x4 (*part)[64] = reinterpret_cast<f32x4 (*)[64]>(sums);
    part[wave][lane] = acc;
    __syncthreads();
    if (wave || i >= a.rows) return;
#pragma unroll
    for (int v = 1; v < 8; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += part[v][lane][e];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] *= sigmoid(gate[e]);
    store_quad((bf16*)a.out_t + (int64_t)i * a.ld_t + (col >> 3) * a.t_oct + (col & 7), acc);
}

extern "C" int tfl_latent_value(const float* ws, int64_t ws_floats, int nsplit, const TflGemm* p, void* stream) {
    if (!ws || !p || !p->wp || !p->gate || !p->out_t || nsplit < 2 || nsplit > 128) return TF_EINVAL;
    const TflGemm a = *p;
    if (a.rows < 1 || a.rows > VALUE_ROWS || a.n < 16 || (a.n & 15) || a.k != 512 || a.groups < 1 || a.chunk_major || a.t_oct < 8 || (a.t_oct & 7) || a.ld_t < 8
        || (a.ld_t & 7) || a.ld_gate < (int64_t)a.groups * a.n || (a.ld_gate & 3)) return TF_EINVAL;
    if (ws_floats < tfl_attn_decode_ws_floats(a.rows, a.groups, 512, nsplit)) return TF_ENOSPC;
    hipLaunchKernelGGL(latent_value_kernel, dim3((a.n >> 4) * ((a.groups + 7) / 8 * 8)), dim3(512), 0, (hipStream_t)stream, ws, nsplit, a);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// --------------------------------------------------------------------------------------------------------------- prefill
// Four waves of 16 query rows, KT keys per tile, up to DK 32-wide chunks of query-key size and DV 16-wide tiles of value size.
template <typename T, int KT, int DK, int DV>
__global__ __launch_bounds__(256, 1) void attn_prefill_kernel(const T* __restrict__ q, const T* __restrict__ kv, const T* __restrict__ ck,
                                                           const int32_t* __restrict__ seq, const int32_t* __restrict__ pos,
                                                           const float* __restrict__ cosb, const float* __restrict__ sinb,
                                                           int half, int max_pos, const T* __restrict__ gate, int64_t ld_gate,
                                                           T* __restrict__ out, int64_t ld_out, int tq, int tk, int H, int N, int R,
                                                           int V, int C, float scale) {
    typedef typename El<T>::Frag Frag;
    constexpr int EPV = 16 / sizeof(T), PADE = EPV, PADV = 2 * EPV, QB = 64, NT = 256;
    extern __shared__ __align__(16) char smem[];
    const int nc = N >> 5, dk = (N + R) >> 5, dv = V >> 4;
    const int D = 32 * dk, ldk = D + PADE, ldv = 16 * dv + PADV;
    T* Ks = (T*)smem;                                         // [KT][ldk], then the values [KT][ldv]
    T* Vs = Ks + KT * ldk;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, i = lane & 15;
    // workgroups go round-robin over the 8 XCDs: all query blocks of a head sit on one of them and share its L2, longest first
    const int nqb = gridDim.x / H, id = blockIdx.x;
    const bool by_xcd = (H & 7) == 0;
    const int j_ = by_xcd ? id >> 3 : id, h = by_xcd ? (j_ / nqb) * 8 + (id & 7) : j_ / nqb;
    const int32_t* sq = seq + 4 * blockIdx.y;
    const int q_at = sq[0], nq = sq[1], k_at = sq[2], nk = sq[3];
    const int qb = (nqb - 1 - j_ % nqb) * QB;
    if (qb >= nq || nq < 1 || nk < nq || q_at < 0 || k_at < 0 || q_at + nq > tq || k_at + nk > tk) return;
    const int past = nk - nq;
    const int64_t ld_kv = (int64_t)H * (N + V), ld_ck = C + R;

    Frag qf[DK];
    const int j = qb + 16 * wave + i, qpos = past + j;        // the lane's own query token: its row, its key index
    const int64_t tok = q_at + min(j, nq - 1);
    const T* src = q + (tok * H + h) * (int64_t)(N + R) + 8 * g;
    int p = pos[tok];
    p = p < 0 ? 0 : (p >= max_pos ? max_pos - 1 : p);
#pragma unroll
    for (int c = 0; c < DK; ++c) {
        if (c >= dk) { qf[c] = Frag{}; continue; }
        Frag f = load_frag(src + 32 * c);
        if (c >= nc) {
            const int pr = (c - nc) * 16 + 4 * g;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (pr + e < half) {
                    const float cs = cosb[(int64_t)p * half + pr + e], sn = sinb[(int64_t)p * half + pr + e];
                    const float u = (float)f[2 * e], v = (float)f[2 * e + 1];
                    f[2 * e] = (T)(u * cs - v * sn);
                    f[2 * e + 1] = (T)(v * cs + u * sn);
                }
        }
        qf[c] = f;
    }
    f32x4 o[DV];
    float m_run = NEG_INF, l_run = 0.f;
#pragma unroll
    for (int d = 0; d < DV; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int last_q = min(qb + QB, nq) - 1;                  // last query row of the workgroup
    const int ntiles = (past + last_q) / KT + 1;
    const int first_qpos = past + qb + 16 * wave;             // the wave's first row: tiles that end before it need no mask
    const int kn = N / EPV, kr = R / EPV, vn = V / EPV, ppr = kn + kr + vn;   // 16-byte pieces per key
    for (int t = 0; t < ntiles; ++t) {
        const int k0 = t * KT;
        for (int p = tid; p < KT * ppr; p += NT) {
            const int key = p / ppr;
            int c = p - key * ppr;
            const int64_t kk = k_at + min(k0 + key, nk - 1);
            const T* src;
            T* dst;
            if (c < kn) {
                src = kv + kk * ld_kv + (int64_t)h * N + EPV * c;
                dst = Ks + key * ldk + EPV * c;
            } else if (c < kn + kr) {
                c -= kn;
                src = ck + kk * ld_ck + C + EPV * c;
                dst = Ks + key * ldk + N + EPV * c;
            } else {
                c -= kn + kr;
                src = kv + kk * ld_kv + (int64_t)H * N + (int64_t)h * V + EPV * c;
                dst = Vs + key * ldv + EPV * c;
            }
            *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(src);
        }
        __syncthreads();
        f32x4 s[KT / 16];
#pragma unroll
        for (int kt = 0; kt < KT / 16; ++kt) {
            s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
            const T* kp = Ks + (16 * kt + i) * ldk + 8 * g;
#pragma unroll
            for (int c = 0; c < DK; ++c) {
                if (c < dk) {
                    const Frag a = load_frag(kp + 32 * c);
                    s[kt] = El<T>::mma(a, qf[c], s[kt]);
                }
            }
        }
        if (k0 + KT - 1 > first_qpos) {
#pragma unroll
            for (int kt = 0; kt < KT / 16; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (k0 + 16 * kt + 4 * g + r > qpos) s[kt][r] = NEG_INF;
        }
        Frag pf[KT / 32];
        float mx = NEG_INF;
#pragma unroll
        for (int kt = 0; kt < KT / 16; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[kt][r]);
        mx = rows_max(mx);
        mx = fmaxf(m_run, mx * scale);                        // (scale > 0; key 0 is visible to every row: finite from tile 0 on)
        const float alpha = __builtin_amdgcn_exp2f((m_run - mx) * LOG2E), sc = scale * LOG2E, mb = mx * LOG2E;
        m_run = mx;
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < KT / 16; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f(fmaf(s[kt][r], sc, -mb));
                sum += p;
                pf[kt >> 1][(kt & 1) * 4 + r] = (T)p;
            }
        l_run = l_run * alpha + sum;
        if (!__all(alpha == 1.0f)) {                          // (most tiles leave every maximum where it was)
#pragma unroll
            for (int d = 0; d < DV; ++d)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[d][r] *= alpha;
        }
#pragma unroll
        for (int d = 0; d < DV; ++d) {
            if (d < dv) {
#pragma unroll
                for (int c = 0; c < KT / 32; ++c) {
                    const Frag a = load_frag_t(Vs, ldv, 32 * c + 4 * g, 32 * c + 16 + 4 * g, 16 * d, i);
                    o[d] = El<T>::mma(a, pf[c], o[d]);
                }
            }
        }
        __syncthreads();
    }
    float l = l_run;
    l = rows_sum(l);
    if (j >= nq) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int d = 0; d < DV; ++d) {
        if (d >= dv) continue;
        const int col = h * V + 16 * d + 4 * g;
        const f32x4 z = load_quad(gate + tok * ld_gate + col);
        f32x4 v = o[d];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= inv * sigmoid(z[r]);
        store_quad(out + tok * ld_out + col, v);
    }
}

// Keys of 128 + 64 and values of 128 in bfloat16, on the loop of flash_tile.h: 80 KB of LDS, two workgroups of 128 query rows per CU (or one of 256).
// Workgroups go round-robin over the 8 XCDs: a head's query blocks sit on one of them and share its L2, the last blocks of all sequences and
// heads first (sequence by sequence six of 222 to 1 333 rows take 106 us, not 98).  That reads every key once per query block from wherever it
// lies, so with more keys than the chip's caches hold (256 MB; from 5 * 2^17 keys times heads, 320 MB, on) and more than one round of workgroups the order is sequence
// by sequence, a block's heads side by side: 32 heads, 16 x 500 rows behind 4 096 keys 1 028 -> 875 us, 16 x 1 333 behind 2 000 1 900 -> 1 557.
// 32 heads, against one workgroup of 256 rows per CU with tiles staged in registers and one product at a time: 4 096 rows 302 -> 243 us, behind
// 4 096 keys 597 -> 568 (907 TFLOP/s), 6 x 666 rows 111 -> 92, 3 x 700 rows behind 4 096 401 -> 335.
template <int NWV>
__global__ __launch_bounds__(64 * NWV, 2) void attn_prefill_sized_kernel(const bf16* __restrict__ q, const bf16* __restrict__ kv, const bf16* __restrict__ ck,
                                                                    const int32_t* __restrict__ seq, const int32_t* __restrict__ pos,
                                                                    const float* __restrict__ cosb, const float* __restrict__ sinb, int half,
                                                                    int max_pos, const bf16* __restrict__ gate, int64_t ld_gate,
                                                                    bf16* __restrict__ out, int64_t ld_out, int tq, int tk, int H, int C,
                                                                    float scale, int by_seq) {
    typedef FlashTile<2, NWV> Flash;
    constexpr int N = 128, R = 64, V = 128, QB = Flash::ROWS, KT = Flash::KT;
    extern __shared__ __align__(16) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, i = lane & 15;
    const bool by_xcd = (H & 7) == 0;
    const int hx = by_xcd ? H >> 3 : H, x = by_xcd ? blockIdx.x & 7 : 0;
    const int at = by_xcd ? blockIdx.x >> 3 : blockIdx.x;     // the XCD's own workgroups, in order
    const SeqBlock o = seq_block(at, by_xcd ? gridDim.x >> 3 : gridDim.x, hx, blockIdx.y, gridDim.y, by_seq);
    const int h = by_xcd ? o.head * 8 + x : o.head, qb = (gridDim.y - 1 - o.block) * QB;
    const int32_t* sq = seq + 4 * o.seq;
    const int q_at = sq[0], nq = sq[1], k_at = sq[2], nk = sq[3];
    if (qb >= nq || nq < 1 || nk < nq || q_at < 0 || k_at < 0 || q_at + nq > tq || k_at + nk > tk) return;
    const int past = nk - nq;
    const int64_t ld_kv = (int64_t)H * (N + V), ld_ck = C + R;

    Flash f;
    int hi[2], lo[2] = {0, 0};                                // last key that the lane's own query token sees
    auto load = [&] {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int j = min(qb + 32 * wave + 16 * u + i, nq - 1);
            hi[u] = past + j;
            const int64_t tok = q_at + j;
            const bf16* src = q + (tok * H + h) * (int64_t)(N + R) + 8 * g;
            int p = pos[tok];
            p = p < 0 ? 0 : (p >= max_pos ? max_pos - 1 : p);
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                bf16x8 v = load_frag(src + 32 * c);
                if (c >= 4 && half > 0) {
                    const int pr = (c - 4) * 16 + 4 * g;
                    float cs[4], sn[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {             // (all loads at once: behind the condition each waited for the one before)
                        const int64_t at = (int64_t)p * half + min(pr + e, half - 1);
                        cs[e] = cosb[at];
                        sn[e] = sinb[at];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float a = (float)v[2 * e], b = (float)v[2 * e + 1];
                        const bf16 x = (bf16)(a * cs[e] - b * sn[e]), y = (bf16)(b * cs[e] + a * sn[e]);
                        v[2 * e] = pr + e < half ? x : v[2 * e];
                        v[2 * e + 1] = pr + e < half ? y : v[2 * e + 1];
                    }
                }
                f.q[u][c] = v;
            }
        }
    };
    const int wave_first = past + qb + 32 * wave;             // the wave's first row: tiles that end before it need no mask
    f.run(smem, 0, (past + min(qb + QB, nq) - 1) / KT + 1, (uint32_t)ld_kv, (uint32_t)ld_ck, scale, lo, hi, load,
          [&](int t) {
              const bf16* base = kv + (int64_t)(k_at + t * KT) * ld_kv;
              return typename Flash::Tile{base + h * N, ck + (int64_t)(k_at + t * KT) * ld_ck + C, base + (int64_t)H * N + h * V, min(KT, nk - t * KT) - 1};
          },
          [&](int k0) { return k0 + KT - 1 <= wave_first; });
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int j = qb + 32 * wave + 16 * u + i;
        const float inv = 1.0f / f.weight(u);
        if (j >= nq) continue;
        const int64_t tok = q_at + j;
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const int col = h * V + 16 * d + 4 * g;
            const f32x4 z = load_quad(gate + tok * ld_gate + col);
            f32x4 v = f.acc[u][d];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= inv * sigmoid(z[r]);
            store_quad(out + tok * ld_out + col, v);
        }
    }
}

template <int NWV>
static int launch_prefill_sized(const void* q, const void* kv, const void* ck, const int32_t* seq, int nseq, int max_new, const int32_t* pos,
                                const float* cosb, const float* sinb, int half, int max_pos, const void* gate, int64_t ld_gate, void* out,
                                int64_t ld_out, int tq, int tk, int H, int C, float scale, hipStream_t st) {
    typedef FlashTile<2, NWV> Flash;
    const int blocks = (max_new + Flash::ROWS - 1) / Flash::ROWS;
    const int64_t all = (int64_t)H * nseq * blocks;
    const bool by_seq = (int64_t)tk * H >= 5 << 17 && all > 2048 / NWV && all < 1 << 30;
    auto k = attn_prefill_sized_kernel<NWV>;
    const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, Flash::LDS);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(k, dim3((unsigned)(H * nseq), blocks), dim3(64 * NWV), Flash::LDS, st, (const bf16*)q,
                       (const bf16*)kv, (const bf16*)ck, seq, pos, cosb, sinb, half, max_pos, (const bf16*)gate, ld_gate, (bf16*)out, ld_out, tq, tk, H,
                       C, scale, (int)by_seq);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

template <typename T, int KT, int DK, int DV>
static int launch_prefill(const void* q, const void* kv, const void* ck, const int32_t* seq, int nseq, int max_new, const int32_t* pos,
                          const float* cosb, const float* sinb, int half, int max_pos, const void* gate, int64_t ld_gate, void* out,
                          int64_t ld_out, int tq, int tk, int H, int N, int R, int V, int C, float scale, hipStream_t st) {
    const int pad = 16 / (int)sizeof(T);
    const size_t lds = sizeof(T) * KT * (size_t)(N + R + V + 3 * pad);
    if (lds > 160 * 1024) return TF_ERANGE;
    auto k = attn_prefill_kernel<T, KT, DK, DV>;
    static bool attr = false;
    if (!attr) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        attr = true;
    }
    hipLaunchKernelGGL(k, dim3((max_new + 63) / 64 * H, nseq), dim3(256), lds, st, (const T*)q, (const T*)kv, (const T*)ck,
                       seq, pos, cosb, sinb, half, max_pos, (const T*)gate, ld_gate, (T*)out, ld_out, tq, tk, H, N, R, V, C, scale);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tfl_attn_prefill(const void* q, const void* kv, const void* ck, const int32_t* seq, int nseq, int max_new,
                                const int32_t* pos, const float* cosb, const float* sinb, int half, int max_pos, const void* gate,
                                int64_t ld_gate, void* out, int64_t ld_out, int tq, int tk, int H, int N, int R, int V, int C,
                                float scale, int dtype, void* stream) {
    if (!q || !kv || !ck || !seq || !pos || !gate || !out || nseq < 1 || nseq > 65535 || max_new < 1 || tq < 1 || tk < 1) return TF_EINVAL;
    if (H < 1 || H > 65535 || N < 32 || (N & 31) || R < 0 || (R & 31) || V < 32 || (V & 31) || C < 32 || (C & 31)) return TF_EINVAL;
    if (half < 0 || 2 * half > R || max_pos < 1 || (half && (!cosb || !sinb)) || !(scale > 0.f)) return TF_EINVAL;
    if ((ld_gate & 3) || (ld_out & 3) || ld_gate < (int64_t)H * V || ld_out < (int64_t)H * V) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
#define GO(T, KT, DK, DV)                                                                                                             \
    return launch_prefill<T, KT, DK, DV>(q, kv, ck, seq, nseq, max_new, pos, cosb, sinb, half, max_pos, gate, ld_gate, \
                                                  out, ld_out, tq, tk, H, N, R, V, C, scale, st)
#define SIZED_ARGS q, kv, ck, seq, nseq, max_new, pos, cosb, sinb, half, max_pos, gate, ld_gate, out, ld_out, tq, tk, H, C, scale, st
    const int D = N + R;
    if (dtype == 0) {
        if (N == 128 && R == 64 && V == 128 && C <= 1 << 24 && (int64_t)H * nseq <= 1 << 30 && max_new <= 1 << 22) {       // (63 rows of
                                                                 // either stay below 2^32 bytes)
            // 256 rows per workgroup read half as much, which tells where the keys of all heads come from memory (from 16 384 per sequence) or
            // are many to a query (8 and more; a causal prompt of 222 rows 27 % slower), but only with whole rounds of 256: 2 048 rows behind 20 000
            // keys 879 -> 853 us, 4 096 1 812 -> 1 758; 32 heads, 16 x 130 behind 4 096 466 -> 410, 8 heads, 32 x 222 behind 10 000 545 -> 477; behind
            // 10 000 471 -> 478, 2 500 behind 20 000 1 322 -> 1 568
            const int64_t wide = (int64_t)((max_new + 255) / 256) * H * nseq;
            if ((tk / nseq >= 16384 || (tk / 8 >= tq && max_new > 128)) && (wide + 255) / 256 * 256 - wide < 48) return launch_prefill_sized<8>(SIZED_ARGS);
            return launch_prefill_sized<4>(SIZED_ARGS);
        }
        if (D <= 96 && V <= 64) GO(bf16, 64, 3, 4);
        if (D <= 192 && V <= 128) GO(bf16, 64, 6, 8);
        if (D <= 384 && V <= 256) GO(bf16, 64, 12, 16);
        return TF_ERANGE;
    }
    if (dtype == 1) {
        if (D <= 96 && V <= 64) GO(float, 32, 3, 4);
        if (D <= 192 && V <= 128) GO(float, 32, 6, 8);
        if (D <= 384 && V <= 256) GO(float, 32, 12, 16);
        return TF_ERANGE;
    }
#undef GO
#undef SIZED_ARGS
    return TF_EINVAL;
}
