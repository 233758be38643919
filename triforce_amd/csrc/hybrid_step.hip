// Decode step of the hybrid family's mixers: one new token per row.
//
// step_kernel runs both halves of a mixer side by side, as workgroups of one launch:
//   attention   per (key / value head, split of the visible keys): norm and rotate the group's queries and the new key, store the cache
//               row, walk the 64-key pages from the chunk's start.  Scores are transposed (rows keys, columns heads); wave w takes
//               keys 16w ..; the weights go through LDS and every wave accumulates its share of the value columns.
//   recurrence  per (head, 64 value columns): short convolution or per-channel decays of the token, then one pass over the state:
//               S = decay S + k v^T, o = S^T q.
// step_out_kernel makes the operand of the output projection: attention merged over the splits and gated, recurrence normed and gated.
#include "hybrid_common.h"
#include <type_traits>

template <typename T> struct StepCfg { static constexpr int PARTS = sizeof(T) == 2 ? 2 : 1; };

// Which part of which row's keys a workgroup takes.  The launch has rows * nsplit slots per key / value head; rows of a batch see
// different numbers of pages (and after a chunk's edge only a few), so up to 64 rows the slots are dealt by pages: the same number of
// them, q, to every slot, row r having ceil(pages / q) slots in a row.  Every workgroup works it out from the rows' lengths (one
// load, three reductions); the first one leaves each row's first slot and slots for the merge.  More rows: nsplit slots each.
struct Slots { int row, first, pages, t0; };                  // the row that owns a slot (-1: none), its first slot, pages per slot, first page

__device__ __forceinline__ int first_visible(int n, int chunk) { return n > 0 && chunk > 0 ? (n - 1) / chunk * chunk : 0; }

__device__ __forceinline__ Slots find_slot(const int32_t* klen, int rows, int nsplit, int chunk, int slot, int32_t* info) {
    const int lane = threadIdx.x & 63;
    Slots f;
    if (rows == 1 || rows > 64) {
        f.row = slot / nsplit;
        const int n = klen[f.row];
        f.t0 = first_visible(n, chunk) / TFL_PAGE;
        f.first = f.row * nsplit;
        f.pages = n > 0 ? ((n - 1) / TFL_PAGE + 1 - f.t0 + nsplit - 1) / nsplit : 1;
        return f;
    }
    const int n = lane < rows ? klen[lane] : 0, t0 = first_visible(n, chunk) / TFL_PAGE;
    const int p = n > 0 ? (n - 1) / TFL_PAGE + 1 - t0 : 0;
    int total = p, most = p;
    total = __builtin_amdgcn_readfirstlane(lanes_sum(total));                            // (one number for the wave, and known to be: see attn_part_sized)
    most = __builtin_amdgcn_readfirstlane(lanes_max(most));
    const int slots = rows * nsplit, least = max(1, (most + 255) / 256);                     // (the merge weighs 256 slots of a row)
    // sum of ceil(p / q) <= total / q + rows: this q always fits, a smaller one often does
    const int fits = max(least, slots > rows ? (total + slots - rows - 1) / (slots - rows) : most);
    int q = max(least, (total + slots - 1) / slots), c = 0, upto = 0;
    for (int k = 0;; ++k) {
        if (k == 3 || q > fits) q = fits;
        c = (p + q - 1) / q;
        upto = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
            if (o < rows) {
                const int t = __shfl_up(upto, o, 64);
                if (lane >= o) upto += t;
            }
        if (q == fits || __builtin_amdgcn_readlane(upto, rows - 1) <= slots) break;
        ++q;
    }
    if (info && threadIdx.x < rows) {                         // (wave 0)
        info[2 * lane] = upto - c;
        info[2 * lane + 1] = c;
    }
    const uint64_t over = __ballot(lane < rows && upto > slot);
    f.row = over ? __ffsll((long long)over) - 1 : -1;
    const int at = over ? f.row : 0;
    f.first = __builtin_amdgcn_readlane(upto - c, at);
    f.t0 = __builtin_amdgcn_readlane(t0, at);
    f.pages = q;
    return f;
}

struct AttnStep : TfhAttnStep {
    int slots;                                                // rows * nsplit
    // ws: partial values [slots][H][V], maxima and sums [slots][H][2], first slot and slots of each row [rows][2]
    __device__ __forceinline__ float* stats() const { return ws + (int64_t)slots * H * V; }
    __device__ __forceinline__ int32_t* info() const { return reinterpret_cast<int32_t*>(ws + (int64_t)slots * H * (V + 2)); }
};

// ------------------------------------------------------------------------------------------------------------ attention
// NTW: 16-wide value tiles per wave at most.
template <typename T, int NTW>
__device__ __forceinline__ void attn_part(const AttnStep& a, const float* raw, int n, int row, int gh, int slot, int p_beg, int p_end, float eps, char* smem) {
    typedef typename El<T>::Frag Frag;
    constexpr int KT = TFL_PAGE, EPV = 16 / sizeof(T), PARTS = StepCfg<T>::PARTS, NT = 256, LDP = KT + EPV;
    const int D = a.D, V = a.V, dk = D >> 5, ldk = D + EPV, ldv = V + 2 * EPV;
    T* Ks = (T*)smem;                                         // [KT][ldk]
    T* Vs = Ks + KT * ldk;                                    // [KT][ldv]
    T* Qs = Vs + KT * ldv;                                    // [16][ldk]
    T* Ps = Qs + 16 * ldk;                                    // [PARTS][16][LDP]
    float* red = (float*)(Ps + PARTS * 16 * LDP);             // [4][16]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, i = lane & 15;
    const int hpg = a.H / a.G, tiles_h = (hpg + 15) >> 4;
    const int grp = gh / tiles_h, ht = gh - grp * tiles_h;
    const int h0 = grp * hpg + 16 * ht, nh = min(16, hpg - 16 * ht);
    const int first_key = first_visible(n, a.chunk), t_beg = p_beg, t_end = p_end;
    float* ml = a.stats();
    const int32_t* tab = a.table + (int64_t)row * a.table_ld;
    const int64_t ld_c = (int64_t)a.G * (D + V);
    auto rows_of = [&](int t) {
        const int pg = tab[t];
        return (T*)a.cache + (int64_t)(pg < 0 ? 0 : (pg >= a.n_pages ? (int)a.n_pages - 1 : pg)) * TFL_PAGE * ld_c;
    };
    const int p = min(n - 1, a.max_pos - 1);
    const float *cs = a.cos + (int64_t)p * a.half, *sn = a.sin + (int64_t)p * a.half;
    for (int r = wave; r < 16; r += 4) {
        float o[4] = {0.f, 0.f, 0.f, 0.f};
        if (r < nh) {
            const float* src = raw + a.q_off + (h0 + r) * D;
            head_norm_rotate([src](int e) { return src[e]; }, D, a.D_real, a.q_norm, eps, cs, sn, a.half, lane, o);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < D) Qs[r * ldk + lane + 64 * j] = (T)o[j];
    }
    f32x4 o[NTW];
#pragma unroll
    for (int x = 0; x < NTW; ++x) o[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = NEG_INF, l_run = 0.f;
    const int kn = D / EPV, vn = V / EPV, ppr = kn + vn;
    for (int t = t_beg; t < t_end; ++t) {
        const int k0 = t * KT;
        T* base = rows_of(t);
        const int fresh = n - 1 - k0;                         // tile row of the new key (< KT: in this tile)
        for (int q = tid; q < KT * ppr; q += NT) {
            const int key = q / ppr, c = q - key * ppr;
            if (key == fresh) continue;
            u32x4 v = {0, 0, 0, 0};
            if (key < fresh) v = *reinterpret_cast<const u32x4*>(base + (int64_t)key * ld_c + (c < kn ? grp * D + EPV * c : a.G * D + grp * V + EPV * (c - kn)));
            *reinterpret_cast<u32x4*>(c < kn ? Ks + key * ldk + EPV * c : Vs + key * ldv + EPV * (c - kn)) = v;
        }
        if (fresh < KT) {
            T* dst = base + (int64_t)fresh * ld_c;
            if (wave == 0) {
                const float* src = raw + a.k_off + grp * D;
                float k[4];
                head_norm_rotate([src](int e) { return src[e]; }, D, a.D_real, a.k_norm, eps, cs, sn, a.half, lane, k);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (lane + 64 * j < D) {
                        Ks[fresh * ldk + lane + 64 * j] = (T)k[j];
                        if (ht == 0) dst[grp * D + lane + 64 * j] = (T)k[j];
                    }
            } else {
                for (int e = tid - 64; e < V; e += 192) {
                    const T v = (T)raw[a.v_off + grp * V + e];
                    Vs[fresh * ldv + e] = v;
                    if (ht == 0) dst[a.G * D + grp * V + e] = v;
                }
            }
        }
        __syncthreads();
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        const T *kp = Ks + (16 * wave + i) * ldk + 8 * g, *qp = Qs + i * ldk + 8 * g;
        for (int c = 0; c < dk; ++c) s = El<T>::mma(load_frag(kp + 32 * c), load_frag(qp + 32 * c), s);
        float mx = NEG_INF;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = k0 + 16 * wave + 4 * g + r;
            s[r] = k < n && k >= first_key ? s[r] * a.scale : NEG_INF;
            mx = fmaxf(mx, s[r]);
        }
        mx = rows_max(mx);
        if (g == 0) red[wave * 16 + i] = mx;
        __syncthreads();
        mx = m_run;
#pragma unroll
        for (int w = 0; w < 4; ++w) mx = fmaxf(mx, red[w * 16 + i]);      // (every tile has a visible key: finite)
        const float alpha = exp2f((m_run - mx) * LOG2E);
        m_run = mx;
        f32x4 w4, lo;
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            w4[r] = exp2f((s[r] - mx) * LOG2E);
            sum += w4[r];
            lo[r] = w4[r] - (float)(T)w4[r];
        }
        l_run = l_run * alpha + sum;
        T* dst = Ps + i * LDP + 16 * wave + 4 * g;
        store_quad(dst, w4);
        if constexpr (PARTS == 2) store_quad(dst + 16 * LDP, lo);
        __syncthreads();
#pragma unroll
        for (int x = 0; x < NTW; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[x][r] *= alpha;
#pragma unroll
        for (int c = 0; c < KT / 32; ++c) {
            Frag b[PARTS];
#pragma unroll
            for (int z = 0; z < PARTS; ++z) b[z] = load_frag(Ps + (z * 16 + i) * LDP + 32 * c + 8 * g);
#pragma unroll
            for (int x = 0; x < NTW; ++x) {
                const int col = 16 * (wave * NTW + x);
                if (col < V) {
                    const Frag f = load_frag_t(Vs, ldv, 32 * c + 8 * g, 32 * c + 8 * g + 4, col, i);
#pragma unroll
                    for (int z = 0; z < PARTS; ++z) o[x] = El<T>::mma(f, b[z], o[x]);
                }
            }
        }
        __syncthreads();
    }
    l_run = rows_sum(l_run);
    if (g == 0) red[wave * 16 + i] = l_run;
    __syncthreads();
    if (i < nh) {
        const int64_t at = (int64_t)slot * a.H + h0 + i;
#pragma unroll
        for (int x = 0; x < NTW; ++x) {
            const int col = 16 * (wave * NTW + x) + 4 * g;
            if (col < V) *reinterpret_cast<f32x4*>(a.ws + at * V + col) = o[x];
        }
        if (wave == 0 && g == 0) {
            ml[2 * at] = m_run;
            ml[2 * at + 1] = red[i] + red[16 + i] + red[32 + i] + red[48 + i];
        }
    }
}

// head_norm_rotate() of D entries (64 or 128) in two parts, loads and arithmetic.
template <int D> struct HeadFactors {                         // this lane's weights of the norm, and its angles
    float w[D / 64], pw[D / 64], cs[D / 64], sn[D / 64];
    __device__ __forceinline__ void load(const float* norm, const float* c, const float* s, int half, int lane) {
#pragma unroll
        for (int j = 0; j < D / 64; ++j) {
            const int e = lane + 64 * j;
            w[j] = norm[e];
            pw[j] = cs[j] = sn[j] = 0.f;
            if (half > 0) {                                   // (no tables without a rotated part)
                const int pe = e < half ? e + half : max(e - half, 0), p = min(e < half ? e : e - half, half - 1);
                pw[j] = norm[pe];
                cs[j] = c[p];
                sn[j] = s[p];
            }
        }
    }
};
template <int D> struct HeadEntries {                         // raw entries, and those of the other half of a rotated pair
    float v[D / 64], pv[D / 64];
    __device__ __forceinline__ void load(const float* src, int half, int lane) {
#pragma unroll
        for (int j = 0; j < D / 64; ++j) {
            const int e = lane + 64 * j;
            v[j] = src[e];
            pv[j] = src[e < half ? e + half : max(e - half, 0)];
        }
    }
    __device__ __forceinline__ void norm_rotate(const HeadFactors<D>& f, int D_real, float eps, int half, int lane, float (&o)[D / 64]) const {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < D / 64; ++j) ss = fmaf(v[j], v[j], ss);
        ss = wave_sum64(ss);
        const float inv = 1.0f / sqrtf(ss / (float)D_real + eps);
#pragma unroll
        for (int j = 0; j < D / 64; ++j) {
            const int e = lane + 64 * j;
            const float u = v[j] * inv * f.w[j], t = pv[j] * inv * f.pw[j];
            o[j] = e < half ? u * f.cs[j] - t * f.sn[j] : e < 2 * half ? u * f.cs[j] + t * f.sn[j] : u;
        }
    }
};

// The same for known sizes, bfloat16: 32 * DK entries of query-key size, 16 * DV of value size.  The waves walk their own 32-key tiles
// without a barrier: rows come from memory whole (the next tile's while this one is used), pass through a piece of LDS that only the wave
// touches, and the result registers of a tile's two score products are the weight operand of its value products.  The waves meet once,
// at the end.  Keys and values of a tile pass through the same piece, one after the other: 41 KB a workgroup, so that with 168
// registers three of them fit a CU and the recurrences' workgroups (all latency) run beside the attention's (all bandwidth) instead
// of behind them.  What is left is a chain of some 12 us (launch, length, page, first rows, norms, merge of the waves) in front of and
// behind the stream.  Step and merge, 41 KB and dealt slots against 77 KB and nsplit slots a row: 1 x 8 192 keys 23.7 -> 20.9 us, 8 x 4 096 51.3 ->
// 46.9, 8 rows of 808 to 8 157 keys 59.1 -> 55.5, 32 around 3 000 139.5 -> 123.8.
// The wave knows that its row, slot and pages are one number (scalar), and holds the ids of 64 pages: an id read in the loop, or a load behind a
// condition, has the compiler wait for every load in flight, the tile ahead too.  G = 8, H = 32 of 128, step and merge, before -> now: 8 x 4 096 keys
// 34.5 -> 32.0 us, 1 x 8 000 18.1 -> 16.6, 16 x 3 000 44.3 -> 40.8, 32 x 3 000 82.4 -> 72.1, 64 x 1 000 61.2 -> 55.1.
template <int DK, int DV>
struct SizedStep {
    static constexpr int KT = 32, D = 32 * DK, V = 16 * DV, LDK = D + 8, LDV = V + 16, TILE = KT * (LDK > LDV ? LDK : LDV);
    static constexpr size_t LDS = sizeof(bf16) * (4 * TILE + 16 * LDK) + sizeof(float) * 128;
    static_assert(4 * 16 * V * sizeof(float) <= sizeof(bf16) * 4 * TILE, "the waves' results reuse the tiles");
};

template <int DK, int DV>
__device__ __forceinline__ void attn_part_sized(const AttnStep& a, const float* raw, int n, int row, int gh, int slot, int p_beg, int p_end, float eps, char* smem) {
    typedef SizedStep<DK, DV> Z;
    constexpr int KT = Z::KT, D = Z::D, V = Z::V, LDK = Z::LDK, LDV = Z::LDV, KP = D / 8, VP = V / 8, NK = KT * KP / 64, NV = KT * VP / 64;
    static_assert(64 % KP == 0 && 64 % VP == 0, "whole rows per load");
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int lane = tid & 63, g = lane >> 4, i = lane & 15;
    bf16* Kt = (bf16*)smem + wave * Z::TILE;                  // this wave's [KT][LDK], then [KT][LDV]
    bf16* Vt = Kt;
    bf16* Qs = (bf16*)smem + 4 * Z::TILE;                     // [16][LDK]
    float* red = (float*)(Qs + 16 * LDK);                     // [4][16] maxima, [4][16] sums
    const int hpg = a.H / a.G, tiles_h = (hpg + 15) >> 4;
    const int grp = gh / tiles_h, ht = gh - grp * tiles_h;
    const int h0 = grp * hpg + 16 * ht, nh = min(16, hpg - 16 * ht);
    const int first_key = first_visible(n, a.chunk);
    constexpr int PT = TFL_PAGE / KT;                         // tiles per page; the chunk may begin inside the first one
    const int t_beg = max(p_beg * PT, first_key / KT), t_end = min(p_end * PT, (n - 1) / KT + 1);
    float* ml = a.stats();
    const int32_t* tab = a.table + (int64_t)row * a.table_ld;
    const int64_t ld_c = (int64_t)a.G * (D + V);
    int ids_from = p_beg, ids = tab[min(p_beg + lane, p_end - 1)];                       // of 64 pages
    auto rows_of = [&](int t) {
        const int page = t * KT / TFL_PAGE;
        if (page >= ids_from + 64) {
            ids_from = page;
            ids = tab[min(page + lane, p_end - 1)];
            asm volatile("" : "+v"(ids));                     // (waited for here: behind the branch all loads would be)
        }
        const int pg = __builtin_amdgcn_readlane(ids, page - ids_from);
        return (bf16*)a.cache + ((int64_t)(pg < 0 ? 0 : (pg >= a.n_pages ? (int)a.n_pages - 1 : pg)) * TFL_PAGE + t * KT % TFL_PAGE) * ld_c;
    };
    // What the norms and the new key need is asked for first: loads return in the order that they were asked for.
    const int p = min(n - 1, a.max_pos - 1);
    HeadFactors<D> qw, kw;
    HeadEntries<D> qr[4], kr;
    qw.load(a.q_norm, a.cos + (int64_t)p * a.half, a.sin + (int64_t)p * a.half, a.half, lane);
#pragma unroll
    for (int h = 0; h < 4; ++h)
        if (wave + 4 * h < nh) qr[h].load(raw + a.q_off + (h0 + wave + 4 * h) * D, a.half, lane);
    const int t_new = (n - 1) / KT;                           // the new key's tile, and whose it is
    const bool newest = t_new < t_end && ((t_new - t_beg) & 3) == wave;
    float vr[V / 64] = {};
    if (newest) {
        kw.load(a.k_norm, a.cos + (int64_t)p * a.half, a.sin + (int64_t)p * a.half, a.half, lane);
        kr.load(raw + a.k_off + grp * D, a.half, lane);
#pragma unroll
        for (int j = 0; j < V / 64; ++j) vr[j] = raw[a.v_off + grp * V + lane + 64 * j];
    }
    u32x4 prek[NK], prev[NV];
    const uint32_t row_bytes = 2 * (uint32_t)ld_c;            // (G * (D + V) elements: a tile stays far below 2^32 bytes)
    auto fetch_k = [&](int t) {
        const char* base = reinterpret_cast<const char*>(rows_of(t) + grp * D);
        const int left = n - 1 - t * KT;                      // rows behind the last key repeat it (masked)
#pragma unroll
        for (int j = 0; j < NK; ++j)
            prek[j] = *reinterpret_cast<const u32x4*>(base + ((uint32_t)min(lane / KP + j * (64 / KP), left) * row_bytes + 16u * (lane % KP)));
    };
    auto fetch_v = [&](int t) {
        const char* base = reinterpret_cast<const char*>(rows_of(t) + a.G * D + grp * V);
        const int left = n - 1 - t * KT;
#pragma unroll
        for (int j = 0; j < NV; ++j)
            prev[j] = *reinterpret_cast<const u32x4*>(base + ((uint32_t)min(lane / VP + j * (64 / VP), left) * row_bytes + 16u * (lane % VP)));
    };
    __builtin_amdgcn_sched_barrier(0);
    if (t_beg + wave < t_end) {
        fetch_k(t_beg + wave);
        fetch_v(t_beg + wave);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int r = wave + 4 * h;
        float o[D / 64] = {};
        if (r < nh) qr[h].norm_rotate(qw, a.D_real, eps, a.half, lane, o);
#pragma unroll
        for (int j = 0; j < D / 64; ++j) Qs[r * LDK + lane + 64 * j] = (bf16)o[j];
    }
    bf16 k_new[D / 64] = {}, v_new[V / 64] = {};              // of the new key
    if (newest) {
        float o[D / 64];
        kr.norm_rotate(kw, a.D_real, eps, a.half, lane, o);
#pragma unroll
        for (int j = 0; j < D / 64; ++j) k_new[j] = (bf16)o[j];
#pragma unroll
        for (int j = 0; j < V / 64; ++j) v_new[j] = (bf16)vr[j];
    }
    __syncthreads();
    bf16x8 qf[DK];
#pragma unroll
    for (int c = 0; c < DK; ++c) qf[c] = load_frag(Qs + i * LDK + 32 * c + 8 * g);
    f32x4 o[DV];
#pragma unroll
    for (int d = 0; d < DV; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = NEG_INF, l_run = 0.f;
    // One tile, and the next one's loads.  The last one apart: only it can hold the new key, and loads behind a condition would be waited for as if
    // they had been left out.
    auto step = [&](int t, auto last) __attribute__((always_inline)) {
        constexpr bool LAST = decltype(last)::value;
        const int k0 = t * KT, fresh = n - 1 - k0;            // tile row of the new key (< KT: in this tile)
        const bool edge = LAST && fresh < KT;
        asm("" : "+v"(lane), "+v"(g), "+v"(i));               // (opaque once per tile: hoisted addresses would take the registers)
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            const int r = lane / KP + j * (64 / KP);
            *reinterpret_cast<u32x4*>(Kt + r * LDK + 8 * (lane % KP)) = edge && r >= fresh ? u32x4{0, 0, 0, 0} : prek[j];
        }
        bf16* dst = edge ? rows_of(t) + (int64_t)fresh * ld_c : nullptr;
        if (edge) {
#pragma unroll
            for (int j = 0; j < D / 64; ++j) {
                Kt[fresh * LDK + lane + 64 * j] = k_new[j];
                if (ht == 0) dst[grp * D + lane + 64 * j] = k_new[j];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");            // (one wave's LDS accesses stay in order; so must the compiler)
        if constexpr (!LAST) fetch_k(t + 4);
        f32x4 s[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DK; ++c) s[kt] = El<bf16>::mma(load_frag(Kt + (16 * kt + i) * LDK + 32 * c + 8 * g), qf[c], s[kt]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");            // the keys are used up: the values take their place
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int r = lane / VP + j * (64 / VP);
            *reinterpret_cast<u32x4*>(Vt + r * LDV + 8 * (lane % VP)) = edge && r >= fresh ? u32x4{0, 0, 0, 0} : prev[j];
        }
        if (edge) {
#pragma unroll
            for (int j = 0; j < V / 64; ++j) {
                Vt[fresh * LDV + lane + 64 * j] = v_new[j];
                if (ht == 0) dst[a.G * D + grp * V + lane + 64 * j] = v_new[j];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if constexpr (!LAST) fetch_v(t + 4);
        float mx = NEG_INF;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = k0 + 16 * kt + 4 * g + r;
                s[kt][r] = (!LAST || k < n) && k >= first_key ? s[kt][r] * a.scale : NEG_INF;
                mx = fmaxf(mx, s[kt][r]);
            }
        mx = rows_max(mx);
        mx = fmaxf(m_run, mx);                                // (every tile has a visible key: finite)
        const float alpha = __builtin_amdgcn_exp2f((m_run - mx) * LOG2E);
        m_run = mx;
        bf16x8 hi, lo;
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float w = __builtin_amdgcn_exp2f((s[kt][r] - mx) * LOG2E);
                sum += w;
                hi[4 * kt + r] = (bf16)w;
                lo[4 * kt + r] = (bf16)(w - (float)(bf16)w);
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
            const bf16x8 f = load_frag_t(Vt, LDV, 4 * g, 16 + 4 * g, 16 * d, i);
            o[d] = El<bf16>::mma(f, hi, o[d]);
            o[d] = El<bf16>::mma(f, lo, o[d]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    if (t_beg + wave < t_end) {
        int t = t_beg + wave;
        for (; t + 4 < t_end; t += 4) step(t, std::false_type());
        step(t, std::true_type());
    }
    l_run = rows_sum(l_run);
    if (g == 0) {
        red[wave * 16 + i] = m_run;
        red[64 + wave * 16 + i] = l_run;
    }
    __syncthreads();                                          // everyone is done with the tiles
    float* po = (float*)smem;                                 // [4][16][V]
    float m = NEG_INF;
#pragma unroll
    for (int w = 0; w < 4; ++w) m = fmaxf(m, red[w * 16 + i]);
    const float f = m_run == NEG_INF ? 0.f : __builtin_amdgcn_exp2f((m_run - m) * LOG2E);
    if (i < nh) {
#pragma unroll
        for (int d = 0; d < DV; ++d) {
#pragma unroll
            for (int r = 0; r < 4; ++r) o[d][r] *= f;
            *reinterpret_cast<f32x4*>(po + (wave * 16 + i) * V + 16 * d + 4 * g) = o[d];
        }
        if (wave == 0 && g == 0) {
            float l = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float mw = red[w * 16 + i];
                l += mw == NEG_INF ? 0.f : red[64 + w * 16 + i] * __builtin_amdgcn_exp2f((mw - m) * LOG2E);
            }
            float* q = ml + ((int64_t)slot * a.H + h0 + i) * 2;
            q[0] = m;
            q[1] = l;
        }
    }
    __syncthreads();
    for (int e = tid; e < nh * V / 4; e += 256) {
        const int h = e / (V / 4), c = 4 * (e % (V / 4));
        f32x4 v = *reinterpret_cast<const f32x4*>(po + h * V + c);
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(po + (w * 16 + h) * V + c);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += x[r];
        }
        *reinterpret_cast<f32x4*>(a.ws + ((int64_t)slot * a.H + h0 + h) * V + c) = v;
    }
}

// ------------------------------------------------------------------------------------------------------------ recurrence
// LDS: q, k, decay [N] each, v [64], one float per (state row group, value) for the read-out.
template <typename T>
__device__ __forceinline__ void rec_part(const TfhRecStep& a, int slice, const float* raw, int n, int row, int bid, char* smem) {
    const int N = a.N, slices = (a.V + slice - 1) / slice, head = bid / slices, v0 = (bid - head * slices) * slice, vs = min(slice, a.V - v0);
    const int seat = a.seat[row];
    if (n < 1 || seat < 0 || seat >= a.seats) return;         // idle row
    float *qs = (float*)smem, *ks = qs + N, *dc = ks + N, *xs = dc + N, *po = xs + 64;
    const int tid = threadIdx.x, pos = n - 1;
    const bool scalar = a.a2 == nullptr, fresh = pos == 0;    // (a seat's earlier owner left its state behind)
    const int nq = vs >> 2, ng = 256 / nq, vq = tid % nq, gr = tid / nq;   // thread: four values, state rows gr, gr + ng, ...
    f32x4* S = reinterpret_cast<f32x4*>(a.state + (((int64_t)seat * a.H + head) * N) * a.V + v0) + vq;
    const int64_t step = a.V >> 2;
    constexpr int U = 8;
    f32x4 s[U];
    auto load = [&](int r0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            s[u] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (gr < ng && r0 + u * ng < N && !fresh) s[u] = S[(r0 + u * ng) * step];
        }
    };
    load(gr);
    float decay = 0.f;
    if (scalar) {
        const int grp = head / a.per_group, inner = a.H * a.V, GN = a.H / a.per_group * N;
        float* ring = a.ring + (int64_t)seat * a.taps * a.channels;
        const bool owner = head % a.per_group == 0 && v0 == 0;            // stores the group's B and C inputs
        const float dt = softplus(raw[a.dt_off + head] + a.dt_bias[head]);
        decay = expf(a.nega[head] * dt);
        for (int e = tid; e < vs + 2 * N; e += 256) {
            const int c = e < vs ? head * a.V + v0 + e : (e < vs + N ? inner + grp * N + e - vs : inner + GN + grp * N + e - vs - N);
            const float now = raw[a.x_off + c];
            float y = fmaf(now, a.conv_w[(int64_t)(a.taps - 1) * a.channels + c], a.conv_b[c]);
            for (int t0 = 1; t0 < a.taps; t0 += 4) {                      // (the loads of four taps at once)
                float in[4], w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int t = t0 + u;
                    const bool use = t < a.taps && t <= pos;
                    in[u] = use ? ring[(int64_t)((pos - t) % a.taps) * a.channels + c] : 0.f;
                    w[u] = use ? a.conv_w[(int64_t)(a.taps - 1 - t) * a.channels + c] : 0.f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) y = fmaf(in[u], w[u], y);
            }
            if (e < vs || owner) ring[(int64_t)(pos % a.taps) * a.channels + c] = now;   // (a slot that no reader of this step uses)
            y = silu(y);
            if (e < vs) xs[e] = y;
            else if (e < vs + N) ks[e - vs] = y * dt;
            else qs[e - vs - N] = y;
        }
    } else {
        for (int e = tid; e < N; e += 256) {
            const int c = head * N + e;
            qs[e] = raw[a.q_off + c] * a.q_scale;
            ks[e] = raw[a.k_off + c];
            const T* w = (const T*)a.a2 + (int64_t)c * a.rank;
            float z = a.a2_b[c];
#pragma unroll 4
            for (int r = 0; r < a.rank; r += 4) {
                const f32x4 w4 = load_quad(w + r), x4 = load_quad(raw + a.a_off + r);
#pragma unroll
                for (int u = 0; u < 4; ++u) z = fmaf(w4[u], x4[u], z);
            }
            dc[e] = expf(log_sigmoid(z) * a.inv_tau);
        }
        for (int e = tid; e < vs; e += 256) xs[e] = raw[a.v_off + head * a.V + v0 + e];
    }
    __syncthreads();
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    if (gr < ng) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(xs + 4 * vq);
        for (int r0 = gr; r0 < N; r0 += U * ng) {
            if (r0 > gr) load(r0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int r = r0 + u * ng;
                if (r >= N) continue;
                const float d = scalar ? decay : dc[r], k = ks[r], q = qs[r];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[u][e] = fmaf(d, s[u][e], k * x[e]);
                    o[e] = fmaf(s[u][e], q, o[e]);
                }
                S[r * step] = s[u];
            }
        }
        *reinterpret_cast<f32x4*>(po + gr * vs + 4 * vq) = o;
    }
    __syncthreads();
    if (tid < vs) {
        float y = 0.f;
        for (int k = 0; k < ng; ++k) y += po[k * vs + tid];
        if (scalar) y = fmaf(a.skip[head], xs[tid], y) * silu_of<T>(raw[a.gate_off + head * a.V + v0 + tid]);
        a.out[((int64_t)row * a.H + head) * a.V + v0 + tid] = y;
    }
}

// All rows' attention first (it takes longer), then the recurrences: attn_blocks and rec_blocks of them in all.  DK > 0: the sized
// attention.
template <typename T, int NTW, int DK, int DV>
__global__ __launch_bounds__(256, DK > 0 ? 3 : 1) void step_kernel(const AttnStep a, const TfhRecStep r, int attn_blocks, int rec_per_row, int slice, int rows,
                                                   const float* __restrict__ raw, int64_t ld_raw, const int32_t* __restrict__ klen, float eps) {
    extern __shared__ __align__(32) char smem[];
    if ((int)blockIdx.x >= attn_blocks) {
        const int id = blockIdx.x - attn_blocks, row = id / rec_per_row;
        rec_part<T>(r, slice, raw + (int64_t)row * ld_raw, klen[row], row, id - row * rec_per_row, smem);
        return;
    }
    const int gh = blockIdx.x / a.slots, slot = blockIdx.x - gh * a.slots;
    const Slots f = find_slot(klen, rows, a.nsplit, a.chunk, slot, blockIdx.x == 0 ? a.info() : nullptr);
    if (f.row < 0) return;
    const int n = klen[f.row], p_beg = f.t0 + (slot - f.first) * f.pages, p_end = n > 0 ? min((n - 1) / TFL_PAGE + 1, p_beg + f.pages) : 0;
    if (p_beg >= p_end) {                                     // (more than 64 rows: slots past the last page)
        const int hpg = a.H / a.G, tiles_h = (hpg + 15) >> 4, grp = gh / tiles_h, h0 = grp * hpg + 16 * (gh - grp * tiles_h), tid = threadIdx.x;
        if (tid < min(16, grp * hpg + hpg - h0)) {
            float* p = a.stats() + ((int64_t)slot * a.H + h0 + tid) * 2;
            p[0] = NEG_INF;
            p[1] = 0.f;
        }
        return;
    }
    const float* rr = raw + (int64_t)f.row * ld_raw;
    if constexpr (DK > 0) attn_part_sized<DK, DV>(a, rr, n, f.row, gh, slot, p_beg, p_end, eps, smem);
    else attn_part<T, NTW>(a, rr, n, f.row, gh, slot, p_beg, p_end, eps, smem);
}

// ------------------------------------------------------------------------------------------------------------ operand
template <typename T>
__global__ __launch_bounds__(256) void step_out_kernel(const AttnStep a, const TfhRecStep r, int attn_blocks, int groups,
                                                       const float* __restrict__ raw, int64_t ld_raw, T* __restrict__ act, int64_t ld_act,
                                                       int64_t act_oct, float eps) {
    __shared__ float wgt[256];
    __shared__ float red[8];
    __shared__ f32x4 acc[256];
    const int row = blockIdx.y, tid = threadIdx.x;
    const float* rr = raw + (int64_t)row * ld_raw;
    T* dst = act + (int64_t)row * ld_act;
    if ((int)blockIdx.x < attn_blocks) {                      // one head: splits merged, output gate
        const bool dealt = gridDim.y > 1 && gridDim.y <= 64;
        const int head = blockIdx.x, V = a.V, first = dealt ? min(a.info()[2 * row], a.slots - 1) : row * a.nsplit, ns = dealt ? a.info()[2 * row + 1] : a.nsplit;
        const int64_t at = (int64_t)first * a.H + head;        // + s * H: slot s of the row
        const float* ml = a.stats() + 2 * at;
        const int nq = V >> 2, ng = 256 / nq, vq = tid % nq, gr = tid / nq, c = head * V + 4 * vq;
        // Bound by round trips: gate and first partial rows are asked for together with the statistics, whose two halves come at once.
        constexpr int U = 2;
        f32x4 z0[U], zg = {0.f, 0.f, 0.f, 0.f};
        const int last = max(ns, 1) - 1;
#pragma unroll
        for (int u = 0; u < U; ++u) z0[u] = *reinterpret_cast<const f32x4*>(a.ws + (at + (int64_t)min(gr + u * ng, last) * a.H) * V + 4 * vq);
        if (gr == 0) zg = *reinterpret_cast<const f32x4*>(rr + a.gate_off + c);
        const float m_have = ml[2 * (int64_t)min(tid, last) * a.H], l_have = ml[2 * (int64_t)min(tid, last) * a.H + 1];
        const float ls = tid < ns ? l_have : 0.f, ms = ls > 0.f ? m_have : NEG_INF;
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
        if (gr < ng) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int s = gr + u * ng;
                const float f = s < ns ? wgt[s] : 0.f;
                if (f > 0.f) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = fmaf(z0[u][e], f, v[e]);
                }
            }
            for (int s = gr + U * ng; s < ns; s += ng) {
                const float f = wgt[s];
                if (f > 0.f) {                                // (an empty split's partial row was never written)
                    const f32x4 z = *reinterpret_cast<const f32x4*>(a.ws + (at + (int64_t)s * a.H) * V + 4 * vq);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = fmaf(z[e], f, v[e]);
                }
            }
        }
        acc[tid] = v;
        __syncthreads();
        if (gr == 0) {
            for (int k = 1; k < ng; ++k) {
                const f32x4 z = acc[k * nq + vq];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += z[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= sigmoid_of<T>(zg[e]) * a.out_scale;
            store_quad(dst + (c >> 3) * act_oct + (c & 7), v);
        }
        return;
    }
    const int grp = blockIdx.x - attn_blocks, size = r.H * r.V_real / groups, first = grp * size, off = a.H * a.V;
    const bool per_channel = r.a2 != nullptr;                 // gate behind the norm, one weight vector for all heads
    const float* src = r.out + (int64_t)row * r.H * r.V;
    auto where = [&](int c) { return c / r.V_real * r.V + c % r.V_real; };
    float ss = 0.f;
    if (r.V == r.V_real && !(size & 3)) {                     // no padding inside a row: quads, the first HOLD of a thread stay in registers
        constexpr int HOLD = 4;
        f32x4 held[HOLD], wt[HOLD], gt[HOLD];
        auto weights = [&](int c) { return *reinterpret_cast<const f32x4*>(r.norm_w + (per_channel ? c : first + c)); };
        auto gates = [&](int c) { return *reinterpret_cast<const f32x4*>(rr + r.gate_off + first + c); };
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            const int c = 4 * (tid + 256 * u);
            held[u] = wt[u] = gt[u] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (c < size) {
                held[u] = *reinterpret_cast<const f32x4*>(src + first + c);
                wt[u] = weights(c);
                if (per_channel) gt[u] = gates(c);
            }
        }
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            ss += held[u][0] * held[u][0] + held[u][1] * held[u][1] + held[u][2] * held[u][2] + held[u][3] * held[u][3];
        }
        for (int c = 4 * (tid + 256 * HOLD); c < size; c += 1024) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(src + first + c);
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        ss = block_sum<4>(ss, red);
        const float inv = r.out_scale / sqrtf(ss / (float)size + eps);
        auto put = [&](int c, f32x4 v, f32x4 w, f32x4 z) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] * inv * w[e];
            if (per_channel) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] *= silu_of<T>(z[e]);
            }
            const int o = off + first + c;
            store_quad(dst + (o >> 3) * act_oct + (o & 7), v);
        };
#pragma unroll
        for (int u = 0; u < HOLD; ++u)
            if (4 * (tid + 256 * u) < size) put(4 * (tid + 256 * u), held[u], wt[u], gt[u]);
        for (int c = 4 * (tid + 256 * HOLD); c < size; c += 1024)
            put(c, *reinterpret_cast<const f32x4*>(src + first + c), weights(c), per_channel ? gates(c) : f32x4{0.f, 0.f, 0.f, 0.f});
        return;
    }
    for (int c = tid; c < size; c += 256) {
        const float v = src[where(first + c)];
        ss = fmaf(v, v, ss);
    }
    ss = block_sum<4>(ss, red);
    const float inv = r.out_scale / sqrtf(ss / (float)size + eps);
    for (int c = tid; c < size; c += 256) {
        const int at = where(first + c);
        float v = src[at] * inv * r.norm_w[per_channel ? c : first + c];
        if (per_channel) v *= silu_of<T>(rr[r.gate_off + at]);
        const int o = off + at;
        dst[(o >> 3) * act_oct + (o & 7)] = (T)v;
        if ((first + c) % r.V_real == r.V_real - 1)
            for (int k = o + 1; k < o - r.V_real + 1 + r.V; ++k) dst[(k >> 3) * act_oct + (k & 7)] = (T)0.f;
    }
}

#define TFH_MAX_SPLIT 256

extern "C" int64_t tfh_attn_step_ws_floats(int rows, int H, int V, int nsplit) {
    if (rows < 1 || H < 1 || V < 1 || nsplit < 1) return 0;
    return (int64_t)rows * H * nsplit * (V + 2) + 2 * (int64_t)rows;
}

static bool sized_step(int D, int V, int dtype) { return dtype == 0 && V == D && (D == 64 || D == 128); }

// Two workgroups per CU (512), at least four splits a row up to 64 rows, whose unequal lengths are dealt by splits, as long as a split keeps a
// page of keys.  us with the merge, recurrences beside it, caches from memory:
//   * the sized attention of 128: one workgroup per CU for a row alone, above 16 splits a row in whole sixteens, three splits above 64 rows.  One row
//     of 300 / 3 000 / 8 000 keys at 32 splits 13.6 / 15.1 / 15.8, at 64 14.6 / 16.9 / 17.9; three of 1 000 at 16 / 21 16.9 / 20.0; 16 rows
//     of 3 000 at 4 / 8 / 16 65.9 / 66.6 / 74.1; 128 rows of 1 000 at 1 / 2 / 3 / 4 / 8 240 / 245 / 243 / 258 / 277, of 3 000 426 / 431 / 431 / 429 /
//     446, 65 rows of up to 8 000 325 / 264 / 252 / 246 / 254;
//   * of 64, and the general one: splits as they come (bfloat16 heads of 96, one row of 30 000 keys at 32 / 64 89 / 59; of 256, five rows at 16 / 25
//     705 / 463);
//   * the general one, 16 to 31 rows: at least eight (16 rows of 8 000 to 4 000 keys, float32 heads of 128 at 4 / 6 / 8 / 16 830 / 694 / 674 / 737,
//     bfloat16 of 96 198 / 125 / 106 / 116); from 32 rows on three where two workgroups or fewer fit a CU (float32 heads of 128, 48 rows of 1 000 to 500
//     keys at 1 / 2 / 3 / 4 384 / 395 / 365 / 400, 128 rows of 300 488 / 544 / 524 / 664), four where more do.
extern "C" int tfh_attn_step_splits(int rows, int H, int G, int D, int V, int max_keys, int dtype) {
    if (rows < 1 || H < 1 || G < 1 || max_keys < 1) return 1;
    const bool sized = sized_step(D, V, dtype), full = sized && D == 128, large = (int64_t)(D + V) * (dtype ? 4 : 2) >= 640;
    const int groups = G * ((H / G + 15) / 16);
    const int least = full ? (rows <= 64 ? 4 : 3) : sized ? 4 : rows < 16 ? 4 : rows < 32 ? 8 : large ? 3 : 4;
    int n = (int)((rows == 1 && full ? 256 : 512) / ((int64_t)rows * groups));
    if (full && n > 16) n &= ~15;
    if (n < least) n = least;
    const int cap = (max_keys + TFL_PAGE - 1) / TFL_PAGE;
    if (n > cap) n = cap;
    if (n > TFH_MAX_SPLIT) n = TFH_MAX_SPLIT;
    return n < 1 ? 1 : n;
}

// The same for bfloat16 heads of 128.
extern "C" int tfh_attn_step_pick_nsplit(int rows, int H, int G, int max_keys) { return tfh_attn_step_splits(rows, H, G, 128, 128, max_keys, 0); }

static int check_attn(const TfhAttnStep& a, int64_t ld_raw) {
    if (!a.q_norm || !a.k_norm || !a.cache || !a.table || !a.ws || a.n_pages < 1 || a.n_pages > (1 << 30) || a.table_ld < 1) return TF_EINVAL;
    if (a.H < 1 || a.G < 1 || a.H % a.G || a.D < 32 || (a.D & 31) || a.D_real < 1 || a.D_real > a.D || a.V < 32 || (a.V & 31)) return TF_EINVAL;
    if (a.half < 0 || 2 * a.half > a.D_real || a.max_pos < 1 || (a.half && (!a.cos || !a.sin)) || a.chunk < 0 || a.nsplit < 1
        || a.nsplit > TFH_MAX_SPLIT) return TF_EINVAL;
    if (a.q_off < 0 || a.k_off < 0 || a.v_off < 0 || a.gate_off < 0 || (a.gate_off & 3) || ld_raw < a.q_off + (int64_t)a.H * a.D
        || ld_raw < a.k_off + (int64_t)a.G * a.D || ld_raw < a.v_off + (int64_t)a.G * a.V || ld_raw < a.gate_off + (int64_t)a.H * a.V) return TF_EINVAL;
    return a.D > 256 || a.V > 256 ? TF_ERANGE : TF_OK;
}

static int check_rec(const TfhRecStep& a, int64_t ld_raw) {
    if (!a.state || !a.seat || !a.out || !a.norm_w || a.seats < 1 || a.H < 1 || a.per_group < 1 || a.H % a.per_group || a.N < 32 || (a.N & 31)
        || a.V < 32 || (a.V & 31) || a.V_real < 1 || a.V_real > a.V || a.norm_groups < 1 || (int64_t)a.H * a.V_real % a.norm_groups) return TF_EINVAL;
    if (a.gate_off < 0 || ld_raw < a.gate_off + (int64_t)a.H * a.V) return TF_EINVAL;
    if (a.a2) {
        if (!a.a2_b || a.rank < 4 || (a.rank & 3) || (a.a_off & 3) || a.q_off < 0 || a.k_off < 0 || a.v_off < 0 || a.a_off < 0 || ld_raw < a.q_off + (int64_t)a.H * a.N
            || ld_raw < a.k_off + (int64_t)a.H * a.N || ld_raw < a.v_off + (int64_t)a.H * a.V || ld_raw < a.a_off + (int64_t)a.rank
            || a.per_group != 1 || a.norm_groups != a.H) return TF_EINVAL;
    } else {
        if (!a.conv_w || !a.conv_b || !a.ring || !a.dt_bias || !a.nega || !a.skip || a.taps < 1 || a.x_off < 0 || a.dt_off < 0
            || a.channels != a.H * a.V + 2 * (a.H / a.per_group) * a.N || ld_raw < a.x_off + (int64_t)a.channels
            || ld_raw < a.dt_off + (int64_t)a.H) return TF_EINVAL;
    }
    return a.N > 1024 ? TF_ERANGE : TF_OK;
}

static size_t step_lds(int dtype, const TfhAttnStep* a, const TfhRecStep* r) {
    size_t need = r ? sizeof(float) * (3 * (size_t)r->N + 64 + 1024) : 0;
    if (a) {
        const size_t e = dtype ? 4 : 2, epv = 16 / e, parts = dtype ? 1 : 2;
        const size_t at = e * (64 * (a->D + epv) + 64 * (a->V + 2 * epv) + 16 * (a->D + epv) + parts * 16 * (64 + epv)) + 4 * 64 * sizeof(float);
        if (at > need) need = at;
    }
    return need;
}

template <typename T, int NTW, int DK, int DV>
static int launch_step(const AttnStep& a, const TfhRecStep& r, int attn_blocks, int rec_blocks, int slice, size_t lds, const float* raw,
                       int64_t ld_raw, const int32_t* klen, int rows, float eps, hipStream_t st) {
    auto k = step_kernel<T, NTW, DK, DV>;
    static bool attr = false;
    if (!attr) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        attr = true;
    }
    if constexpr (DK > 0) lds = SizedStep<DK, DV>::LDS > lds ? SizedStep<DK, DV>::LDS : lds;
    hipLaunchKernelGGL(k, dim3((unsigned)((int64_t)(attn_blocks + rec_blocks) * rows)), dim3(256), lds, st, a, r, attn_blocks * rows, rec_blocks, slice, rows, raw, ld_raw, klen, eps);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tfh_step(const TfhAttnStep* pa, const TfhRecStep* pr, const float* raw, int64_t ld_raw, const int32_t* klen, int rows, float eps,
                        int dtype, void* stream) {
    if ((!pa && !pr) || !raw || !klen || rows < 1 || rows > 65535 || (ld_raw & 3) || (dtype != 0 && dtype != 1)) return TF_EINVAL;
    AttnStep a = {};
    TfhRecStep r = {};
    int ab = 0, rb = 0, slice = 64, rc;
    if (pa) {
        static_cast<TfhAttnStep&>(a) = *pa;
        a.slots = rows * a.nsplit;
        if ((rc = check_attn(a, ld_raw)) != TF_OK) return rc;
        ab = a.G * ((a.H / a.G + 15) / 16) * a.nsplit;
    }
    if (pr) {
        r = *pr;
        if ((rc = check_rec(r, ld_raw)) != TF_OK) return rc;
        while (slice > 16 && (int64_t)rows * r.H * ((r.V + slice - 1) / slice) < 256) slice /= 2;      // (fill the chip)
        rb = r.H * ((r.V + slice - 1) / slice);
    }
    hipStream_t st = (hipStream_t)stream;
#define GO(T, NTW, DK, DV) return launch_step<T, NTW, DK, DV>(a, r, ab, rb, slice, lds, raw, ld_raw, klen, rows, eps, st)
    if (pa && sized_step(a.D, a.V, dtype)) {
        const size_t lds = step_lds(dtype, nullptr, pr);
        if (a.D == 64) GO(bf16, 1, 2, 4);
        GO(bf16, 2, 4, 8);
    }
    const size_t lds = step_lds(dtype, pa, pr);
    if (lds > 160 * 1024) return TF_ERANGE;
    const int V = pa ? a.V : 32;
    if (dtype == 0) {
        if (V <= 64) GO(bf16, 1, 0, 0);
        if (V <= 128) GO(bf16, 2, 0, 0);
        GO(bf16, 4, 0, 0);
    }
    if (V <= 64) GO(float, 1, 0, 0);
    if (V <= 128) GO(float, 2, 0, 0);
    GO(float, 4, 0, 0);
#undef GO
}

extern "C" int tfh_step_out(const TfhAttnStep* pa, const TfhRecStep* pr, const float* raw, int64_t ld_raw, void* act, int64_t ld_act,
                            int64_t act_oct, int rows, float eps, int dtype, void* stream) {
    if ((!pa && !pr) || !raw || !act || rows < 1 || rows > 65535 || (ld_raw & 3) || ld_act < 8 || (ld_act & 7) || act_oct < 8 || (act_oct & 7)
        || (dtype != 0 && dtype != 1)) return TF_EINVAL;
    AttnStep a = {};
    TfhRecStep r = {};
    int ab = 0, groups = 0, rc;
    if (pa) {
        static_cast<TfhAttnStep&>(a) = *pa;
        a.slots = rows * a.nsplit;
        if ((rc = check_attn(a, ld_raw)) != TF_OK) return rc;
        ab = a.H;
    }
    if (pr) {
        r = *pr;
        if ((rc = check_rec(r, ld_raw)) != TF_OK) return rc;
        groups = r.norm_groups;
    }
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid(ab + groups, rows);
    if (dtype == 0) hipLaunchKernelGGL((step_out_kernel<bf16>), grid, dim3(256), 0, st, a, r, ab, groups, raw, ld_raw, (bf16*)act, ld_act, act_oct, eps);
    else hipLaunchKernelGGL((step_out_kernel<float>), grid, dim3(256), 0, st, a, r, ab, groups, raw, ld_raw, (float*)act, ld_act, act_oct, eps);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}
