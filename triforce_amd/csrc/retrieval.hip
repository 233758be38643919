// Retrieval-cache build and KV row movement for gfx950.
//
// Replaces RetrievalCache.init_graph_cache (models/cache.py:146-178; distributed twin :517-556):
//   chunk_k = K[:prefill].view(C, chunk, H, D).mean(dim=-3)            -> tf_retrieval_score
//   chunk_attn = q @ chunk_k^T   (fp16, un-scaled)                      -> tf_retrieval_score
//   topk(chunk_attn[:, :, 1:], k = sets-1) + 1, chunk 0 prepended       -> tf_retrieval_topk
//   gather of whole chunks for K and V                                  -> tf_retrieval_gather
// and RetrievalCache.update_graph_cache / StreamingLLMEvictionCache.evict_* (cache.py:180-182,
// 252-265) -> tf_kv_copy_rows / tf_kv_shift_rows.
//
// All of it is HBM-bound byte work: K is streamed exactly once (16-B loads, 256-B row segments
// per 16-lane group), nothing is staged in a temporary, the top-k runs in LDS.
#include "common.h"

#include <type_traits>

#ifndef TF_RSCORE_CAP_CEIL
#define TF_RSCORE_CAP_CEIL 0
#endif

// ---- scoring ------------------------------------------------------------------------------
// One 16-lane group per chunk (a wave scores 4 chunks per step); lane (c4, li) owns 8 d's.
// Rounding points follow the reference: mean -> fp16, dot -> fp16.
template <int D>
__global__ __launch_bounds__(256) void retrieval_score_kernel(const h16* __restrict__ k, int64_t stride_t,
                                                              int64_t stride_h, const h16* __restrict__ q,
                                                              h16* __restrict__ scores, int C, int chunk) {
    static_assert(D == 128 || D == 64, "head_dim");
    constexpr int LPR = D / 8;                   // lanes per row (16 for D=128, 8 for D=64)
    constexpr int GPB = 256 / LPR;               // chunk groups per block
    const int h = blockIdx.y;
    const int grp = threadIdx.x / LPR, li = threadIdx.x % LPR;
    const h16* kb = k + (int64_t)h * stride_h + 8 * li;
    float qf[8];
    {
        const half8 qv = load_half8(q + (int64_t)h * D + 8 * li);
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[e] = (float)qv[e];
    }
    const float inv = 1.0f / (float)chunk;
    for (int c = blockIdx.x * GPB + grp; c < C; c += gridDim.x * GPB) {
        float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        const h16* kp = kb + (int64_t)c * chunk * stride_t;
        for (int r = 0; r < chunk; ++r) {          // sequential fp32 accumulation over the chunk rows
            const half8 kv = load_half8_stream(kp + (int64_t)r * stride_t);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += (float)kv[e];
        }
        float dot = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const h16 mean = (h16)(acc[e] * inv);    // chunk mean rounded to fp16 (cache.py:154)
            dot = fmaf(qf[e], (float)mean, dot);
        }
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) dot += __shfl_xor(dot, o, 64);
        if (li == 0) scores[(int64_t)h * C + c] = (h16)dot;
    }
}

// The same for chunks of CH rows (known at compile time): a group's next chunk is requested before the current one is summed up, so
// that a few resident waves keep the stream going.  A plain read is fastest on this chip with about 32 KB in flight per CU and loses
// 10-25 % at half or at several times that; the general kernel above holds 8 workgroups per CU with 8 KB per wave.
template <int D, int CH>
__global__ __launch_bounds__(256) void retrieval_score_ahead_kernel(const h16* __restrict__ k, int64_t stride_t,
                                                                    int64_t stride_h, const h16* __restrict__ q,
                                                                    h16* __restrict__ scores, int C) {
    constexpr int LPR = D / 8, GPB = 256 / LPR;
    const int h = blockIdx.y;
    const int grp = threadIdx.x / LPR, li = threadIdx.x % LPR;
    const h16* kb = k + (int64_t)h * stride_h + 8 * li;
    float qf[8];
    {
        const half8 qv = load_half8(q + (int64_t)h * D + 8 * li);
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[e] = (float)qv[e];
    }
    const float inv = 1.0f / (float)CH;
    const int step = gridDim.x * GPB;
    auto fetch = [&](half8 (&r)[CH], int c) {                    // (past the end: the last chunk again, not used)
        const h16* kp = kb + (int64_t)min(c, C - 1) * CH * stride_t;
#pragma unroll
        for (int j = 0; j < CH; ++j) r[j] = load_half8_stream(kp + (int64_t)j * stride_t);
    };
    auto score = [&](const half8 (&r)[CH], int c) {
        float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < CH; ++j) {                           // sequential fp32 accumulation over the chunk rows
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += (float)r[j][e];
        }
        float dot = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = fmaf(qf[e], (float)(h16)(acc[e] * inv), dot);
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) dot += __shfl_xor(dot, o, 64);
        if (li == 0 && c < C) scores[(int64_t)h * C + c] = (h16)dot;
    };
    half8 a[CH], b[CH];
    const int c0 = blockIdx.x * GPB;                             // (uniform bound: the waves of a workgroup go together)
    fetch(a, c0 + grp);
    for (int c = c0; c < C; c += 2 * step) {
        fetch(b, c + grp + step);
        score(a, c + grp);
        if (c + step >= C) break;
        fetch(a, c + grp + 2 * step);
        score(b, c + grp + step);
    }
}

// ---- per-head top-k: full bitonic sort of (score, chunk) keys in LDS ------------------------
__device__ __forceinline__ uint32_t sortable_fp16(uint32_t b) {
    return (b & 0x8000u) ? ((~b) & 0xFFFFu) : (b | 0x8000u);
}

__global__ __launch_bounds__(1024) void retrieval_topk_kernel(const uint16_t* __restrict__ scores,
                                                               int32_t* __restrict__ idx, int C, int sets,
                                                               int npow2) {
    extern __shared__ uint32_t keys[];
    const int h = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const uint16_t* sc = scores + (int64_t)h * C;
    // candidates are chunks 1..C-1; key = sortable(score) << 16 | (65535 - chunk): descending key
    // order == descending score, ascending chunk among equal scores.  Padding sorts last.
    for (int i = tid; i < npow2; i += nt) {
        const int c = i + 1;
        keys[i] = (c < C) ? ((sortable_fp16(sc[c]) << 16) | (uint32_t)(65535 - (c & 0xFFFF))) : 0u;
    }
    __syncthreads();
    for (int kk = 2; kk <= npow2; kk <<= 1) {
        for (int j = kk >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < npow2; i += nt) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const bool desc = ((i & kk) == 0);
                    const uint32_t a = keys[i], b = keys[ixj];
                    if ((a < b) == desc) {
                        keys[i] = b;
                        keys[ixj] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
    int32_t* out = idx + (int64_t)h * sets;
    if (tid == 0) out[0] = 0;
    for (int i = tid; i < sets - 1; i += nt) out[1 + i] = 65535 - (int32_t)(keys[i] & 0xFFFFu);
}

// ---- per-head top-k, select-then-sort form ---------------------------------------------------
// The keys are distinct 32-bit integers, so the m-th largest one is found EXACTLY by a radix select (integer histograms in LDS:
// deterministic), the m keys >= it are compacted and only those are sorted.  Same output, bit for bit, as the full sort.
//
// One workgroup per head; a latency chain, not a bandwidth one (15 615 keys are 31 KB), so every serial piece is what counts:
//   * the keys stay in registers (NK a thread), all asked for at once;
//   * digits of 11 / 11 / 10 bits: 2 048 bins spread a head's scores (an fp16's sign, exponent and five mantissa bits) where 256 bins made
//     the waves queue on a handful of LDS counters;
//   * the bin that holds the m-th key is found by one wave with two 64-wide scans, in registers;
//   * as soon as that bin holds kTopkNear keys at most (nearly always after the first digit: some 65 of 15 615 normal scores) they are ranked
//     against each other, instead of two more passes over all keys; more of them, and a pass costs less than the ranks;
//   * a wave counts what it keeps by ballots and takes its places with one atomic;
//   * bitonic stages below 64 exchange inside a wave, without LDS; the others alternate between two buffers, one barrier each.
// 32 heads x 15 616 chunks, m = 511: 46.9 us as one sort, 17.0 with three passes over keys in LDS and exchanges through it, 10.7 now; scores that need
// a second digit 19.5 -> 14.4; 32 x 4 000 12.6 -> 7.9, 32 x 1 000 (m = 255) 9.4 -> 6.5, 32 x 32 768 23.7 -> 16.7, 8 x 20 000 (m = 4 095) 36.9 -> 31.1.
constexpr int kTopkBins = 2048, kTopkNear = 256;
__device__ __forceinline__ int topk_bin(int b) { return b + (b >> 5); }      // (a lane sums 32 neighbouring bins: no bank twice)

template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ uint32_t lane_dpp(uint32_t v) {       // 0 from outside
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
// Inclusive sums over the lanes of a wave: 1, 2, 4, 8 places within a row of 16, then a row's last lane for the rows behind it.
__device__ __forceinline__ int lanes_scan(int v) {
    v += lane_dpp<0x111>(v);
    v += lane_dpp<0x112>(v);
    v += lane_dpp<0x114>(v);
    v += lane_dpp<0x118>(v);
    v += lane_dpp<0x142, 0xa>(v);
    v += lane_dpp<0x143, 0xc>(v);
    return v;
}
// The larger and the smaller key of lanes l and l ^ J.
template <int J> __device__ __forceinline__ LanePair<uint32_t> lane_order(uint32_t v) {
    uint32_t b;
    if constexpr (J == 32 || J == 16) {
        const LanePair<uint32_t> p = J == 32 ? lane_halves(v) : lane_rows(v);
        return {max(p.a, p.b), min(p.a, p.b)};
    } else if constexpr (J == 8) {
        b = lane_rotated<8>(v);
    } else if constexpr (J == 4) {
        b = lane_dpp<0x1b>(lane_dpp<0x141>(v));                          // l ^ 7 (a half row mirrored), then ^ 3
    } else {
        b = lane_dpp<J == 2 ? 0x4e : 0xb1>(v);
    }
    return {max(v, b), min(v, b)};
}

// The digit (of `bins` of them) at which the count from the top reaches `rem`, the keys in its bin and what is left to find among them.  One wave.
__device__ __forceinline__ void topk_digit(const int* hist, int bins, int rem, int lane, int* digit, int* keys, int* left) {
    const int per = bins >> 6;                                           // 32 or 16
    int own = 0;
#pragma unroll 8
    for (int j = 0; j < per; ++j) own += hist[topk_bin(bins - 1 - (lane * per + j))];
    const int upto = lanes_scan(own);                                    // inclusive count of the lanes before (higher digits)
    const int owner = __ffsll((long long)__ballot(upto >= rem)) - 1;     // (rem <= keys in the histogram: some lane reaches it)
    const int before = __builtin_amdgcn_readlane(upto - own, owner);
    const int cnt = lane < per ? hist[topk_bin(bins - 1 - (owner * per + lane))] : 0;
    const int in = lanes_scan(cnt);
    const int at = __ffsll((long long)__ballot(before + in >= rem)) - 1;
    *digit = bins - 1 - (owner * per + at);
    *keys = __builtin_amdgcn_readlane(cnt, at);
    *left = rem - before - __builtin_amdgcn_readlane(in - cnt, at);
}

// E = winners per thread (the sort's size / 1024, at least 1): element e * 1024 + tid sits in register e of thread tid, so stages
// below 64 are lane exchanges, stages of 1024 and more are register exchanges and only those between go through LDS.
// NK = keys per thread (n <= 1024 * NK).
template <int E, int NK>
__global__ __launch_bounds__(1024) void retrieval_topk_select_kernel(const uint16_t* __restrict__ scores,
                                                                      int32_t* __restrict__ idx, int C, int sets,
                                                                      int n, int mpow2) {
    extern __shared__ uint32_t sel[];        // [2][mpow2] the winners
    __shared__ __align__(16) int hist[kTopkBins + kTopkBins / 32];
    __shared__ uint32_t s_prefix;
    __shared__ int s_remaining, s_keys, s_count;
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    constexpr int nt = 1024;
    const uint16_t* sc = scores + (int64_t)h * C;
    const int m = sets - 1;
    int32_t* out = idx + (int64_t)h * sets;
    if (tid == 0) out[0] = 0;
    if (m == 0) return;
    uint32_t key[NK];                                                    // of chunks 1..C-1; 0 behind the last (no key is 0)
#pragma unroll
    for (int u = 0; u < NK; ++u) key[u] = sc[min(tid + u * nt, n - 1) + 1];
    for (int i = tid + m; i < mpow2; i += nt) sel[i] = 0u;               // padding sorts last
    if (tid == 0) { s_remaining = m; s_count = 0; }
    uint32_t prefix = 0u, known = 0u, open = 0u;                         // the bits of the m-th key found so far, and those to find
    int keys = 0, left = 0;                                              // with these bits, and how many of them win
#pragma unroll
    for (int pass = 0; pass < 3; ++pass) {
        const int shift = pass == 0 ? 21 : (pass == 1 ? 10 : 0), bins = pass == 2 ? 1024 : kTopkBins;
        for (int i = tid; i < kTopkBins + kTopkBins / 32; i += nt) hist[i] = 0;
        __syncthreads();
        if (pass == 0) {
#pragma unroll
            for (int u = 0; u < NK; ++u) {
                const int i = tid + u * nt;
                key[u] = i < n ? (sortable_fp16(key[u]) << 16) | (uint32_t)(65535 - ((i + 1) & 0xFFFF)) : 0u;
            }
        }
#pragma unroll
        for (int u = 0; u < NK; ++u)
            if (key[u] && (key[u] & known) == prefix) atomicAdd(&hist[topk_bin((key[u] >> shift) & (bins - 1))], 1);
        __syncthreads();
        if (tid < 64) {
            int digit, in, rest;
            topk_digit(hist, bins, s_remaining, lane, &digit, &in, &rest);
            if (tid == 0) {
                s_remaining = rest;
                s_keys = in;
                s_prefix = prefix | ((uint32_t)digit << shift);
            }
        }
        __syncthreads();
        prefix = s_prefix;
        known |= (uint32_t)(bins - 1) << shift;
        open = (1u << shift) - 1u;
        keys = s_keys;
        left = s_remaining;
        if (keys <= kTopkNear) break;                                    // (the last digit leaves one key: keys are distinct)
    }
    uint32_t* near = reinterpret_cast<uint32_t*>(hist);                  // [keys], zeros up to a multiple of 16 (the counts are used up)
    if (tid < 16) near[keys + tid] = 0u;
    const uint32_t least = max(prefix, 1u), most = prefix | open;        // keys above `most` win, m - left of them
    uint32_t total = 0;                                                  // of this wave: winners, and keys of the bin << 16
#pragma unroll
    for (int u = 0; u < NK; ++u)
        total += (uint32_t)__popcll(__ballot(key[u] > most)) + ((uint32_t)__popcll(__ballot(key[u] >= least && key[u] <= most)) << 16);
    uint32_t at = 0;
    if (lane == 0 && total) at = (uint32_t)atomicAdd(&s_count, (int)total);
    at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    uint32_t at_sel = at & 0xFFFFu, at_near = at >> 16;
    auto below = [](uint64_t b) { return (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u)); };
#pragma unroll
    for (int u = 0; u < NK; ++u) {
        const bool wins = key[u] > most, in = key[u] >= least && key[u] <= most;
        const uint64_t bw = __ballot(wins), bi = __ballot(in);
        if (wins) sel[at_sel + below(bw)] = key[u];
        if (in) near[at_near + below(bi)] = key[u];
        at_sel += (uint32_t)__popcll(bw);
        at_near += (uint32_t)__popcll(bi);
    }
    __syncthreads();
    if (tid < keys) {
        const uint32_t own = near[tid];
        int rank = 0;
        for (int j = 0; j < keys; j += 16) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint4 v = *reinterpret_cast<const uint4*>(near + j + 4 * e);
                rank += (int)(v.x > own) + (int)(v.y > own) + (int)(v.z > own) + (int)(v.w > own);
            }
        }
        if (rank < left) sel[m - left + rank] = own;
    }
    __syncthreads();
    uint32_t v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = e * nt + tid < mpow2 ? sel[e * nt + tid] : 0u;
    uint32_t* spare = sel + mpow2;           // a stage's buffer: written before its barrier and read behind it, the next stage takes the other
    for (int kk = 2; kk <= mpow2; kk <<= 1) {
        int j = kk >> 1;
        if constexpr (E > 1) {
            for (; j >= nt; j >>= 1) {                                   // both elements of a pair sit in this thread
                const int je = j / nt;
#pragma unroll
                for (int e = 0; e < E; ++e) {
#pragma unroll
                    for (int f = e + 1; f < E; ++f) {
                        if ((e ^ f) == je) {
                            const bool desc = ((e * nt + tid) & kk) == 0;
                            const uint32_t a = v[e], b = v[f];
                            v[e] = (a < b) == desc ? b : a;
                            v[f] = (a < b) == desc ? a : b;
                        }
                    }
                }
            }
        }
        for (; j >= 64; j >>= 1) {                                       // other waves hold the partners
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (e * nt + tid < mpow2) spare[e * nt + tid] = v[e];
            __syncthreads();
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = e * nt + tid;
                if (i < mpow2) {
                    const uint32_t b = spare[i ^ j];
                    const bool larger = ((i & kk) == 0) == ((i & j) == 0);   // this place keeps the larger key of the pair
                    v[e] = larger ? max(v[e], b) : min(v[e], b);
                }
            }
            spare = spare == sel ? sel + mpow2 : sel;
        }
        if (tid < mpow2) {                                               // (whole waves: mpow2 is 64 at least)
            auto stage = [&](auto J) __attribute__((always_inline)) {
                constexpr int j = decltype(J)::value;
                if (kk > j)
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        const int i = e * nt + tid;
                        const LanePair<uint32_t> p = lane_order<j>(v[e]);
                        v[e] = ((i & kk) == 0) == ((i & j) == 0) ? p.a : p.b;
                    }
            };
            stage(std::integral_constant<int, 32>{});
            stage(std::integral_constant<int, 16>{});
            stage(std::integral_constant<int, 8>{});
            stage(std::integral_constant<int, 4>{});
            stage(std::integral_constant<int, 2>{});
            stage(std::integral_constant<int, 1>{});
        }
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
        if (e * nt + tid < m) out[1 + e * nt + tid] = 65535 - (int32_t)(v[e] & 0xFFFFu);
}

// ---- gather ---------------------------------------------------------------------------------
// One 128-thread workgroup per (slot, head, K | V): a 2-KiB chunk, one 16-byte vector per thread.  Bound by the mixed stream, not by loads in
// flight: whole lines that nobody reads soon are written past the caches, whose place the reads keep.  32 heads x 512 chunks of 15 616 (67 MB read and
// 67 written, four layers in turn) plain -> this way 29.3 -> 22.2 us (6.0 TB/s; behind a build's scores 29.3 -> 25.4), 1 536 chunks, two layers 39.4 -> 34.1, 32 x 256 of 1 000
// 12.3 -> 10.1, 5 x 513 of 5 003 10.2 -> 8.9, one layer from the caches 4.5 -> 4.3 and 2.5 -> 2.2.  Reads past the caches instead 21.7, but 5.3 and
// 3.0 where the chunks are in them; both 23.3; two, four or eight slots a workgroup 20.5 to 30, the same order.
__global__ __launch_bounds__(128) void retrieval_gather_kernel(
    const h16* __restrict__ k_src, const h16* __restrict__ v_src, int64_t sst, int64_t ssh,
    const int32_t* __restrict__ idx, h16* __restrict__ k_dst, h16* __restrict__ v_dst, int64_t dst_t, int64_t dsh,
    int sets, int chunk, int D) {
    const int slot = blockIdx.x, h = blockIdx.y;
    const bool is_v = blockIdx.z != 0;
    const h16* src = (is_v ? v_src : k_src) + (int64_t)h * ssh;
    h16* dst = (is_v ? v_dst : k_dst) + (int64_t)h * dsh;
    const int c = idx[(int64_t)h * sets + slot];
    const int vec_per_row = D / 8;
    for (int e = threadIdx.x; e < chunk * vec_per_row; e += blockDim.x) {
        const int r = e / vec_per_row, dv = e - r * vec_per_row;
        const half8 x = load_half8(src + ((int64_t)c * chunk + r) * sst + 8 * dv);
        __builtin_nontemporal_store(x, reinterpret_cast<half8*>(dst + ((int64_t)slot * chunk + r) * dst_t + 8 * dv));
    }
}

// ---- row copies -----------------------------------------------------------------------------
// (blockIdx.z = 1: the second (src, dst) pair of the same geometry — K and V of one cache in one launch)
__global__ __launch_bounds__(256) void kv_copy_rows_kernel(const h16* __restrict__ src, int64_t ssl, int64_t sst,
                                                           int64_t ssh, h16* __restrict__ dst, int64_t dsl,
                                                           int64_t dst_t, int64_t dsh, int src_t0, int dst_t0, int n,
                                                           int H, int D, const h16* __restrict__ src2,
                                                           h16* __restrict__ dst2) {
    const int l = blockIdx.y / H, h = blockIdx.y % H;
    const h16* s = (blockIdx.z ? src2 : src) + (int64_t)l * ssl + (int64_t)h * ssh;
    h16* d = (blockIdx.z ? dst2 : dst) + (int64_t)l * dsl + (int64_t)h * dsh;
    const int vpr = D / 8;
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n * vpr; e += gridDim.x * blockDim.x) {
        const int r = e / vpr, dv = e - r * vpr;
        store_half8(d + (int64_t)(dst_t0 + r) * dst_t + 8 * dv, load_half8(s + (int64_t)(src_t0 + r) * sst + 8 * dv));
    }
}

// In-place downward shift (dst_t0 <= src_t0), overlap allowed: one workgroup per (layer, head)
// walks the rows in ascending blocks; inside a block every thread reads before anyone writes.
__global__ __launch_bounds__(256) void kv_shift_rows_kernel(h16* __restrict__ cache, int64_t sl, int64_t st,
                                                            int64_t sh, int src_t0, int dst_t0, int n, int H, int D,
                                                            h16* __restrict__ cache2) {
    const int l = blockIdx.x / H, h = blockIdx.x % H;
    h16* base = (blockIdx.y ? cache2 : cache) + (int64_t)l * sl + (int64_t)h * sh;
    const int vpr = D / 8;
    const int rows_per_blk = 256 / vpr;
    const int r_in = threadIdx.x / vpr, dv = threadIdx.x % vpr;
    for (int r0 = 0; r0 < n; r0 += rows_per_blk) {
        const int r = r0 + r_in;
        half8 x;
        const bool ok = (r < n) && (r_in < rows_per_blk);
        if (ok) x = load_half8(base + (int64_t)(src_t0 + r) * st + 8 * dv);
        __syncthreads();
        if (ok) store_half8(base + (int64_t)(dst_t0 + r) * st + 8 * dv, x);
        __syncthreads();
    }
}

// ---- C ABI ------------------------------------------------------------------------------------
extern "C" int tf_retrieval_score(const void* k, int64_t stride_t, int64_t stride_h, const void* q, void* scores,
                                  int C, int chunk, int H, int D, void* stream) {
    if (!k || !q || !scores || C < 1 || chunk < 1 || H < 1) return TF_EINVAL;
    if ((stride_t % 8) || (stride_h % 8)) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const int gpb = 256 / (D / 8);
    int gx = (C + gpb - 1) / gpb;
#if TF_RSCORE_CAP_CEIL
    const int cap = (2048 + H - 1) / H;              // round 1-3 rule: 2 080 workgroups at H = 40, 2 050 at H = 5
#else
    // 8 resident workgroups per CU and NOT ONE MORE: with ceil(2048 / H) the 32 (H = 40) or 2 (H = 5) workgroups past
    // 2 048 start when the others retire and stream their share alone, latency-bound (0.59 of peak at H = 40 against
    // 0.81 at H = 32, profiles/r03_bench_13b_cfg4_world1.json); grid-stride beyond
    const int cap = H <= 2048 ? 2048 / H : 1;
#endif
    if (gx > cap) gx = cap;
    if (gx < 1) gx = 1;
    if (D == 128 && chunk == 8) {
        // Workgroups per CU.  One (16 KB asked for ahead of 16 KB in use per wave quartet) is the best stream where every CU gets the
        // same share and enough of it to pay for its start: 32 x 15 616 chunks 158.3 us at the general kernel's 8, 155.4 at two,
        // 150.2 at one (6.81 TB/s); 40 heads (240 of 256 CUs with work) 198 / 194 / 199, 32 x 4 000 46.4 / 42.0 / 43.1,
        // 32 x 1 000 12.6 / 12.1 / 13.0, 5 x 5 003 10.3 / 10.3 / 11.0.
        const bool one = 256 % H == 0 && (int64_t)C * H >= (1 << 18);
        const int room = one ? 256 : 512, few = H <= room ? room / H : 1;
        // Three or four rounds and a little: the general kernel has every chunk on its way at once, a last round here is nearly a round
        // (32 x 800, 3.1 rounds, 9.9 us there against 10.5, 40 x 600 9.5 against 10.4, 64 x 450, 3.5 rounds, 11.0 against 11.7; 40 x 700, 3.6
        // rounds, 10.7 both; 32 x 600, 2.3 rounds, 8.4 and 8.7 from memory, 7.7 and 7.4 from the caches; more workgroups here 11.4 for 32 x 800).
        const int round = few * gpb, whole = C / round, rest = C - whole * round;
        const bool at_once = (int64_t)H * ((C + gpb - 1) / gpb) <= 2048 && whole >= 3 && rest > 0 && 5 * rest < 3 * round;
        if (!at_once) {
            hipLaunchKernelGGL((retrieval_score_ahead_kernel<128, 8>), dim3(gx < few ? gx : few, H), dim3(256), 0, st, (const h16*)k,
                               stride_t, stride_h, (const h16*)q, (h16*)scores, C);
            TF_LAUNCH_CHECK();
            return TF_OK;
        }
    }
    if (D == 128)
        hipLaunchKernelGGL((retrieval_score_kernel<128>), dim3(gx, H), dim3(256), 0, st, (const h16*)k, stride_t,
                           stride_h, (const h16*)q, (h16*)scores, C, chunk);
    else if (D == 64)
        hipLaunchKernelGGL((retrieval_score_kernel<64>), dim3(gx, H), dim3(256), 0, st, (const h16*)k, stride_t,
                           stride_h, (const h16*)q, (h16*)scores, C, chunk);
    else
        return TF_EINVAL;
    TF_LAUNCH_CHECK();
    return TF_OK;
}

template <int E, int NK>
static int launch_topk_select(const void* scores, int32_t* idx, int C, int sets, int H, int mpow2, void* stream) {
    const size_t lds = 2 * (size_t)mpow2 * sizeof(uint32_t);
    if (lds > 48 * 1024) {
        static bool raised = false;
        if (!raised) {
            hipError_t e = hipFuncSetAttribute((const void*)retrieval_topk_select_kernel<E, NK>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024);
            if (e != hipSuccess) return (int)e;
            raised = true;
        }
    }
    hipLaunchKernelGGL((retrieval_topk_select_kernel<E, NK>), dim3(H), dim3(1024), lds, (hipStream_t)stream,
                       (const uint16_t*)scores, idx, C, sets, C - 1, mpow2);
    TF_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tf_retrieval_topk(const void* scores, int32_t* idx, int C, int sets, int H, void* stream) {
    if (!scores || !idx || C < 2 || sets < 1 || sets > C || H < 1) return TF_EINVAL;
    if (C > 32768) return TF_ERANGE;
    // select-then-sort up to 8 192 winners (two buffers of them, 64 KB)
    int mpow2 = 64;
    while (mpow2 < sets - 1) mpow2 <<= 1;
    if (mpow2 <= 8192) {
#define GO(E, NK) return launch_topk_select<E, NK>(scores, idx, C, sets, H, mpow2, stream)
#define GO_N(E) do { if (C - 1 <= 8192) GO(E, 8); if (C - 1 <= 16384) GO(E, 16); GO(E, 32); } while (0)
        switch (mpow2 <= 1024 ? 1 : mpow2 / 1024) {
            case 1: GO_N(1);
            case 2: GO_N(2);
            case 4: GO_N(4);
            default: GO_N(8);
        }
#undef GO_N
#undef GO
    }
    int npow2 = 2;
    while (npow2 < C - 1) npow2 <<= 1;
    const size_t lds = (size_t)npow2 * sizeof(uint32_t);
    if (lds > 64 * 1024) {
        static bool raised = false;
        if (!raised) {
            hipError_t e = hipFuncSetAttribute((const void*)retrieval_topk_kernel,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
            if (e != hipSuccess) return (int)e;
            raised = true;
        }
    }
    hipLaunchKernelGGL(retrieval_topk_kernel, dim3(H), dim3(1024), lds, (hipStream_t)stream,
                       (const uint16_t*)scores, idx, C, sets, npow2);
    TF_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tf_retrieval_gather(const void* k_src, const void* v_src, int64_t src_stride_t, int64_t src_stride_h,
                                   const int32_t* idx, void* k_dst, void* v_dst, int64_t dst_stride_t,
                                   int64_t dst_stride_h, int sets, int chunk, int H, int D, void* stream) {
    if (!k_src || !v_src || !idx || !k_dst || !v_dst || sets < 1 || chunk < 1 || H < 1 || (D % 8)) return TF_EINVAL;
    if ((src_stride_t % 8) || (src_stride_h % 8) || (dst_stride_t % 8) || (dst_stride_h % 8)) return TF_EINVAL;
    hipLaunchKernelGGL(retrieval_gather_kernel, dim3(sets, H, 2), dim3(128), 0, (hipStream_t)stream,
                       (const h16*)k_src, (const h16*)v_src, src_stride_t, src_stride_h, idx, (h16*)k_dst, (h16*)v_dst,
                       dst_stride_t, dst_stride_h, sets, chunk, D);
    TF_LAUNCH_CHECK();
    return TF_OK;
}

// Compaction of accepted tree nodes (DistributedSimpleCache.gather_kv_incremental, models/cache.py:333-343):
// rows offset + idx[j] -> offset + j for j in [0, n), K and V, every layer and head.  idx must be strictly
// increasing (a root-to-leaf path of the Sequoia tree: node ids grow with depth), so idx[j] >= j and walking the
// rows in ascending batches with read-all / barrier / write-all is overlap-safe without the reference's clone().
__global__ __launch_bounds__(256) void kv_gather_rows_kernel(h16* __restrict__ kc, h16* __restrict__ vc, int64_t sl,
                                                             int64_t st, int64_t sh, int offset,
                                                             const int32_t* __restrict__ idx, int n, int H, int D) {
    const int l = blockIdx.x / H, h = blockIdx.x % H;
    h16* base = (blockIdx.y ? vc : kc) + (int64_t)l * sl + (int64_t)h * sh;
    const int vpr = D / 8;
    const int rows_per_blk = 256 / vpr;
    const int r_in = threadIdx.x / vpr, dv = threadIdx.x % vpr;
    for (int r0 = 0; r0 < n; r0 += rows_per_blk) {
        const int r = r0 + r_in;
        half8 x;
        const bool ok = (r < n) && (r_in < rows_per_blk);
        if (ok) x = load_half8(base + (int64_t)(offset + idx[r]) * st + 8 * dv);
        __syncthreads();
        if (ok) store_half8(base + (int64_t)(offset + r) * st + 8 * dv, x);
        __syncthreads();
    }
}

extern "C" int tf_kv_gather_rows(void* k_cache, void* v_cache, int64_t stride_l, int64_t stride_t, int64_t stride_h,
                                 int offset, const int32_t* idx, int n, int L, int H, int D, void* stream) {
    if (!k_cache || !v_cache || !idx || n < 1 || offset < 0 || L < 1 || H < 1 || D < 8 || (D % 8) || D > 2048)
        return TF_EINVAL;
    hipLaunchKernelGGL(kv_gather_rows_kernel, dim3(L * H, 2), dim3(256), 0, (hipStream_t)stream, (h16*)k_cache,
                       (h16*)v_cache, stride_l, stride_t, stride_h, offset, idx, n, H, D);
    TF_LAUNCH_CHECK();
    return TF_OK;
}

static int kv_copy_rows_launch(const void* src, const void* src2, int64_t src_stride_l, int64_t src_stride_t,
                               int64_t src_stride_h, void* dst, void* dst2, int64_t dst_stride_l, int64_t dst_stride_t,
                               int64_t dst_stride_h, int src_t0, int dst_t0, int n, int L, int H, int D, void* stream) {
    if (n == 0) return TF_OK;
    if (!src || !dst || n < 0 || L < 1 || H < 1 || (D % 8) || src_t0 < 0 || dst_t0 < 0) return TF_EINVAL;
    if ((src_stride_t % 8) || (src_stride_h % 8) || (src_stride_l % 8) || (dst_stride_t % 8) || (dst_stride_h % 8) ||
        (dst_stride_l % 8))
        return TF_EINVAL;
    int gx = (n * (D / 8) + 255) / 256;
    if (gx > 64) gx = 64;
    hipLaunchKernelGGL(kv_copy_rows_kernel, dim3(gx, L * H, src2 ? 2 : 1), dim3(256), 0, (hipStream_t)stream,
                       (const h16*)src, src_stride_l, src_stride_t, src_stride_h, (h16*)dst, dst_stride_l, dst_stride_t,
                       dst_stride_h, src_t0, dst_t0, n, H, D, (const h16*)src2, (h16*)dst2);
    TF_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tf_kv_copy_rows(const void* src, int64_t src_stride_l, int64_t src_stride_t, int64_t src_stride_h,
                               void* dst, int64_t dst_stride_l, int64_t dst_stride_t, int64_t dst_stride_h,
                               int src_t0, int dst_t0, int n, int L, int H, int D, void* stream) {
    return kv_copy_rows_launch(src, nullptr, src_stride_l, src_stride_t, src_stride_h, dst, nullptr, dst_stride_l,
                               dst_stride_t, dst_stride_h, src_t0, dst_t0, n, L, H, D, stream);
}

// K and V rows of one cache pair in ONE launch (same strides and row ranges for both): the decode step's tail copies
extern "C" int tf_kv_copy_rows_pair(const void* src_k, const void* src_v, int64_t src_stride_l, int64_t src_stride_t,
                                    int64_t src_stride_h, void* dst_k, void* dst_v, int64_t dst_stride_l,
                                    int64_t dst_stride_t, int64_t dst_stride_h, int src_t0, int dst_t0, int n, int L, int H,
                                    int D, void* stream) {
    if (n != 0 && (!src_v || !dst_v)) return TF_EINVAL;
    return kv_copy_rows_launch(src_k, src_v, src_stride_l, src_stride_t, src_stride_h, dst_k, dst_v, dst_stride_l,
                               dst_stride_t, dst_stride_h, src_t0, dst_t0, n, L, H, D, stream);
}

static int kv_shift_rows_launch(void* cache, void* cache2, int64_t stride_l, int64_t stride_t, int64_t stride_h,
                                int src_t0, int dst_t0, int n, int L, int H, int D, void* stream) {
    if (n == 0 || src_t0 == dst_t0) return TF_OK;
    if (!cache || n < 0 || L < 1 || H < 1 || (D % 8) || D > 2048 || dst_t0 > src_t0 || dst_t0 < 0) return TF_EINVAL;
    if ((stride_t % 8) || (stride_h % 8) || (stride_l % 8)) return TF_EINVAL;
    hipLaunchKernelGGL(kv_shift_rows_kernel, dim3(L * H, cache2 ? 2 : 1), dim3(256), 0, (hipStream_t)stream, (h16*)cache,
                       stride_l, stride_t, stride_h, src_t0, dst_t0, n, H, D, (h16*)cache2);
    TF_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tf_kv_shift_rows(void* cache, int64_t stride_l, int64_t stride_t, int64_t stride_h, int src_t0,
                                int dst_t0, int n, int L, int H, int D, void* stream) {
    return kv_shift_rows_launch(cache, nullptr, stride_l, stride_t, stride_h, src_t0, dst_t0, n, L, H, D, stream);
}

extern "C" int tf_kv_shift_rows_pair(void* k_cache, void* v_cache, int64_t stride_l, int64_t stride_t, int64_t stride_h,
                                     int src_t0, int dst_t0, int n, int L, int H, int D, void* stream) {
    if (n != 0 && src_t0 != dst_t0 && !v_cache) return TF_EINVAL;
    return kv_shift_rows_launch(k_cache, v_cache, stride_l, stride_t, stride_h, src_t0, dst_t0, n, L, H, D, stream);
}
