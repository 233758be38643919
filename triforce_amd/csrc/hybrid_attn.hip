// Prefill attention of the hybrid family: grouped-query flash attention over the paged cache with chunked visibility (key j is seen
// by query i only inside the same chunk of positions).
//
// Keys and values of 128 in bfloat16: attn_chunk_sized_kernel on the loop of flash_tile.h; a tile is a page.  Anything else: attn_chunk_kernel,
// 16 query rows per wave, the waves of a workgroup share a 64-key tile; scores are computed transposed, so the result registers of two 16-key
// tiles are the weight operand of one value product.
// A workgroup starts at the chunk of its first query, so keys of earlier chunks are never read.
#include "flash_tile.h"
#include "hybrid_common.h"

// Workgroups go round-robin over the 8 XCDs: the query blocks of a key / value head stay on one of them (its heads side by side), the last
// blocks of all sequences and heads first (sequence by sequence six of 222 to 1 333 rows take 82 us, not 73).  That reads every key once per
// query block from wherever it lies: with more keys than the caches keep for it (2^18 visible keys times key / value heads, 128 MB) and more
// than one round of workgroups (the caller's by_seq) the order is sequence by sequence, a block's heads side by side: 32 heads on 32, 16 x
// 1 333 rows behind 2 000 keys 1 668 -> 1 299 us, 32 x 700 behind 500 723 -> 550; 8 on 2, 32 x 700 behind 4 096 552 -> 522.  32 heads on 8, against
// workgroups of 256 rows with tiles staged in registers, head by head: 4 096 rows 276 -> 197 us, 3 904 behind 4 096 531 -> 478 (810
// TFLOP/s), 4 096 behind 6 000 with a chunk's edge at 8 192 569 -> 453, 6 x 1 000 behind 500 in chunks of 640 140 -> 94.
__global__ __launch_bounds__(256, 2) void attn_chunk_sized_kernel(const bf16* __restrict__ q, int64_t ld_q, const bf16* __restrict__ cache, int n_pages,
                                                                  const int32_t* __restrict__ table, int table_ld, const int32_t* __restrict__ seq,
                                                                  const bf16* __restrict__ gate, int64_t ld_gate, bf16* __restrict__ out,
                                                                  int64_t ld_out, int tokens, int H, int G, int chunk, float scale, float out_scale,
                                                                  int nseq, int by_seq) {
    typedef FlashTile<0, 4> Flash;
    constexpr int D = 128, QB = Flash::ROWS, KT = Flash::KT;
    extern __shared__ __align__(16) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, i = lane & 15;
    if (by_seq) {                                             // (the lengths are on the device: every wave adds them up)
        int64_t keys = 0;
        for (int s = lane; s < nseq; s += 64) keys += max(0, seq[4 * s + 1]) + max(0, chunk > 0 ? seq[4 * s + 2] % chunk : seq[4 * s + 2]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) keys += __shfl_xor(keys, o, 64);
        by_seq = __builtin_amdgcn_readfirstlane(keys * G >= 1 << 18);     // (scalar, and with it every tile address)
    }
    const bool by_xcd = (H & 7) == 0;
    const int hx = by_xcd ? H >> 3 : H, at = by_xcd ? blockIdx.x >> 3 : blockIdx.x;      // the XCD's own workgroups, in order
    const SeqBlock o = seq_block(at, by_xcd ? gridDim.x >> 3 : gridDim.x, hx, blockIdx.y, gridDim.y, by_seq);
    const int h = (by_xcd ? (blockIdx.x & 7) * hx : 0) + o.head, b = o.seq, qb = (gridDim.y - 1 - o.block) * QB;
    const int32_t* sq = seq + 4 * b;
    const int q_at = sq[0], nq = sq[1], past = sq[2];
    if (qb >= nq || nq < 1 || past < 0 || q_at < 0 || q_at + nq > tokens) return;
    const int nk = past + nq, kvh = h / (H / G);
    const int64_t ld_c = (int64_t)G * 2 * D;
    const int32_t* tab = table + (int64_t)b * table_ld;

    Flash f;
    int lo[2], hi[2];                                         // first and last key that the lane's own query sees
    auto load = [&] {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int j = min(qb + 32 * wave + 16 * u + i, nq - 1);
            hi[u] = past + j;
            lo[u] = chunk > 0 ? hi[u] / chunk * chunk : 0;
            const bf16* src = q + (int64_t)(q_at + j) * ld_q + h * D + 8 * g;
#pragma unroll
            for (int c = 0; c < 4; ++c) f.q[u][c] = load_frag(src + 32 * c);
        }
    };
    const int first_q = past + qb, last_q = past + min(qb + QB, nq) - 1;       // positions of the workgroup's rows
    const int wave_first = min(first_q + 32 * wave, nk - 1), wave_last = min(wave_first + 31, nk - 1);
    const int wave_chunk = chunk > 0 ? wave_last / chunk * chunk : 0;          // tiles from here to wave_first need no mask
    f.run(smem, (chunk > 0 ? first_q / chunk * chunk : 0) / KT, last_q / KT + 1, (uint32_t)ld_c, 0, scale, lo, hi, load,
          [&](int t) {
              const int pg = tab[t];
              const bf16* base = cache + (int64_t)(pg < 0 ? 0 : (pg >= n_pages ? n_pages - 1 : pg)) * TFL_PAGE * ld_c + kvh * D;
              return Flash::Tile{base, nullptr, base + G * D, min(KT, nk - t * KT) - 1};
          },
          [&](int k0) { return k0 + KT - 1 <= wave_first && k0 >= wave_chunk; });
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int j = qb + 32 * wave + 16 * u + i;
        const float inv = out_scale / f.weight(u);
        if (j >= nq) continue;
        const int64_t tok = q_at + j;
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const int col = h * D + 16 * d + 4 * g;
            const f32x4 z = load_quad(gate + tok * ld_gate + col);
            f32x4 v = f.acc[u][d];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= inv * sigmoid_of<bf16>(z[r]);
            store_quad(out + tok * ld_out + col, v);
        }
    }
}

template <typename T, int DK, int DV>
__global__ __launch_bounds__(256, 1) void attn_chunk_kernel(const T* __restrict__ q, int64_t ld_q, const T* __restrict__ cache, int n_pages,
                                                            const int32_t* __restrict__ table, int table_ld, const int32_t* __restrict__ seq,
                                                            const T* __restrict__ gate, int64_t ld_gate, T* __restrict__ out, int64_t ld_out,
                                                            int tokens, int H, int G, int D, int V, int chunk, float scale, float out_scale) {
    typedef typename El<T>::Frag Frag;
    constexpr int KT = 64, EPV = 16 / sizeof(T), QB = 64, NT = 256;
    const int dk = D >> 5, dv = V >> 4, ldk = D + EPV, ldv = V + 2 * EPV;
    extern __shared__ __align__(16) char smem[];
    T* Ks = (T*)smem;                                         // [KT][ldk], then the values
    T* Vs = Ks + KT * ldk;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, i = lane & 15;
    // workgroups go round-robin over the 8 XCDs: the query blocks of a key / value head stay on one of them, longest first
    const int nqb = gridDim.x / H, id = blockIdx.x;
    const bool by_xcd = (H & 7) == 0;
    const int j_ = by_xcd ? id >> 3 : id, h = by_xcd ? (id & 7) * (H >> 3) + j_ / nqb : j_ / nqb;
    const int32_t* sq = seq + 4 * blockIdx.y;
    const int q_at = sq[0], nq = sq[1], past = sq[2];
    const int qb = (nqb - 1 - j_ % nqb) * QB;
    if (qb >= nq || nq < 1 || past < 0 || q_at < 0 || q_at + nq > tokens) return;
    const int nk = past + nq, kvh = h / (H / G);
    const int64_t ld_c = (int64_t)G * (D + V);
    const int32_t* tab = table + (int64_t)blockIdx.y * table_ld;

    Frag qf[DK];
    const int own = min(qb + 16 * wave + i, nq - 1), qpos = past + own;        // the lane's own query: row, position, first key it sees
    const int first_key = chunk > 0 ? qpos / chunk * chunk : 0;
    const T* src = q + (int64_t)(q_at + own) * ld_q + h * D + 8 * g;
#pragma unroll
    for (int c = 0; c < DK; ++c) qf[c] = c < dk ? load_frag(src + 32 * c) : Frag{};
    f32x4 o[DV];
    float m_run = NEG_INF, l_run = 0.f;
#pragma unroll
    for (int d = 0; d < DV; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int first_q = past + qb, last_q = past + min(qb + QB, nq) - 1;       // positions of the workgroup's rows
    const int t_beg = (chunk > 0 ? first_q / chunk * chunk : 0) / KT, t_end = last_q / KT + 1;
    const int wave_first = min(first_q + 16 * wave, nk - 1), wave_last = min(wave_first + 15, nk - 1);
    const int wave_chunk = chunk > 0 ? wave_last / chunk * chunk : 0;          // tiles from here to wave_first need no mask
    auto rows_of = [&](int t) {
        const int pg = tab[t];
        return cache + (int64_t)(pg < 0 ? 0 : (pg >= n_pages ? n_pages - 1 : pg)) * TFL_PAGE * ld_c;
    };
    for (int t = t_beg; t < t_end; ++t) {
        const int k0 = t * KT;
        const T* base = rows_of(t);
        const int kn = D / EPV, vn = V / EPV, ppr = kn + vn, left = nk - k0 - 1;
        for (int p = tid; p < KT * ppr; p += NT) {
            const int key = p / ppr, c = p - key * ppr;
            const T* src = base + (int64_t)min(key, left) * ld_c + (c < kn ? kvh * D + EPV * c : G * D + kvh * V + EPV * (c - kn));
            *reinterpret_cast<u32x4*>(c < kn ? Ks + key * ldk + EPV * c : Vs + key * ldv + EPV * (c - kn)) = *reinterpret_cast<const u32x4*>(src);
        }
        __syncthreads();
        f32x4 s[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
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
        if (k0 + KT - 1 > wave_first || k0 < wave_chunk) {
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int k = k0 + 16 * kt + 4 * g + r;
                    if (k > qpos || k < first_key) s[kt][r] = NEG_INF;
                }
        }
        Frag pf[2];
        float mx = NEG_INF;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[kt][r]);
        mx = rows_max(mx);
        mx = fmaxf(m_run, mx * scale);
        // a row may have seen no key yet (its chunk starts in a later tile): its maximum is -inf, every weight 0
        const float ref = mx == NEG_INF ? 0.f : mx;
        const float alpha = __builtin_amdgcn_exp2f((m_run - ref) * LOG2E), sc = scale * LOG2E, mb = ref * LOG2E;
        m_run = mx;
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f(fmaf(s[kt][r], sc, -mb));
                sum += p;
                pf[kt >> 1][(kt & 1) * 4 + r] = (T)p;
            }
        l_run = l_run * alpha + sum;
        if (!__all(alpha == 1.0f)) {
#pragma unroll
            for (int d = 0; d < DV; ++d)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[d][r] *= alpha;
        }
#pragma unroll
        for (int d = 0; d < DV; ++d) {
            if (d < dv) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const Frag a = load_frag_t(Vs, ldv, 32 * c + 4 * g, 32 * c + 16 + 4 * g, 16 * d, i);
                    o[d] = El<T>::mma(a, pf[c], o[d]);
                }
            }
        }
        __syncthreads();
    }
    const int j = qb + 16 * wave + i;
    float l = l_run;
    l = rows_sum(l);
    if (j >= nq) return;
    const float inv = out_scale / l;
    const int64_t tok = q_at + j;
#pragma unroll
    for (int d = 0; d < DV; ++d) {
        if (d >= dv) continue;
        const int col = h * V + 16 * d + 4 * g;
        const f32x4 z = load_quad(gate + tok * ld_gate + col);
        f32x4 v = o[d];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= inv * sigmoid_of<T>(z[r]);
        store_quad(out + tok * ld_out + col, v);
    }
}

template <typename T, int DK, int DV>
static int launch_chunk(const void* q, int64_t ld_q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* seq, int nseq,
                        int max_new, const void* gate, int64_t ld_gate, void* out, int64_t ld_out, int tokens, int H, int G, int D, int V,
                        int chunk, float scale, float out_scale, hipStream_t st) {
    const int epv = 16 / (int)sizeof(T);
    const size_t lds = sizeof(T) * 64 * (size_t)(D + V + 3 * epv);
    if (lds > 160 * 1024) return TF_ERANGE;
    auto k = attn_chunk_kernel<T, DK, DV>;
    static bool attr = false;
    if (!attr) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        attr = true;
    }
    hipLaunchKernelGGL(k, dim3((max_new + 63) / 64 * H, nseq), dim3(256), lds, st, (const T*)q, ld_q,
                       (const T*)cache, n_pages, table, table_ld, seq, (const T*)gate, ld_gate, (T*)out, ld_out, tokens, H, G, D, V, chunk, scale,
                       out_scale);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

extern "C" int tfh_attn_prefill(const void* q, int64_t ld_q, const void* cache, int64_t n_pages, const int32_t* table, int table_ld,
                                const int32_t* seq, int nseq, int max_new, const void* gate, int64_t ld_gate, void* out, int64_t ld_out,
                                int tokens, int H, int G, int D, int V, int chunk, float scale, float out_scale, int dtype, void* stream) {
    if (!q || !cache || !table || !seq || !gate || !out || nseq < 1 || nseq > 65535 || max_new < 1 || tokens < 1 || n_pages < 1
        || n_pages > (1 << 30) || table_ld < 1) return TF_EINVAL;
    if (H < 1 || G < 1 || H % G || D < 32 || (D & 31) || V < 32 || (V & 31) || chunk < 0 || !(scale > 0.f)) return TF_EINVAL;
    if ((ld_q & 7) || (ld_gate & 3) || (ld_out & 3) || ld_q < (int64_t)H * D || ld_gate < (int64_t)H * V || ld_out < (int64_t)H * V) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
#define GO(T, DK, DV)                                                                                                                \
    return launch_chunk<T, DK, DV>(q, ld_q, cache, (int)n_pages, table, table_ld, seq, nseq, max_new, gate, ld_gate, out, ld_out, \
                                                tokens, H, G, D, V, chunk, scale, out_scale, st)
    if (dtype == 0) {
        if (D == 128 && V == 128 && G <= 1 << 16 && (int64_t)H * nseq <= 1 << 30 && max_new <= 1 << 22) {       // (63 cache rows stay below 2^32 bytes)
            constexpr int LDS = FlashTile<0, 4>::LDS;
            const int blocks = (max_new + 127) / 128;
            const bool by_seq = nseq > 1 && (int64_t)H * nseq * blocks > 512 && (int64_t)H * nseq * blocks < 1 << 30;
            const hipError_t e = hipFuncSetAttribute((const void*)attn_chunk_sized_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
            if (e != hipSuccess) return (int)e;
            hipLaunchKernelGGL(attn_chunk_sized_kernel, dim3((unsigned)(H * nseq), blocks), dim3(256), LDS, st, (const bf16*)q, ld_q,
                               (const bf16*)cache, (int)n_pages, table, table_ld, seq, (const bf16*)gate, ld_gate, (bf16*)out, ld_out, tokens, H, G,
                               chunk, scale, out_scale, nseq, (int)by_seq);
            TFL_LAUNCH_CHECK();
            return TF_OK;
        }
        if (D <= 64 && V <= 64) GO(bf16, 2, 4);
        if (D <= 128 && V <= 128) GO(bf16, 4, 8);
        if (D <= 256 && V <= 256) GO(bf16, 8, 16);
        return TF_ERANGE;
    }
    if (dtype == 1) {
        if (D <= 64 && V <= 64) GO(float, 2, 4);
        if (D <= 128 && V <= 128) GO(float, 4, 8);
        if (D <= 256 && V <= 256) GO(float, 8, 16);
        return TF_ERANGE;
    }
#undef GO
    return TF_EINVAL;
}
