// Row kernels of the hybrid family: residual streams + norm between sublayers, the prefill halves of the mixers' input projections
// (query / key norm, rotation, cache append; short convolution, step sizes; per-channel decays), group norm and the gated unit.
#include "hybrid_common.h"

extern "C" int tfh_abi_version(void) { return 1; }

// ------------------------------------------------------------------------------------------------------------ streams
// One workgroup per row.  S streams at most (streams is the real number); the sublayer input u stays in LDS between its two uses.
// PREP: a step's first launch, with decode_prep_row() of all rows as one more workgroup.
template <typename T, typename Y, int S, int NW, bool PREP = false>
__global__ __launch_bounds__(64 * NW) void connect_kernel(const T* __restrict__ embed, const int64_t* __restrict__ ids, int vocab,
                                                          const float* __restrict__ embed_w, const Y* __restrict__ y, int64_t ld_y,
                                                          const float* __restrict__ out, const float* __restrict__ mix,
                                                          const float* __restrict__ in, const float* __restrict__ norm_w,
                                                          float* __restrict__ x, int streams, int keep, T* __restrict__ h, int64_t ld_h,
                                                          int64_t h_oct, int width, int width_real, float eps, const TflDecodePrep prep) {
    constexpr int NT = 64 * NW;
    if constexpr (PREP) {
        if ((int)blockIdx.x == prep.rows) {
            for (int m = threadIdx.x; m < prep.rows; m += NT) decode_prep_row(prep, m);
            return;
        }
    }
    extern __shared__ __align__(16) float us[];              // [width]
    __shared__ float red[NW];
    __shared__ float cf[S * S + 2 * S];                      // mix | out | in
    const int row = blockIdx.x, nq = width >> 2;
    float* xr = x + (int64_t)row * streams * width;
    const Y* yr = y ? y + (int64_t)row * ld_y : nullptr;
    // Few rows are bound by round trips: what a thread's first quad needs is asked for together with the coefficients (8 rows of 4 x 4 096
    // 6.0 -> 5.3 us).  More rows are bound by memory, and more streams do not fit the registers.
    constexpr bool EARLY = NW == 16 && S <= 4;
    f32x4 x0[S], y0 = {0.f, 0.f, 0.f, 0.f}, w0 = {0.f, 0.f, 0.f, 0.f};
    auto streams_of = [&](f32x4 (&v)[S], int q) {
#pragma unroll
        for (int s = 0; s < S; ++s)
            v[s] = s < streams ? *reinterpret_cast<const f32x4*>(xr + (int64_t)s * width + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
    };
    if (EARLY && (int)threadIdx.x < nq) {
        if (!embed) streams_of(x0, threadIdx.x);
        if (yr) y0 = load_quad(yr + 4 * threadIdx.x);
        w0 = *reinterpret_cast<const f32x4*>(norm_w + 4 * threadIdx.x);
    }
    for (int t = threadIdx.x; t < S * S; t += NT) {
        const int s = t / S, d = t - s * S;
        cf[t] = y && s < streams && d < streams ? mix[s * streams + d] : 0.f;
    }
    for (int t = threadIdx.x; t < S; t += NT) {
        cf[S * S + t] = y && t < streams ? out[t] : 0.f;
        cf[S * S + S + t] = t < streams ? in[t] : 0.f;
    }
    __syncthreads();
    float ss = 0.f;
    if (embed) {
        int64_t id = ids[row];
        id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
        const T* er = embed + id * (int64_t)width;
        float e2 = 0.f;
        for (int q = threadIdx.x; q < nq; q += NT) {
            const f32x4 v = load_quad(er + 4 * q);
            e2 += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        e2 = block_sum<NW>(e2, red);
        const float inv = 1.0f / sqrtf(e2 / (float)width_real + eps);
        float share = 0.f;
#pragma unroll
        for (int s = 0; s < S; ++s) share += cf[S * S + S + s];
        for (int q = threadIdx.x; q < nq; q += NT) {
            f32x4 v = load_quad(er + 4 * q);
            const f32x4 w = *reinterpret_cast<const f32x4*>(embed_w + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = v[r] * inv * w[r];
            for (int s = 0; s < streams; ++s) *reinterpret_cast<f32x4*>(xr + (int64_t)s * width + 4 * q) = v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= share;
            *reinterpret_cast<f32x4*>(us + 4 * q) = v;
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
    } else {
        for (int q = threadIdx.x; q < nq; q += NT) {
            const bool have = EARLY && q == (int)threadIdx.x;
            f32x4 v[S];
            if (have) {
#pragma unroll
                for (int s = 0; s < S; ++s) v[s] = x0[s];
            } else {
                streams_of(v, q);
            }
            f32x4 u = {0.f, 0.f, 0.f, 0.f};
            if (yr) {
                const f32x4 z = have ? y0 : load_quad(yr + 4 * q);
#pragma unroll
                for (int t = 0; t < S; ++t) {
                    const float o = cf[S * S + t], g = cf[S * S + S + t];
                    f32x4 n;
#pragma unroll
                    for (int r = 0; r < 4; ++r) n[r] = o * z[r];
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        const float m = cf[s * S + t];
#pragma unroll
                        for (int r = 0; r < 4; ++r) n[r] = fmaf(m, v[s][r], n[r]);
                    }
                    if (keep && t < streams) *reinterpret_cast<f32x4*>(xr + (int64_t)t * width + 4 * q) = n;
#pragma unroll
                    for (int r = 0; r < 4; ++r) u[r] = fmaf(g, n[r], u[r]);
                }
            } else {
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const float g = cf[S * S + S + s];
#pragma unroll
                    for (int r = 0; r < 4; ++r) u[r] = fmaf(g, v[s][r], u[r]);
                }
            }
            *reinterpret_cast<f32x4*>(us + 4 * q) = u;
            ss += u[0] * u[0] + u[1] * u[1] + u[2] * u[2] + u[3] * u[3];
        }
    }
    ss = block_sum<NW>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)width_real + eps);
    for (int q = threadIdx.x; q < nq; q += NT) {              // (each thread reads back what it wrote itself)
        f32x4 u = *reinterpret_cast<const f32x4*>(us + 4 * q);
        const f32x4 w = EARLY && q == (int)threadIdx.x ? w0 : *reinterpret_cast<const f32x4*>(norm_w + 4 * q);
#pragma unroll
        for (int r = 0; r < 4; ++r) u[r] = u[r] * inv * w[r];
        store_quad(h + (int64_t)row * ld_h + (q >> 1) * h_oct + 4 * (q & 1), u);
    }
}

template <typename T, typename Y, int S, int NW, bool PREP>
static int launch_connect(const void* embed, const int64_t* ids, int vocab, const float* embed_w, const void* y, int64_t ld_y, const float* out,
                          const float* mix, const float* in, const float* norm_w, float* x, int streams, int keep, void* h, int64_t ld_h,
                          int64_t h_oct, int rows, int width, int width_real, float eps, const TflDecodePrep& prep, hipStream_t st) {
    auto k = connect_kernel<T, Y, S, NW, PREP>;
    static bool attr = false;
    if (!attr) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 144 * 1024);
        if (e != hipSuccess) return (int)e;
        attr = true;
    }
    hipLaunchKernelGGL(k, dim3(rows + PREP), dim3(64 * NW), sizeof(float) * width, st, (const T*)embed, ids, vocab, embed_w, (const Y*)y, ld_y, out, mix,
                       in, norm_w, x, streams, keep, (T*)h, ld_h, h_oct, width, width_real, eps, prep);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

static int connect(const void* embed, const int64_t* ids, int vocab, const float* embed_w, const void* y, int y_f32, int64_t ld_y,
                           const float* out, const float* mix, const float* in, const float* norm_w, float* x, int streams, int keep,
                           void* h, int64_t ld_h, int64_t h_oct, int rows, int width, int width_real, float eps, const TflDecodePrep* prep, int dtype, void* stream) {
    if (!x || !h || !norm_w || !in || rows < 1 || width < 8 || (width & 7) || ld_h < 8 || (ld_h & 7) || h_oct < 8 || (h_oct & 7)
        || width_real < 1 || width_real > width || streams < 1) return TF_EINVAL;
    if (embed && (!ids || !embed_w || vocab < 1 || y)) return TF_EINVAL;
    if (y && (!out || !mix || ld_y < width || (ld_y & 3))) return TF_EINVAL;
    if ((dtype != 0 && dtype != 1) || (dtype == 1 && y && !y_f32)) return TF_EINVAL;
    if (streams > 16 || width > 32768) return TF_ERANGE;
    hipStream_t st = (hipStream_t)stream;
    const TflDecodePrep d = prep ? *prep : TflDecodePrep{};
#define GO(T, Y, S, NW, PREP) \
    return launch_connect<T, Y, S, NW, PREP>(embed, ids, vocab, embed_w, y, ld_y, out, mix, in, norm_w, x, streams, keep, h, ld_h, h_oct, rows, \
                                       width, width_real, eps, d, st)
#define GO_S(T, Y, NW, PREP) do { if (streams <= 2) GO(T, Y, 2, NW, PREP); if (streams <= 4) GO(T, Y, 4, NW, PREP); if (streams <= 8) GO(T, Y, 8, NW, PREP); GO(T, Y, 16, NW, PREP); } while (0)
#define GO_W(T, Y, PREP) do { if (rows <= 256 && width >= 2048) GO_S(T, Y, 16, PREP); GO_S(T, Y, 4, PREP); } while (0)
    if (prep) {
        if (dtype == 1) GO_W(float, float, true);
        GO_W(bf16, bf16, true);
    }
    if (dtype == 1) GO_W(float, float, false);
    if (y_f32) GO_W(bf16, float, false);
    GO_W(bf16, bf16, false);
#undef GO_W
#undef GO_S
#undef GO
}

extern "C" int tfh_connect(const void* embed, const int64_t* ids, int vocab, const float* embed_w, const void* y, int y_f32, int64_t ld_y,
                           const float* out, const float* mix, const float* in, const float* norm_w, float* x, int streams, int keep,
                           void* h, int64_t ld_h, int64_t h_oct, int rows, int width, int width_real, float eps, int dtype, void* stream) {
    return connect(embed, ids, vocab, embed_w, y, y_f32, ld_y, out, mix, in, norm_w, x, streams, keep, h, ld_h, h_oct, rows, width, width_real, eps, nullptr, dtype, stream);
}

extern "C" int tfh_connect_first(const void* embed, const int64_t* ids, int vocab, const float* embed_w, const float* in, const float* norm_w, float* x, int streams,
                                 void* h, int64_t ld_h, int64_t h_oct, int rows, int width, int width_real, float eps, const TflDecodePrep* prep, int dtype, void* stream) {
    if (!embed || !decode_prep_ok(prep, rows)) return TF_EINVAL;
    return connect(embed, ids, vocab, embed_w, nullptr, 0, 0, nullptr, nullptr, in, norm_w, x, streams, 1, h, ld_h, h_oct, rows, width, width_real, eps, prep, dtype, stream);
}

// ------------------------------------------------------------------------------------------------------------ q | k | v
// One workgroup per new token.  OCT (rotated halves of whole octets): L lanes per head, an octet each; otherwise a wave per head.
template <typename T, bool OCT, int L>
__global__ __launch_bounds__(256) void qkv_prepare_kernel(T* __restrict__ y, int64_t ld_y, int q_off, int k_off, int v_off,
                                                          const float* __restrict__ q_norm, const float* __restrict__ k_norm,
                                                          const float* __restrict__ cosb, const float* __restrict__ sinb, int half, int max_pos,
                                                          const int32_t* __restrict__ pos, const int32_t* __restrict__ slot, T* __restrict__ cache,
                                                          int64_t cache_rows, int H, int G, int D, int D_real, int V, float eps) {
    const int row = blockIdx.x;
    T* yr = y + (int64_t)row * ld_y;
    int p = pos[row];
    p = p < 0 ? 0 : (p >= max_pos ? max_pos - 1 : p);
    const float *cs = cosb + (int64_t)p * half, *sn = sinb + (int64_t)p * half;
    const int64_t sl = slot[row];
    T* dst = sl >= 0 && sl < cache_rows ? cache + sl * (int64_t)(G * (D + V)) : nullptr;
    if constexpr (OCT) {
        typedef typename El<T>::Frag Frag;
        const int l = threadIdx.x % L, e = 8 * l;
        const bool own = e < D, turned = e < 2 * half, low = e < half;
        const int pe = low ? e + half : e - half;             // the octet this one turns with
        f32x8 c = f32x8{}, sg = f32x8{};
        if (turned) {
            c = load_frag(cs + (low ? e : e - half));
            sg = load_frag(sn + (low ? e : e - half));
        }
        for (int hd = threadIdx.x / L; hd < H + G; hd += 256 / L) {
            T* src = hd < H ? yr + q_off + hd * D : yr + k_off + (hd - H) * D;
            const float* w = hd < H ? q_norm : k_norm;
            const Frag x = own ? load_frag(src + e) : Frag{}, q = turned ? load_frag(src + pe) : Frag{};
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = fmaf((float)x[j], (float)x[j], ss);
#pragma unroll
            for (int o = L / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
            const float inv = 1.0f / sqrtf(ss / (float)D_real + eps);
            T* to = hd < H ? src : (dst ? dst + (hd - H) * D : nullptr);
            if (!own || !to) continue;
            const f32x8 wx = load_frag(w + e);
            Frag o;
            if (turned) {
                const f32x8 wq = load_frag(w + pe);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float u = (float)x[j] * inv * wx[j], t = (float)q[j] * inv * wq[j];
                    o[j] = (T)(low ? u * c[j] - t * sg[j] : u * c[j] + t * sg[j]);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = (T)((float)x[j] * inv * wx[j]);
            }
            *reinterpret_cast<Frag*>(to + e) = o;
        }
    } else {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        for (int hd = wave; hd < H + G; hd += 4) {
            T* src = hd < H ? yr + q_off + hd * D : yr + k_off + (hd - H) * D;
            float o[4];
            head_norm_rotate([src](int e) { return (float)src[e]; }, D, D_real, hd < H ? q_norm : k_norm, eps, cs, sn, half, lane, o);
            T* to = hd < H ? src : (dst ? dst + (hd - H) * D : nullptr);
            if (to) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (lane + 64 * j < D) to[lane + 64 * j] = (T)o[j];
            }
        }
    }
    if (dst)
        for (int c = threadIdx.x; c < G * V / 8; c += 256)
            *reinterpret_cast<typename El<T>::Frag*>(dst + G * D + 8 * c) = load_frag(yr + v_off + 8 * c);
}

extern "C" int tfh_qkv_prepare(void* y, int64_t ld_y, int q_off, int k_off, int v_off, const float* q_norm, const float* k_norm,
                               const float* cosb, const float* sinb, int half, int max_pos, const int32_t* pos, const int32_t* slot,
                               void* cache, int64_t cache_rows, int rows, int H, int G, int D, int D_real, int V, float eps, int dtype,
                               void* stream) {
    if (!y || !q_norm || !k_norm || !pos || !slot || !cache || rows < 1 || cache_rows < 1 || H < 1 || G < 1 || H % G) return TF_EINVAL;
    if (D < 8 || (D & 7) || V < 8 || (V & 7) || D_real < 1 || D_real > D || half < 0 || 2 * half > D_real || max_pos < 1
        || (half && (!cosb || !sinb)) || (ld_y & 7) || (q_off & 7) || (k_off & 7) || (v_off & 7) || q_off < 0 || k_off < 0 || v_off < 0) return TF_EINVAL;
    if (ld_y < q_off + (int64_t)H * D || ld_y < k_off + (int64_t)G * D || ld_y < v_off + (int64_t)G * V) return TF_EINVAL;
    if (D > 256) return TF_ERANGE;
    hipStream_t st = (hipStream_t)stream;
#define GO(T, OCT, L) hipLaunchKernelGGL((qkv_prepare_kernel<T, OCT, L>), dim3(rows), dim3(256), 0, st, (T*)y, ld_y, q_off, k_off, v_off, q_norm, \
                                         k_norm, cosb, sinb, half, max_pos, pos, slot, (T*)cache, cache_rows, H, G, D, D_real, V, eps)
#define GO_L(T) do { if (half % 8) GO(T, false, 64); else if (D <= 64) GO(T, true, 8); else if (D <= 128) GO(T, true, 16); else GO(T, true, 32); } while (0)
    if (dtype == 0) GO_L(bf16);
    else if (dtype == 1) GO_L(float);
    else return TF_EINVAL;
#undef GO_L
#undef GO
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// ------------------------------------------------------------------------------------------------------------ convolution
#define CONV_TOKENS 16
// Workgroup: 64 channel octets by 4 runs of CONV_TOKENS / 4 tokens; the first one of a row makes the step sizes.  TAPS > 0: that many,
// inputs and taps in registers.
template <typename T, int TAPS>
__global__ __launch_bounds__(256) void conv_kernel(const T* __restrict__ y, int64_t ld_y, int x_off, int dt_off, const float* __restrict__ conv_w,
                                                   const float* __restrict__ conv_b, int taps_, int channels,
                                                   const float* __restrict__ dt_bias, int heads, const float* __restrict__ ring, int seats,
                                                   T* __restrict__ xbc, float* __restrict__ dt, const int32_t* __restrict__ seq, int tokens) {
    typedef typename El<T>::Frag Frag;
    constexpr int RUN = CONV_TOKENS / 4;
    const int taps = TAPS > 0 ? TAPS : taps_;
    const int32_t* sq = seq + 4 * blockIdx.z;
    const int at = sq[0], n = sq[1], past = sq[2], seat = sq[3];
    const int j0 = blockIdx.y * CONV_TOKENS;
    if (j0 >= n || at < 0 || at + n > tokens || past < 0 || seat < 0 || seat >= seats) return;
    if (blockIdx.x == 0) {
        for (int t = threadIdx.x; t < heads * min(CONV_TOKENS, n - j0); t += 256) {
            const int64_t row = at + j0 + t / heads;
            const int hd = t % heads;
            dt[row * heads + hd] = softplus((float)y[row * ld_y + dt_off + hd] + dt_bias[hd]);
        }
        return;
    }
    const float* rg = ring + (int64_t)seat * taps * channels;
    const int oct = (blockIdx.x - 1) * 64 + (threadIdx.x & 63), c = 8 * oct, j1 = j0 + RUN * (threadIdx.x >> 6);
    if (c < channels && j1 < n) {
        const T* col = y + (int64_t)at * ld_y + x_off + c;
        const f32x8 b = load_frag(conv_b + c);
        auto input = [&](int r) {                             // raw input of new token r (negative: an earlier one)
            f32x8 v = f32x8{};
            if (r >= 0) {
                const Frag x = load_frag(col + (int64_t)min(r, n - 1) * ld_y);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = (float)x[e];
            } else if (past + r >= 0) {
                v = load_frag(rg + (int64_t)((past + r) % taps) * channels + c);
            }
            return v;
        };
        auto finish = [&](int j, f32x8 s) {
            Frag o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (T)silu_of<T>(s[e]);
            *reinterpret_cast<Frag*>(xbc + (int64_t)(at + j) * channels + c) = o;
        };
        if constexpr (TAPS > 0) {
            f32x8 in[RUN + TAPS - 1], w[TAPS];
#pragma unroll
            for (int k = 0; k < RUN + TAPS - 1; ++k) in[k] = input(j1 + k - (TAPS - 1));
#pragma unroll
            for (int t = 0; t < TAPS; ++t) w[t] = load_frag(conv_w + (int64_t)t * channels + c);
#pragma unroll
            for (int j = 0; j < RUN; ++j) {
                f32x8 s = b;
#pragma unroll
                for (int t = 0; t < TAPS; ++t)
#pragma unroll
                    for (int e = 0; e < 8; ++e) s[e] = fmaf(in[j + t][e], w[t][e], s[e]);
                if (j1 + j < n) finish(j1 + j, s);
            }
        } else {
            for (int j = j1; j < min(j1 + RUN, n); ++j) {
                f32x8 s = b;
                for (int t = 0; t < taps; ++t) {
                    const f32x8 v = input(j - (taps - 1) + t), w = load_frag(conv_w + (int64_t)t * channels + c);
#pragma unroll
                    for (int e = 0; e < 8; ++e) s[e] = fmaf(v[e], w[e], s[e]);
                }
                finish(j, s);
            }
        }
    }
}

// The last inputs of every sequence into its ring (a launch of its own: the convolution above still reads the older ones).
template <typename T>
__global__ __launch_bounds__(256) void conv_ring_kernel(const T* __restrict__ y, int64_t ld_y, int x_off, int taps, int channels,
                                                        float* __restrict__ ring, int seats, const int32_t* __restrict__ seq, int tokens) {
    const int32_t* sq = seq + 4 * blockIdx.y;
    const int at = sq[0], n = sq[1], past = sq[2], seat = sq[3];
    if (n < 1 || at < 0 || at + n > tokens || past < 0 || seat < 0 || seat >= seats) return;
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= channels) return;
    for (int r = max(0, n - taps); r < n; ++r)
        ring[((int64_t)seat * taps + (past + r) % taps) * channels + c] = (float)y[(int64_t)(at + r) * ld_y + x_off + c];
}

extern "C" int tfh_conv_prepare(const void* y, int64_t ld_y, int x_off, int dt_off, const float* conv_w, const float* conv_b, int taps,
                                int channels, const float* dt_bias, int heads, float* ring, int seats, void* xbc, float* dt,
                                const int32_t* seq, int nseq, int max_new, int tokens, int dtype, void* stream) {
    if (!y || !conv_w || !conv_b || !dt_bias || !ring || !xbc || !dt || !seq || nseq < 1 || nseq > 65535 || max_new < 1 || tokens < 1) return TF_EINVAL;
    if (taps < 1 || channels < 8 || (channels & 7) || heads < 1 || seats < 1 || (ld_y & 7) || (x_off & 7) || x_off < 0 || dt_off < 0
        || ld_y < x_off + (int64_t)channels || ld_y < dt_off + (int64_t)heads) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid(1 + (channels / 8 + 63) / 64, (max_new + CONV_TOKENS - 1) / CONV_TOKENS, nseq);
#define GO_TAPS(T, TAPS) hipLaunchKernelGGL((conv_kernel<T, TAPS>), grid, dim3(256), 0, st, (const T*)y, ld_y, x_off, dt_off, conv_w, conv_b, taps, \
                                            channels, dt_bias, heads, ring, seats, (T*)xbc, dt, seq, tokens)
#define GO(T) do { \
    if (taps == 4) GO_TAPS(T, 4); else GO_TAPS(T, 0); \
    TFL_LAUNCH_CHECK(); \
    hipLaunchKernelGGL((conv_ring_kernel<T>), dim3((channels + 255) / 256, nseq), dim3(256), 0, st, (const T*)y, ld_y, x_off, taps, channels, ring, \
                       seats, seq, tokens); } while (0)
    if (dtype == 0) GO(bf16);
    else if (dtype == 1) GO(float);
    else return TF_EINVAL;
#undef GO_TAPS
#undef GO
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// ------------------------------------------------------------------------------------------------------------ channel decays
// Workgroup: 16 channel quads by 16 runs of 4 tokens of one chunk; a run's own sums, then the runs before it.
template <typename T>
__global__ __launch_bounds__(256) void decay_kernel(const T* __restrict__ z, int64_t ld_z, const float* __restrict__ bias, float inv_tau,
                                                    float* __restrict__ gcum, const int32_t* __restrict__ seq, int tokens, int channels) {
    __shared__ f32x4 sums[16][17];
    const int32_t* sq = seq + 4 * blockIdx.z;
    const int at = sq[0], n = sq[1], run = threadIdx.x >> 4, q = threadIdx.x & 15, c = 64 * blockIdx.x + 4 * q, j0 = blockIdx.y * TFH_CHUNK + 4 * run;
    if ((int)blockIdx.y * TFH_CHUNK >= n || at < 0 || at + n > tokens) return;
    f32x4 s[4], own = {0.f, 0.f, 0.f, 0.f};
    if (c < channels) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(bias + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 x = load_quad(z + (int64_t)(at + min(j0 + j, n - 1)) * ld_z + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) own[e] += fmaxf(log_sigmoid_of<T>(x[e] + b[e]) * inv_tau, -60.f);
            s[j] = own;
        }
    }
    sums[run][q] = own;
    __syncthreads();
    if (c >= channels) return;
    f32x4 before = {0.f, 0.f, 0.f, 0.f};
    for (int r = 0; r < run; ++r) {
        const f32x4 x = sums[r][q];
#pragma unroll
        for (int e = 0; e < 4; ++e) before[e] += x[e];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[j][e] += before[e];
        if (j0 + j < n) *reinterpret_cast<f32x4*>(gcum + (int64_t)(at + j0 + j) * channels + c) = s[j];
    }
}

extern "C" int tfh_decay_prepare(const void* z, int64_t ld_z, const float* bias, float inv_tau, float* gcum, const int32_t* seq, int nseq,
                                 int max_new, int tokens, int channels, int dtype, void* stream) {
    if (!z || !bias || !gcum || !seq || nseq < 1 || nseq > 65535 || max_new < 1 || tokens < 1 || channels < 4 || (channels & 3) || ld_z < channels || (ld_z & 3)
        || !(inv_tau > 0.f))
        return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((channels + 63) / 64, (max_new + TFH_CHUNK - 1) / TFH_CHUNK, nseq);
    if (dtype == 0) hipLaunchKernelGGL((decay_kernel<bf16>), grid, dim3(256), 0, st, (const bf16*)z, ld_z, bias, inv_tau, gcum, seq, tokens, channels);
    else if (dtype == 1) hipLaunchKernelGGL((decay_kernel<float>), grid, dim3(256), 0, st, (const float*)z, ld_z, bias, inv_tau, gcum, seq, tokens, channels);
    else return TF_EINVAL;
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

// ------------------------------------------------------------------------------------------------------------ group norm
// NW waves per group, 4 / NW groups per workgroup.  QUADS: no padding inside a row and sizes in fours.
template <typename T, typename F, int NW, bool QUADS>
__global__ __launch_bounds__(256) void group_norm_kernel(const F* __restrict__ src, int64_t ld_src, const F* __restrict__ gate, int64_t ld_gate,
                                                         const float* __restrict__ w, int shared_w, T* __restrict__ out, int64_t ld_out,
                                                         int64_t out_oct, int groups, int size, int V_real, int V, float eps, float scale) {
    constexpr int NT = 64 * NW;
    __shared__ float red[4];
    const int row = blockIdx.y, sub = threadIdx.x / NT, tid = threadIdx.x % NT, grp = blockIdx.x * (4 / NW) + sub;
    const bool live = grp < groups;                          // (idle waves stay for the barriers)
    const int first = grp * size;
    const F* sr = src + (int64_t)row * ld_src;
    const F* gr = gate ? gate + (int64_t)row * ld_gate : nullptr;
    T* dst = out + (int64_t)row * ld_out;
    auto where = [&](int c) { return QUADS ? c : c / V_real * V + c % V_real; };
    float ss = 0.f;
    if (live) {
        if constexpr (QUADS) {
            for (int c = 4 * tid; c < size; c += 4 * NT) {
                const f32x4 v = load_quad(sr + first + c);
                ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
            }
        } else {
            for (int c = tid; c < size; c += NT) {
                const float v = (float)sr[where(first + c)];
                ss = fmaf(v, v, ss);
            }
        }
    }
    if constexpr (NW == 4) ss = block_sum<4>(ss, red);
    else ss = wave_sum64(ss);
    if (!live) return;
    const float inv = scale / sqrtf(ss / (float)size + eps);
    const float* wr = w + (shared_w ? 0 : first);
    if constexpr (QUADS) {
        for (int c = 4 * tid; c < size; c += 4 * NT) {
            f32x4 v = load_quad(sr + first + c);
            const f32x4 wv = *reinterpret_cast<const f32x4*>(wr + c);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = v[r] * inv * wv[r];
            if (gr) {
                const f32x4 z = load_quad(gr + first + c);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= silu_of<T>(z[r]);
            }
            store_quad(dst + ((first + c) >> 3) * out_oct + ((first + c) & 7), v);
        }
    } else {
        for (int c = tid; c < size; c += NT) {
            const int at = where(first + c);
            float v = (float)sr[at] * inv * wr[c];
            if (gr) v *= silu_of<T>((float)gr[at]);
            dst[(at >> 3) * out_oct + (at & 7)] = (T)v;
            if ((first + c) % V_real == V_real - 1)
                for (int k = at + 1; k < at - V_real + 1 + V; ++k) dst[(k >> 3) * out_oct + (k & 7)] = (T)0.f;
        }
    }
}

extern "C" int tfh_group_norm(const void* src, int64_t ld_src, const void* gate, int64_t ld_gate, int f32, const float* w, int shared_w,
                              void* out, int64_t ld_out, int64_t out_oct, int rows, int groups, int size, int V_real, int V, float eps,
                              float scale, int dtype, void* stream) {
    if (!src || !w || !out || rows < 1 || rows > 65535 * 16 || groups < 1 || size < 1 || V_real < 1 || V < V_real || (int64_t)groups * size % V_real) return TF_EINVAL;
    const int64_t span = (int64_t)groups * size / V_real * V;
    if (ld_src < span || (ld_src & 3) || (gate && (ld_gate < span || (ld_gate & 3))) || ld_out < 8 || (ld_out & 7) || out_oct < 8 || (out_oct & 7)) return TF_EINVAL;
    if (dtype != 0 && dtype != 1) return TF_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const bool quads = V == V_real && size % 4 == 0;
    for (int r0 = 0; r0 < rows; r0 += 65535) {
        const int nr = rows - r0 < 65535 ? rows - r0 : 65535;
#define GO(T, F, NW, Q) hipLaunchKernelGGL((group_norm_kernel<T, F, NW, Q>), dim3((groups + 4 / NW - 1) / (4 / NW), nr), dim3(256), 0, st, \
                                           (const F*)src + r0 * ld_src, ld_src, gate ? (const F*)gate + r0 * ld_gate : nullptr, ld_gate, w, shared_w, \
                                           (T*)out + r0 * ld_out, ld_out, out_oct, groups, size, V_real, V, eps, scale)
#define GO_Q(T, F) do { if (size > 512) { if (quads) GO(T, F, 4, true); else GO(T, F, 4, false); } \
                        else { if (quads) GO(T, F, 1, true); else GO(T, F, 1, false); } } while (0)
        if (dtype == 1) GO_Q(float, float);
        else if (f32) GO_Q(bf16, float);
        else GO_Q(bf16, bf16);
#undef GO_Q
#undef GO
        TFL_LAUNCH_CHECK();
    }
    return TF_OK;
}

// ------------------------------------------------------------------------------------------------------------ gated unit
template <typename T>
__global__ __launch_bounds__(256) void glu_kernel(const T* __restrict__ s, T* __restrict__ out, int64_t octets) {
    for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < octets; p += (int64_t)gridDim.x * 256) {
        const typename El<T>::Frag g = load_frag(s + 16 * p), u = load_frag(s + 16 * p + 8);
        typename El<T>::Frag o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (T)(gelu_tanh((float)g[e]) * (float)u[e]);
        *reinterpret_cast<typename El<T>::Frag*>(out + 8 * p) = o;
    }
}

extern "C" int tfh_glu(const void* s, void* out, int rows, int n, int dtype, void* stream) {
    if (!s || !out || rows < 1 || n < 8 || (n & 7)) return TF_EINVAL;
    const int64_t octets = (int64_t)rows * n / 8;
    const unsigned gx = (unsigned)((octets + 255) / 256 < 16384 ? (octets + 255) / 256 : 16384);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == 0) hipLaunchKernelGGL((glu_kernel<bf16>), dim3(gx), dim3(256), 0, st, (const bf16*)s, (bf16*)out, octets);
    else if (dtype == 1) hipLaunchKernelGGL((glu_kernel<float>), dim3(gx), dim3(256), 0, st, (const float*)s, (float*)out, octets);
    else return TF_EINVAL;
    TFL_LAUNCH_CHECK();
    return TF_OK;
}
