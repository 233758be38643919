/* C ABI of libtriforce_hybrid.so: chunked grouped-query attention, linear recurrences (scalar and per-channel decay) and several
 * residual streams (models/modeling_kemurax.py), for gfx950.
 *
 * Every entry point enqueues on `stream` and returns TF_OK, a TF_E* code (nothing launched) or a hipError_t.
 * dtype: 0 = bfloat16 operands with fp32 accumulation, 1 = everything in fp32.  "T" below is that element type.
 *
 * Padded sizes.  Every dimension that a matrix product contracts or tiles is padded to a multiple of 32 with zeros when the
 * weights are loaded; the kernels below only see padded sizes unless a parameter is called "real".
 * Attention: H query heads on G key / value heads, D / V = query-key / value size of a head; one cached row is [G*D keys][G*V values],
 * pages of TFL_PAGE rows.  Recurrences: per head a state of N x V fp32 that lives in the sequence's seat.
 *
 * Prefill batches are packed: seq [nseq][4] int32 = {first new token, new tokens, tokens before them, seat}.
 */
#ifndef TRIFORCE_HYBRID_H
#define TRIFORCE_HYBRID_H
#include "triforce_tile.h"
#ifdef __cplusplus
extern "C" {
#endif

#define TFH_CHUNK 64                /* tokens a recurrence takes at a time in prefill */

int tfh_abi_version(void);

/* Between two sublayers, per row, x fp32 [rows][streams][width]:
 *   embed != NULL: every stream = rms-norm(embed[ids]) * embed_w;   y != NULL: x_t = sum_s mix[s*streams + t] x_s + out[t] * y
 *   u = sum_s in[s] x_s;   h = u / rms(u) * norm_w   (T)
 * x is written back unless keep == 0.  y is fp32 when y_f32, else T.  width_real elements carry data; h is an activation block. */
int tfh_connect(const void* embed, const int64_t* ids, int vocab, const float* embed_w, const void* y, int y_f32, int64_t ld_y,
                const float* out, const float* mix, const float* in, const float* norm_w, float* x, int streams, int keep, void* h,
                int64_t ld_h, int64_t h_oct, int rows, int width, int width_real, float eps, int dtype, void* stream);
/* The first of a decode step (embed given, y not, x kept), with tfl_decode_prep of its rows in the same launch. */
int tfh_connect_first(const void* embed, const int64_t* ids, int vocab, const float* embed_w, const float* in, const float* norm_w, float* x, int streams, void* h,
                      int64_t ld_h, int64_t h_oct, int rows, int width, int width_real, float eps, const TflDecodePrep* prep, int dtype, void* stream);

/* tfh_connect of rows whose next reader is a wide product, in that product's launch (bfloat16, one row of up to 4 streams of up to 4 096): every
 * workgroup makes the normed row for itself, beside the beginning of its weights.  x_out (NULL: the streams are not kept) is another block than x;
 * product->x is not read.  epilogue TFL_EPI_F32 or TFL_EPI_GLU, chunk-major weights, 16-byte aligned pointers.  TF_ERANGE: not a size of this form (nothing launched);
 * tfh_connect_gemm_takes says so beforehand. */
typedef struct TfhConnect {
    const float* y;                 /* [rows], row stride ld_y */
    const float* out;               /* [streams] */
    const float* mix;               /* [streams][streams] */
    const float* in;                /* [streams] */
    const float* norm_w;
    const float* x;                 /* [rows][streams][width] */
    float* x_out;
    int64_t ld_y;
    int32_t streams, width, width_real;
    float eps;
} TfhConnect;
int tfh_connect_gemm_takes(int rows, int streams, int width, int n, int k, int epilogue);
int tfh_connect_gemm(const TfhConnect* f, const TflGemm* product, int epilogue, void* stream);

/* The same between two wide products of any number of rows, up to 4 streams, without a launch of its own (bfloat16, chunk-major weights, 16-byte aligned pointers).
 * tfh_streams_gemm: y = product->x . W^T of a sublayer's last product (n = width) goes into the streams (f->y is not read; f->x_out: x itself, another block, or
 *   NULL), product->out_t = u * norm_w, an activation block without the norm's scale, and product->ss_out[m*ss_ld + n/16] = sums of u^2 over each panel.
 * tfh_scaled_gemm: TFL_EPI_F32 or TFL_EPI_GLU of rows that are scaled by 1 / sqrt(sum(ss_in[m][:ss_n]) / k_real + eps) behind the product; ss_n and ss_ld in fours,
 *   up to 512.
 * TF_ERANGE: not a size of these forms; the _takes functions say so beforehand. */
int tfh_streams_gemm_takes(int rows, int streams, int n, int k);
int tfh_streams_gemm(const TfhConnect* f, const TflGemm* product, void* stream);
int tfh_scaled_gemm_takes(int rows, int n, int epilogue);
int tfh_scaled_gemm(const TflGemm* a, int epilogue, void* stream);

/* ---- prefill ----------------------------------------------------------------------------------------------------------- */

/* Queries and keys of new tokens: per head x / rms * norm, then entries i and i + half of the first 2 * half turn at pos[token];
 * queries in place, keys and values into cache row slot[token].  y [rows] at stride ld_y, columns q_off (H*D), k_off (G*D), v_off (G*V). */
int tfh_qkv_prepare(void* y, int64_t ld_y, int q_off, int k_off, int v_off, const float* q_norm, const float* k_norm, const float* cos,
                    const float* sin, int half, int max_pos, const int32_t* pos, const int32_t* slot, void* cache, int64_t cache_rows,
                    int rows, int H, int G, int D, int D_real, int V, float eps, int dtype, void* stream);

/* Causal attention of packed new tokens over the paged cache (the new rows are in it); key j is visible to query i only when
 * i / chunk == j / chunk (chunk = 0: no chunks).  table [nseq][table_ld].
 *   out [tokens] at stride ld_out: o[h*V + d] * sigmoid(gate[token*ld_gate + h*V + d]) * out_scale */
int tfh_attn_prefill(const void* q, int64_t ld_q, const void* cache, int64_t n_pages, const int32_t* table, int table_ld,
                     const int32_t* seq, int nseq, int max_new, const void* gate, int64_t ld_gate, void* out, int64_t ld_out, int tokens,
                     int H, int G, int D, int V, int chunk, float scale, float out_scale, int dtype, void* stream);

/* Short causal convolution (+ bias, silu) over `channels` columns of y, and the recurrence's step sizes softplus(y_dt + dt_bias).
 * conv_w fp32 [taps][channels]; ring fp32 [seats][taps][channels]: slot position % taps holds the raw input of a position. */
int tfh_conv_prepare(const void* y, int64_t ld_y, int x_off, int dt_off, const float* conv_w, const float* conv_b, int taps,
                     int channels, const float* dt_bias, int heads, float* ring, int seats, void* xbc, float* dt, const int32_t* seq,
                     int nseq, int max_new, int tokens, int dtype, void* stream);

/* Log decays per key channel, max(logsigmoid(z + bias) * inv_tau, -60), summed up inside chunks of TFH_CHUNK new tokens. */
int tfh_decay_prepare(const void* z, int64_t ld_z, const float* bias, float inv_tau, float* gcum, const int32_t* seq, int nseq, int max_new,
                      int tokens, int channels, int dtype, void* stream);

/* S = decay * S + k v^T, o = S^T q over packed new tokens; segments of a sequence run side by side: their own contributions first,
 * then a scan over them, then the outputs.  seg [nseg][4] = {first token, tokens, sequence, 0}, segments of a sequence in order,
 * each a multiple of TFH_CHUNK tokens but the last; span [nseq][2] = {first segment, segments}. */
typedef struct TfhRecurrence {
    const void* q;                  /* T; head h reads columns (h / per_group) * N of a token's row */
    const void* k;
    const void* v;                  /* T; head h reads columns h*V */
    const float* gcum;              /* per-channel decay: [tokens][H*N] of tfh_decay_prepare; NULL: scalar decay */
    const float* dt;                /* scalar decay: [tokens][H] step sizes (k is multiplied by them) */
    const float* nega;              /* [H] log decay per unit of step */
    const float* skip;              /* [H]: o += skip * v (NULL: none) */
    const void* gate;               /* o *= silu(gate[token*ld_gate + h*V + v]) (NULL: none) */
    float* state;                   /* [seats][H][N][V] */
    float* part;                    /* [nseg][H][N][V], when some sequence has several segments */
    float* decay;                   /* [nseg][H] or [nseg][H*N], likewise */
    void* out;                      /* T, [tokens] at stride ld_out, columns h*V */
    const int32_t* seq;
    const int32_t* seg;
    const int32_t* span;
    int64_t ld_q, ld_k, ld_v, ld_gate, ld_out;
    int32_t nseq, nseg, max_segs, tokens, seats, H, per_group, N, V;
    float q_scale;
} TfhRecurrence;
int tfh_recurrence(const TfhRecurrence* a, int dtype, void* stream);

/* Groups of `size` values / rms * w * scale into activation block columns 0 .. : the real values of a row are heads of V_real in
 * strides of V (zeros are written between).  shared_w: w has `size` entries, used by every group.  gate != NULL: the result is
 * multiplied by silu(gate).  src / gate: T, or fp32 when f32. */
int tfh_group_norm(const void* src, int64_t ld_src, const void* gate, int64_t ld_gate, int f32, const float* w, int shared_w, void* out,
                   int64_t ld_out, int64_t out_oct, int rows, int groups, int size, int V_real, int V, float eps, float scale, int dtype,
                   void* stream);

/* s [rows][2n] in blocks of 8 gate | 8 up columns -> out [rows][n] = gelu_tanh(gate) * up. */
int tfh_glu(const void* s, void* out, int rows, int n, int dtype, void* stream);

/* ---- decode: one token per row; raw = fp32 projections of the row's token, klen = keys including it (<= 0: idle row) ------- */
typedef struct TfhAttnStep {
    const float* q_norm;
    const float* k_norm;
    const float* cos;
    const float* sin;
    void* cache;
    const int32_t* table;
    float* ws;                      /* tfh_attn_step_ws_floats */
    int64_t n_pages;
    int32_t q_off, k_off, v_off, gate_off, half, max_pos, table_ld, H, G, D, D_real, V, chunk, nsplit;
    float scale, out_scale;
} TfhAttnStep;
typedef struct TfhRecStep {
    const float* conv_w;            /* scalar decay: convolution over x | B | C at x_off, step sizes at dt_off, gate at gate_off */
    const float* conv_b;
    float* ring;
    const float* dt_bias;
    const float* nega;
    const float* skip;
    const void* a2;                 /* per-channel decay (NULL: scalar): T [H*N][rank] (rank in fours), z = a2 . raw[a_off ..] + a2_b */
    const float* a2_b;
    const float* norm_w;
    float* state;
    const int32_t* seat;
    float* out;                     /* fp32 [rows][H*V] */
    int32_t x_off, dt_off, gate_off, q_off, k_off, v_off, a_off, taps, channels, rank, seats, H, per_group, N, V, V_real, norm_groups;
    float inv_tau, q_scale, out_scale;
} TfhRecStep;

int64_t tfh_attn_step_ws_floats(int rows, int H, int V, int nsplit);
/* The nsplit to take for rows that see up to max_keys keys (tfh_attn_step_pick_nsplit: for bfloat16 heads of 128). */
int tfh_attn_step_splits(int rows, int H, int G, int D, int V, int max_keys, int dtype);
int tfh_attn_step_pick_nsplit(int rows, int H, int G, int max_keys);
/* Both parts of a layer's mixer in one launch, either may be NULL: norm / rotation / cache append / attention over the splits of the
 * visible keys; convolution / decay / state update / read-out. */
int tfh_step(const TfhAttnStep* attn, const TfhRecStep* rec, const float* raw, int64_t ld_raw, const int32_t* klen, int rows, float eps,
             int dtype, void* stream);
/* The operand of the output projection: [attention merged over the splits, gated | recurrence normed, gated], an activation block. */
int tfh_step_out(const TfhAttnStep* attn, const TfhRecStep* rec, const float* raw, int64_t ld_raw, void* act, int64_t ld_act,
                 int64_t act_oct, int rows, float eps, int dtype, void* stream);

#ifdef __cplusplus
}
#endif
#endif
