/* C ABI of libtriforce_latent.so: kernels of the latent-attention model family (models/modeling_befidra.py) for gfx950.
 *
 * Every entry point enqueues on `stream` and returns TF_OK, a TF_E* code (nothing launched) or a hipError_t.
 * dtype: 0 = bfloat16 operands with fp32 accumulation, 1 = everything in fp32.  "T" below is that element type.
 *
 * Padded sizes.  Every dimension that a matrix product contracts or tiles is padded to a multiple of 32 with zeros when the
 * weights are loaded; the kernels below only see padded sizes unless a parameter is called "real".  Names: H heads, N / R =
 * unrotated / rotated query-key size of a head, V = value size of a head, C = latent size (all padded), W = C + R = one
 * cached row: [latent C][rotated key R].
 */
#ifndef TRIFORCE_LATENT_H
#define TRIFORCE_LATENT_H
#include "triforce_tile.h"
#ifdef __cplusplus
extern "C" {
#endif

int tfl_abi_version(void);          /* 2: as tfl_tile_abi_version 3 */

/* x (fp32 residual) of one row per workgroup, in this order, each part optional:
 *   x = embed[ids]            (embed != NULL)
 *   x += y / rms(y) * y_w     (y != NULL; fp32 when y_f32, else T)
 *   x += step                 (step != NULL)
 *   h = x / rms(x) * norm_w   (T)
 * width_real elements carry data, rows have stride width (padded with zeros); h is an activation block (triforce_tile.h). */
int tfl_finish(const void* embed, const int64_t* ids, int vocab, const void* y, int y_f32, int64_t ld_y, const float* y_w,
               const float* step, const float* norm_w, float* x, void* h, int64_t ld_h, int64_t h_oct, int rows, int width,
               int width_real, float eps, int dtype, void* stream);
/* The first of a decode step (embed given, y not), with tfl_decode_prep of its rows in the same launch. */
int tfl_finish_first(const void* embed, const int64_t* ids, int vocab, const float* step, const float* norm_w, float* x, void* h, int64_t ld_h, int64_t h_oct,
                     int rows, int width, int width_real, float eps, const TflDecodePrep* prep, int dtype, void* stream);

/* tfl_finish of rows whose next reader is a wide product, in that product's launch (bfloat16, up to 2 rows of up to 4 096): every workgroup makes the normed
 * rows for itself, beside the beginning of its weights.  x_out = x + y / rms(y) * y_w [+ step] is another block than x; product->x is not read.
 * epilogue TFL_EPI_IN or TFL_EPI_F32, chunk-major weights, 16-byte aligned pointers.  TF_ERANGE: not a size of this form (nothing launched); tfl_finish_gemm_takes says so beforehand. */
typedef struct TflFinish {
    const float* y;                 /* [rows], row stride ld_y */
    const float* y_w;
    const float* step;              /* NULL: none */
    const float* norm_w;
    const float* x;                 /* [rows][width] */
    float* x_out;
    int64_t ld_y;
    int32_t width, width_real;
    float eps;
} TflFinish;
int tfl_finish_gemm_takes(int rows, int width, int n, int k, int epilogue, int n_raw);
int tfl_finish_gemm(const TflFinish* f, const TflGemm* product, int epilogue, void* stream);

/* x += d (T); xt = T(x)  (xt may be NULL). */
int tfl_residual(const void* d, float* x, void* xt, int64_t n, int dtype, void* stream);

/* out = gelu_tanh(s) * tok_table[ids[m]*ld_tok + n] for n < n_real, 0 behind. */
int tfl_token_gate(const void* s, int64_t ld_s, const void* tok_table, int64_t ld_tok, const int64_t* ids, int vocab, void* out,
                   int rows, int n, int n_real, int dtype, void* stream);

/* Both products of a token's side input for up to 16 rows in bfloat16: out[m*ld_out + n] = sum over s of (gelu_tanh(x . Wg^T)[m][s] * tok_table[ids[m]*ld_tok
 * + s]) * Wp[n][s], n < n_real (TFL_EPI_TOKEN, then TFL_EPI_F32).  gate_packed [side, width] and proj_packed [width, side] panel-major; x an activation block;
 * ws: tfl_token_side_ws_floats(rows, side) floats. */
int64_t tfl_token_side_ws_floats(int rows, int side);
int tfl_token_side(const void* gate_packed, const void* proj_packed, const void* x, int64_t ld_x, int64_t x_oct, const void* table,
                   int64_t ld_tok, const int64_t* ids, int vocab, float* out, int64_t ld_out, float* ws, int64_t ws_floats, int rows,
                   int width, int side, int side_real, int n_real, void* stream);

/* Prefill half of the input projection: y [rows][q + C + R + gate + up] (T) ->
 *   cq [rows][q] = y_q / rms * q_norm;  cache row slot[m] = latent / rms * kv_norm | rotated key;  ck [rows][C + R] the same
 *   row again (NULL: not wanted);  act [rows] at stride ld_act = gelu_tanh(up) (n_up = 0: none). */
int tfl_prepare(const void* y, int64_t ld_y, int q, int q_real, int C, int c_real, int R, int up_off, int n_up,
                const float* q_norm, const float* kv_norm, float eps, const float* cos, const float* sin, int half, int max_pos,
                const int32_t* pos, const int32_t* slot, void* cache, int cache_rows, void* cq, void* ck, void* act,
                int64_t ld_act, int rows, int dtype, void* stream);

/* dst[t] = cache[src[t]]: the cached rows of whole prefixes, packed. */
int tfl_gather_rows(const void* cache, int cache_rows, const int32_t* src, void* dst, int rows, int W, int dtype, void* stream);

/* Causal attention of packed new tokens over up-projected keys and values.
 *   q [tq][H*(N + R)] unrotated; the R part is rotated here at pos[token].
 *   kv [tk][H*N + H*V]: unrotated keys of all heads, then values;  ck [tk][C + R]: the rotated keys sit at column C.
 *   seq [nseq][4] int32: {first new token, new tokens, first key, keys}; new token j sees keys 0 .. keys - new + j.
 *   out [tq] at stride ld_out: o[h*V + d] * sigmoid(gate[token*ld_gate + h*V + d]) */
int tfl_attn_prefill(const void* q, const void* kv, const void* ck, const int32_t* seq, int nseq, int max_new, const int32_t* pos,
                     const float* cos, const float* sin, int half, int max_pos, const void* gate, int64_t ld_gate, void* out,
                     int64_t ld_out, int tq, int tk, int H, int N, int R, int V, int C, float scale, int dtype, void* stream);

/* One query token per sequence over the paged latent cache: q [rows][H][C + R] (keys are the cached rows themselves, values
 * their first C entries), len[row] keys (<= 0: output 0), page table [rows][table_ld].  out [rows][H][C] (T).
 * ws: tfl_attn_decode_ws_floats floats when nsplit > 1.  tfl_attn_decode_splits: the nsplit to take for rows of up to max_len keys
 * (tfl_attn_decode_pick_nsplit: for bfloat16 rows of 512 + 64). */
int64_t tfl_attn_decode_ws_floats(int rows, int H, int C, int nsplit);
int tfl_attn_decode_splits(int rows, int H, int C, int R, int max_len, int dtype);
int tfl_attn_decode_pick_nsplit(int rows, int H, int max_len);
int tfl_attn_decode(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len,
                    void* out, float* ws, int64_t ws_floats, int rows, int H, int C, int R, float scale, int nsplit, int dtype,
                    void* stream);

/* The same for bfloat16 rows of 512 + 64, 17 to 32 heads and up to 32 rows, with a product in the same launch that needs nothing of it:
 * product->out_f += x . W^T (TFL_EPI_RESIDUAL without out_t, chunk-major weights; include/triforce_tile.h).  workers CUs do the attention, its
 * splits dealt over the rows' pages (at most nsplit, 2 .. 128, of a row); the others take panels_each panels (2 .. 4) of the product.
 * out NULL: the splits stay in ws, for tfl_latent_value.
 * tfl_attn_beside_plan: workers, panels_each and nsplit for rows with `pages` pages in all, 0 where the two are better launched apart; parts: how
 * many splits all rows have together.  tfl_attn_beside_plan_of: the same, `longest` of the pages in one row. */
int tfl_attn_beside_plan(int rows, int H, int C, int R, int64_t pages, int n, int k, int32_t* panels_each, int32_t* nsplit, int32_t* parts);
int tfl_attn_beside_plan_of(int rows, int H, int C, int R, int64_t pages, int64_t longest, int n, int k, int32_t* panels_each, int32_t* nsplit,
                            int32_t* parts);
int tfl_attn_decode_beside(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len, void* out, float* ws,
                           int64_t ws_floats, int rows, int H, float scale, int nsplit, int workers, int panels_each, const TflGemm* product, void* stream);
/* The same for 17 to 32 rows with the product's panels in eights over `parts` (1 .. 4) ranges of k each, whose sums go to product->out_f [parts][rows][n]
 * (product->n_real = ld_f = n): parts * ceil(n / 128) workgroups.  tfl_beside_parts: how many parts, with the workers and nsplit to them, 0 where that is not the faster way.  TFL_EPI_RESIDUAL of a later product adds them (TflGemm.also). */
int tfl_beside_parts(int rows, int H, int C, int R, int64_t pages, int64_t longest, int n, int k, int32_t* workers, int32_t* nsplit);
int tfl_attn_decode_beside_parts(const void* q, const void* cache, int n_pages, const int32_t* table, int table_ld, const int32_t* len, void* out, float* ws,
                                 int64_t ws_floats, int rows, int H, float scale, int nsplit, int workers, int parts, const TflGemm* product, void* stream);

/* Columns of the product (n of k) beside the attention, from the last on, that the query to latent product in front of it carries (tfl_gemm_carry); 0: none. */
int tfl_latent_carry(int rows, int H, int C, int R, int64_t pages, int64_t longest, int n, int k);

/* TFL_EPI_GATED in bfloat16 (include/triforce_tile.h; k 512, up to 4 rows) of what the splits in ws merge to: product->x is not read. */
int tfl_latent_value(const float* ws, int64_t ws_floats, int nsplit, const TflGemm* product, void* stream);

#ifdef __cplusplus
}
#endif
#endif
