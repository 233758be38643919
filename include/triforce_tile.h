/* C ABI of libtriforce_tile.so: what the batch-served model families share (models/latent_core.py, models/hybrid_core.py) - the
 * skinny GEMM over packed weights with its epilogues, and the set-up of a paged decode step.  gfx950.
 *
 * Every entry point enqueues on `stream` and returns TF_OK, a TF_E* code (nothing launched) or a hipError_t.
 * dtype: 0 = bfloat16 operands with fp32 accumulation, 1 = everything in fp32.  "T" below is that element type.  Sizes are padded
 * to multiples of 32 with zeros unless a parameter is called "real".
 *
 * Packed weights: a [n, k] matrix is stored as [n/16][k/32][64][8]: piece (g*16 + i) of a 16x32 tile holds
 * w[16a + i][32b + 8g .. +7] - one wavefront load per tile.  chunk_major: the same tiles as [k/32][n/16], so that neighbouring panels
 * are neighbours in memory (what a launch with one workgroup per CU streams fastest).
 */
#ifndef TRIFORCE_TILE_H
#define TRIFORCE_TILE_H
#include <stdint.h>
#ifndef TF_OK
#define TF_OK 0
#define TF_EINVAL (-22)
#define TF_ENOSPC (-28)
#define TF_ERANGE (-34)
#endif
#ifdef __cplusplus
extern "C" {
#endif

#define TFL_PAGE 64                 /* cache rows per page */

int tfl_tile_abi_version(void);     /* 3: TflGemm with n_also and also */

/* Activation blocks: element (m, k) lives at m*ld + (k/8)*oct + k%8.  Row-major rows have oct = 8; decode keeps its norm output
 * and the output projection's input octet-major (ld = 8, oct = 8 * rows), where a 16-row operand is four contiguous runs. */

/* What a skinny GEMM does with its fp32 result (row m of x, output n of the group). */
enum {
    TFL_EPI_F32 = 0,                /* out_f[m*ld_f + n] = acc, n < n_real */
    TFL_EPI_IN = 1,                 /* n < n_raw: out_f[m*ld_f + n] = acc and ss[m*(n_raw/16) + n/16] = sum over the panel of
                                       acc^2, and for n < n_scaled out_t2 = acc * norm_w[n]
                                       (octet-major); else out_t(m, n - n_raw) = gelu_tanh(acc) */
    TFL_EPI_QUERY = 2,              /* acc *= 1 / sqrt(sum(ss_in[m][:ss_n]) / k_real + eps); heads of N + R outputs: out_t2[(m*H + h)*N + n] unrotated;
                                       out_t[(m*H + h)*(C + R) + C + n] rotated at pos[m] */
    TFL_EPI_LATENT = 3,             /* group h: out_t[(m*H + h)*(C + R) + n] = acc */
    TFL_EPI_GATED = 4,              /* group h: out_t(m, h*ppg*16 + n) = acc * sigmoid(gate[m*ld_gate + h*ppg*16 + n]) */
    TFL_EPI_RESIDUAL = 5,           /* out_f[m*ld_f + n] += acc; out_t(m, n) = the sum when out_t is given */
    TFL_EPI_TOKEN = 6,              /* out_t[m*ld_t + n] = gelu_tanh(acc) * tok_table[ids[m]*ld_tok + n], n < n_real (0 behind) */
    TFL_EPI_GLU = 7                 /* panels of 8 gate rows | 8 up rows: out_t(m, n) = gelu_tanh(gate) * up, n < n/2 */
};
typedef struct TflGemm {
    const void* wp;                 /* packed weights, groups back to back */
    const void* x;
    const float* norm_w;            /* [n_scaled] */
    const float* ss_in;             /* [rows][ss_n]: the first ss_n panels' sums of squares, row stride ss_ld */
    void* out_t;
    void* out_t2;
    float* out_f;
    float* ss_out;
    const float* gate;
    const void* tok_table;
    const int64_t* ids;
    const int32_t* pos;
    const float* cos;               /* [max_pos][half] */
    const float* sin;
    /* key half of TFL_EPI_QUERY: extra workgroups normalise / rotate / store the cache row of every batch row */
    const float* kv_raw;            /* [rows] raw [latent C][rotated R] rows (NULL: none), row stride ld_kv */
    const float* kv_norm_w;         /* fp32 [C] */
    void* cache;                    /* [cache rows][C + R] */
    const int32_t* slot;            /* cache row per batch row; negative: nothing is stored */
    int64_t ld_x, x_oct, x_group, ld_t, t_oct, ld_f, ld_gate, ld_tok, ld_kv;
    int32_t rows, n, k, groups;     /* n = outputs per group, all groups alike */
    int32_t n_real, k_real, n_raw, n_scaled, ss_n, ss_ld;
    int32_t H, N, R, C, half, c_real, max_pos, cache_rows, vocab;
    float eps;
    int32_t chunk_major;            /* packed weights as [k/32][n/16][64][8] (one group) */
    int32_t n_also;                 /* RESIDUAL of the one-workgroup-per-CU form, 17 rows and more: also[p][m][n] is added too, p < n_also (0 .. 4), blocks of [rows][n] */
    const float* also;
} TflGemm;

int tfl_gemm(const TflGemm* a, int dtype, int epilogue, void* stream);

/* tfl_gemm in bfloat16 with LATENT, up to 16 rows and n a multiple of 64, and beside it, on workgroups of their own in the same launch, another product
 * that waits for nothing of it: carried->out_f += carried->x . W^T (chunk-major weights, one group, as many rows, no out_t). */
int tfl_gemm_carry(const TflGemm* a, const TflGemm* carried, void* stream);

/* Start of a decode step: pos = len; slot = table[len/64]*64 + len%64; klen = len + 1; len += 1.  Rows with len < 0 (or past
 * their table) stay idle: pos 0, slot -1, klen 0. */
int tfl_decode_prep(int32_t* len, const int32_t* table, int table_ld, int table_cols, int32_t* pos, int32_t* slot, int32_t* klen,
                    int rows, void* stream);
typedef struct TflDecodePrep {      /* the same as part of a step's first launch (tfl_finish_first, tfh_connect_first) */
    int32_t* len;
    const int32_t* table;
    int32_t *pos, *slot, *klen;
    int32_t table_ld, table_cols, rows;
} TflDecodePrep;

/* float32 products of many rows on the bfloat16 matrix cores (csrc/split_gemm.hip): out[m*ld_out + n] = sum over k of x[m*ld_x + k] * w[n*k_total + k].
 * n % 16 == 0, k % 32 == 0, 16-byte aligned pointers and rows; k is cut into `splits` parts (0: the library's choice).
 * ws: tfl_split_gemm_ws_floats floats for the same sizes and splits. */
int64_t tfl_split_gemm_ws_floats(int rows, int n, int k, int splits);
int tfl_split_gemm(const float* w, const float* x, int64_t ld_x, float* out, int64_t ld_out, float* ws, int64_t ws_floats, int rows, int n, int k,
                   int splits, void* stream);

/* bfloat16 products of many rows (csrc/rows_gemm.h): out[m*ld_out + n] = sum over k of x[m*ld_x + k] * w[n*k_total + k], or with form
 * TFL_ROWS_GELU_EIGHTS, w being blocks of 8 gate rows | 8 up rows, out[m*ld_out + n] = gelu_tanh(gate n) * up n for n < n_total/2.
 * n % 16 == 0 (32 with a gated unit), k % 64 == 0, ld_x and ld_out % 8 == 0, 16-byte aligned pointers, x and w below 4 GiB.
 * shape, splits: the tile and the parts of k, tfl_rows_gemm_plan's or any other of 0 .. TFL_ROWS_SHAPES - 1 with a step of 64 for every part;
 * the plan returns the floats of ws they need (parts * rows * n from two parts on). */
#define TFL_ROWS_SHAPES 8
enum { TFL_ROWS_PLAIN = 0, TFL_ROWS_GELU_EIGHTS = 2 };
int64_t tfl_rows_gemm_plan(int rows, int n, int k, int32_t* shape, int32_t* splits);
int tfl_rows_gemm(const void* x, int64_t ld_x, const void* w, void* out, int64_t ld_out, float* ws, int64_t ws_floats, int rows, int n, int k,
                  int form, int shape, int splits, void* stream);

/* table[row * table_ld + column] = page for n (at most TFL_MAX_ENTRIES) host triples {row, column, page}: pages handed out between
 * two decode steps.  The triples are kernel arguments (nothing is read after the call returns). */
#define TFL_MAX_ENTRIES 64
int tfl_set_pages(int32_t* table, int table_ld, int rows, int cols, const int32_t* entries, int n, void* stream);

#ifdef __cplusplus
}
#endif
#endif
