// bfloat16 products of many rows for the prefill of the batch-served families: see rows_gemm.h.
#include "tile_common.h"
#include "rows_gemm.h"

extern "C" int64_t tfl_rows_gemm_plan(int rows, int n, int k, int32_t* shape, int32_t* splits) { return rg::entry_plan(rows, n, k, shape, splits); }

extern "C" int tfl_rows_gemm(const void* x, int64_t ld_x, const void* w, void* out, int64_t ld_out, float* ws, int64_t ws_floats, int rows, int n, int k,
                             int form, int shape, int splits, void* stream) {
    return rg::entry<__bf16, rg::GELU_EIGHTS>(x, ld_x, w, out, ld_out, ws, ws_floats, rows, n, k, form, shape, splits, stream);
}
