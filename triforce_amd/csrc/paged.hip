// Set-up of a paged decode step on the device (no host upload while neither the sequences nor their pages change).
#include "tile_common.h"

static_assert(sizeof(TflGemm) == 312, "another struct is another version, here and in latent_ops.hip and hybrid_ops.hip");
extern "C" int tfl_tile_abi_version(void) { return 3; }

__global__ void decode_prep_kernel(int32_t* __restrict__ len, const int32_t* __restrict__ table, int table_ld, int table_cols,
                                   int32_t* __restrict__ pos, int32_t* __restrict__ slot, int32_t* __restrict__ klen, int rows) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < rows) decode_prep_row(TflDecodePrep{len, table, pos, slot, klen, table_ld, table_cols, rows}, m);
}

extern "C" int tfl_decode_prep(int32_t* len, const int32_t* table, int table_ld, int table_cols, int32_t* pos, int32_t* slot,
                               int32_t* klen, int rows, void* stream) {
    if (!len || !table || !pos || !slot || !klen || rows < 1 || table_cols < 1 || table_ld < table_cols) return TF_EINVAL;
    hipLaunchKernelGGL(decode_prep_kernel, dim3((rows + 63) / 64), dim3(64), 0, (hipStream_t)stream, len, table, table_ld, table_cols,
                       pos, slot, klen, rows);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}

struct PageEntries { int32_t e[3 * TFL_MAX_ENTRIES]; };

__global__ void set_pages_kernel(int32_t* __restrict__ table, int table_ld, const PageEntries entries, int n) {
    const int j = threadIdx.x;
    if (j < n) table[(int64_t)entries.e[3 * j] * table_ld + entries.e[3 * j + 1]] = entries.e[3 * j + 2];
}

extern "C" int tfl_set_pages(int32_t* table, int table_ld, int rows, int cols, const int32_t* entries, int n, void* stream) {
    if (!table || !entries || rows < 1 || cols < 1 || table_ld < cols || n < 1 || n > TFL_MAX_ENTRIES) return TF_EINVAL;
    PageEntries p;
    for (int j = 0; j < n; ++j) {
        if (entries[3 * j] < 0 || entries[3 * j] >= rows || entries[3 * j + 1] < 0 || entries[3 * j + 1] >= cols) return TF_EINVAL;
        for (int i = 0; i < 3; ++i) p.e[3 * j + i] = entries[3 * j + i];
    }
    hipLaunchKernelGGL(set_pages_kernel, dim3(1), dim3(TFL_MAX_ENTRIES), 0, (hipStream_t)stream, table, table_ld, p, n);
    TFL_LAUNCH_CHECK();
    return TF_OK;
}
