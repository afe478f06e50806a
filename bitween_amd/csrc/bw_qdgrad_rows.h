// bw_qdgrad_rows.h - the input gradient of up to 48 rows (bw_qdgrad_rows.hip), as bw_qdgrad.hip calls it.
#pragma once
#include "bw_common.h"

struct DgradRowsArgs {
    const void* go;
    const void* qweight;
    const void* scale;
    const void* zp;
    _Float16* gx;
    float* ws;                                   // [splits][M][K] partial sums
    int M, N, K, ldg, ldx, groups, row_bytes;
    int splits, steps_per_split;                 // slices of N (two and more), in steps of 32
    uint32_t go_bytes, w_bytes, meta_bytes;
};

// M <= 48 (bfloat16: 32), N a multiple of 8, an even number of groups a row; go aligned to 16 bytes and ldg a multiple of 8, scale and zp aligned to 4 bytes,
// gx to 8 and ldx a multiple of 4; extents below 2^31 bytes.
int bw_launch_dgrad_rows(const DgradRowsArgs& a, int bits, int group, int dtype, hipStream_t stream);
