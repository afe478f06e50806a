// bw_qgemm_cols.hip - the prefill kernel's 128- and 256-row tiles of 192 columns (natural-order schedule, three column tiles a wave), in a
// translation unit of their own so that they compile beside the others.  Which tile a call gets is decided in bw_qgemm.hip (gemm_tile).
#include "bw_qgemm_kernel.h"

int bw_launch_gemm_cols192(int bits, int group, int rows, const GemmArgs& a, void* workspace, size_t workspace_bytes, hipStream_t stream) {
#define BW_CASE(B, G)                                                                                \
    if (bits == B && group == G)                                                                      \
        return rows == 256 ? launch_gemm<B, G, 16, true, 3>(a, workspace, workspace_bytes, stream)    \
             : rows == 128 ? launch_gemm<B, G, 8, true, 3>(a, workspace, workspace_bytes, stream)     \
                           : BW_EUNSUPPORTED;
    BW_CASE(4, 128) BW_CASE(4, 64) BW_CASE(4, 32)
    BW_CASE(8, 128) BW_CASE(8, 64) BW_CASE(8, 32)
    BW_CASE(2, 128) BW_CASE(2, 64) BW_CASE(2, 32)
#undef BW_CASE
    return BW_EUNSUPPORTED;
}
