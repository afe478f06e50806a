// The batch kernel at 4 bits (template and reasons: bw_qbatch_kernel.h).
#include "bw_qbatch_kernel.h"

int bw_launch_qbatch_w4(int group, int mt, int ntw, const BatchArgs& a, hipStream_t stream) {
    return launch_qbatch_bits<4>(group, mt, ntw, a, stream);
}
