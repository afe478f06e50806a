// The batch kernel at 2 bits (template and reasons: bw_qbatch_kernel.h).
#include "bw_qbatch_kernel.h"

int bw_launch_qbatch_w2(int group, int mt, int ntw, const BatchArgs& a, hipStream_t stream) {
    return launch_qbatch_bits<2>(group, mt, ntw, a, stream);
}
