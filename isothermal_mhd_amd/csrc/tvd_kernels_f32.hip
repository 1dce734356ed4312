// FP32 instantiation of the K98 TVD + CTU + CT kernels (FMA contraction; fdiv/fsqrt use the
// hardware reciprocal and square root).  Face B, corner and centre EMFs and the CFL speed
// stay FP64.
#include "tvd_kernels_impl.hpp"

namespace imhd {
IMHD_INST_TVD(float)
int tvd_sweep_waves_per_cu() {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_tvd_sweep_m<float>, 256, 0);
    return 4 * (e == hipSuccess && n > 0 ? n : 1);
}
}  // namespace imhd
