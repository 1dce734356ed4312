// FP32 characteristic PPM corrector: FMA contraction as in the other FP32 kernels, except
// where char_edge and ppm_edge write their fused operations out.
#include "vl_kernels_impl.hpp"
#include "vl_char_impl.hpp"

namespace imhd {
IMHD_INST_CHAR(float, RS_ROE)
IMHD_INST_CHAR(float, RS_HLLD)
IMHD_INST_CHAR(float, RS_HLLE)
}  // namespace imhd
