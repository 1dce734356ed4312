// FP64 predictor and PLM corrector (no FMA contraction: the reference's arithmetic bit for
// bit); the PLM corrector with the Roe solver runs k_vl_stage (vs_near).
#include "vl_kernels_impl.hpp"
#include "vl_near_impl.hpp"

namespace imhd {
IMHD_INST_NEAR(RS_ROE, true)
IMHD_INST_NEAR(RS_HLLD, true)
IMHD_INST_NEAR(RS_HLLE, true)
IMHD_INST_NEAR(RS_HLLD, false)
IMHD_INST_NEAR(RS_HLLE, false)
}  // namespace imhd
