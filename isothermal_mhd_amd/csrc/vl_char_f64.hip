// FP64 characteristic PPM corrector (no FMA contraction: the reference's arithmetic bit for
// bit).
#include "vl_kernels_impl.hpp"
#include "vl_char_impl.hpp"

namespace imhd {
IMHD_INST_CHAR(double, RS_ROE)
IMHD_INST_CHAR(double, RS_HLLD)
IMHD_INST_CHAR(double, RS_HLLE)
}  // namespace imhd
