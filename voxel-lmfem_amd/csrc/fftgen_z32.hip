// FP32 z pass for axes of any length (vxl_fftgen.h).
#include "vxl_fftgen.h"

namespace vxl {
VXL_FFTGEN_Z_INSTANCES(float)
}  // namespace vxl
