// FP64 FFT passes for axes of any length (vxl_fftgen.h).
#include "vxl_fftgen.h"

namespace vxl {
VXL_FFTGEN_INSTANCES(double)
}  // namespace vxl
