// pp_line_mm_nd.hip -- instantiates the dense-product ND line transforms (pp_line_mm.h): x and y
// axes, forward and inverse, FP64 and FP32 forms.
#include "pp_line_mm.h"

namespace pp {
template hipError_t launch_line_mm_kind<KIND_ND>(int, int, int, const LineArgs &, hipStream_t);
}  // namespace pp
