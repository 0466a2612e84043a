// The few-row LUT GEMM over float16 LUTs, one weight in a launch.
#include "gemm_few_launch.h"

namespace flute {
flute_status gemm_few_f16(int mb, const GemmParams &p, dim3 grid, hipStream_t stream) {
    return launch_few_shape<false, false>(mb, p, grid, stream);
}
}  // namespace flute
