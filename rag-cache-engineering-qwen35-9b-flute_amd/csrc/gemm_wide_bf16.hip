// bfloat16 instantiations of the many-row LUT GEMM (gemm_wide_kernel.h).
#include "gemm_wide_launch.h"

namespace flute {
flute_status gemm_wide_bf16(int mb, int b1, int b2, int slices, const WideParams &p, hipStream_t stream) {
    return mb == 4 ? launch_wide_bits<true, 4>(b1, b2, slices, p, stream) : launch_wide_bits<true, 2>(b1, b2, slices, p, stream);
}
}  // namespace flute
