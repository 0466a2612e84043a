// Several weights in one launch of the small-M LUT GEMM.
#include "gemm_launch.h"

namespace flute {

flute_status gemm_launch_segs(int bf16, int mb, int mw, const GemmParams &p, dim3 grid, int lds, hipStream_t stream) {
    return bf16 ? launch_gemm_shape<true, true>(mb, mw, p, grid, lds, stream)
                : launch_gemm_shape<false, true>(mb, mw, p, grid, lds, stream);
}

}  // namespace flute
