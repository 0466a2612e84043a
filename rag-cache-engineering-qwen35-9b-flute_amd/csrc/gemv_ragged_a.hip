// Instantiations of the lean GEMV kernel for K ranges that do not divide evenly: one 4-bit width, (1, 4) and (4, 1).
#include "gemv_pair_launch.h"

namespace flute {

flute_status launch_gemv_ragged_a(const GemvParams &p, int pair, int grid_x, int nw, size_t lds_bytes, bool lut_bf16,
                                  hipStream_t stream) {
    switch (pair) {
        case 0:
            return lut_bf16 ? launch_ragged<true, 4, 4>(p, grid_x, nw, lds_bytes, stream)
                            : launch_ragged<false, 4, 4>(p, grid_x, nw, lds_bytes, stream);
        case 14:
            return lut_bf16 ? launch_ragged<true, 1, 4>(p, grid_x, nw, lds_bytes, stream)
                            : launch_ragged<false, 1, 4>(p, grid_x, nw, lds_bytes, stream);
        default:
            return lut_bf16 ? launch_ragged<true, 4, 1>(p, grid_x, nw, lds_bytes, stream)
                            : launch_ragged<false, 4, 1>(p, grid_x, nw, lds_bytes, stream);
    }
}

}  // namespace flute
