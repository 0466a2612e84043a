// Instantiations of the lean GEMV kernel for K ranges that do not divide evenly: (3, 3), (2, 4) and (2, 3).
#include "gemv_pair_launch.h"

namespace flute {

flute_status launch_gemv_ragged_b(const GemvParams &p, int pair, int grid_x, int nw, size_t lds_bytes, bool lut_bf16,
                                  hipStream_t stream) {
    switch (pair) {
        case 33:
            return lut_bf16 ? launch_ragged<true, 3, 3>(p, grid_x, nw, lds_bytes, stream)
                            : launch_ragged<false, 3, 3>(p, grid_x, nw, lds_bytes, stream);
        case 24:
            return lut_bf16 ? launch_ragged<true, 2, 4>(p, grid_x, nw, lds_bytes, stream)
                            : launch_ragged<false, 2, 4>(p, grid_x, nw, lds_bytes, stream);
        default:
            return lut_bf16 ? launch_ragged<true, 2, 3>(p, grid_x, nw, lds_bytes, stream)
                            : launch_ragged<false, 2, 3>(p, grid_x, nw, lds_bytes, stream);
    }
}

}  // namespace flute
