// Launch of gemm_kernel's instantiations.  Included by gemm.hip (one weight) and
// gemm_segs.hip (several), which compile side by side.
#pragma once

#include <atomic>

#include "gemm_kernel.h"
#include "host_common.h"

namespace flute {

template <int MB, int KW, int MW, bool BF16, int B1, bool PERM = false, bool LEAN = false, bool SEGS = false>
flute_status launch_gemm(const GemmParams &p, dim3 grid, int lds, hipStream_t stream) {
    static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
    if (!attr_done) {
        FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)gemm_kernel<MB, KW, MW, BF16, B1, PERM, LEAN, SEGS>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize,
                                            (int)kLdsPerCU));
        attr_done = true;
    }
    hipLaunchKernelGGL((gemm_kernel<MB, KW, MW, BF16, B1, PERM, LEAN, SEGS>), grid, dim3(64 * KW * MW), lds,
                       stream, p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

template <int MB, int KW, int MW, bool BF16, bool SEGS>
flute_status launch_gemm_bits(const GemmParams &p, dim3 grid, int lds, hipStream_t stream) {
    if (p.nstreams == 1) {
        switch (p.bits[0]) {
            case 4:
                if (p.rep_log2[0] == 6 && p.lean) return launch_gemm<MB, KW, MW, BF16, 4, true, true, SEGS>(p, grid, lds, stream);
                if (p.rep_log2[0] == 6) return launch_gemm<MB, KW, MW, BF16, 4, true, false, SEGS>(p, grid, lds, stream);
                return launch_gemm<MB, KW, MW, BF16, 4, false, false, SEGS>(p, grid, lds, stream);
            case 3: return launch_gemm<MB, KW, MW, BF16, 3, false, false, SEGS>(p, grid, lds, stream);
            case 2: return launch_gemm<MB, KW, MW, BF16, 2, false, false, SEGS>(p, grid, lds, stream);
            default: return launch_gemm<MB, KW, MW, BF16, 1, false, false, SEGS>(p, grid, lds, stream);
        }
    }
    set_error("flute_gemm: two streams at this size run as one launch per stream");
    return FLUTE_ERR_UNSUPPORTED;
}

// SEGS: several weights in the launch
template <bool BF16, bool SEGS>
flute_status launch_gemm_shape(int mb, int mw, const GemmParams &p, dim3 grid, int lds, hipStream_t stream) {
    if (mb != 4) {
        set_error("flute_gemm: %d blocks of rows per wavefront", mb);
        return FLUTE_ERR_UNSUPPORTED;
    }
    if (mw == 1) return launch_gemm_bits<4, 8, 1, BF16, SEGS>(p, grid, lds, stream);
    return launch_gemm_bits<4, 4, 2, BF16, SEGS>(p, grid, lds, stream);
}

}  // namespace flute
