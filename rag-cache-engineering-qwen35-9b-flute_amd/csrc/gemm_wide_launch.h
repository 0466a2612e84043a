// Launch of one element type's instantiations of gemm_wide_kernel.  Included by gemm_wide_f16.hip
// and gemm_wide_bf16.hip, which compile side by side.
#pragma once

#include <atomic>

#include "gemm_wide_kernel.h"
#include "host_common.h"

namespace flute {

template <bool BF16, int B1, int B2, int MB>
flute_status launch_wide(int slices, const WideParams &p, hipStream_t stream) {
    constexpr int lds = wide_lds_bytes<B1, B2>();
    static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
    if (!attr_done) {
        FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)gemm_wide_kernel<BF16, B1, B2, MB>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        attr_done = true;
    }
    hipLaunchKernelGGL((gemm_wide_kernel<BF16, B1, B2, MB>), dim3(p.mtiles * p.ntiles, slices), dim3(512), lds, stream, p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

// b1 >= b2 (0: no second stream)
template <bool BF16, int MB>
flute_status launch_wide_bits(int b1, int b2, int slices, const WideParams &p, hipStream_t stream) {
    switch (b1 * 8 + b2) {
        case 8 * 1 + 0: return launch_wide<BF16, 1, 0, MB>(slices, p, stream);
        case 8 * 1 + 1: return launch_wide<BF16, 1, 1, MB>(slices, p, stream);
        case 8 * 2 + 0: return launch_wide<BF16, 2, 0, MB>(slices, p, stream);
        case 8 * 2 + 1: return launch_wide<BF16, 2, 1, MB>(slices, p, stream);
        case 8 * 2 + 2: return launch_wide<BF16, 2, 2, MB>(slices, p, stream);
        case 8 * 3 + 0: return launch_wide<BF16, 3, 0, MB>(slices, p, stream);
        case 8 * 3 + 1: return launch_wide<BF16, 3, 1, MB>(slices, p, stream);
        case 8 * 3 + 2: return launch_wide<BF16, 3, 2, MB>(slices, p, stream);
        case 8 * 3 + 3: return launch_wide<BF16, 3, 3, MB>(slices, p, stream);
        case 8 * 4 + 0: return launch_wide<BF16, 4, 0, MB>(slices, p, stream);
        case 8 * 4 + 1: return launch_wide<BF16, 4, 1, MB>(slices, p, stream);
        case 8 * 4 + 2: return launch_wide<BF16, 4, 2, MB>(slices, p, stream);
        case 8 * 4 + 3: return launch_wide<BF16, 4, 3, MB>(slices, p, stream);
        default: return launch_wide<BF16, 4, 4, MB>(slices, p, stream);
    }
}

}  // namespace flute
