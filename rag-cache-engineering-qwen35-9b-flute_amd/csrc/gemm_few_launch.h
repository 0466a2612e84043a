// Launch of one element type's instantiations of gemm_few_kernel.  Included by gemm_few_f16.hip and
// gemm_few_bf16.hip (one weight) and their _segs counterparts (several), which compile side by side.
#pragma once

#include <atomic>

#include "gemm_few_kernel.h"
#include "host_common.h"

namespace flute {

template <int FORM, bool BF16, int B1, int B2, bool SEGS>
flute_status launch_few(const GemmParams &p, dim3 grid, hipStream_t stream) {
    constexpr int lds = few_lds_total<B1, B2, FORM>();
    static_assert(lds <= kLdsPerCU, "tables, staging or sums exceed a CU's LDS");
    static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
    if (!attr_done) {
        FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)gemm_few_kernel<FORM, BF16, B1, B2, SEGS>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        attr_done = true;
    }
    hipLaunchKernelGGL((gemm_few_kernel<FORM, BF16, B1, B2, SEGS>), grid, dim3(512), lds, stream, p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

template <int FORM, bool BF16, bool SEGS>
flute_status launch_few_bits(const GemmParams &p, dim3 grid, hipStream_t stream) {
    switch (p.nstreams == 2 ? p.bits[0] * 8 + p.bits[1] : p.bits[0] * 8) {
        case 8 * 1: return launch_few<FORM, BF16, 1, 0, SEGS>(p, grid, stream);
        case 8 * 2: return launch_few<FORM, BF16, 2, 0, SEGS>(p, grid, stream);
        case 8 * 3: return launch_few<FORM, BF16, 3, 0, SEGS>(p, grid, stream);
        case 8 * 4: return launch_few<FORM, BF16, 4, 0, SEGS>(p, grid, stream);
        case 8 * 1 + 1: return launch_few<FORM, BF16, 1, 1, SEGS>(p, grid, stream);
        case 8 * 2 + 1: return launch_few<FORM, BF16, 2, 1, SEGS>(p, grid, stream);
        case 8 * 2 + 2: return launch_few<FORM, BF16, 2, 2, SEGS>(p, grid, stream);
        case 8 * 3 + 1: return launch_few<FORM, BF16, 3, 1, SEGS>(p, grid, stream);
        case 8 * 3 + 2: return launch_few<FORM, BF16, 3, 2, SEGS>(p, grid, stream);
        case 8 * 3 + 3: return launch_few<FORM, BF16, 3, 3, SEGS>(p, grid, stream);
        case 8 * 4 + 1: return launch_few<FORM, BF16, 4, 1, SEGS>(p, grid, stream);
        case 8 * 4 + 2: return launch_few<FORM, BF16, 4, 2, SEGS>(p, grid, stream);
        case 8 * 4 + 3: return launch_few<FORM, BF16, 4, 3, SEGS>(p, grid, stream);
    }
    set_error("flute_gemm: no few-row kernel for widths (%d, %d)", p.bits[0], p.bits[1]);
    return FLUTE_ERR_UNSUPPORTED;
}

template <bool BF16, bool SEGS>
flute_status launch_few_shape(int mb, const GemmParams &p, dim3 grid, hipStream_t stream) {
    if (p.seg[0].resB) return mb == 1 ? launch_few_bits<4, BF16, SEGS>(p, grid, stream) : launch_few_bits<5, BF16, SEGS>(p, grid, stream);
    if (mb == 1) return launch_few_bits<1, BF16, SEGS>(p, grid, stream);
    return p.A8 ? launch_few_bits<3, BF16, SEGS>(p, grid, stream) : launch_few_bits<2, BF16, SEGS>(p, grid, stream);
}

}  // namespace flute
