// Standalone Walsh-Hadamard rotation: one workgroup per row, the butterfly of
// fht_dev.h in LDS, fp32 throughout, one rounding to the I/O type.
#include "fht_dev.h"
#include "host_common.h"

#include <atomic>

#include <cmath>
#include <cstdlib>

namespace flute {

namespace {

constexpr int kFhtThreads = 512;

struct FhtParams {
    const void *x;
    void *out;
    const float *signs;
    const float *awq;
    int64_t ldx, ldo;   // row strides of x and out in elements
    int K;
    int dtype;      // flute_dtype of x and out
    int adjoint;
    int block;      // > 0: equal blocks
    int chunk;      // columns transformed per pass in block mode
    int *shift;     // bfloat16 rows: bf16_row_shift of each result row's largest exponent, or NULL
    // Operand-order output for the LUT GEMM instead of rows (ap != NULL): the rotated row
    // m is rounded to `dtype`, converted to the LUT's 16-bit type and written where the
    // GEMM's activation pre-pass would put it, Ap[g][j][m / 16][lane][8]; rows from M up
    // to the padded count are written as zeros.
    uint32_t *ap;
    int ap_M, ap_mblk_pad, ap_bf16, ap_block_xor;
    int vec_io;     // x and out rows allow 16-byte accesses (16-bit types only)
    int vec_mul;    // signs and awq allow 16-byte loads
};

__device__ __forceinline__ float load_any(const void *p, int64_t i, int dtype) {
    if (dtype == FLUTE_F32) return ((const float *)p)[i];
    return load_act(p, i, dtype == FLUTE_BF16);
}
__device__ __forceinline__ void store_any(void *p, int64_t i, int dtype, float v) {
    if (dtype == FLUTE_F32) ((float *)p)[i] = v;
    else ((uint16_t *)p)[i] = round_act(v, dtype == FLUTE_BF16);
}

// forward:  out = ((x [*awq]) @ H) * signs * inv [/ awq]   (fht.py:206-222, 646-651 upstream)
// adjoint:  out = ((x * signs) @ H) * inv                  (fht.py:225-238 upstream)
// Eight consecutive columns k0...k0+7 (k0 a multiple of 8) of row m in operand order:
// k = g*64 + (2j + ktl)*16 + 2*kg + 8*s2 + e lives in lane kg*16 + m%16 of block m/16,
// dword ktl*2 + s2, half e; so the eight values are the (e = 0, 1) pairs of the four
// lanes kg = 0...3 at one dword position.
__device__ __forceinline__ void store_operand_order(const FhtParams &p, int m, int k0,
                                                    const uint16_t (&v)[8]) {
    const int g = k0 >> 6, kl = k0 & 63;
    const int jh = kl >> 5, s = ((kl >> 4) & 1) * 2 + ((kl >> 3) & 1);
    const int64_t unit = ((int64_t)(g * 2 + jh) * p.ap_mblk_pad + ((m >> 4) ^ image_block_xor(g, p.ap_block_xor))) * 64 + (m & 15);
#pragma unroll
    for (int kg = 0; kg < 4; ++kg)
        p.ap[(unit + kg * 16) * 4 + s] = (uint32_t)v[2 * kg] | ((uint32_t)v[2 * kg + 1] << 16);
}

__device__ __forceinline__ void load_mul8(const float *m, int k, int vec, float (&v)[8]) {
    if (vec) {
        const float4 a = *(const float4 *)(m + k), b = *(const float4 *)(m + k + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = m[k + q];
    }
}

// Eight consecutive columns of a row as fp32, already multiplied by what the direction
// applies before the butterfly (signs for the adjoint, the scale for the compensated
// forward transform); sg/sc keep the multipliers the output needs.
__device__ __forceinline__ void load_cols8(const FhtParams &p, int64_t row, int k, float (&f)[8],
                                           float (&sg)[8], float (&sc)[8]) {
    const int bf16 = p.dtype == FLUTE_BF16;
    if (p.vec_io) {
        const uint4 raw = *(const uint4 *)((const uint16_t *)p.x + row + k);
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint16_t h = (uint16_t)(w[q >> 1] >> (16 * (q & 1)));
            f[q] = bf16 ? bf2f(h) : h2f(h);
        }
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) f[q] = load_any(p.x, row + k + q, p.dtype);
    }
    load_mul8(p.signs, k, p.vec_mul, sg);
    if (p.awq) load_mul8(p.awq, k, p.vec_mul, sc);
    if (p.adjoint || p.awq) {
#pragma unroll
        for (int q = 0; q < 8; ++q) f[q] *= p.adjoint ? sg[q] : sc[q];
    }
}

// The transformed eight columns out: scaled, (forward) signed and de-scaled, one rounding
// to the I/O type, as rows or in the GEMM's operand order.
__device__ __forceinline__ void store_cols8(const FhtParams &p, int64_t orow, int k, float inv,
                                            const float (&f)[8], const float (&sg)[8],
                                            const float (&sc)[8], uint32_t &top) {
    const int bf16 = p.dtype == FLUTE_BF16;
    uint16_t op[8];
    float t[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) t[q] = p.adjoint ? f[q] * inv : f[q] * sg[q] * inv;
    if (!p.adjoint && p.awq) {          // one uniform branch: as a select per value every launch paid for the divisions
#pragma unroll
        for (int q = 0; q < 8; ++q) t[q] = t[q] / sc[q];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        if (p.dtype != FLUTE_F32) {
            uint16_t a = round_act(t[q], bf16);
            if (p.ap && bf16 != p.ap_bf16) a = round_act(bf16 ? bf2f(a) : h2f(a), p.ap_bf16);
            op[q] = a;
        }
    }
    if (p.shift) {
#pragma unroll
        for (int q = 0; q < 8; ++q) top = max(top, (uint32_t)(op[q] >> 7) & 0xffu);
    }
    if (p.ap) {
        store_operand_order(p, blockIdx.x, k, op);
    } else if (p.dtype == FLUTE_F32) {
#pragma unroll
        for (int q = 0; q < 8; ++q) ((float *)p.out)[orow + k + q] = t[q];
    } else if (p.vec_io) {
        *(uint4 *)((uint16_t *)p.out + orow + k) =
            make_uint4((uint32_t)op[0] | ((uint32_t)op[1] << 16),
                       (uint32_t)op[2] | ((uint32_t)op[3] << 16),
                       (uint32_t)op[4] | ((uint32_t)op[5] << 16),
                       (uint32_t)op[6] | ((uint32_t)op[7] << 16));
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) ((uint16_t *)p.out)[orow + k + q] = op[q];
    }
}

// One workgroup per row, eight consecutive columns a thread and piece, all segments of the row side by
// side (transform_row).  What bounds it: for few rows the chain load -> stages -> barriers -> store, so
// a row's values and multipliers are one memory round trip; for many rows the loads and stores.  P pieces
// of eight columns a thread in as few registers as K needs, so a CU holds several rows.
template <int P>
__global__ void __launch_bounds__(kFhtThreads) fht_row_kernel(const FhtParams p) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x;
    const int64_t row = (int64_t)blockIdx.x * p.ldx;
    const int64_t orow = (int64_t)blockIdx.x * p.ldo;
    if (p.ap && (int)blockIdx.x >= p.ap_M) {           // padding row of the operand image
        const uint16_t zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int j = tid * 8; j < p.K; j += kFhtThreads * 8)
            store_operand_order(p, blockIdx.x, j, zero);
        return;
    }
    uint32_t top = 0;
    float sg[P][8];
    transform_row<P>(
        (float *)lds, p.K, p.block, tid, kFhtThreads,
        [&](int h, int j, float (&f)[8]) {
            float sc[8];
            load_cols8(p, row, j, f, sg[h], sc);
        },
        [&](int h, int j, float (&f)[8], int nst) {
            float sc[8];
            if (p.awq) load_mul8(p.awq, j, p.vec_mul, sc);
            store_cols8(p, orow, j, inv_sqrt_pow2(nst), f, sg[h], sc, top);
        });
    if (p.shift) {
        __shared__ uint32_t slots[kFhtThreads / 64];
        top = workgroup_max(top, slots, tid, kFhtThreads);
        if (tid == 0) p.shift[blockIdx.x] = bf16_row_shift(top);
    }
}

template <int P>
flute_status launch_row(const FhtParams &p, int rows, size_t lds_bytes, hipStream_t stream) {
    static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
    if (!attr_done) {
        FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)fht_row_kernel<P>, hipFuncAttributeMaxDynamicSharedMemorySize, 98304));
        attr_done = true;
    }
    hipLaunchKernelGGL(fht_row_kernel<P>, dim3(rows), dim3(kFhtThreads), lds_bytes, stream, p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

// Rows beyond 16384 columns: their segments (chunks of blocks) one after the other, eight consecutive
// columns a thread and step.  The first nine stages stay in
// registers (fht_head: between a thread's columns, then between lanes), the rest are one or two
// passes over an fp32 buffer in LDS; blocks and segments of up to 512 columns never touch it.
__global__ void __launch_bounds__(kFhtThreads) fht_kernel(const FhtParams p) {
    extern __shared__ __align__(16) uint8_t lds[];
    float *buf = (float *)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t row = (int64_t)blockIdx.x * p.ldx;
    const int64_t orow = (int64_t)blockIdx.x * p.ldo;
    constexpr int STEP = kFhtThreads * 8;
    if (p.ap && (int)blockIdx.x >= p.ap_M) {           // padding row of the operand image
        const uint16_t zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int j = tid * 8; j < p.K; j += STEP)
            store_operand_order(p, blockIdx.x, j, zero);
        return;
    }
    uint32_t top = 0;
    // block mode: chunks of whole blocks; otherwise the descending power-of-two
    // segments of K (fht.py:118-134 upstream)
    for (int off = 0; off < p.K;) {
        int count, nst;
        if (p.block > 0) {
            count = min(p.chunk, p.K - off);
            nst = 31 - __builtin_clz((unsigned)p.block);
        } else {
            nst = 31 - __builtin_clz((unsigned)(p.K - off));
            count = 1 << nst;
        }
        const float inv = inv_sqrt_pow2(nst);
        float f[8], sg[8], sc[8];
        for (int j = tid * 8; j < count; j += STEP) {
            load_cols8(p, row, off + j, f, sg, sc);
            fht_head(f, lane, nst);
            if (nst <= 9) {
                store_cols8(p, orow, off + j, inv, f, sg, sc, top);
            } else {
                const int s0 = fht_slot(j);            // a multiple of 8: slot(j + q) = s0 ^ q
#pragma unroll
                for (int q = 0; q < 8; ++q) buf[s0 ^ q] = f[q];
            }
        }
        if (nst > 9) {
            __syncthreads();
            fht_tail(buf, count, nst, 9, tid, kFhtThreads);
            for (int j = tid * 8; j < count; j += STEP) {
                if (count > STEP) {                    // (one step: the multipliers are still here)
                    load_mul8(p.signs, off + j, p.vec_mul, sg);
                    if (p.awq) load_mul8(p.awq, off + j, p.vec_mul, sc);
                }
                const int s0 = fht_slot(j);
#pragma unroll
                for (int q = 0; q < 8; ++q) f[q] = buf[s0 ^ q];
                store_cols8(p, orow, off + j, inv, f, sg, sc, top);
            }
            __syncthreads();                           // the next segment reuses the buffer
        }
        off += count;
    }
    if (p.shift) {
        __shared__ uint32_t slots[kFhtThreads / 64];
        top = workgroup_max(top, slots, tid, kFhtThreads);
        if (tid == 0) p.shift[blockIdx.x] = bf16_row_shift(top);
    }
}

}  // namespace

}  // namespace flute

namespace flute {

flute_status fht_launch(const void *x, int64_t ldx, const float *signs, const float *awq, void *out,
                        int64_t ldo, int M, int K, int dtype, int adjoint, int block,
                        hipStream_t stream, const FhtOperandOut *operand, int *shift) {
    FhtParams p;
    p.x = x;
    p.out = out;
    p.signs = signs;
    p.awq = awq;
    p.ldx = ldx;
    p.ldo = ldo;
    p.K = K;
    p.dtype = dtype;
    p.adjoint = adjoint ? 1 : 0;
    p.block = block;
    p.chunk = 0;
    p.shift = shift;
    p.ap = operand ? operand->ap : nullptr;
    p.ap_M = M;
    p.ap_mblk_pad = operand ? operand->mblk_pad : 0;
    p.ap_block_xor = operand ? operand->block_xor : 0;
    p.ap_bf16 = operand ? operand->lut_bf16 : 0;
    const bool io16 = dtype != FLUTE_F32;
    p.vec_io = io16 && ((uintptr_t)x & 15) == 0 && ldx % 8 == 0 &&
               (operand || (((uintptr_t)out & 15) == 0 && ldo % 8 == 0));
    p.vec_mul = ((uintptr_t)signs & 15) == 0 && (!awq || ((uintptr_t)awq & 15) == 0);
    size_t lds_bytes;
    if (block > 0) {
        FLUTE_REQUIRE(is_pow2(block) && block >= 32 && block <= 16384 && K % block == 0,
                      FLUTE_ERR_INVALID,
                      "flute_fht: block must be a power of two in [32, 16384] dividing K (got %d)",
                      block);
        p.chunk = K <= 16384 ? K : (16384 / block) * block;
        lds_bytes = block > 512 ? (size_t)p.chunk * 4 : 0;
    } else {
        const Segs segs = make_segments(K, 0);
        FLUTE_REQUIRE(segs.len[0] <= 16384, FLUTE_ERR_UNSUPPORTED,
                      "flute_fht: segment of %d columns exceeds the 16384-column LDS tile",
                      segs.len[0]);
        lds_bytes = segs.len[0] > 512 ? (size_t)segs.len[0] * 4 : 0;
    }
    const int rows = operand ? operand->mblk_pad * 16 : M;
    if (rows == 0) return FLUTE_OK;
    if (K <= transform_reach(4, kFhtThreads)) {
        lds_bytes = lds_bytes ? (size_t)K * 4 : 0;
        switch ((K + kFhtThreads * 8 - 1) / (kFhtThreads * 8)) {
            case 1: return launch_row<1>(p, rows, lds_bytes, stream);
            case 2: return launch_row<2>(p, rows, lds_bytes, stream);
            case 3: return launch_row<3>(p, rows, lds_bytes, stream);
            default: return launch_row<4>(p, rows, lds_bytes, stream);
        }
    }
    static std::atomic<bool> attr_done{false};   // threads may race to the first call: the call is idempotent
    if (!attr_done) {
        FLUTE_HIP_CHECK(hipFuncSetAttribute((const void *)fht_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 98304));
        attr_done = true;
    }
    hipLaunchKernelGGL(fht_kernel, dim3(rows), dim3(kFhtThreads), lds_bytes, stream, p);
    FLUTE_HIP_CHECK(hipGetLastError());
    return FLUTE_OK;
}

}  // namespace flute

using namespace flute;

extern "C" flute_status flute_fht(const void *x, const float *signs, const float *awq, void *out,
                                  int M, int K, int dtype, int adjoint, int block, void *stream) {
    FLUTE_REQUIRE(x && out && signs, FLUTE_ERR_INVALID, "flute_fht: x, signs and out must not be NULL");
    FLUTE_REQUIRE(dtype == FLUTE_F16 || dtype == FLUTE_BF16 || dtype == FLUTE_F32, FLUTE_ERR_INVALID,
                  "flute_fht: dtype must be float16, bfloat16 or float32");
    FLUTE_REQUIRE(M >= 0, FLUTE_ERR_INVALID, "flute_fht: M must be >= 0");
    {
        const uintptr_t elem = dtype == FLUTE_F32 ? 3 : 1;
        FLUTE_REQUIRE(((uintptr_t)x & elem) == 0 && ((uintptr_t)out & elem) == 0, FLUTE_ERR_INVALID,
                      "flute_fht: x and out must be aligned to their element size");
        FLUTE_REQUIRE(((uintptr_t)signs & 3) == 0 && ((uintptr_t)awq & 3) == 0, FLUTE_ERR_INVALID,
                      "flute_fht: signs and awq are fp32 and must be 4-byte aligned");
    }
    FLUTE_REQUIRE(K >= 32 && K % 32 == 0 && K <= 65504, FLUTE_ERR_INVALID,
                  "flute_fht: K must be a multiple of 32 in [32, 65504] (got %d)", K);
    FLUTE_REQUIRE(!(awq && adjoint), FLUTE_ERR_INVALID,
                  "flute_fht: the awq-compensated transform exists in the forward direction only");
    return fht_launch(x, K, signs, awq, out, K, M, K, dtype, adjoint, block, (hipStream_t)stream,
                      nullptr);
}
