// What the two LUT GEMM kernels share: operand types and the matrix instruction.
#pragma once

#include <type_traits>

#include "common.h"

namespace flute {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

// Activation image of the many-row kernel: operand (g, half j of the 64-k tile, 16-row block mb) is
// 1 KB, lane kg*16 + row holding A[mb*16 + row][g*64 + j*32 + kg*8 ... + 7].  The 16-byte piece
// that starts at column k (a multiple of 8) of row m:
__host__ __device__ inline int64_t wide_piece(int m, int k, int mblk) {
    return ((int64_t)(k >> 5) * mblk + (m >> 4)) * 64 + ((k >> 3) & 3) * 16 + (m & 15);
}

template <bool BF16>
__device__ __forceinline__ f4_t mfma16(u4_t w, u4_t a, f4_t acc) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, w),
                                                       __builtin_bit_cast(bf8_t, a), acc, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, w),
                                                      __builtin_bit_cast(h8_t, a), acc, 0, 0, 0);
}

// silu(a) * b of eight 16-bit values: fp32 inside, one rounding.
template <bool BF16>
__device__ __forceinline__ u4_t silu_mul8(u4_t a, u4_t b) {
    u4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t r = 0;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const uint16_t x = (uint16_t)(a[e] >> (16 * s)), y = (uint16_t)(b[e] >> (16 * s));
            const float f = BF16 ? bf2f(x) : h2f(x);
            const float t = f / (1.0f + expf(-f)) * (BF16 ? bf2f(y) : h2f(y));
            r |= (uint32_t)round_act(t, BF16) << (16 * s);
        }
        o[e] = r;
    }
    return o;
}

// Partial sums cross workgroups (and so the per-XCD L2s) inside one launch: they are
// written through and read around the L2 with device-scope (sc1) accesses, the same
// instructions a relaxed agent-scope atomic compiles to, but 16 bytes at a time.
__device__ __forceinline__ void ws_store16(float *p, f4_t v) {
    // s_nop: a store of more than 8 bytes reads its data registers after issue, and the
    // compiler does not know what this statement is, so it would not keep the next write to
    // those registers away from it
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void ws_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Four 16-byte device-scope loads in flight, complete on return.
__device__ __forceinline__ void ws_load16x4(const float *p0, const float *p1, const float *p2,
                                            const float *p3, f4_t &a, f4_t &b, f4_t &c, f4_t &d) {
    asm volatile(
        "global_load_dwordx4 %0, %4, off sc1\n"
        "global_load_dwordx4 %1, %5, off sc1\n"
        "global_load_dwordx4 %2, %6, off sc1\n"
        "global_load_dwordx4 %3, %7, off sc1\n"
        "s_waitcnt vmcnt(0)"
        : "=&v"(a), "=&v"(b), "=&v"(c), "=&v"(d)
        : "v"(p0), "v"(p1), "v"(p2), "v"(p3)
        : "memory");
}

// Eight of them, `step` floats apart.
__device__ __forceinline__ void ws_load16x8(const float *p, int64_t step, f4_t (&v)[8]) {
    asm volatile(
        "global_load_dwordx4 %0, %8, off sc1\n"
        "global_load_dwordx4 %1, %9, off sc1\n"
        "global_load_dwordx4 %2, %10, off sc1\n"
        "global_load_dwordx4 %3, %11, off sc1\n"
        "global_load_dwordx4 %4, %12, off sc1\n"
        "global_load_dwordx4 %5, %13, off sc1\n"
        "global_load_dwordx4 %6, %14, off sc1\n"
        "global_load_dwordx4 %7, %15, off sc1\n"
        "s_waitcnt vmcnt(0)"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
        : "v"(p), "v"(p + step), "v"(p + 2 * step), "v"(p + 3 * step), "v"(p + 4 * step), "v"(p + 5 * step),
          "v"(p + 6 * step), "v"(p + 7 * step)
        : "memory");
}

// Dword b of the lane whose bits (5, 4) are a changes places with dword a of the one whose are b.
__device__ __forceinline__ void transpose_lanes16(uint32_t (&q)[4]) {
    auto p = __builtin_amdgcn_permlane32_swap(q[0], q[2], false, false);
    q[0] = p[0]; q[2] = p[1];
    p = __builtin_amdgcn_permlane32_swap(q[1], q[3], false, false);
    q[1] = p[0]; q[3] = p[1];
    p = __builtin_amdgcn_permlane16_swap(q[0], q[1], false, false);
    q[0] = p[0]; q[1] = p[1];
    p = __builtin_amdgcn_permlane16_swap(q[2], q[3], false, false);
    q[2] = p[0]; q[3] = p[1];
}

// The same between the four lanes of a quad.
__device__ __forceinline__ void transpose_quad(uint32_t (&q)[4], int lane) {
    auto swap = [](uint32_t &lo, uint32_t &hi, auto ctrl, bool odd) {
        const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, decltype(ctrl)::value, 0xf, 0xf, true);
        const uint32_t h = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, decltype(ctrl)::value, 0xf, 0xf, true);
        hi = odd ? hi : l;
        lo = odd ? h : lo;
    };
    const std::integral_constant<int, 0x4e> by2;        // quad_perm [2, 3, 0, 1]
    const std::integral_constant<int, 0xb1> by1;        // quad_perm [1, 0, 3, 2]
    swap(q[0], q[2], by2, lane & 2);
    swap(q[1], q[3], by2, lane & 2);
    swap(q[0], q[1], by1, lane & 1);
    swap(q[2], q[3], by1, lane & 1);
}

}  // namespace flute
