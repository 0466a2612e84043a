// Walsh-Hadamard butterfly on an fp32 LDS buffer, shared by the standalone
// rotation kernel and the GEMV prologue so that both produce the same bits.
//
// The transform is the stage-doubling butterfly of fht.py:174-192 upstream: for
// len = 1, 2, 4, ... every pair (i, i + len) whose index i has bit log2(len)
// clear becomes (a + b, a - b).  Each pair operation is a single fp32 add and a
// single fp32 subtract, and a value is touched by exactly one pair per stage, so
// the result does not depend on which thread executes which pair: it is
// bit-identical to the scalar loop as long as the stages run in ascending order.
//
// Stages are executed four at a time in registers (radix-16 passes): a thread
// gathers the 16 values whose indices differ only in the four bits of the pass,
// runs the four stages locally, and scatters them back.  One barrier per pass
// instead of one per stage.
#pragma once

#include "common.h"

namespace flute {

// float(1 / sqrt(2^n)), identical to rounding the fp64 quotient: the value is
// 2^-(n/2) for even n and float(sqrt(2)) * 2^-((n+1)/2) for odd n, and scaling
// by a power of two is exact.
__device__ __forceinline__ float inv_sqrt_pow2(int n) {
    return ldexpf((n & 1) ? 1.41421356237309504880f : 1.0f, -((n + 1) >> 1));
}

// Physical LDS slot of logical element i: a linear XOR swizzle of the five bank
// bits by higher index bits.  In the first radix-16 pass 32 consecutive lanes
// differ in index bits 4..8, in the second in bits 0..3 and 8; the swizzle maps
// both patterns (and plain consecutive indices) onto 32 distinct banks.
__device__ __forceinline__ int fht_slot(int i) {
    return i ^ ((i >> 5) & 7) ^ (((i >> 8) & 1) * 24);
}

template <int R>
__device__ __forceinline__ void fht_pass(float *buf, int b, int sh0, int tid, int nthreads) {
    constexpr int E = 1 << R;
    const int ngroups = b >> R;
    const int lowmask = (1 << sh0) - 1;
    for (int gi = tid; gi < ngroups; gi += nthreads) {
        const int base = ((gi >> sh0) << (sh0 + R)) | (gi & lowmask);
        float v[E];
#pragma unroll
        for (int j = 0; j < E; ++j) v[j] = buf[fht_slot(base + (j << sh0))];
#pragma unroll
        for (int q = 0; q < R; ++q) {
#pragma unroll
            for (int j = 0; j < E; ++j) {
                if ((j & (1 << q)) == 0) {
                    const float a = v[j], c = v[j | (1 << q)];
                    v[j] = a + c;
                    v[j | (1 << q)] = a - c;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < E; ++j) buf[fht_slot(base + (j << sh0))] = v[j];
    }
}

// In-place transform of `count` values held at buf[fht_slot(0..count-1)], as
// count / b independent blocks of b = 2^nstages consecutive values (count a
// multiple of b; b >= 2).  Must be called by every thread of the workgroup; the
// buffer must be complete (barrier) on entry and is complete on exit.
template <int RMAX = 4>
__device__ __forceinline__ void fht_lds(float *buf, int count, int nstages, int tid,
                                        int nthreads) {
    // RMAX = stages per pass: 4 keeps 16 values in registers, 3 keeps 8 (for callers
    // that are short of registers); the order of the stages, and so every bit of the
    // result, is the same.
    int sh0 = 0;
    while (nstages - sh0 >= RMAX) {
        fht_pass<RMAX>(buf, count, sh0, tid, nthreads);
        __syncthreads();
        sh0 += RMAX;
    }
    const int rem = nstages - sh0;
    if (RMAX > 3 && rem == 3) fht_pass<3>(buf, count, sh0, tid, nthreads);
    else if (rem == 2) fht_pass<2>(buf, count, sh0, tid, nthreads);
    else if (rem == 1) fht_pass<1>(buf, count, sh0, tid, nthreads);
    if (rem) __syncthreads();
}

// ---- stages between a thread's own columns and across the lanes of a wavefront ----------------
// Same butterflies, same single rounding per value and stage as above, so a transform may take its
// first stages in registers and the rest in LDS and keep every bit.

// Stages of length 1 ... N/2 between a thread's own N consecutive columns.
template <int N>
__device__ __forceinline__ void stages_in_thread(float (&f)[N]) {
#pragma unroll
    for (int len = 1; len < N; len <<= 1) {
#pragma unroll
        for (int q = 0; q < N; ++q) {
            if ((q & len) == 0) {
                const float a = f[q], c = f[q | len];
                f[q] = a + c;
                f[q | len] = a - c;
            }
        }
    }
}

// One stage against the lane whose number differs in bit M.  1, 2 and 8 are row permutations of the
// vector pipe (quad_perm, row_ror), 4 and 16 ds_swizzle, 32 ds_bpermute (the LDS crossbar without a
// memory access).  The lower lane of a pair keeps a + b and the upper a - b, formed as
// fma(mine, +-1, other): the product is exact, so every value sees the same single rounding per
// stage as in the buffered butterfly.
template <int M, int N>
__device__ __forceinline__ void stage_across_lanes(float (&f)[N], int lane) {
    const float sgn = (lane & M) ? -1.0f : 1.0f;
    const int partner = (lane ^ 32) << 2;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const int own = __float_as_int(f[q]);
        int other;
        if constexpr (M == 1) other = __builtin_amdgcn_mov_dpp(own, 0xb1, 0xf, 0xf, false);
        else if constexpr (M == 2) other = __builtin_amdgcn_mov_dpp(own, 0x4e, 0xf, 0xf, false);
        else if constexpr (M == 8) other = __builtin_amdgcn_mov_dpp(own, 0x128, 0xf, 0xf, false);
        else if constexpr (M == 32) other = __builtin_amdgcn_ds_bpermute(partner, own);
        else other = __builtin_amdgcn_ds_swizzle(own, (M << 10) | 0x1f);
        f[q] = fmaf(f[q], sgn, __int_as_float(other));
    }
}

// The first stages of a transform of 2^nst >= N consecutive columns (nst uniform): those between a
// thread's N columns and between lanes, all of them where N * 64 columns cover the block.  The
// lanes of a block hold its columns in order and are active together.
template <int N>
__device__ __forceinline__ void fht_head(float (&f)[N], int lane, int nst) {
    constexpr int own = N == 8 ? 3 : 4;
    static_assert(N == 8 || N == 16, "columns of a thread");
    stages_in_thread(f);
    if (nst > own) stage_across_lanes<1>(f, lane);
    if (nst > own + 1) stage_across_lanes<2>(f, lane);
    if (nst > own + 2) stage_across_lanes<4>(f, lane);
    if (nst > own + 3) stage_across_lanes<8>(f, lane);
    if (nst > own + 4) stage_across_lanes<16>(f, lane);
    if (nst > own + 5) stage_across_lanes<32>(f, lane);
}

// The stages that fht_head left, sh0 = 9 or 10 on, over the buffer: barriers as in fht_lds.
__device__ __forceinline__ void fht_tail(float *buf, int count, int nst, int sh0, int tid, int nthreads) {
    while (nst - sh0 >= 4) {
        fht_pass<4>(buf, count, sh0, tid, nthreads);
        __syncthreads();
        sh0 += 4;
    }
    const int rem = nst - sh0;
    if (rem == 3) fht_pass<3>(buf, count, sh0, tid, nthreads);
    else if (rem == 2) fht_pass<2>(buf, count, sh0, tid, nthreads);
    else if (rem == 1) fht_pass<1>(buf, count, sh0, tid, nthreads);
    if (rem > 0) __syncthreads();
}

}  // namespace flute
