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

#include <type_traits>

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

// ---- a whole row at once -----------------------------------------------------------------------
// The same stage for wavefronts whose lanes are all active, shared out over the two pipes: 1, 2 and 8
// are row permutations of the vector pipe, 4 goes through ds_swizzle, and for 16 and 32 two values
// change halves with each other (v_permlane16_swap, v_permlane32_swap), so that sum and difference
// are each formed once, for half the lanes of either, and change back.
template <int M, int N>
__device__ __forceinline__ void stage_all_lanes(float (&f)[N], int lane) {
    if constexpr (M == 16 || M == 32) {
#pragma unroll
        for (int q = 0; q < N; q += 2) {
            auto swap = [](float a, float b) {
                const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
                if constexpr (M == 32) return __builtin_amdgcn_permlane32_swap(x, y, false, false);
                else return __builtin_amdgcn_permlane16_swap(x, y, false, false);
            };
            const auto in = swap(f[q], f[q + 1]);
            const float a = __uint_as_float(in[0]), c = __uint_as_float(in[1]);
            const auto out = swap(a + c, a - c);
            f[q] = __uint_as_float(out[0]);
            f[q + 1] = __uint_as_float(out[1]);
        }
    } else {
        const float sgn = (lane & M) ? -1.0f : 1.0f;
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int own = __float_as_int(f[q]);
            int other;
            if constexpr (M == 1) other = __builtin_amdgcn_mov_dpp(own, 0xb1, 0xf, 0xf, false);
            else if constexpr (M == 2) other = __builtin_amdgcn_mov_dpp(own, 0x4e, 0xf, 0xf, false);
            else if constexpr (M == 8) other = __builtin_amdgcn_mov_dpp(own, 0x128, 0xf, 0xf, false);
            else other = __builtin_amdgcn_ds_swizzle(own, (M << 10) | 0x1f);
            f[q] = fmaf(f[q], sgn, __int_as_float(other));
        }
    }
}

// Stages of the transform that column j of a row of K takes part in: its block's, or those of its
// descending power-of-two segment (the highest bit in which j and K differ: K has it, j has not).
__device__ __forceinline__ int column_stages(int j, int K, int block) {
    return 31 - __builtin_clz((unsigned)(block > 0 ? block : K ^ j));
}

// Stage `s` for the lanes whose columns take part in it.
template <int M, int N>
__device__ __forceinline__ void stage_some_lanes(float (&f)[N], int lane, bool takes) {
    float g[N];
#pragma unroll
    for (int q = 0; q < N; ++q) g[q] = f[q];
    stage_all_lanes<M>(g, lane);
#pragma unroll
    for (int q = 0; q < N; ++q) f[q] = takes ? g[q] : f[q];
}

// Where transform_row keeps column i in LDS: 16-byte pieces stay whole, and pieces that a thread's
// neighbours access together lie on different banks, as do the consecutive columns of a pass.
__device__ __forceinline__ int row_slot(int i) { return i ^ ((i >> 3) & 4); }

// R stages of length 2^SH0 (512 columns, or sixteen times that) and up over the 2^nst columns
// from `off` on (a multiple of 2^nst).  Bits of a column above row_slot's reach are apart from it, so
// the columns of a group lie at constant distances from the first: one address, the rest immediates.
template <int R, int SH0>
__device__ __forceinline__ void row_pass(float *buf, int off, int nst, int tid, int nthreads) {
    constexpr int E = 1 << R;
    static_assert(SH0 >= 9, "above the slots' permutation");
    const int groups = 1 << (nst - R);
#pragma unroll 1
    for (int g = tid; g < groups; g += nthreads) {
        float *const at = buf + row_slot(off + (((g >> SH0) << (SH0 + R)) | (g & ((1 << SH0) - 1))));
        float v[E];
#pragma unroll
        for (int j = 0; j < E; ++j) v[j] = at[j << SH0];
        stages_in_thread(v);
#pragma unroll
        for (int j = 0; j < E; ++j) at[j << SH0] = v[j];
    }
}

// Columns of a row that transform_row reaches with P pieces of eight columns a thread.
constexpr int transform_reach(int P, int nthreads) { return 8 * P * nthreads; }

// Transform of a whole row of K columns (K and the block multiples of 32, K up to transform_reach),
// all its segments side by side: thread `tid` holds the eight consecutive columns at (h * nthreads + tid) * 8
// for h = 0 ... P - 1, load(h, j, f) fetches them and store(h, j, f, stages) gets them back.  The
// first stages stay in registers, the rest are one or two passes over `buf` (K floats of LDS, needed
// for blocks and segments beyond 512 columns), with two or three barriers whatever the number of
// segments.  Every value goes through the same single roundings as in the buffered butterfly.
// Called by all threads; on return no wavefront reads another's columns in the buffer any more.
// What bounds it, for one row: vector instructions of one CU (about thirty a column over 64 lanes) and
// the trip to memory in front.  Segments one after the other (a chain of loads, barriers and passes
// each), eight dword accesses a thread and column-wise addresses: 1 x 12288 9.0 -> 7.6 us, 800 x 11072
// 22.8 -> 20.0, 1000 x 4096 9.2 -> 8.1; the fused prologue, one token: 11072 -> 4096 22.5 -> 14.4 us
// (with the ragged GEMV), 12288 -> 4096, (3, 3) bits 17.2 -> 15.9.
template <int P, class Load, class Store>
__device__ __forceinline__ void transform_row(float *buf, int K, int block, int tid, int nthreads, Load load, Store store) {
    constexpr int N = 8, own = 3, sh = own + 6;         // columns of a thread; stages in it, in a wavefront
    const int lane = tid & 63;
    float f[P][N];
#pragma unroll
    for (int h = 0; h < P; ++h)
        if (h * nthreads * N < K) load(h, min((h * nthreads + tid) * N, K - N), f[h]);
#pragma unroll
    for (int h = 0; h < P; ++h) {
        if (h * nthreads * N >= K) break;               // uniform
        const int nst = column_stages(min((h * nthreads + tid) * N, K - N), K, block);
        stages_in_thread(f[h]);
        stage_all_lanes<1>(f[h], lane);
        if (__all(nst >= sh)) {
            stage_all_lanes<2>(f[h], lane);
            stage_all_lanes<4>(f[h], lane);
            stage_all_lanes<8>(f[h], lane);
            stage_all_lanes<16>(f[h], lane);
            stage_all_lanes<32>(f[h], lane);
        } else {
            stage_some_lanes<2>(f[h], lane, nst > own + 1);
            stage_some_lanes<4>(f[h], lane, nst > own + 2);
            stage_some_lanes<8>(f[h], lane, nst > own + 3);
            stage_some_lanes<16>(f[h], lane, nst > own + 4);
            stage_some_lanes<32>(f[h], lane, nst > own + 5);
        }
    }
    const int top = column_stages(0, K, block);         // the longest segment is the first
    if (top > sh) {
#pragma unroll
        for (int h = 0; h < P; ++h) {
            const int j = (h * nthreads + tid) * N;
            if (j < K && column_stages(j, K, block) > sh) {
                // (j + q and j agree above bit 3: the pieces' slots differ as the columns do)
#pragma unroll
                for (int q = 0; q < N; q += 4)
                    *(float4 *)(buf + (row_slot(j) ^ q)) = make_float4(f[h][q], f[h][q + 1], f[h][q + 2], f[h][q + 3]);
            }
        }
        __syncthreads();
        auto level = [&](auto first, int nst, int off) {
            constexpr int SH0 = decltype(first)::value;
            switch (min(nst - SH0, 4)) {
                case 4: row_pass<4, SH0>(buf, off, nst, tid, nthreads); break;
                case 3: row_pass<3, SH0>(buf, off, nst, tid, nthreads); break;
                case 2: row_pass<2, SH0>(buf, off, nst, tid, nthreads); break;
                default: row_pass<1, SH0>(buf, off, nst, tid, nthreads); break;
            }
        };
        auto levels = [&](auto first) {
            constexpr int SH0 = decltype(first)::value;
            if (block > 0) {
                for (int off = 0; off < K; off += block) level(first, top, off);
            } else {
                for (int b = top, off = 0; b > SH0; --b) {
                    if (!((K >> b) & 1)) continue;
                    level(first, b, off);
                    off += 1 << b;
                }
            }
        };
        levels(std::integral_constant<int, sh>());
        if (top > sh + 4) {
            __syncthreads();
            levels(std::integral_constant<int, sh + 4>());
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < P; ++h) {
            const int j = (h * nthreads + tid) * N;
            if (j < K && column_stages(j, K, block) > sh) {
#pragma unroll
                for (int q = 0; q < N; q += 4) {
                    const float4 v = *(const float4 *)(buf + (row_slot(j) ^ q));
                    f[h][q] = v.x;
                    f[h][q + 1] = v.y;
                    f[h][q + 2] = v.z;
                    f[h][q + 3] = v.w;
                }
            }
        }
    }
#pragma unroll
    for (int h = 0; h < P; ++h) {
        const int j = (h * nthreads + tid) * N;
        if (j < K) store(h, j, f[h], column_stages(j, K, block));
    }
}

}  // namespace flute
